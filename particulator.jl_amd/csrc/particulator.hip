// particulator.hip -- kernels and C ABI of the null-collision Monte Carlo step on
// MI355X (gfx950).
//
// Data layout in HBM (per species): records of ten FP64 fields x,y,z,px,py,pz,w,t,s,r (80
// bytes a slot), and columns of a u8 active flag, a u64 uid and an i32 swarm, each `capacity`
// long.  A device counter n holds the slots in use; secondaries are appended at n with an
// atomic claim.
//
// One step (pt_advance), or up to MAX_SUB steps of a run in one launch:
//   k_snapshot   -- pass range [0, n) of every species (the advance_init!/iup state) and the
//                   final times of the launch's steps
//   k_advance    -- lanes take particles of all three species one after another: ratebound,
//                   then the reference's `while trem > eps` loop of push / null-collision
//                   selection / sampling, appending secondaries, which the wave's free lanes
//                   take up at once; droplow!'s energy cut at the end of each step.  Rate
//                   tables live in LDS.
//   k_advance again and k_tail -- only when secondaries found no room: whole-grid passes over
//                   them, then one workgroup until no new particle appears (the reference's
//                   further advance1! passes).
// Compaction (pt_compact) fills holes below the active count with active particles from
// above it (repack!), found by wave-ballot prefix sums over the active flags.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <thread>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <new>
#include <string>
#include <mutex>
#include <vector>

#include "pt_device.h"
#include "pt_mlp.h"

namespace pt {
// the message of the last failed context-free call on this host thread (pt_tables.cpp)
const char* host_last_error();
void host_set_error(const char* msg);
}  // namespace pt

using namespace pt;

typedef unsigned long long ull;

// ------------------------------------------------------------------ device parameters
// The ten FP64 fields of a particle (x, y, z, px, py, pz, w, t, s, r) form one 80-byte
// record: f[k] points at field k of slot 0 and successive slots are PT_NFIELDS doubles
// apart, so the state a lane writes back when its particle finishes is 72 contiguous bytes
// (whole sectors) instead of nine words in nine columns.  PF(f[k], i) is field k of slot i.
#define PF(col, i) ((col)[(size_t)(i) * PT_NFIELDS])
struct SpeciesDev {
    double* f[PT_NFIELDS];  // field k of slot 0 (one allocation: f[k] = f[0] + k)
    uint8_t* active;
    uint64_t* uid;
    int32_t* swarm;
    double* trem;     // time left in the step of a particle waiting in a queue
    uint32_t* draw;   // its position in its random stream
    uint8_t* evp;     // the process selected for its pending collision
    ull* n;
    ull cap;
    int tracked;
    int pad;
};

enum { FLAG_RATEBOUND = 0, FLAG_CAPACITY = 1, FLAG_RANGE = 2, FLAG_SAMPLER = 3, FLAG_TAIL = 4, NFLAGS = 5 };
enum {
    W_PSTEPS = 0, W_SECONDARIES = 1, W_MOVED = 2, W_EVENTS = 3, W_TAIL = 4, W_MAIN_SEC = 5,
    NWORK = 8
};
constexpr int NCOUNT = MAX_PROCS + 1;

// Step clock in device memory.  pt_advance writes tfinal and the step number; a captured
// run derives them on the device (tfinal = t + dt, then t = tfinal and step + 1 at the end
// of the step: the same arithmetic as the host loop t += dt), so replays of one graph
// advance the time.
constexpr int MAX_SUB = 16;  // steps of one launch at most
struct Clock {
    double t, dt, tfinal;
    uint32_t step, qpar;  // qpar: which work queue of each species is the input
    ull cursor;           // work items claimed by the push/select kernel
    ull ecur;             // queued collisions claimed by the sampling kernel
    ull nmark[PT_NSPECIES];  // population counts where the last secondary pass starts
    uint32_t pass;           // 0: the launch's main pass; > 0: passes over its secondaries
    uint32_t nsub;           // steps of this launch
    ull tcur;                // items claimed in the current pass of the one-workgroup tail
    ull left;                // secondaries that found their wave's stack full
    uint32_t done, pad;      // workgroups that have ended the current pass
    double tf[MAX_SUB];      // their final times
};

// Work queues of the event rounds: per species two ping-pong queues of particles to
// advance and one queue of pending collisions per sampler kind present in its table.
// Entries are slot indices; bit 31 marks a particle born in this step.
constexpr int NKQ = 6;
constexpr uint32_t CHILD_BIT = 0x80000000u;
struct Queues {
    uint32_t* work[PT_NSPECIES][2];
    uint32_t* ev[PT_NSPECIES][NKQ];
    ull* cnt;  // [3][2] work counts, then [3][NKQ] collision counts
    int8_t kq[PT_NSPECIES][16];  // sampler kind -> collision queue (-1: none)
    int8_t qkind[PT_NSPECIES][NKQ];  // collision queue -> sampler kind
    int nkq[PT_NSPECIES];
};
__host__ __device__ constexpr int QWK(int s, int par) { return 2 * s + par; }
__host__ __device__ constexpr int QEV(int s, int k) { return 2 * PT_NSPECIES + NKQ * s + k; }
constexpr int NQCNT = 2 * PT_NSPECIES + NKQ * PT_NSPECIES;

// WallCallback (src/callback.jl:146-184) of each species: coord < 0 for none
struct WallDev {
    int coord[PT_NSPECIES];
    int drop[PT_NSPECIES];
    double v[PT_NSPECIES];
    pt_wall_record* rec;
    ull* n;
    ull cap;
    int on;
    int pad;
};

// What the host reads after nearly every call, written by the kernels into pinned host memory,
// so that a call ends with one synchronisation and no copies.
constexpr int NSTAT = 8;
struct Report {
    ull n[PT_NSPECIES];  // slots in use
    ull flags[NFLAGS];
    ull left;            // secondaries the last pass left to a further one
    double stat[NSTAT];  // population statistics (k_stats)
};

struct Params {
    SpeciesDev sp[PT_NSPECIES];
    DevTable tab[PT_NSPECIES];
    DevSB sb[MAX_SB];
    DevPE pe[MAX_PE];
    const Field* fields;
    int nswarm;
    int rb_in_lds;
    int field_lds;      // every swarm's field is homogeneous E, B without loss: in LDS
    int lds_field_off;  // its offset in doubles: six per swarm (E, then B)
    uint64_t seed;
    ull* counts;  // [3][NCOUNT]
    ull* flags;   // [NFLAGS]
    ull* work;    // [NWORK]
    double* tally;  // [3][tally_bins + 2]
    int tally_bins;
    double tally_lo, tally_hi;
    int tally_tracked;  // births of tracked species are tallied too
    int dose_bins;      // depth-dose tally: dose[dose_bins] under, [+1] over, [+2] total
    double* dose;
    double dose_zlo, dose_zhi;
    ull* range;  // [3][2]
    Clock* clock;
    Queues q;
    uint32_t defer_mask;  // sampler kinds (bit = pt_proc_kind) queued in collision rounds
    MlpDev mlp[NLEARN];   // learned samplers (bremsstrahlung, Moller) used by the sampling kernel
    WallDev wall;         // WallCallback per species
    int lds_coop_off;     // byte offset of the step kernels' per-wave RBEB job area
    uint32_t forcing_off;  // restrictions of the forcing and the pusher (off_em / off_cl / off_push)
    int lds_rate_off[PT_NSPECIES];
    int lds_rb_off[PT_NSPECIES];
    int lds_proc_off[PT_NSPECIES];
    int lds_dose_off;     // the depth-dose bins in LDS (when there are any, at most DOSE_LDS)
    int lds_doubles;      // even
    Report* report;       // pinned host memory
    ull* image;           // what a workgroup stages: the Staged block, then lds_doubles doubles
};

// ------------------------------------------------------------------ LDS state
// doubles of a swarm's homogeneous fields in LDS: E, and B unless there is none
__host__ __device__ __forceinline__ int field_doubles(uint32_t off) { return (off & OFF_NO_B) ? 3 : 6; }

// the selection scan evaluates SCAN_GROUP processes at a time; zeros after each species' rate
// table in LDS for what it reads past the last one (10^7 electrons, 18 processes: three 34.9 ms,
// four 35.2, six 35.5; by subtraction, process after process, 35.6)
constexpr int SCAN_GROUP = 3;
constexpr int SCAN_PAD = 3 * SCAN_GROUP;

template <typename T>
using gptr = T PT_GLOBAL*;

// Per-species pointers, table metadata and process records are staged in LDS once per
// workgroup; the Chebyshev rate tables (and the rate bounds of a single swarm) follow in
// dynamic LDS.  The particle columns are typed as global memory and the tables are read
// through LDS-typed pointers, so that neither becomes a flat access.
struct SpLite {
    gptr<double> f[PT_NFIELDS];
    gptr<uint8_t> active;
    gptr<uint64_t> uid;
    gptr<int32_t> swarm;
    gptr<double> trem;
    gptr<uint32_t> draw;
    gptr<uint8_t> evp;
    ull* n;
    ull cap;
    const double* rb;  // rate bounds in global memory (several swarms)
    int rate_off;      // the rate table in the dynamic LDS (doubles)
    int rb_off;        // the rate bounds there (one swarm)
    int proc_off;      // the process records there
    double cut, xmax, ixmax, two_k1;  // ixmax = 1 / xmax, two_k1 = 2^(k+1)
    // |p|^2 above which the kinetic energy is certainly above the cut: the cut's |p|^2
    // times 1 + 1e-9, far beyond the rounding of the energy computed from |p|^2
    double ppcut_hi;
    int tracked, valid, nprocs, k, nswarm, rb_lds;
};

// block-local counters, flushed once per block (the depth-dose histogram too, in the dynamic
// LDS, when it has at most DOSE_LDS bins: deposits are frequent and would otherwise contend in
// global memory)
constexpr int DOSE_LDS = 512;
struct BlockCounters {
    ull counts[PT_NSPECIES * NCOUNT];
    ull flags[NFLAGS];
    ull work[NWORK];
};

// What every workgroup needs of the parameters, in the form it needs it: built once in global
// memory when parameters change (k_build_image) with the doubles of the dynamic LDS behind it,
// so that staging is one coalesced copy with all its loads in flight.  (Built by each workgroup
// from the parameters, with its dependent loads and the serial work of one thread, it took
// about 20 us of a launch.)
struct __attribute__((aligned(16))) Staged {
    SpLite sp[PT_NSPECIES];
    double cut[PT_NSPECIES];  // new particles at or below the cut are not stored
    int stored[PT_NSPECIES];  // species whose new particles are stored (tracked, with a table)
    // the field of swarm 0 (the push of a one-swarm population reads it here: from global
    // memory each read would be a vector load whose wait also waits for every memory
    // operation issued before it)
    Field field0;
};

struct Shared : Staged {
    BlockCounters bc;
    double tf[MAX_SUB];  // the final times of the launch's steps (nsub of them)
    int nsub, pad;
};

// what is staged in the dynamic LDS at most: the math table, three species' rates and process
// records, and either one swarm's rate bounds and fields or the fields of many; the dose bins
constexpr size_t table_doubles(int bounds, int swarms) {
    return MATH_DOUBLES +
           PT_NSPECIES * (MAX_INTERVALS * (MAX_PROCS * 3 + bounds) + SCAN_PAD + MAX_PROCS * sizeof(DevProc) / sizeof(double)) +
           6 * swarms + DOSE_LDS + 2 + 2;
}
constexpr size_t MAX_TABLE_BYTES = sizeof(double) * std::max(table_doubles(3, 1), table_doubles(0, MAX_LDS_FIELDS));
constexpr size_t IMAGE_BYTES = sizeof(Staged) + MAX_TABLE_BYTES;
constexpr size_t LDS_BYTES = 160 * 1024;  // of a CU, and what a workgroup may have

constexpr int IMAGE_BLOCKS = 32;  // one workgroup took 28 us, which each of many fields set in a row waits for
__global__ void __launch_bounds__(256) k_build_image(const Params* __restrict__ Pp) {
    const Params& P = *Pp;
    const int t0 = blockIdx.x * blockDim.x + threadIdx.x, nt = gridDim.x * blockDim.x;
    Staged& st = *(Staged*)P.image;
    double* const lds = (double*)(&st + 1);
    for (int q = t0; q < MATH_DOUBLES; q += nt) lds[q] = g_math[q];
    if (P.field_lds)
        for (int q = t0, m = field_doubles(P.forcing_off); q < m * P.nswarm; q += nt) {
            const FieldFn& f = (q % m) < 3 ? P.fields[q / m].e : P.fields[q / m].b;
            lds[P.lds_field_off + q] = f.v[q % 3];
        }
    if (P.dose_bins > 0 && P.dose_bins <= DOSE_LDS)
        for (int q = t0; q < P.dose_bins + 2; q += nt) lds[P.lds_dose_off + q] = 0.0;
    if (t0 == 0) st.field0 = P.fields[0];
    for (int s = 0; s < PT_NSPECIES; s++) {
        const DevTable& tb = P.tab[s];
        const SpeciesDev& S = P.sp[s];
        if (threadIdx.x == 0 && blockIdx.x == (s + 1) % gridDim.x) {
            SpLite& L = st.sp[s];
            for (int f = 0; f < PT_NFIELDS; f++) L.f[f] = (gptr<double>)S.f[f];
            L.active = (gptr<uint8_t>)S.active;
            L.uid = (gptr<uint64_t>)S.uid;
            L.swarm = (gptr<int32_t>)S.swarm;
            L.trem = (gptr<double>)S.trem;
            L.draw = (gptr<uint32_t>)S.draw;
            L.evp = (gptr<uint8_t>)S.evp;
            L.n = S.n;
            L.cap = S.cap;
            L.tracked = S.tracked;
            L.valid = tb.valid;
            L.nprocs = tb.nprocs;
            L.k = tb.k;
            L.nswarm = tb.nswarm;
            L.cut = tb.cut;
            {
                const double pc = s == PT_PHOTON ? tb.cut / C
                                                 : sqrt((tb.cut + MC2) * (tb.cut + MC2) - MC2 * MC2) / C;
                L.ppcut_hi = tb.cut > 0.0 ? pc * pc * (1.0 + 1e-9) : -1.0;
            }
            L.xmax = tb.xmax;
            L.ixmax = 1.0 / tb.xmax;
            L.two_k1 = ldexp(1.0, tb.k + 1);
            L.rate_off = P.lds_rate_off[s];
            L.rb_off = P.lds_rb_off[s];
            L.proc_off = P.lds_proc_off[s];
            L.rb = tb.ratebound;
            L.rb_lds = P.rb_in_lds;
            st.cut[s] = tb.cut;
            st.stored[s] = S.tracked && tb.valid;
        }
        if (!tb.valid) continue;
        for (int q = t0; q < tb.nprocs; q += nt)
            ((DevProc*)(lds + P.lds_proc_off[s]))[q] = tb.procs[q];
        int nr = (tb.k + 1) * tb.nprocs * 3;
        double* dst = lds + P.lds_rate_off[s];
        // the coefficients of the cumulative rates: sums over the row's processes so far, with
        // the rounding error of each addition carried along
        for (int q = t0; q < (tb.k + 1) * 3; q += nt) {
            double sum = 0.0, err = 0.0;
            for (int j = 0; j < tb.nprocs; j++) {
                const int at = ((q / 3) * tb.nprocs + j) * 3 + q % 3;
                const double v = tb.rate[at], n = sum + v, b = n - sum;
                err += (sum - (n - b)) + (v - b);
                sum = n;
                dst[at] = err == err ? sum + err : sum;  // (an infinite sum has no error)
            }
        }
        for (int q = nr + t0; q < nr + SCAN_PAD; q += nt) dst[q] = 0.0;
        if (P.rb_in_lds) {
            int nb = (tb.k + 1) * 3;
            double* d2 = lds + P.lds_rb_off[s];
            for (int q = t0; q < nb; q += nt) d2[q] = tb.ratebound[q];
        }
    }
}

// process j of species s
__device__ __forceinline__ const DevProc& process(const Shared& sh, int s, int j) {
    return ((const DevProc*)(pt_lds + sh.sp[s].proc_off))[j];
}

__device__ __forceinline__ void stage(const Params& P, Shared& sh) {
    typedef uint32_t word4 __attribute__((ext_vector_type(4)));
    const PT_GLOBAL word4* src = (const PT_GLOBAL word4*)P.image;
    const int n0 = sizeof(Staged) / 16, n = n0 + P.lds_doubles / 2;
    PT_LDS word4* const d0 = (PT_LDS word4*)(Staged*)&sh;
    PT_LDS word4* const d1 = (PT_LDS word4*)pt_lds;
    constexpr int U = 8;  // loads in flight per thread
    for (int q0 = threadIdx.x; q0 < n; q0 += U * blockDim.x) {
        word4 v[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int q = q0 + u * (int)blockDim.x;
            v[u] = src[q < n ? q : 0];
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int q = q0 + u * (int)blockDim.x;
            if (q < n0) d0[q] = v[u];
            else if (q < n) d1[q - n0] = v[u];
        }
    }
    if (threadIdx.x < MAX_SUB) sh.tf[threadIdx.x] = P.clock->tf[threadIdx.x];
    if (threadIdx.x == 0) sh.nsub = (int)P.clock->nsub;
    ull* const z = (ull*)&sh.bc;
    for (int q = threadIdx.x; q < (int)(sizeof(BlockCounters) / sizeof(ull)); q += blockDim.x) z[q] = 0;
    __syncthreads();
}

// setr!, src/collisions.jl:63-74
__device__ __forceinline__ double setr(const SpLite& L, double E, int swarm, bool& oob) {
    if (E < L.cut) return 0.0;
    double t1, t2;
    bool o;
    int i = precheb(E, L.k, L.xmax, L.ixmax, L.two_k1, t1, t2, o);
    oob |= o;
    const size_t off = (size_t)(L.nswarm > 1 ? swarm : 0) * (L.k + 1) * 3 + i * 3;
    return L.rb_lds ? cheb3(as_lds(pt_lds) + L.rb_off + off, t1, t2) : cheb3(as_global(L.rb) + off, t1, t2);
}

// The selection scan of do_one_collision! (src/collisions.jl:160-186): the first process j
// whose rate exceeds what is left of xi after subtracting the rates of processes 0..j-1, that
// is, the first whose cumulative rate exceeds xi; np or more for a null collision.  The row
// holds the coefficients of the cumulative rates, so a process costs two multiplications, two
// additions, a comparison and a selection, and nothing is carried from one to the next.  A
// group may run past the row's end into the next row or the table's padding (SCAN_PAD): what
// it finds there stands for the null collision.  (The sums differ from those of subtracting
// one rate after another by rounding: a draw within that of a cumulative rate may fall on
// the other side.)
__device__ __forceinline__ int select_process(const PT_LDS double* rt, int np, double t1, double t2, double xi) {
    constexpr int G = SCAN_GROUP;
    int sel = np;
    double c[3 * G];
#pragma unroll
    for (int u = 0; u < 3 * G; u++) c[u] = rt[u];
    for (int j = 0; j < np; j += G) {
        double cu[G];
#pragma unroll
        for (int u = 0; u < G; u++) cu[u] = (c[3 * u] + c[3 * u + 1] * t1) + c[3 * u + 2] * t2;
        const PT_LDS double* nx = rt + (j + G < np ? 3 * (j + G) : 0);
#pragma unroll
        for (int u = 0; u < 3 * G; u++) c[u] = nx[u];
        bool any = false;
#pragma unroll
        for (int u = G - 1; u >= 0; u--) {
            const bool hit = cu[u] > xi;
            any = any || hit;
            sel = hit ? j + u : sel;
        }
        if (any) break;
    }
    return sel;
}
// whether a null collision's remainder of xi is a number
__device__ __forceinline__ bool null_remains(const PT_LDS double* rt, int np, double t1, double t2, double xi) {
    return np == 0 ? xi >= 0.0 : cheb3(rt + 3 * (np - 1), t1, t2) <= xi;
}

__device__ void flush_counters(const Params& P, BlockCounters* bc) {
    __syncthreads();
    if (P.dose_bins > 0 && P.dose_bins <= DOSE_LDS)
        for (int q = threadIdx.x; q < P.dose_bins + 2; q += blockDim.x) {
            const double v = pt_lds[P.lds_dose_off + q];
            if (v != 0.0) atomicAdd(&P.dose[q], v);
        }
    for (int q = threadIdx.x; q < PT_NSPECIES * NCOUNT; q += blockDim.x)
        if (bc->counts[q]) atomicAdd(&P.counts[q], bc->counts[q]);
    for (int q = threadIdx.x; q < NFLAGS; q += blockDim.x)
        if (bc->flags[q]) atomicAdd(&P.flags[q], bc->flags[q]);
    for (int q = threadIdx.x; q < NWORK; q += blockDim.x)
        if (bc->work[q]) atomicAdd(&P.work[q], bc->work[q]);
}

// energy e (weight x J) left at depth z: the depth-dose tally (bins, then under- and
// overflow; the total is their sum)
__device__ __forceinline__ void deposit(const Params& P, BlockCounters& bc, double e, double z) {
    if (P.dose_bins <= 0 || e == 0.0) return;
    double f = (z - P.dose_zlo) / (P.dose_zhi - P.dose_zlo);
    int b = f < 0.0 ? P.dose_bins : (f >= 1.0 ? P.dose_bins + 1 : (int)floor(f * P.dose_bins));
    if (b < 0 || b > P.dose_bins + 1) b = P.dose_bins + 1;
    if (P.dose_bins <= DOSE_LDS) __hip_atomic_fetch_add((PT_LDS double*)pt_lds + P.lds_dose_off + b, e, __ATOMIC_RELAXED,
                                                        __HIP_MEMORY_SCOPE_WORKGROUP);
    else __hip_atomic_fetch_add((PT_GLOBAL double*)P.dose + b, e, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// ------------------------------------------------------------------ append
// add_particle!, src/population.jl:103-113 (+ birth tallies of untracked species; the energy
// of a particle born below the cut is left where it is born)
constexpr ull NO_SLOT = ~0ull;

// A slot of species sp2's store for each lane here with `want`: the lanes that call this
// together and want a slot of the same species share one atomic on its counter and take
// consecutive slots in lane order.  Lanes without `want` get NO_SLOT.  Called by every lane
// active at the call site (not under a lane-dependent branch).
__device__ __forceinline__ ull claim_slots(const Shared& sh, int sp2, bool want) {
    const int lane = threadIdx.x & 63;
    const uint64_t ltmask = lane ? (~0ull >> (64 - lane)) : 0ull;
    ull slot = NO_SLOT;
    uint64_t pend = __ballot(want);
    while (pend) {
        const int leader = __ffsll((unsigned long long)pend) - 1;
        const int key = __shfl(sp2, leader);
        const bool mine = want && sp2 == key;
        const uint64_t m = __ballot(mine);
        ull base = 0;
        if (lane == leader) base = global_add(sh.sp[key].n, (ull)__popcll(m));
        base = __shfl(base, leader);
        if (mine) slot = base + (ull)__popcll(m & ltmask);
        pend &= ~m;
    }
    return slot;
}

// add_particle! (src/population.jl:99-122) of the k-th new particle of the event of
// particle puid that ended at stream position dend; its uid is computed only when it is
// stored.  The lanes of a wave that append together claim their slots with one atomic per
// species.
__device__ __forceinline__ ull append(const Params& P, Shared& sh, int sp2, const V3& x,
                                      const V3& p, double w, double t, double s, uint64_t puid,
                                      uint32_t step, uint32_t dend, int k, int swarm, bool main_pass,
                                      uint32_t mark) {
    const SpLite& L = sh.sp[sp2];
    double E = kinenergy(sp2, p);
    bool store = true;
    if (E <= L.cut) {
        deposit(P, sh.bc, E * w, x.z);
        store = false;
    } else {
        if (!L.tracked || P.tally_tracked) {
            if (P.tally) {
                double* h = P.tally + (size_t)sp2 * (P.tally_bins + 2);
                atomicAdd(&h[P.tally_bins], 1.0);
                atomicAdd(&h[P.tally_bins + 1], w);
                if (P.tally_bins > 0) {
                    double lx = log(E / P.tally_lo) / log(P.tally_hi / P.tally_lo);
                    int b = (int)floor(lx * P.tally_bins);
                    if (b >= 0 && b < P.tally_bins) atomicAdd(&h[b], w);
                }
            }
            store = L.tracked != 0;
        }
        if (store && !L.valid) {
            atomicAdd(&sh.bc.flags[FLAG_CAPACITY], 1ull);
            store = false;
        }
    }
    const ull slot = claim_slots(sh, sp2, store);
    if (!store) return NO_SLOT;
    if (slot >= L.cap) {
        atomicAdd(&sh.bc.flags[FLAG_CAPACITY], 1ull);
        return NO_SLOT;
    }
    bool oob = false;
    double r = setr(L, E, swarm, oob);
    if (oob) atomicAdd(&sh.bc.flags[FLAG_RANGE], 1ull);
    PF(L.f[PT_X], slot) = x.x;
    PF(L.f[PT_Y], slot) = x.y;
    PF(L.f[PT_Z], slot) = x.z;
    PF(L.f[PT_PX], slot) = p.x;
    PF(L.f[PT_PY], slot) = p.y;
    PF(L.f[PT_PZ], slot) = p.z;
    PF(L.f[PT_W], slot) = w;
    PF(L.f[PT_T], slot) = t;
    PF(L.f[PT_S], slot) = s;
    PF(L.f[PT_R], slot) = r;
    L.uid[slot] = child_uid(P.seed, puid, step, dend, k);
    L.swarm[slot] = swarm;
    L.active[slot] = 1;
    L.draw[slot] = mark;
    atomicAdd(&sh.bc.work[W_SECONDARIES], 1ull);
    if (main_pass) atomicAdd(&sh.bc.work[W_MAIN_SEC], 1ull);
    return slot;
}

// ------------------------------------------------------------------ particle loop
// The body of advance1!'s @batch loop (src/mixed_population.jl:61-87), with
// do_one_collision! (src/collisions.jl:142-199) and apply! (:83-133) inlined, run as an
// event loop: each iteration advances a lane's particle by one push (and at most one
// collision); a lane whose particle has reached tfinal takes its next particle at once, so
// lanes of a wave stay busy whatever their particles' collision counts.  r is recomputed
// when a particle enters the step (advance_init!) and droplow!'s cut is applied when it
// is done.
//
// Work items q index the concatenation of the three species' item lists: slot ranges
// [rb[s], re[s]) (SRC_RANGE) or the entries of the species' input work queues
// (SRC_QUEUE).  A wave claims chunks of consecutive items from `cursor` and hands
// them out in order to its free lanes (ballot rank), so the particles a wave holds lie in
// a short window of consecutive slots: refills read whole cache lines and neighbouring
// write-backs meet in L2.
//
// A launch carries its particles through up to MAX_SUB steps (MULTI): particles do not
// interact, and a step's stream and rate bound depend on the particle alone, so a lane goes
// on to the next step of its particle in registers, with the arithmetic of the step
// boundary (droplow!'s cut, the times t += dt, setr!, a fresh stream) and without the record's
// way to memory and back, the launches between steps and the wait for the step's slowest
// wave.  10^7 electrons, 8 steps a launch: 2.50 -> 2.36 ms a step; 41,000 electrons: 253 ->
// 168 us; a pencil beam of 2 x 10^6 photons, where the wait is for the electron with the most
// collisions: 75 -> 26 ms.
//
// Collisions are sampled in the lane.  The secondaries it stores go on a stack in LDS that
// the wave's free lanes take from before new items; those that find it full are left to the
// passes over the launch's secondaries (the `draw` column holds the step each was born in,
// and the number of steps once it is done).
//
// Lanes reach their next collision at different times: of a wave's 64, about 40 end a push in
// a collision and 24 at the end of a step.  When enough lanes could still reach theirs, they
// push once more before the wave goes through the collision code: in wide workgroups (WIDE),
// 10^7 electrons 36.6 -> 35.0 ms with 12 to 20 lanes, 37.4 with 28.  Smaller populations do
// without: they are as long as their longest chain of collisions, and asking alone costs it
// 2 to 4% (a beam of 2 x 10^6 photons 153 -> 147 ms, 10^4 electrons 9.4 -> 9.1; 3.2 x 10^5
// electrons, the other way, 19.6 -> 19.9).
// EVENT = true (collision rounds): a selected real collision of a sampler kind in
// P.defer_mask is not sampled here; the particle is written back with its time left and
// stream position and queued for that sampler kind (wave-aggregated appends), and the
// lane moves on.  The sampling kernel then runs each queued kind with whole waves of the
// same kind (no divergence between samplers; the learned samplers need it).
// Items a wave claims at a time: 128 in workgroups of up to 256 threads, 256 in larger ones
// (512, and the 768 of large populations; 64 and 128 there: 16.35 and 19.2 ms against 16.1 for
// 8 launches of one step of 10^7 electrons), and a quarter of the wave's share of what is left
// when that is less, so that the waves end together.
constexpr ull LEAST_CHUNK = 16;
__device__ __forceinline__ ull claim_chunk(ull left, ull nwaves, ull least) {
    const ull most = blockDim.x > 256 ? 256ull : 128ull, share = left / (4 * nwaves);
    return share > most ? most : share < least ? least : share;
}
// Lanes of a wave that take items.  An iteration of a wave whose lanes are in different
// branches takes up to three times as long as that of a single lane (14 against 5 us), so a
// population with fewer particles than the launch has lanes is spread over all its waves.
__device__ __forceinline__ int lanes_used(ull total, ull nwaves) {
    return total >= 64 * nwaves ? 64 : (int)((total + nwaves - 1) / nwaves);
}
enum { SRC_RANGE = 0, SRC_QUEUE = 1 };
// a further push round before the collisions, when at least MORE_LANES lanes can use it
constexpr int MORE_ROUNDS = 1, MORE_LANES = 20;

struct Loaded {
    V3 x, p;
    double w, t, s;
    uint64_t uid;
    int swarm;
    uint32_t act;  // the active byte as read (nonzero: active), tested where it is used
};

// A record seen as five 16-byte pairs: (x,y) (z,px) (py,pz) (w,t) (s,r).  Records are 80
// bytes from a 256-byte aligned base, so every pair is 16-byte aligned and moves in one
// global_load_dwordx4 / global_store_dwordx4 instead of two 8-byte accesses.
typedef double pair2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ PT_GLOBAL pair2* rec_pairs(const SpLite& L, ull idx) {
    return (PT_GLOBAL pair2*)&PF(L.f[PT_X], idx);
}

// s_waitcnt vmcnt(0) (expcnt and lgkmcnt left at their maxima): every vector memory
// operation of the wave issued so far has completed
__device__ __forceinline__ void wait_vmem() { __builtin_amdgcn_s_waitcnt(0x0F70); }

// one round trip: every column of slot idx is read before any is tested
__device__ __forceinline__ Loaded load_slot(const SpLite& L, ull idx) {
    Loaded a;
    a.act = L.active[idx];
    const PT_GLOBAL pair2* r2 = rec_pairs(L, idx);
    const pair2 q0 = r2[0], q1 = r2[1], q2 = r2[2], q3 = r2[3];
    const double sv = PF(L.f[PT_S], idx);  // r is not read: the step sets it afresh
    a.x = V3{q0.x, q0.y, q1.x};
    a.p = V3{q1.y, q2.x, q2.y};
    a.w = q3.x;
    a.t = q3.y;
    a.s = sv;
    a.uid = L.uid[idx];
    a.swarm = L.swarm[idx];
    return a;
}

// Append `val` to the queue (arr, cnt) each lane names (cnt == nullptr: none).  Lanes
// naming the same queue share one atomic and write consecutive entries.  Must be called
// by the whole wave.
__device__ __forceinline__ void wave_push(ull* cnt, uint32_t* arr, uint32_t val, int lane, uint64_t ltmask) {
    uint64_t pend = __ballot(cnt != nullptr);
    while (pend) {
        int leader = __ffsll((unsigned long long)pend) - 1;
        ull key = __shfl((ull)(uintptr_t)cnt, leader);
        bool mine = cnt != nullptr && (ull)(uintptr_t)cnt == key;
        uint64_t m = __ballot(mine);
        ull base = 0;
        if (lane == leader) base = global_add((ull*)(uintptr_t)key, (ull)__popcll(m));
        base = __shfl(base, leader);
        if (mine) arr[base + (ull)__popcll(m & ltmask)] = val;
        pend &= ~m;
    }
}

// A lane's RBEB collision waiting for the wave's cooperative rejection loop (LDS, one slot
// per lane of the wave, then a 64-entry rank table)
struct __attribute__((aligned(16))) RbebJob {
    RbebSetup s;
    double first;  // uniform number d0 of the stream when d0 is odd (a cached block's half)
    uint64_t uid;
    uint32_t d0, step;  // stream position before the loop, step of the stream
};
// a wave's LDS area: the RBEB jobs and their rank table, then its stack of secondaries
constexpr int STACK = 64;
constexpr int COOP_JOB_BYTES = 64 * (int)sizeof(RbebJob) + 64;
constexpr int COOP_WAVE_BYTES = COOP_JOB_BYTES + 8 * STACK;

// v of the lane before (lane 0: anything): a wave-wide shift by one on the vector unit, without
// the round trip through LDS of a shuffle
__device__ __forceinline__ double lane_before(double v) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), 0x138, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), 0x138, 0xf, 0xf, false);
    return __hiloint2double(hi, lo);
}

// The rejection loops of the wave's pending RBEB collisions (_rbeb_sample,
// src/rbeb.jl:170-196), run by every lane of the wave together.  Trip k of a particle uses
// draws d0 + 2k and d0 + 2k + 1 of its stream, so any lane can evaluate it: each round the
// lanes are shared out over the particles still waiting (64 / n trips each, in order), and
// a particle takes its first accepting trip.  Result and stream position are those of the
// sequential loop; the wave runs about log(n) rounds instead of the longest particle's
// trip count.  Called by the whole wave; `pending` lanes have written their job.  Every
// particle still waiting has evaluated the same number of trips, so a round's stream
// positions need no memory, and its only shuffles are the accepted w and the second half of
// the last block looked at (LDS round trips take about 130 cycles each).
__device__ __forceinline__ void rbeb_coop(const Params& P, PT_LDS char* wlds, int lane, uint64_t ltmask,
                                          bool& pending, double& wout, StepStream& g) {
    PT_LDS RbebJob* jobs = (PT_LDS RbebJob*)wlds;
    PT_LDS uint8_t* rank_lane = (PT_LDS uint8_t*)(wlds + 64 * sizeof(RbebJob));
    const uint32_t k0 = (uint32_t)P.seed, k1 = (uint32_t)(P.seed >> 32);
    uint64_t U = __ballot(pending);
    uint32_t done = 0;  // trips of each waiting particle so far
    while (U) {
        const int nU = __popcll(U);
        // m = 64 / nU and gi = lane / m: the quotients are at least 1/128 away from the next
        // integers, far more than the error of the reciprocals
        const int m = (int)(64.5f * __builtin_amdgcn_rcpf((float)nU));
        const int myrank = __popcll(U & ltmask);
        if (pending) rank_lane[myrank] = (uint8_t)lane;
        wave_lds_order();
        const int gi = (int)(((float)lane + 0.5f) * __builtin_amdgcn_rcpf((float)m)), j = lane - gi * m;
        const bool act = gi < nU;
        double c0b = 0.0, c1b = 0.0, wv = 0.0;
        uint32_t D = 0;
        RbebSetup js;
        double jfirst = 0.0;
        if (act) {
            const PT_LDS RbebJob& J = jobs[rank_lane[gi]];
            js.t = J.s.t;
            js.A = J.s.A;
            js.Cc = J.s.Cc;
            js.M = J.s.M;
            js.pbn = J.s.pbn;
            js.ratio = J.s.ratio;
            js.iratio = J.s.iratio;
            jfirst = J.first;
            D = J.d0 + 2u * (done + (uint32_t)j);
            // the block of the trip's second draw
            uint32_t a = (uint32_t)J.uid, b = (uint32_t)(J.uid >> 32), c = J.step, e = (D + 1) >> 1;
            philox10(a, b, c, e, k0, k1);
            c0b = u01(a, b);
            c1b = u01(c, e);
        }
        const double prev = lane_before(c1b);  // the previous trip's block (same particle when j > 0)
        bool acc = false;
        if (act) {
            const bool odd = (D & 1) != 0;
            const double u = odd ? (j == 0 ? jfirst : prev) : c0b;
            acc = rbeb_trip(js, u, odd ? c0b : c1b, wv) || D + 2u >= DRAW_LIMIT;
        }
        const uint64_t Acc = __ballot(act && acc);
        // the first accepting trip, or the last one
        int hit = m - 1;
        bool got = false;
        if (pending) {
            const uint64_t gm = m >= 64 ? ~0ull : ((1ull << m) - 1ull);
            const uint64_t bits = (Acc >> (myrank * m)) & gm;
            got = bits != 0;
            if (got) hit = __ffsll((unsigned long long)bits) - 1;
        }
        const int src = pending ? myrank * m + hit : lane;
        const double w_s = __shfl(wv, src), c1_s = __shfl(c1b, src);
        if (pending) {
            if (got) {
                wout = w_s;
                // (at an odd position the second half of the last block is the next draw)
                g.draw += 2u * (done + (uint32_t)hit) + 2u;
                g.c1 = c1_s;
                g.cblk = (g.draw >> 1) + (g.draw & 1);
                pending = false;
            } else {
                jobs[lane].first = c1_s;
            }
        }
        done += (uint32_t)m;
        wave_lds_order();
        U = __ballot(pending);
    }
}

// onadvance of WallCallback (src/callback.jl:166-182): an upward crossing of x[coord] = v
// records lincomb(new, old, w) (src/electron.jl:127-132), w = (v - old) / (new - old); the
// particle is dropped if the wall says so.  The recorded state's s and r are not drawn.
__device__ __forceinline__ void wall_check(const Params& P, int sp, const V3& xo, const V3& po, double to,
                                           const V3& x, const V3& p, double w, double t, uint64_t uid,
                                           int swarm, bool& active) {
    const int c = P.wall.coord[sp];
    if (c < 0) return;
    const double v = P.wall.v[sp];
    const double a0 = c == 0 ? xo.x : (c == 1 ? xo.y : xo.z);
    const double a1 = c == 0 ? x.x : (c == 1 ? x.y : x.z);
    if (!(a0 < v && v < a1)) return;
    const double a = (v - a0) / (a1 - a0);
    ull slot = atomicAdd(P.wall.n, 1ull);
    if (slot < P.wall.cap) {
        pt_wall_record& r = P.wall.rec[slot];
        r.x[0] = x.x * a + xo.x * (1.0 - a);
        r.x[1] = x.y * a + xo.y * (1.0 - a);
        r.x[2] = x.z * a + xo.z * (1.0 - a);
        r.p[0] = p.x * a + po.x * (1.0 - a);
        r.p[1] = p.y * a + po.y * (1.0 - a);
        r.p[2] = p.z * a + po.z * (1.0 - a);
        r.w = w * a + w * (1.0 - a);
        r.t = t * a + to * (1.0 - a);
        r.uid = uid;
        r.species = sp;
        r.swarm = swarm;
    }
    if (P.wall.drop[sp]) active = false;
}

// The learned sampler's outputs for the lanes whose collision uses the network `which`
// (use): each draws its two uniforms (u1, u2) from its own stream, and the wave evaluates
// the network for all of them on the matrix cores.  Called by the whole wave.  y0, y1: the
// outputs (network + closed-form baseline) of the lanes with `use`.
template <class G>
__device__ __forceinline__ void learned_pass(const Params& P, const Shared& sh, int which, bool use, int sp, int sel,
                                             double E, G& g, float& y0, float& y1) {
    float xin[MLP_IN];
    for (int q = 0; q < MLP_IN; q++) xin[q] = 0.0f;
    if (use) {
        const double u1 = g.next(), u2 = g.next();
        const DevProc& pr = process(sh, sp, sel);
        const double ph =
            which == LEARN_SB ? sb_phase(P.sb[pr.slot].log_energy, P.sb[pr.slot].thr, P.sb[pr.slot].ne, E) : 0.0;
        mlp_features(E / EV, pr.Z, u1, u2, ph, xin);
    }
    float a0, a1;
    mlp_wave(P.mlp[which].w, P.mlp[which].b, xin, use, a0, a1);
    if (use) {
        float b0, b1;
        mlp_baseline(which, xin, b0, b1);
        y0 = a0 + b0;
        y1 = a1 + b1;
    }
}

// the swarm a particle's statistics go to (out-of-range values count as swarm 0)
__device__ __forceinline__ int swarm_of(const Params& P, int32_t sw) { return (sw < 0 || sw >= P.nswarm) ? 0 : sw; }

template <int SRC, bool EVENT, bool WALL = false, bool MLP = false, bool LEAN = false>
__device__ __forceinline__ void select_loop(const Params& P, Shared& sh, PT_LDS char* wlds, const ull* rb, const ull* re,
                                            ull* cursor, uint32_t step0, bool main_pass, int par) {
    // range passes with every collision in place advance their particles through several
    // steps; the others through one
    constexpr bool MULTI = SRC == SRC_RANGE && !EVENT;
    constexpr bool MORE = MULTI && LEAN;
    const int K = MULTI ? sh.nsub : 1;
    const ull n0 = re[0] - rb[0], n1 = re[1] - rb[1], n2 = re[2] - rb[2];
    const ull total = n0 + n1 + n2;
    const uint32_t foff = P.forcing_off;  // read once: the loop below does not reload it
    const int lane = threadIdx.x & 63;
    const uint64_t ltmask = lane ? (~0ull >> (64 - lane)) : 0ull;
    // wave-uniform chunk state
    const ull nwaves = (ull)gridDim.x * (blockDim.x >> 6);
    const int lanes = lanes_used(total, nwaves);
    const ull least = lanes < LEAST_CHUNK ? lanes : LEAST_CHUNK;
    // The first one fills the wave's lanes.  With one step a launch it is more, up to the wave's
    // share, as each further claim is a round trip (2 x 10^5 electrons 6.8 -> 6.5 ms for 24
    // such launches); an item of several steps takes far longer than that, and the waves end
    // closer together if little is given out beforehand (32 swarms of 10^4 electrons 20.1 ->
    // 18.9 ms, 1.2 x 10^6 7.3 -> 7.0; a beam of 2 x 10^6 photons, whose electrons no longer
    // crowd in a wave's first items, 147 -> 124).
    ull chunk = K == 1 && total / nwaves > 64 ? claim_chunk(4 * total, nwaves, least) : (ull)lanes;
    ull cbeg = 0, cend = 0;
    bool drained = false;
    // the wave's next chunk of items; false when they are all claimed
    auto claim = [&]() {
        int fl = __ffsll((unsigned long long)__ballot(1)) - 1;
        ull b = 0;
        if (lane == fl) b = global_add(cursor, chunk);
        b = __shfl(b, fl);
        if (b >= total) {
            drained = true;
            return false;
        }
        cbeg = b;
        cend = b + chunk < total ? b + chunk : total;
        chunk = claim_chunk(total - cend, nwaves, least);
        return true;
    };
    // the wave's secondaries waiting to be advanced (LDS, last in first out)
    PT_LDS uint64_t* const stk = (PT_LDS uint64_t*)(wlds + COOP_JOB_BYTES);
    int nstk = 0;  // wave-uniform
    int extra = 0;  // push rounds since the wave's last collision phase (wave-uniform)
    // lane state
    bool have = false;
    int sp = 0, swarm = 0;
    uint32_t idx = 0;
    V3 x{0, 0, 0}, p{0, 0, 0};
    double w = 0, t = 0, s = 0, r = 0, trem = 0;
    StepStream g;
    g.init(P.seed, 0, 0);
    uint32_t iters = 0;
    uint32_t n_events = 0, n_psteps = 0, n_tail = 0;  // the lane's work counts
    bool active = false, oob = false;
    bool child = false;  // born in the step it is in (counted apart)
    bool born = false;   // born in this launch: marked when it is done
    bool half = false;   // its next draw is the second half of the block cached in g.c1
    bool pend = false;   // its push ended in a collision, which is still to be selected
    bool new_r = false;  // its rate bound is to be recomputed
    double cE = 0.0;     // kinetic energy at the pending collision
    int ks = 0;          // the step it is in (0..K-1)
    // what the lane's particle needs of its species and swarm, in registers while it has the
    // lane (each read from LDS is a round trip in the chain of dependent operations that an
    // iteration is): table grid, cut, offsets of its tables, and with a uniform electric field
    // and no magnetic one its force
    double cut = 0, pphi = 0, xmax = 1, ixmax = 1, two_k1 = 1;
    int kint = 0, nprocs = 0, rate_off = 0, rb_off = 0;
    V3 F{0, 0, 0};
    const bool ffree = P.field_lds && (foff & OFF_NO_B);
    const bool falong = (foff & OFF_E_Z) != 0;
    // the rate bound's coefficients in the interval ci of its energy
    int ci = -1;
    double rc0 = 0, rc1 = 0, rc2 = 0;
    auto cut_of = [&]() { return LEAN ? sh.sp[sp].cut : cut; };
    auto grid = [&](double E, double& t1, double& t2, bool& o) {
        const SpLite& L = sh.sp[sp];
        return LEAN ? precheb(E, L.k, L.xmax, L.ixmax, L.two_k1, t1, t2, o)
                    : precheb(E, kint, xmax, ixmax, two_k1, t1, t2, o);
    };
    // setr! of the lane's particle (src/collisions.jl:63-74)
    auto rate_bound = [&](double E) {
        if (E < cut_of()) return 0.0;
        double t1, t2;
        bool o;
        const int i = grid(E, t1, t2, o);
        oob |= o;
        if constexpr (LEAN) {
            const SpLite& L = sh.sp[sp];
            if (P.rb_in_lds) return cheb3(as_lds(pt_lds) + L.rb_off + 3 * i, t1, t2);
            return cheb3(as_global(L.rb) + ((size_t)(P.nswarm > 1 ? swarm : 0) * (L.k + 1) + i) * 3, t1, t2);
        }
        if (i != ci) {
            ci = i;
            if (P.rb_in_lds) {
                const PT_LDS double* c = as_lds(pt_lds) + rb_off + 3 * i;
                rc0 = c[0];
                rc1 = c[1];
                rc2 = c[2];
            } else {
                const PT_GLOBAL double* c =
                    as_global(sh.sp[sp].rb) + ((size_t)(P.nswarm > 1 ? swarm : 0) * (kint + 1) + i) * 3;
                rc0 = c[0];
                rc1 = c[1];
                rc2 = c[2];
            }
        }
        return (rc0 * 1.0 + rc1 * t1) + rc2 * t2;
    };
    // with no dose tally nothing is left of a secondary below the cut; with one, its energy
    const double dropcut = sh.cut[PT_ELECTRON] * (1.0 - 1e-9);
    // the particle that has just been given to the lane: its species' and swarm's constants
    auto settle = [&]() {
        if constexpr (LEAN) return;
        const SpLite& L = sh.sp[sp];
        cut = L.cut;
        pphi = L.ppcut_hi;
        xmax = L.xmax;
        ixmax = L.ixmax;
        two_k1 = L.two_k1;
        kint = L.k;
        nprocs = L.nprocs;
        rate_off = L.rate_off;
        rb_off = L.rb_off;
        ci = -1;
        if (ffree) {
            const PT_LDS double* e = as_lds(pt_lds) + P.lds_field_off + field_doubles(P.forcing_off) * swarm;
            const double q = (sp == PT_ELECTRON ? -1.0 : 1.0) * QE;
            const bool none = sp == PT_PHOTON || (foff & off_em(sp));
            F = V3{none ? 0.0 : q * e[0], none ? 0.0 : q * e[1], none ? 0.0 : q * e[2]};
        }
    };
    // an item that was just read becomes the lane's particle if it has a step to do from
    // step k0 on; `ch`: it was born in step k0
    auto take = [&](int qs, ull qi, const Loaded& a, int k0, bool ch, bool bo) {
        int k = k0;
        double cr = sh.tf[k] - a.t;
        if constexpr (MULTI) {
            while (!(cr > EPS64) && ++k < K) {
                cr = sh.tf[k] - a.t;
                ch = false;
            }
        }
        if (a.act == 0 || !(cr > EPS64)) return;
        sp = qs;
        idx = (uint32_t)qi;
        x = a.x;
        p = a.p;
        w = a.w;
        t = a.t;
        s = a.s;
        swarm = swarm_of(P, a.swarm);
        trem = cr;
        oob = false;
        new_r = true;
        ks = k;
        g.init(P.seed, a.uid, step0 + (uint32_t)k);
        half = false;
        iters = 0;
        active = true;
        have = true;
        child = ch;
        born = bo;
        settle();
    };
    for (;;) {
        const bool first = !MORE || extra == 0;
        // A. the end of a particle's step: droplow!'s cut, then its next step, or back to memory
        if (have && !pend && (!(trem > EPS64) || !active)) {
            // droplow!: the energy is computed only where |p|^2 does not settle the test
            if (active && !(dot3(p, p) > (LEAN ? sh.sp[sp].ppcut_hi : pphi))) {
                double Ek = kinenergy(sp, p);
                if (Ek < cut_of()) {
                    active = false;
                    deposit(P, sh.bc, Ek * w, x.z);
                }
            }
            // a collision at the very end of the step: the record gets the new rate bound
            if (new_r) {
                r = rate_bound(kinenergy(sp, p));
                new_r = false;
            }
            if (oob) atomicAdd(&sh.bc.flags[FLAG_RANGE], 1ull);
            if (child)
                n_tail++;
            else
                n_psteps++;
            bool cont = false;
            if constexpr (MULTI) {
                if (active) {
                    while (++ks < K) {
                        trem = sh.tf[ks] - t;
                        if (trem > EPS64) {
                            cont = true;
                            break;
                        }
                    }
                }
            }
            if (cont) {
                // the next step's advance_init!: a new rate bound and random stream
                g.restart(step0 + (uint32_t)ks);
                half = false;
                iters = 0;
                oob = false;
                child = false;
                new_r = true;
            } else {
                // the particle's record: 72 contiguous bytes (w unchanged), written in whole
                // sectors, four of the five stores 16 bytes wide
                const SpLite& L = sh.sp[sp];
                {
                    PT_GLOBAL pair2* w2 = rec_pairs(L, idx);
                    const pair2 v0 = {x.x, x.y}, v1 = {x.z, p.x}, v2 = {p.y, p.z}, v4 = {s, r};
                    w2[0] = v0;
                    w2[1] = v1;
                    w2[2] = v2;
                    PF(L.f[PT_T], idx) = t;
                    w2[4] = v4;
                }
                if (!active) L.active[idx] = 0;
                if (MULTI && born && K > 1) L.draw[idx] = (uint32_t)K;
                have = false;
            }
        }
        // B. free lanes take the wave's waiting secondaries, then the next items of its chunk,
        //    in lane order
        if (first) {
            uint64_t need = __ballot(!have);
            while (need) {
                const int rank = __popcll(need & ltmask), nfree = __popcll(need);
                const int pop = nfree < nstk ? nfree : nstk;
                bool mine = false, ch = !main_pass, bo = false;
                int qs = 0, k0 = 0;
                ull qi = 0;
                if (!have && rank < pop) {
                    const uint64_t e = stk[nstk - 1 - rank];
                    qi = e & 0xFFFFFFFFull;
                    qs = (int)(e >> 32) & 0xFF;
                    k0 = (int)(e >> 40);
                    ch = bo = true;
                    mine = true;
                }
                nstk -= pop;
                const uint64_t open = __ballot(!have && rank >= pop && lane < lanes);
                if (open && !drained && (cbeg < cend || claim())) {
                    const ull want = (ull)__popcll(open);
                    const ull q = cbeg + (ull)__popcll(open & ltmask);
                    if (((open >> lane) & 1) && q < cend) {
                        if (q < n0) {
                            qs = 0;
                            qi = rb[0] + q;
                        } else if (q < n0 + n1) {
                            qs = 1;
                            qi = rb[1] + (q - n0);
                        } else {
                            qs = 2;
                            qi = rb[2] + (q - n0 - n1);
                        }
                        mine = true;
                    }
                    cbeg = cbeg + want < cend ? cbeg + want : cend;
                }
                if (__ballot(mine) == 0) break;
                if (mine) {
                    if constexpr (SRC == SRC_QUEUE) {
                        // queued particles are active and always enter (one with no time left
                        // is only finished); secondaries on the stack enter as in a range
                        const bool queued = !bo;
                        if (queued) {
                            const uint32_t e = P.q.work[qs][par][qi];
                            ch = (e & CHILD_BIT) != 0;
                            qi = e & ~CHILD_BIT;
                        }
                        const SpLite& Lq = sh.sp[qs];
                        const Loaded a = load_slot(Lq, qi);
                        if (queued) {
                            const double cr = Lq.trem[qi];
                            const uint32_t d0 = Lq.draw[qi];
                            sp = qs;
                            idx = (uint32_t)qi;
                            x = a.x;
                            p = a.p;
                            w = a.w;
                            t = a.t;
                            s = a.s;
                            swarm = swarm_of(P, a.swarm);
                            trem = cr;
                            oob = false;
                            r = PF(Lq.f[PT_R], qi);  // set by the sampler (setr! of apply!) or at birth
                            new_r = false;
                            g.init(P.seed, a.uid, step0);
                            g.resume(d0);
                            half = (d0 & 1) != 0;
                            iters = 0;
                            active = true;
                            have = true;
                            child = ch;
                            born = false;
                            settle();
                        } else {
                            take(qs, qi, a, 0, ch, false);
                        }
                    } else {
                        const Loaded a = load_slot(sh.sp[qs], qi);
                        // a pass over secondaries of several steps: the step each was born in,
                        // or K when it has been advanced already
                        if (MULTI && K > 1 && !main_pass && !bo) {
                            k0 = (int)sh.sp[qs].draw[qi];
                            bo = true;
                        }
                        if (k0 < K) take(qs, qi, a, k0, ch, bo);
                    }
                }
                need = __ballot(!have);
            }
            // C. the wave leaves when its items are claimed and no lane holds a particle
            if (drained && nstk == 0 && __ballot(have) == 0) break;
        }
        // setr! for a particle that changed: after its collision, at the start of a step, or
        // newly taken (one evaluation for all these lanes)
        if (new_r) {
            r = rate_bound(kinenergy(sp, p));
            new_r = false;
        }
        const double tnext = qdiv_any(s, r);
        // D. one push of this lane's particle
        if (have && !pend && trem > EPS64 && active) {
            if (++iters > ITER_LIMIT || g.exhausted()) {
                atomicAdd(&sh.bc.flags[FLAG_SAMPLER], 1ull);
                trem = 0.0;
            } else {
                double dt;
                bool coll;
                if (trem > tnext) {
                    dt = tnext;
                    coll = true;
                } else {
                    dt = trem;
                    coll = false;
                    s -= dt * r;
                }
                const V3 xo = x, po = p;
                const double to = t;
                V3 dx{0, 0, 0}, dp{0, 0, 0};
                if (ffree) {
                    if constexpr (LEAN) {
                        const PT_LDS double* e = as_lds(pt_lds) + P.lds_field_off + field_doubles(P.forcing_off) * swarm;
                        const double q = (sp == PT_ELECTRON ? -1.0 : 1.0) * QE;
                        const bool none = sp == PT_PHOTON || (foff & off_em(sp));
                        F = V3{none || falong ? 0.0 : q * e[0], none || falong ? 0.0 : q * e[1], none ? 0.0 : q * e[2]};
                    }
                    push_uniform(sp, F, falong, p, dt, dx, dp);
                } else if (P.field_lds) {
                    const PT_LDS double* fv = as_lds(pt_lds) + P.lds_field_off + field_doubles(P.forcing_off) * swarm;
                    const HomField hf{{fv}, {fv + 3}, {{nullptr, nullptr}}};
                    push_delta(sp, hf, x, p, dt, foff, dx, dp);
                } else if (P.nswarm == 1) {
                    push_delta(sp, sh.field0, x, p, dt, foff, dx, dp);
                } else {
                    push_delta(sp, as_global(P.fields)[swarm], x, p, dt, foff, dx, dp);
                }
                if (foff & off_push(sp)) {
                    dx = V3{0, 0, 0};  // only its time advances
                } else {
                    x = V3{x.x + dx.x, x.y + dx.y, x.z + dx.z};
                    p = V3{p.x + dp.x, p.y + dp.y, p.z + dp.z};
                }
                t = t + dt;
                if constexpr (WALL) wall_check(P, sp, xo, po, to, x, p, w, t, g.uid(), swarm, active);
                trem -= dt;
                if (coll && r != 0.0 && (!WALL || active)) {
                    const double E = kinenergy(sp, p);
                    if (E >= cut_of()) {
                        n_events++;
                        cE = E;
                        pend = true;
                    }
                }
            }
        }
        if constexpr (MULTI) {
            // E. another push round before the collisions: when no lane has one, or when
            //    enough lanes can still reach theirs
            if (__ballot(pend) == 0) {
                extra = 0;
                continue;
            }
        }
        if constexpr (MORE) {
            const bool ready = have && !pend && active && (trem > EPS64 || ks < K - 1);
            if (extra < MORE_ROUNDS && __popcll(__ballot(ready)) >= MORE_LANES) {
                extra++;
                continue;
            }
            extra = 0;
        }
        // F. the selection; a real collision is finished in H, after the wave's RBEB rejection
        //    loops (G)
        ull* qc = nullptr;
        uint32_t* qa = nullptr;
        uint32_t qv = 0;
        int qsel = -1;          // collision queued for the sampling kernel
        int csel = -1;          // collision sampled in H
        bool rb_wait = false;   // an RBEB collision waiting for the cooperative loop
        double rb_w = -1.0;
        ProcVals cp{0, 0.0, 0.0};  // what the common samplers need of its process
        g.cblk = half ? (g.draw >> 1) + 1u : 0u;
        if (pend) {
            pend = false;
            double t1, t2;
            bool o;
            const int iv = grid(cE, t1, t2, o);
            oob |= o;
            const double xi = g.next() * r;
            const int np = LEAN ? sh.sp[sp].nprocs : nprocs, at = LEAN ? sh.sp[sp].rate_off : rate_off;
            const PT_LDS double* const row = as_lds(pt_lds) + at + iv * np * 3;
            const int sel = select_process(row, np, t1, t2, xi);
            if (sel >= np) {
                if (!null_remains(row, np, t1, t2, xi)) atomicAdd(&sh.bc.flags[FLAG_RATEBOUND], 1ull);
                atomicAdd(&sh.bc.counts[sp * NCOUNT], 1ull);
                new_r = true;  // setr! of the null collision (p unchanged)
                s = nextcoll(g);
            } else {
                const DevProc& pr = process(sh, sp, sel);
                cp.kind = pr.kind;
                cp.B = pr.B;
                cp.c0 = pr.c[0];
                const double c1 = pr.c[1], c2 = pr.c[2];
                atomicAdd(&sh.bc.counts[sp * NCOUNT + 1 + sel], 1ull);
                if (EVENT && ((P.defer_mask >> cp.kind) & 1u)) {
                    qsel = sel;
                } else {
                    csel = sel;
                    if (cp.kind == PT_PROC_RBEB) {
                        PT_LDS RbebJob& J = ((PT_LDS RbebJob*)wlds)[lane];
                        const RbebSetup js = rbeb_setup(cE, cp.B, cp.c0, c1, c2, g.tab());
                        J.s.t = js.t;
                        J.s.A = js.A;
                        J.s.Cc = js.Cc;
                        J.s.M = js.M;
                        J.s.pbn = js.pbn;
                        J.s.ratio = js.ratio;
                        J.s.iratio = js.iratio;
                        J.first = g.c1;
                        J.uid = g.uid();
                        J.d0 = g.draw;
                        J.step = g.step;
                        rb_wait = true;
                    }
                }
            }
        }
        // G. every lane of the wave runs the pending RBEB rejection loops
        rbeb_coop(P, wlds, lane, ltmask, rb_wait, rb_w, g);
        // learned samplers: the wave's bremsstrahlung and Moller collisions whose network
        // is in use go through it on the matrix cores, one kind at a time
        float ly0 = 0.0f, ly1 = 0.0f;
        bool lnet = false;
        if constexpr (MLP) {
            int lw = -1;
            if (csel >= 0) {
                const int kd = cp.kind;
                lw = kd == PT_PROC_SB ? LEARN_SB : (kd == PT_PROC_MOLLER ? LEARN_MOLLER : -1);
            }
            lnet = lw >= 0 && P.mlp[lw].on && cE >= P.mlp[lw].emin && cE <= P.mlp[lw].emax;
            for (int which = 0; which < NLEARN; which++)
                if (__ballot(lnet && lw == which)) learned_pass(P, sh, which, lnet && lw == which, sp, csel, cE, g, ly0, ly1);
        }
        // H. the sampled collision
        ull sl0 = NO_SLOT, sl1 = NO_SLOT;  // slots of the secondaries it stored
        int cs0 = 0, cs1 = 0;
        // elastic scattering and ionisation are nearly all collisions of electrons: the lanes
        // of both kinds go through one straight path together
        const bool common = csel >= 0 && ((cp.kind == PT_PROC_ELASTIC && sp != PT_PHOTON) ||
                                          (cp.kind == PT_PROC_RBEB && rb_w >= 0.0));
        if (common) {
            const bool el = cp.kind == PT_PROC_ELASTIC;
            const double E2 = cp.B * rb_w;
            const bool drop = el || E2 < dropcut;
            V3 m0, m1;
            double s0, s1;
            const bool ok = common_event(el, cp, p, cE, E2, drop, g, m0, m1, s0, s1);
            if (!el) {
                if (!ok) atomicAdd(&sh.bc.flags[FLAG_SAMPLER], 1ull);
                // left here: the binding energy, and that of a secondary below the cut
                deposit(P, sh.bc, (drop ? cp.B + E2 : cp.B) * w, x.z);
                if (!drop) {
                    cs1 = PT_ELECTRON;
                    sl1 = append(P, sh, PT_ELECTRON, x, m1, w, t, s1, g.uid(), g.step, g.draw, 0, swarm, main_pass,
                                 (uint32_t)ks);
                }
            }
            p = m0;
            s = s0;
            new_r = true;  // setr! of apply!
        } else if (csel >= 0) {
            const double E = cE;
            const double pn = norm3(p);
            Ev e;
            if (MLP && lnet) learned_event(process(sh, sp, csel), sp, E, ly0, ly1, g, e);
            else sample_event(process(sh, sp, csel), sp, p, pn, E, P.sb, P.pe, g, e, dropcut);
            if (e.err) atomicAdd(&sh.bc.flags[FLAG_SAMPLER], 1ull);
            if (e.dep != 0.0) deposit(P, sh.bc, e.dep * w, x.z);
            V3 m0, m1;
            double s0, s1;
            bool drop1;
            finish_event(p, pn, e, g, m0, m1, s0, s1, sh.cut, sh.stored, dropcut, drop1);
            if (drop1) deposit(P, sh.bc, e.eB * w, x.z);
            const uint32_t dend = g.draw;
            if (e.keep) {
                p = m0;
                s = s0;
                new_r = true;  // setr! of apply!
            } else {
                active = false;
                cs0 = e.sp0;
                sl0 = append(P, sh, e.sp0, x, m0, w, t, s0, g.uid(), g.step, dend, 0, swarm, main_pass, (uint32_t)ks);
            }
            if (e.ne == 2 && !drop1) {
                cs1 = e.sp1;
                sl1 = append(P, sh, e.sp1, x, m1, w, t, s1, g.uid(), g.step, dend, e.keep ? 0 : 1, swarm, main_pass,
                             (uint32_t)ks);
            }
        }
        // what the streams keep between collisions
        half = (g.draw & 1) && g.cblk == (g.draw >> 1) + 1u;
        g.c0 = 0.0;
        g.cblk = 0;
        // the secondaries wait on the wave's stack for its free lanes; those that find it full
        // are left to the passes over the step's secondaries
        if (__ballot(sl0 != NO_SLOT || sl1 != NO_SLOT)) {
#pragma unroll
            for (int q = 0; q < 2; q++) {
                const ull sl = q ? sl1 : sl0;
                const uint64_t m = __ballot(sl != NO_SLOT);
                const int at = nstk + __popcll(m & ltmask);
                if (sl != NO_SLOT && at < STACK)
                    stk[at] = sl | (uint64_t)(q ? cs1 : cs0) << 32 | (uint64_t)(uint32_t)ks << 40;
                const int all = nstk + __popcll(m);
                nstk = all < STACK ? all : STACK;
                if (all > STACK && lane == 0) global_add(&P.clock->left, (ull)(all - STACK));
            }
            wave_lds_order();
        }
        if constexpr (EVENT) {
            if (qsel >= 0) {
                const SpLite& L = sh.sp[sp];
                // queued for its sampler: the state after the push, the time left and the
                // stream position (r and s are replaced when the collision is applied)
                PF(L.f[PT_X], idx) = x.x;
                PF(L.f[PT_Y], idx) = x.y;
                PF(L.f[PT_Z], idx) = x.z;
                PF(L.f[PT_PX], idx) = p.x;
                PF(L.f[PT_PY], idx) = p.y;
                PF(L.f[PT_PZ], idx) = p.z;
                PF(L.f[PT_T], idx) = t;
                L.trem[idx] = trem;
                L.draw[idx] = g.draw;
                L.evp[idx] = (uint8_t)qsel;
                int k = P.q.kq[sp][process(sh, sp, qsel).kind];
                qc = P.q.cnt + QEV(sp, k);
                qa = P.q.ev[sp][k];
                qv = idx | (child ? CHILD_BIT : 0u);
                if (oob) atomicAdd(&sh.bc.flags[FLAG_RANGE], 1ull);
                have = false;
            }
            wave_push(qc, qa, qv, lane, ltmask);
        }
    }
    // the lane's work counts, kept in registers (an LDS atomic per retiring lane on one
    // address would serialise the wave's lanes every iteration)
    if (n_events) atomicAdd(&sh.bc.work[W_EVENTS], (ull)n_events);
    if (n_psteps) atomicAdd(&sh.bc.work[W_PSTEPS], (ull)n_psteps);
    if (n_tail) atomicAdd(&sh.bc.work[W_TAIL], (ull)n_tail);
}

// ------------------------------------------------------------------ step kernels
__global__ void k_snapshot(const Params* __restrict__ Pp, int clocked, double tfinal, double dt, uint32_t step,
                           int nsub) {
    const Params& P = *Pp;
    int s = threadIdx.x;
    Clock& C = *P.clock;
    if (s < PT_NSPECIES) {
        ull n = *P.sp[s].n;
        if (n > P.sp[s].cap) n = P.sp[s].cap;
        P.range[2 * s] = 0;
        P.range[2 * s + 1] = n;
        C.nmark[s] = n;
    }
    for (int q = threadIdx.x; q < NQCNT; q += blockDim.x) P.q.cnt[q] = 0;
    if (s == 0) {
        // the steps' final times, by the host loop's arithmetic (t += dt)
        double tf = clocked ? C.t + C.dt : tfinal;
        const double d = clocked ? C.dt : dt;
        for (int k = 0; k < MAX_SUB; k++) {
            C.tf[k] = tf;
            if (k == nsub - 1) C.tfinal = tf;
            tf = tf + d;
        }
        C.nsub = (uint32_t)nsub;
        if (!clocked) C.step = step;
        C.cursor = 0;
        C.ecur = 0;
        C.qpar = 0;
        C.pass = 0;
        C.left = 0;
        C.done = 0;
    }
}

template <class T>
__device__ __forceinline__ void to_host(T* p, T v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
__device__ __forceinline__ void report_state(const Params& P, ull left) {
    Report& R = *P.report;
    for (int s = 0; s < PT_NSPECIES; s++)
        to_host(&R.n[s], __hip_atomic_load(P.sp[s].n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
    for (int q = 0; q < NFLAGS; q++)
        to_host(&R.flags[q], __hip_atomic_load(&P.flags[q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
    to_host(&R.left, left);
}
__global__ void k_report(const Params* __restrict__ Pp) {
    if (threadIdx.x == 0) report_state(*Pp, 0);
}

// The end of a pass, called by every workgroup of its launch: the last one to end sets up the
// next advance1! pass (src/mixed_population.jl:43-46) over the particles appended since the
// last mark, for the whole grid.  When every secondary found room on its wave's stack there is
// nothing left to do, and the next pass is empty.  What the last workgroup reads was written
// by atomics, which have all been performed once every wave has waited for its own: no cache
// is written back (a __threadfence() in each of the 512 workgroups takes 13 us).
__device__ __forceinline__ void end_pass(const Params& P) {
    wait_vmem();
    __syncthreads();
    if (threadIdx.x != 0) return;
    Clock& C = *P.clock;
    const uint32_t k = __hip_atomic_fetch_add(&C.done, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (k != gridDim.x - 1) return;
    const ull left = __hip_atomic_load(&C.left, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    for (int s = 0; s < PT_NSPECIES; s++) {
        ull n = __hip_atomic_load(P.sp[s].n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (n > P.sp[s].cap) n = P.sp[s].cap;
        P.range[2 * s] = left ? C.nmark[s] : n;
        P.range[2 * s + 1] = n;
        if (left) C.nmark[s] = n;
    }
    C.cursor = 0;
    C.pass += 1;
    C.left = 0;
    C.done = 0;
    report_state(P, left);
}

__global__ void k_tick(const Params* __restrict__ Pp) {
    Clock& C = *Pp->clock;
    if (threadIdx.x == 0) {
        C.t = C.tfinal;
        C.step += C.nsub;
    }
}

// after a sampling round: its output queue becomes the input of the next push/select
// round; the consumed input and the collision queues are emptied.  The secondary passes
// that follow the rounds start where the step's secondaries start (the mark k_snapshot
// set): a secondary stored when its wave's stack was full, in any round, is advanced there;
// the others have reached the end of the step and are skipped.
__global__ void k_rotate(const Params* __restrict__ Pp) {
    const Params& P = *Pp;
    Clock& C = *P.clock;
    __shared__ uint32_t par;
    if (threadIdx.x == 0) par = C.qpar;
    __syncthreads();
    int s = threadIdx.x;
    if (s < PT_NSPECIES) {
        P.q.cnt[QWK(s, par)] = 0;
        for (int k = 0; k < NKQ; k++) P.q.cnt[QEV(s, k)] = 0;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        C.qpar = par ^ 1u;
        C.cursor = 0;
        C.ecur = 0;
    }
}

// push/select over the step's particles (first round) or the input work queues
template <int BS, int SRC, bool EVENT, bool WALL = false, bool MLP = false>
__global__ void __launch_bounds__(BS) __attribute__((amdgpu_waves_per_eu(BS > 512 ? 3 : 2)))
k_advance(const Params* __restrict__ Pp) {
    __shared__ Shared sh;
    __shared__ int skip;
    const Params& P = *Pp;
    const Clock& C = *P.clock;
    const int par = (int)C.qpar;
    ull rb[PT_NSPECIES], re[PT_NSPECIES];
    ull total = 0;
    for (int s = 0; s < PT_NSPECIES; s++) {
        if (SRC == SRC_RANGE) {
            rb[s] = P.range[2 * s];
            re[s] = P.range[2 * s + 1];
        } else {
            rb[s] = 0;
            re[s] = P.q.cnt[QWK(s, par)];
        }
        total += re[s] - rb[s];
    }
    // workgroups that start after every item is claimed leave before staging the tables
    if (threadIdx.x == 0)
        skip = __hip_atomic_load(&P.clock->cursor, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >= total;
    __syncthreads();
    if (skip) {
        if constexpr (!EVENT) {
            // (a further pass over nothing leaves the next one empty, too)
            if (total > 0 || C.pass == 0) end_pass(P);
        }
        return;
    }
    stage(P, sh);
    PT_LDS char* wlds = (PT_LDS char*)pt_lds + P.lds_coop_off + (threadIdx.x >> 6) * COOP_WAVE_BYTES;
    select_loop<SRC, EVENT, WALL, MLP, (BS > 512)>(P, sh, wlds, rb, re, &P.clock->cursor, C.step,
                                                   SRC == SRC_RANGE && C.pass == 0, par);
    flush_counters(P, &sh.bc);
    if constexpr (!EVENT) end_pass(P);
}

// Sampling round: each wave takes 64 queued collisions of one sampler kind (the queues are
// laid out back to back, each padded to whole tiles), samples and applies them (collide /
// apply!, src/collisions.jl:83-133), and queues the surviving primary and the new
// particles for the next push/select round.
template <int BS>
__global__ void __launch_bounds__(BS) __attribute__((amdgpu_waves_per_eu(2))) k_sample(const Params* __restrict__ Pp) {
    __shared__ Shared sh;
    __shared__ ull seg[PT_NSPECIES * NKQ + 1];
    __shared__ int skip;
    const Params& P = *Pp;
    const Clock& C = *P.clock;
    const double tfinal = C.tfinal;
    const uint32_t step = C.step;
    const int par = (int)C.qpar, nxt = par ^ 1;
    if (threadIdx.x == 0) {
        ull acc = 0;
        for (int q = 0; q < PT_NSPECIES * NKQ; q++) {
            seg[q] = acc;
            acc += (P.q.cnt[2 * PT_NSPECIES + q] + 63) & ~63ull;
        }
        seg[PT_NSPECIES * NKQ] = acc;
        skip = __hip_atomic_load(&P.clock->ecur, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >= acc;
    }
    __syncthreads();
    if (skip) return;
    stage(P, sh);
    const int lane = threadIdx.x & 63;
    const uint64_t ltmask = lane ? (~0ull >> (64 - lane)) : 0ull;
    const ull total = seg[PT_NSPECIES * NKQ];
    for (;;) {
        int fl = __ffsll((unsigned long long)__ballot(1)) - 1;
        ull b = 0;
        if (lane == fl) b = atomicAdd(&P.clock->ecur, 64ull);
        b = __shfl(b, fl);
        if (b >= total) break;
        int qi = 0;
        while (qi + 1 < PT_NSPECIES * NKQ && seg[qi + 1] <= b) qi++;
        const int sp = qi / NKQ, kq = qi % NKQ;
        const ull pos = b - seg[qi] + (ull)lane;
        const bool valid = pos < P.q.cnt[QEV(sp, kq)];
        const int kind = P.q.qkind[sp][kq];
        const int lw = kind == PT_PROC_SB ? LEARN_SB : (kind == PT_PROC_MOLLER ? LEARN_MOLLER : -1);
        const bool learned = lw >= 0 && P.mlp[lw].on;  // uniform over the wave (one kind per tile)
        ull* c0 = nullptr;
        ull* c1 = nullptr;
        ull* c2 = nullptr;
        uint32_t* a0 = nullptr;
        uint32_t* a1 = nullptr;
        uint32_t* a2 = nullptr;
        uint32_t v0 = 0, v1 = 0, v2 = 0;
        const SpLite& L = sh.sp[sp];
        uint32_t ent = 0;
        ull idx = 0;
        V3 x{0, 0, 0}, p{1, 0, 0};
        double w = 0, t = 0, E = 0, pn = 1;
        uint64_t uid = 0;
        int swarm = 0, sel = 0;
        StepStream g;
        g.init(0, 0, 0);
        if (valid) {
            ent = P.q.ev[sp][kq][pos];
            idx = ent & ~CHILD_BIT;
            x = V3{PF(L.f[PT_X], idx), PF(L.f[PT_Y], idx), PF(L.f[PT_Z], idx)};
            p = V3{PF(L.f[PT_PX], idx), PF(L.f[PT_PY], idx), PF(L.f[PT_PZ], idx)};
            w = PF(L.f[PT_W], idx);
            t = PF(L.f[PT_T], idx);
            uid = L.uid[idx];
            swarm = L.swarm[idx];
            if (swarm < 0 || swarm >= P.nswarm) swarm = 0;
            sel = L.evp[idx];
            g.init(P.seed, uid, step);
            g.resume(L.draw[idx]);
            E = kinenergy(sp, p);
            pn = norm3(p);
        }
        float y0 = 0.0f, y1 = 0.0f;
        // the network is used in the energy range its KS gate covered; outside it the
        // rejection sampler runs
        const bool use_net = learned && valid && E >= P.mlp[lw].emin && E <= P.mlp[lw].emax;
        if (learned) learned_pass(P, sh, lw, use_net, sp, sel, E, g, y0, y1);
        if (valid) {
            const bool child = (ent & CHILD_BIT) != 0;
            Ev e;
            if (use_net) learned_event(process(sh, sp, sel), sp, E, y0, y1, g, e);
            else sample_event(process(sh, sp, sel), sp, p, pn, E, P.sb, P.pe, g, e);
            if (e.err) atomicAdd(&sh.bc.flags[FLAG_SAMPLER], 1ull);
            if (e.dep != 0.0) deposit(P, sh.bc, e.dep * w, x.z);
            V3 m0, m1;
            double s0, s1;
            bool drop1;
            finish_event(p, pn, e, g, m0, m1, s0, s1, sh.cut, sh.stored, -1.0, drop1);
            const uint32_t dend = g.draw;
            if (e.keep) {
                bool oob = false;
                double r = setr(L, kinenergy(sp, m0), swarm, oob);
                if (oob) atomicAdd(&sh.bc.flags[FLAG_RANGE], 1ull);
                PF(L.f[PT_PX], idx) = m0.x;
                PF(L.f[PT_PY], idx) = m0.y;
                PF(L.f[PT_PZ], idx) = m0.z;
                PF(L.f[PT_S], idx) = s0;
                PF(L.f[PT_R], idx) = r;
                L.draw[idx] = dend;
                c0 = P.q.cnt + QWK(sp, nxt);
                a0 = P.q.work[sp][nxt];
                v0 = ent;
            } else {
                L.active[idx] = 0;
                atomicAdd(&sh.bc.work[child ? W_TAIL : W_PSTEPS], 1ull);
                ull sl = append(P, sh, e.sp0, x, m0, w, t, s0, uid, step, dend, 0, swarm, false, 0);
                if (sl != NO_SLOT) {
                    sh.sp[e.sp0].trem[sl] = tfinal - t;
                    c1 = P.q.cnt + QWK(e.sp0, nxt);
                    a1 = P.q.work[e.sp0][nxt];
                    v1 = (uint32_t)sl | CHILD_BIT;
                }
            }
            if (e.ne == 2) {
                ull sl = append(P, sh, e.sp1, x, m1, w, t, s1, uid, step, dend, e.keep ? 0 : 1, swarm, false, 0);
                if (sl != NO_SLOT) {
                    sh.sp[e.sp1].trem[sl] = tfinal - t;
                    c2 = P.q.cnt + QWK(e.sp1, nxt);
                    a2 = P.q.work[e.sp1][nxt];
                    v2 = (uint32_t)sl | CHILD_BIT;
                }
            }
        }
        wave_push(c0, a0, v0, lane, ltmask);
        wave_push(c1, a1, v1, lane, ltmask);
        wave_push(c2, a2, v2, lane, ltmask);
    }
    flush_counters(P, &sh.bc);
}

// Secondaries not yet advanced after those passes: one workgroup repeats passes over the range
// the last one left and then over what it appends itself, until a pass appends nothing (the
// `while n > 0` loop of advance!, src/mixed_population.jl:43-46).
template <bool WALL, bool MLP>
__global__ void __launch_bounds__(512) k_tail(const Params* __restrict__ Pp, int maxpasses) {
    __shared__ Shared sh;
    __shared__ ull beg[PT_NSPECIES], end[PT_NSPECIES];
    __shared__ int done;
    const Params& P = *Pp;
    bool none = true;
    for (int s = 0; s < PT_NSPECIES; s++) none = none && P.range[2 * s + 1] <= P.range[2 * s];
    if (none) return;
    // the passes' claim counter: in global memory, since the loop claims its chunks with
    // global atomics (an LDS address used as a global one is an invalid access)
    ull* const cur = &P.clock->tcur;
    stage(P, sh);
    const uint32_t step = P.clock->step;
    if (threadIdx.x == 0) done = 0;
    for (int pass = 0; pass < maxpasses; pass++) {
        __threadfence();
        __syncthreads();
        if (threadIdx.x == 0) {
            done = 1;
            __hip_atomic_store(cur, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __threadfence();
            for (int s = 0; s < PT_NSPECIES; s++) {
                ull n = __hip_atomic_load(P.sp[s].n, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT);
                if (n > P.sp[s].cap) n = P.sp[s].cap;
                beg[s] = pass == 0 ? P.range[2 * s] : end[s];
                end[s] = pass == 0 ? P.range[2 * s + 1] : n;
                if (end[s] > beg[s]) done = 0;
            }
        }
        __syncthreads();
        if (done) break;
        ull rb[PT_NSPECIES], re[PT_NSPECIES];
        for (int s = 0; s < PT_NSPECIES; s++) {
            rb[s] = beg[s];
            re[s] = end[s];
        }
        select_loop<SRC_RANGE, false, WALL, MLP>(P, sh, (PT_LDS char*)pt_lds + P.lds_coop_off + (threadIdx.x >> 6) * COOP_WAVE_BYTES,
                                                 rb, re, cur, step, false, 0);
    }
    // the pass limit was reached with work left: report it
    if (threadIdx.x == 0 && !done) sh.bc.flags[FLAG_TAIL] += 1;
    flush_counters(P, &sh.bc);
}

// ------------------------------------------------------------------ learned samplers
// Training data: exact samples of the step's own samplers at rows (T_r, Z_r), transformed
// to the network's outputs (see pt_mlp.h).  Sample k of row r uses the stream
// (seed, uid = r * K + k, step = GEN_STEP).
constexpr uint32_t GEN_STEP = 0xFFFFFFF0u;

__global__ void __launch_bounds__(256) k_mlp_gen(const Params* __restrict__ Pp, int which, const double* __restrict__ T,
                                                 const int* __restrict__ slot, int nrows, int K, uint64_t seed,
                                                 double tcut, float* __restrict__ o0, float* __restrict__ o1) {
    const Params& P = *Pp;
    ull n = (ull)nrows * K;
    for (ull q = (ull)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += (ull)gridDim.x * blockDim.x) {
        const int r = (int)(q / K);
        PhiloxStream g;
        g.init(seed, q, GEN_STEP);
        const double eng = T[r];
        float y0, y1;
        if (which == LEARN_SB) {
            double kf = sb_sample(P.sb[slot[r]], eng, g);
            double cost = sample_tsai(eng, g);
            y0 = kf > 0.0 ? (float)log(kf) : -100.0f;
            double omc = 1.0 - cost;
            y1 = (float)log(omc > 1e-300 ? omc : 1e-300);
        } else {
            double e0 = tcut / eng;
            double eps = moller_sample(tcut, eng, g) / eng;
            y0 = (float)(log(eps / e0) / log(0.5 / e0));
            y1 = 0.0f;
        }
        o0[q] = y0;
        o1[q] = y1;
    }
}

// sort each row of K floats (K a power of two <= 4096) in LDS: bitonic network
__global__ void __launch_bounds__(1024) k_mlp_sort_rows(float* __restrict__ data, int K) {
    __shared__ float v[4096];
    float* row = data + (size_t)blockIdx.x * K;
    for (int q = threadIdx.x; q < K; q += blockDim.x) v[q] = row[q];
    __syncthreads();
    for (int size = 2; size <= K; size <<= 1) {
        for (int stride = size >> 1; stride > 0; stride >>= 1) {
            for (int q = threadIdx.x; q < K / 2; q += blockDim.x) {
                int lo = 2 * q - (q & (stride - 1));
                int hi = lo + stride;
                bool up = (lo & size) == 0;
                float a = v[lo], b = v[hi];
                if ((a > b) == up) {
                    v[lo] = b;
                    v[hi] = a;
                }
            }
            __syncthreads();
        }
    }
    for (int q = threadIdx.x; q < K; q += blockDim.x) row[q] = v[q];
}

// quantile table: Q[r][i] = sorted row r at level (i + 1/2) / Kq
__global__ void k_mlp_quantiles(const float* __restrict__ sorted, int nrows, int K, int Kq, float* __restrict__ Q) {
    ull n = (ull)nrows * Kq;
    for (ull q = (ull)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += (ull)gridDim.x * blockDim.x) {
        ull r = q / Kq, i = q % Kq;
        ull k = (2 * i + 1) * (ull)K / (2 * (ull)Kq);
        Q[q] = sorted[r * K + k];
    }
}

// a training batch: random rows and quantile levels (independent for the two outputs)
__global__ void k_mlp_batch(int which, const float* __restrict__ Q0, const float* __restrict__ Q1,
                            const float* __restrict__ rowx, int nrows, int Kq, int B, uint64_t seed,
                            const uint32_t* __restrict__ stepc, float* __restrict__ X, float* __restrict__ Tg) {
    int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= B) return;
    uint32_t c0 = (uint32_t)b, c1 = 0x4D4C5000u, c2 = *stepc, c3 = 0;
    philox10(c0, c1, c2, c3, (uint32_t)seed, (uint32_t)(seed >> 32));
    int r = (int)(((ull)c0 * (ull)nrows) >> 32);
    int i = (int)(((ull)c1 * (ull)Kq) >> 32);
    int j = (int)(((ull)c2 * (ull)Kq) >> 32);
    float* x = X + (size_t)b * MLP_IN;
    for (int q = 0; q < 4; q++) x[q] = rowx[r * 5 + q];
    x[4] = 2.0f * ((float)i + 0.5f) / (float)Kq - 1.0f;
    x[5] = 2.0f * ((float)j + 0.5f) / (float)Kq - 1.0f;
    x[6] = rowx[r * 5 + 4];
    for (int q = 7; q < MLP_IN; q++) x[q] = 0.0f;
    float b0, b1;
    mlp_baseline(which, x, b0, b1);
    Tg[2 * b] = Q0[(size_t)r * Kq + i] - b0;
    Tg[2 * b + 1] = Q1[(size_t)r * Kq + j] - b1;
}

// The training products on the matrix cores: C = A B in FP32 (v_mfma_f32_32x32x2f32, FP32
// products and accumulation), one wave per 32x32 tile of C.  A(m, k) = A[m sam + k sak],
// B(k, n) = B[k sbk + n sbn]; entries outside [0, M) x [0, K) and [0, K) x [0, N) read as 0,
// and column n == ones of B reads as 1 (the bias column of the weight gradients).  The K
// range is [kz klen, (kz + 1) klen) for workgroup z (slices of the batch).  Epilogues:
//   GEMM_FWD   Z = C + bias[n], H = gelu(Z) (act) or Z            (dense layer forward)
//   GEMM_DATA  D = C * gelu'(Zp) (Zp given) or C                  (gradient of the input)
//   GEMM_PART  part[z][m][n] = C                                   (weight-gradient slices)
// Every wave adds its K terms in the same order, so the results do not depend on timing.
enum { GEMM_FWD = 0, GEMM_DATA = 1, GEMM_PART = 2 };
typedef float f32x16_mfma __attribute__((ext_vector_type(16)));
struct MlpGemm {
    const float* A;
    const float* B;
    long long sam, sak, sbk, sbn;
    int M, N, K, ones, klen;
    int epi, act;
    const float* bias;
    const float* Zp;
    float* C;   // Z, D or part
    float* C2;  // H
    long long ldc;
};
__global__ void __launch_bounds__(64) k_mlp_gemm(const MlpGemm a) {
    const int lane = threadIdx.x & 63, r32 = lane & 31, h = lane >> 5;
    const int m = 32 * blockIdx.x + r32;  // this lane's row of A
    const int n = 32 * blockIdx.y + r32;  // its column of B
    const int kb = blockIdx.z * a.klen, ke = min(a.K, kb + a.klen);
    const bool mok = m < a.M, nok = n < a.N;
    f32x16_mfma acc = f32x16_mfma{};
    // eight K steps per trip: their sixteen loads are issued before the first product
    for (int k0 = kb; k0 < ke; k0 += 16) {
        float av[8], bv[8];
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const int k = k0 + 2 * j + h;
            const bool kok = k < ke;
            av[j] = (mok && kok) ? a.A[(long long)m * a.sam + (long long)k * a.sak] : 0.0f;
            bv[j] = !(nok && kok) ? 0.0f : (n == a.ones ? 1.0f : a.B[(long long)k * a.sbk + (long long)n * a.sbn]);
        }
#pragma unroll
        for (int j = 0; j < 8; j++) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(av[j], bv[j], acc, 0, 0, 0);
    }
    // element r of this lane: C[32 bx + mfma_row(r, lane)][32 by + lane % 32]
    const int cn = 32 * blockIdx.y + r32;
    if (cn >= a.N) return;
#pragma unroll
    for (int r = 0; r < 16; r++) {
        const int cm = 32 * blockIdx.x + mfma_row(r, lane);
        if (cm >= a.M) continue;
        const long long q = (long long)cm * a.ldc + cn;
        if (a.epi == GEMM_FWD) {
            const float z = acc[r] + a.bias[cn];
            a.C[q] = z;
            a.C2[q] = a.act ? gelu(z, false) : z;
        } else if (a.epi == GEMM_DATA) {
            a.C[q] = a.Zp ? acc[r] * gelu_grad(a.Zp[q]) : acc[r];
        } else {
            a.C[(long long)blockIdx.z * a.M * a.ldc + q] = acc[r];
        }
    }
}

// squared-error loss: dY = 2 w_o (Y - T) / B; per-block partial sums of the loss
__global__ void __launch_bounds__(256) k_mlp_loss(const float* __restrict__ Y, const float* __restrict__ Tg,
                                                  float w0, float w1, int B, float* __restrict__ dY,
                                                  float* __restrict__ lpart) {
    __shared__ float red[256];
    int b = blockIdx.x * blockDim.x + threadIdx.x;
    float l = 0.0f;
    if (b < B) {
        float d0 = Y[2 * b] - Tg[2 * b], d1 = Y[2 * b + 1] - Tg[2 * b + 1];
        dY[2 * b] = 2.0f * w0 * d0 / (float)B;
        dY[2 * b + 1] = 2.0f * w1 * d1 / (float)B;
        l = (w0 * d0 * d0 + w1 * d1 * d1) / (float)B;
    }
    red[threadIdx.x] = l;
    __syncthreads();
    for (int off = 128; off > 0; off >>= 1) {
        if ((int)threadIdx.x < off) red[threadIdx.x] += red[threadIdx.x + off];
        __syncthreads();
    }
    if (threadIdx.x == 0) lpart[blockIdx.x] = red[0];
}

// sum of the loss partials of a batch into out[0] (one workgroup, fixed order)
// (out[*at] when `at` is given: the training step's entry of the loss history)
__global__ void __launch_bounds__(256) k_mlp_sum(const float* __restrict__ part, int n, float* __restrict__ out,
                                                 const uint32_t* __restrict__ at) {
    __shared__ float red[256];
    float s = 0.0f;
    for (int q = threadIdx.x; q < n; q += blockDim.x) s += part[q];
    red[threadIdx.x] = s;
    __syncthreads();
    for (int off = 128; off > 0; off >>= 1) {
        if ((int)threadIdx.x < off) red[threadIdx.x] += red[threadIdx.x + off];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[at ? *at : 0u] = red[0];
}

// the batch slices whose weight-gradient partial sums are added in slice order
constexpr int MLP_SLICE = 256;

// g[dst(q)] = sum over slices of part[s][q], in slice order (deterministic)
__global__ void k_mlp_reduce(const float* __restrict__ part, int nslices, int nin, int nout, int pw, int pb,
                             float* __restrict__ g) {
    const int m = nout * (nin + 1);
    int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= m) return;
    float s = 0.0f;
#pragma unroll 8
    for (int k = 0; k < nslices; k++) s += part[(size_t)k * m + q];
    const int o = q / (nin + 1), i = q % (nin + 1);
    g[i < nin ? pw + o * nin + i : pb + o] = s;
}

// Adam step number *stepc (0-based) of `steps`: cosine-decayed learning rate from lr0 to
// lr0 / 100, bias corrections 1 - b^(step + 1)
__global__ void k_mlp_adam(float* __restrict__ p, const float* __restrict__ g, float* __restrict__ m,
                           float* __restrict__ v, int n, double lr0, int steps, const uint32_t* __restrict__ stepc,
                           float b1, float b2, float eps) {
    int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= n) return;
    const uint32_t it = *stepc;
    const float lr = (float)(lr0 * (0.01 + 0.99 * 0.5 * (1.0 + cos(M_PI * (double)it / (double)steps))));
    const float c1 = (float)(1.0 - pow((double)b1, (double)it + 1.0));
    const float c2 = (float)(1.0 - pow((double)b2, (double)it + 1.0));
    float gq = g[q];
    float mq = b1 * m[q] + (1.0f - b1) * gq;
    float vq = b2 * v[q] + (1.0f - b2) * gq * gq;
    m[q] = mq;
    v[q] = vq;
    p[q] -= lr * (mq / c1) / (sqrtf(vq / c2) + eps);
}

// the training loop's step counter, advanced after each Adam step (the batch, the loss
// history and the learning-rate schedule read it on the device)
__global__ void k_mlp_tick(uint32_t* __restrict__ stepc) {
    if (threadIdx.x == 0 && blockIdx.x == 0) stepc[0] += 1u;
}

// FP32 parameters -> BF16 inference image
__global__ void k_mlp_image(const float* __restrict__ p, uint16_t* __restrict__ w, float* __restrict__ b) {
    int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q < MLP_H * MLP_IN) w[I_W1 + q] = f2bf(p[P_W1 + q]);
    // hidden and output layers: column 16 c + vk of row o holds input feature mlp_kperm(c, vk)
    const int o = q / MLP_H, col = q % MLP_H, src = o * MLP_H + mlp_kperm(col >> 4, col & 15);
    if (q < MLP_H * MLP_H) {
        w[I_W2 + q] = f2bf(p[P_W2 + src]);
        w[I_W3 + q] = f2bf(p[P_W3 + src]);
    }
    if (q < MLP_OUTP * MLP_H) w[I_W4 + q] = q < MLP_OUT * MLP_H ? f2bf(p[P_W4 + src]) : (uint16_t)0;
    if (q < MLP_H) {
        b[q] = p[P_B1 + q];
        b[MLP_H + q] = p[P_B2 + q];
        b[2 * MLP_H + q] = p[P_B3 + q];
    }
    if (q < MLP_OUTP) b[3 * MLP_H + q] = q < MLP_OUT ? p[P_B4 + q] : 0.0f;
}

// matrix-core inference: Y[s] for the n input rows X[s] (64 rows per wave)
__global__ void __launch_bounds__(256) k_mlp_infer(int which, const uint16_t* __restrict__ wimg,
                                                   const float* __restrict__ bimg, const float* __restrict__ X, int n,
                                                   float* __restrict__ Y) {
    const int lane = threadIdx.x & 63;
    const int waves = (gridDim.x * blockDim.x) >> 6;
    for (int base = ((blockIdx.x * blockDim.x + threadIdx.x) >> 6) * 64; base < n; base += waves * 64) {
        int s = base + lane;
        float x[MLP_IN];
        for (int q = 0; q < MLP_IN; q++) x[q] = s < n ? X[(size_t)s * MLP_IN + q] : 0.0f;
        float y0, y1;
        mlp_wave(wimg, bimg, x, s < n, y0, y1);
        if (s < n) {
            float b0 = 0.0f, b1 = 0.0f;
            if (which >= 0) mlp_baseline(which, x, b0, b1);
            Y[2 * (size_t)s] = y0 + b0;
            Y[2 * (size_t)s + 1] = y1 + b1;
        }
    }
}

// network inputs for `reps` samples at each of n (T, Z) rows: uniforms from the stream
// (seed, uid = sample index, GEN_STEP + 1)
__global__ void k_mlp_features(const Params* __restrict__ Pp, int which, const double* __restrict__ T,
                               const int32_t* __restrict__ Z, const int32_t* __restrict__ slot, ull n, int reps,
                               uint64_t seed, float* __restrict__ X) {
    const Params& P = *Pp;
    for (ull q = (ull)blockIdx.x * blockDim.x + threadIdx.x; q < n * reps; q += (ull)gridDim.x * blockDim.x) {
        ull r = q / reps;
        PhiloxStream g;
        g.init(seed, q, GEN_STEP + 1);
        double u1 = g.next(), u2 = g.next();
        double ph = which == LEARN_SB ? sb_phase(P.sb[slot[r]].log_energy, P.sb[slot[r]].thr, P.sb[slot[r]].ne, T[r]) : 0.0;
        mlp_features(T[r] / EV, Z[r], u1, u2, ph, X + q * MLP_IN);
    }
}

// init! / advance_init!: r of every active particle (src/mixed_population.jl:20-35)
__global__ void __launch_bounds__(256) k_setr(const Params* __restrict__ Pp, int sp) {
    __shared__ Shared sh;
    const Params& P = *Pp;
    stage(P, sh);
    const SpLite& L = sh.sp[sp];
    ull n = *L.n;
    if (n > L.cap) n = L.cap;
    for (ull i = (ull)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (ull)gridDim.x * blockDim.x) {
        if (!L.active[i]) continue;
        V3 p{PF(L.f[PT_PX], i), PF(L.f[PT_PY], i), PF(L.f[PT_PZ], i)};
        int sw = L.swarm[i];
        if (sw < 0 || sw >= P.nswarm) sw = 0;
        bool oob = false;
        PF(L.f[PT_R], i) = setr(L, kinenergy(sp, p), sw, oob);
        if (oob) atomicAdd(&P.flags[FLAG_RANGE], 1ull);
    }
}

// initial particles generated on the device (same draws as the CPU restatement's
// initialisation): energy, randsphere (src/util.jl:4-12), s = nextcoll()
__global__ void __launch_bounds__(256) k_init_particles(const Params* __restrict__ Pp, int sp,
                                                        ull base, ull n, double e1, double e2,
                                                        int loguniform, int swarm, uint64_t uid0,
                                                        double t0) {
    const Params& P = *Pp;
    const SpeciesDev& S = P.sp[sp];
    for (ull i = (ull)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (ull)gridDim.x * blockDim.x) {
        ull slot = base + i;
        uint64_t uid = uid0 + i;
        PhiloxStream g;
        g.init(P.seed, uid, 0xFFFFFFFFu);
        double E = e1;
        if (loguniform) {
            double la = log(e1), lb = log(e2);
            E = exp(la + g.next() * (lb - la));
        }
        V3 d = randsphere(g);
        double pn = mom_from_kin(sp, E);
        PF(S.f[PT_X], slot) = 0.0;
        PF(S.f[PT_Y], slot) = 0.0;
        PF(S.f[PT_Z], slot) = 0.0;
        PF(S.f[PT_PX], slot) = pn * d.x;
        PF(S.f[PT_PY], slot) = pn * d.y;
        PF(S.f[PT_PZ], slot) = pn * d.z;
        PF(S.f[PT_W], slot) = 1.0;
        PF(S.f[PT_T], slot) = t0;
        PF(S.f[PT_S], slot) = nextcoll(g);
        PF(S.f[PT_R], slot) = 0.0;
        S.uid[slot] = uid;
        S.swarm[slot] = swarm;
        S.active[slot] = 1;
    }
}

// a pencil beam: n particles of kinetic energy e at the origin along the unit vector d
__global__ void __launch_bounds__(256) k_init_beam(const Params* __restrict__ Pp, int sp, ull base, ull n, double e,
                                                   double dx, double dy, double dz, int swarm, uint64_t uid0,
                                                   double t0) {
    const Params& P = *Pp;
    const SpeciesDev& S = P.sp[sp];
    const double pn = mom_from_kin(sp, e);
    for (ull i = (ull)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (ull)gridDim.x * blockDim.x) {
        ull slot = base + i;
        uint64_t uid = uid0 + i;
        PhiloxStream g;
        g.init(P.seed, uid, 0xFFFFFFFFu);
        PF(S.f[PT_X], slot) = 0.0;
        PF(S.f[PT_Y], slot) = 0.0;
        PF(S.f[PT_Z], slot) = 0.0;
        PF(S.f[PT_PX], slot) = pn * dx;
        PF(S.f[PT_PY], slot) = pn * dy;
        PF(S.f[PT_PZ], slot) = pn * dz;
        PF(S.f[PT_W], slot) = 1.0;
        PF(S.f[PT_T], slot) = t0;
        PF(S.f[PT_S], slot) = nextcoll(g);
        PF(S.f[PT_R], slot) = 0.0;
        S.uid[slot] = uid;
        S.swarm[slot] = swarm;
        S.active[slot] = 1;
    }
}

// roulette! (src/population.jl:291-309): a particle survives with probability q (the
// constant q, or qv[i] of slot i when the caller evaluated an energy-dependent f(E)) and
// its weight is divided by q.  Stream: key seed ^ ROUL_KEY, counter (uid, step).
constexpr uint64_t ROUL_KEY = 0x524F554C45545445ull, SPLIT_KEY = 0x53504C4954535054ull;
__global__ void __launch_bounds__(256) k_roulette(const Params* __restrict__ Pp, int sp, double q0,
                                                  const double* __restrict__ qv, uint32_t step, ull n0) {
    const Params& P = *Pp;
    const SpeciesDev& S = P.sp[sp];
    for (ull i = (ull)blockIdx.x * blockDim.x + threadIdx.x; i < n0; i += (ull)gridDim.x * blockDim.x) {
        if (!S.active[i]) continue;
        const double q = qv ? qv[i] : q0;
        PhiloxStream g;
        g.init(P.seed ^ ROUL_KEY, S.uid[i], step);
        if (g.next() < q) PF(S.f[PT_W], i) /= q;
        else S.active[i] = 0;
    }
}

// split! (src/population.jl:316-330): every particle's weight is divided by 1 + f and
// Poisson(f) copies of it are appended (same state, new uids derived from the parent's);
// f is the constant f0 or fv[i] of slot i (a state-dependent f evaluated by the caller).
// Stream: key seed ^ SPLIT_KEY, counter (uid, step).
__global__ void __launch_bounds__(256) k_split(const Params* __restrict__ Pp, int sp, double f0,
                                               const double* __restrict__ fv, uint32_t step, ull n0) {
    const Params& P = *Pp;
    const SpeciesDev& S = P.sp[sp];
    for (ull i = (ull)blockIdx.x * blockDim.x + threadIdx.x; i < n0; i += (ull)gridDim.x * blockDim.x) {
        if (!S.active[i]) continue;
        const double f = fv ? fv[i] : f0;
        const double e0 = exp(-f);
        const double w = PF(S.f[PT_W], i) / (1.0 + f);
        PF(S.f[PT_W], i) = w;
        PhiloxStream g;
        g.init(P.seed ^ SPLIT_KEY, S.uid[i], step);
        // Poisson(f) by sequential inversion (Knuth's product of uniforms for small f)
        int k = 0;
        double prod = g.next();
        while (prod > e0 && k < 1000) {
            k++;
            prod *= g.next();
        }
        for (int c = 0; c < k; c++) {
            ull slot = atomicAdd(S.n, 1ull);
            if (slot >= S.cap) {
                atomicAdd(&P.flags[FLAG_CAPACITY], 1ull);
                break;
            }
            for (int fi = 0; fi < PT_NFIELDS; fi++) PF(S.f[fi], slot) = PF(S.f[fi], i);
            PF(S.f[PT_W], slot) = w;
            S.uid[slot] = child_uid(P.seed ^ SPLIT_KEY, S.uid[i], step, (uint32_t)(c >> 1), c & 1);
            S.swarm[slot] = S.swarm[i];
            S.active[slot] = 1;
        }
    }
}

// ------------------------------------------------------------------ compaction
// repack! of the species in `mask` (bit s), three launches for all of them: count the actives
// of each chunk and, in the last workgroup of a species, the prefix sums; list the k-th hole
// below the active count and the k-th active above it; move.  Counts are read on the device,
// so that the launches can be captured; a workgroup without a chunk in use ends at once.
// (One launch per kernel and species, with a grid over the whole capacity, and a copy of the
// counts: a call took 118 us for three species of 2^27 slots, whatever they held; now 17 us up
// to 16384 slots, 22 for 10^6.)
constexpr int CH = 4096;  // slots per chunk: one 16-byte read of flags per thread of a workgroup
// chunks that one workgroup compacts alone, in one launch (16384 slots: a call 17 us, with
// three launches 20; one launch of 10^3 slots 6.4 us of GPU time, three 13)
constexpr int CMP_SMALL = 4;
struct Compaction {
    SpeciesDev sp[PT_NSPECIES];
    unsigned* cnt[PT_NSPECIES];   // actives of each chunk
    unsigned* hole[PT_NSPECIES];  // holes below the active count before each chunk
    unsigned* tail[PT_NSPECIES];  // actives at or above it before each chunk
    unsigned* hpos[PT_NSPECIES];
    unsigned* tpos[PT_NSPECIES];
    ull* info;  // per species: active count, moves, slots in use before, workgroups done
    ull* work;
    Report* report;
};

// bit i: flag i of the 16 from slot i0 is set (slots from n on: not)
__device__ __forceinline__ unsigned flags16(const uint8_t* __restrict__ active, ull i0, ull n) {
    if (i0 >= n) return 0;
    unsigned m = 0;
    if (i0 + 16 <= n) {
        const uint4 v = *(const uint4*)(active + i0);
        const unsigned w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int q = 0; q < 4; q++) {
            // the top bit of each nonzero byte, gathered into four bits
            const unsigned t = (((w[q] & 0x7F7F7F7Fu) + 0x7F7F7F7Fu) | w[q]) & 0x80808080u;
            m |= (((t >> 7) * 0x10204080u) >> 28) << (4 * q);
        }
    } else {
        for (int q = 0; q < 16 && i0 + q < n; q++) m |= active[i0 + q] ? 1u << q : 0u;
    }
    return m;
}

// exclusive prefix sum over the 256 threads of a workgroup, and the total
__device__ __forceinline__ unsigned block_prefix(unsigned v, unsigned* wsum, unsigned& total) {
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    unsigned inc = v;
    for (int off = 1; off < 64; off <<= 1) {
        const unsigned o = __shfl_up(inc, off, 64);
        if (lane >= off) inc += o;
    }
    if (lane == 63) wsum[wv] = inc;
    __syncthreads();
    unsigned base = 0, all = 0;
    for (int q = 0; q < 4; q++) {
        if (q < wv) base += wsum[q];
        all += wsum[q];
    }
    __syncthreads();
    total = all;
    return base + inc - v;
}

// positions of the k-th hole and the k-th active above, in chunk order
__device__ __forceinline__ void fill_chunk(const Compaction& cp, int s, int c, int nchunks, ull A, ull n, ull moves,
                                           unsigned* wsum) {
    const unsigned h0 = cp.hole[s][c], t0 = cp.tail[s][c];
    const unsigned h1 = c + 1 < nchunks ? cp.hole[s][c + 1] : (unsigned)moves;
    const unsigned t1 = c + 1 < nchunks ? cp.tail[s][c + 1] : (unsigned)moves;
    if (h1 == h0 && t1 == t0) return;
    const ull i0 = (ull)c * CH + 16 * threadIdx.x;
    const unsigned act = flags16(cp.sp[s].active, i0, n);
    const unsigned below = i0 >= A ? 0u : i0 + 16 <= A ? 0xFFFFu : (1u << (A - i0)) - 1u;
    unsigned holes = below & ~act, tails = act & ~below, tot;
    unsigned hk = h0 + block_prefix(__popc(holes), wsum, tot), tk = t0 + block_prefix(__popc(tails), wsum, tot);
    for (; holes; holes &= holes - 1) cp.hpos[s][hk++] = (unsigned)(i0 + __ffs(holes) - 1);
    for (; tails; tails &= tails - 1) cp.tpos[s][tk++] = (unsigned)(i0 + __ffs(tails) - 1);
}

// the k-th active above the active count into the k-th hole below it, k = k0, k0 + step, ...
__device__ __forceinline__ void move_slots(const Compaction& cp, int s, ull m, ull k0, ull step) {
    const SpeciesDev& S = cp.sp[s];
    for (ull k = k0; k < m; k += step) {
        const unsigned d = cp.hpos[s][k], q = cp.tpos[s][k];
        const PT_GLOBAL pair2* from = (const PT_GLOBAL pair2*)&PF(S.f[0], q);
        PT_GLOBAL pair2* to = (PT_GLOBAL pair2*)&PF(S.f[0], d);
        pair2 v[PT_NFIELDS / 2];
#pragma unroll
        for (int f = 0; f < PT_NFIELDS / 2; f++) v[f] = from[f];
        const uint64_t u = S.uid[q];
        const int32_t w = S.swarm[q];
#pragma unroll
        for (int f = 0; f < PT_NFIELDS / 2; f++) to[f] = v[f];
        S.uid[d] = u;
        S.swarm[d] = w;
        S.active[d] = 1;
    }
    if (m && k0 == 0) atomicAdd(&cp.work[W_MOVED], m);
}

__global__ void __launch_bounds__(256) k_cmp_count(const Compaction cp, unsigned mask) {
    const int s = blockIdx.y;
    if (!((mask >> s) & 1)) return;
    const SpeciesDev& S = cp.sp[s];
    ull* const info = cp.info + 4 * s;
    unsigned* const cnt = cp.cnt[s];
    ull n = *S.n;
    if (n > S.cap) n = S.cap;
    const int nchunks = (int)((n + CH - 1) / CH);
    // the workgroups that have a chunk (the first one always takes part); a few chunks are left
    // to one workgroup, which then does the moves as well
    const int parts = nchunks <= CMP_SMALL ? 1 : nchunks < (int)gridDim.x ? nchunks : (int)gridDim.x;
    if ((int)blockIdx.x >= parts) return;
    __shared__ unsigned wsum[4];
    __shared__ bool last;
    for (int c = blockIdx.x; c < nchunks; c += parts) {
        unsigned tot;
        (void)block_prefix(__popc(flags16(S.active, (ull)c * CH + 16 * threadIdx.x, n)), wsum, tot);
        // (read by the last workgroup, which may be on another die)
        if (threadIdx.x == 0) __hip_atomic_store(&cnt[c], tot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if (threadIdx.x == 0) {
        wait_vmem();
        last = __hip_atomic_fetch_add(&info[3], 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (ull)(parts - 1);
    }
    __syncthreads();
    if (!last) return;
    // prefix sums over the chunks, a run of them per thread
    unsigned* const hole = cp.hole[s];
    unsigned* const tail = cp.tail[s];
    const int per = (nchunks + 255) / 256;
    const int c0 = min(nchunks, (int)threadIdx.x * per), c1 = min(nchunks, c0 + per);
    unsigned mine = 0, total = 0;
    for (int c = c0; c < c1; c++) {
        const unsigned v = __hip_atomic_load(&cnt[c], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        hole[c] = v;  // kept for the next loop (the same thread reads it)
        mine += v;
    }
    (void)block_prefix(mine, wsum, total);
    const ull A = total;
    const int sc = (int)(A / CH);  // the chunk that holds slot A
    unsigned low = 0;              // actives of that chunk below A
    if (sc < nchunks) (void)block_prefix(__popc(flags16(S.active, (ull)sc * CH + 16 * threadIdx.x, A)), wsum, low);
    auto split = [&](int c, unsigned v, unsigned& h, unsigned& t) {
        h = c < sc ? CH - v : c == sc ? (unsigned)(A - (ull)sc * CH) - low : 0u;
        t = c < sc ? 0u : c == sc ? v - low : v;
    };
    unsigned hs = 0, ts = 0, h, t, htot, ttot;
    for (int c = c0; c < c1; c++) {
        split(c, hole[c], h, t);
        hs += h;
        ts += t;
    }
    unsigned hrun = block_prefix(hs, wsum, htot), trun = block_prefix(ts, wsum, ttot);
    for (int c = c0; c < c1; c++) {
        split(c, hole[c], h, t);
        hole[c] = hrun;
        tail[c] = trun;
        hrun += h;
        trun += t;
    }
    if (threadIdx.x == 0) {
        info[0] = A;
        info[1] = parts == 1 ? 0 : htot;  // holes below A == actives from A on, still to be moved
        info[2] = n;
        info[3] = 0;
        *S.n = A;
        __hip_atomic_store(&cp.report->n[s], A, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
    if (parts == 1 && htot) {
        __syncthreads();
        for (int c = 0; c < nchunks; c++) fill_chunk(cp, s, c, nchunks, A, n, htot, wsum);
        __syncthreads();
        move_slots(cp, s, htot, threadIdx.x, blockDim.x);
    }
}

__global__ void __launch_bounds__(256) k_cmp_fill(const Compaction cp, unsigned mask) {
    const int s = blockIdx.y;
    const ull* const info = cp.info + 4 * s;
    const ull moves = info[1], n = info[2], A = info[0];
    if (!((mask >> s) & 1) || moves == 0) return;
    __shared__ unsigned wsum[4];
    const int nchunks = (int)((n + CH - 1) / CH);
    for (int c = blockIdx.x; c < nchunks; c += gridDim.x) fill_chunk(cp, s, c, nchunks, A, n, moves, wsum);
}

__global__ void __launch_bounds__(256) k_cmp_move(const Compaction cp, unsigned mask) {
    const int s = blockIdx.y;
    if (!((mask >> s) & 1)) return;
    move_slots(cp, s, cp.info[4 * s + 1], (ull)blockIdx.x * blockDim.x + threadIdx.x, (ull)gridDim.x * blockDim.x);
}

// ------------------------------------------------------------------ copies of the state
// byte ranges copied together (16-byte aligned; dst <- src)
constexpr int MAX_COPIES = 4 * PT_NSPECIES + 6;
struct Copies {
    void* dst[MAX_COPIES];
    const void* src[MAX_COPIES];
    ull bytes[MAX_COPIES];
    int n;
};
__global__ void __launch_bounds__(256) k_copy_ranges(const Copies c) {
    for (int q = 0; q < c.n; q++) {
        const ull words = c.bytes[q] / 16, tid = (ull)blockIdx.x * blockDim.x + threadIdx.x;
        const uint4* from = (const uint4*)c.src[q];
        uint4* to = (uint4*)c.dst[q];
        for (ull i = tid; i < words; i += (ull)gridDim.x * blockDim.x) to[i] = from[i];
        if (tid < (c.bytes[q] & 15)) ((uint8_t*)to)[16 * words + tid] = ((const uint8_t*)from)[16 * words + tid];
    }
}

// ------------------------------------------------------------------ statistics
// sums over active particles: count, w, w*E, w*x, w*y, w*z, w*|x|^2, and max E; each workgroup
// leaves its part and the last one adds them up and reports them.  Bound by memory (a record's
// first 64 bytes: the whole line): every lane reads its particle with 16-byte loads, two
// particles at a time.  2 x 10^6 particles: 38 us (160 MB in whole lines take 33 at the rate of a
// copy); a call 79 -> 48 us without the host's sum of the parts, of 10^4 particles 44 -> 17.
__device__ __forceinline__ double agent_load(const double* p) {
    return __longlong_as_double(
        (long long)__hip_atomic_load((const ull*)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}
__device__ __forceinline__ void agent_store(double* p, double v) {
    __hip_atomic_store((ull*)p, (ull)__double_as_longlong(v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// sums of a[] over the workgroup (the last one: maximum), in threads 0..NSTAT-1
__device__ __forceinline__ double stat_reduce(double a[NSTAT]) {
    __shared__ double red[4][NSTAT];
#pragma unroll
    for (int q = 0; q < NSTAT; q++)
        for (int off = 32; off > 0; off >>= 1) {
            const double o = __shfl_down(a[q], off, 64);
            a[q] = q == NSTAT - 1 ? fmax(a[q], o) : a[q] + o;
        }
    if ((threadIdx.x & 63) == 0)
        for (int q = 0; q < NSTAT; q++) red[threadIdx.x >> 6][q] = a[q];
    __syncthreads();
    double v = 0.0;
    if (threadIdx.x < NSTAT)
        for (int k = 0; k < 4; k++)
            v = threadIdx.x == NSTAT - 1 ? fmax(v, red[k][threadIdx.x]) : v + red[k][threadIdx.x];
    __syncthreads();
    return v;
}
constexpr int STAT_BLOCKS = 1024;
__global__ void __launch_bounds__(256) k_stats(const Params* __restrict__ Pp, int sp, double* __restrict__ part,
                                               ull* __restrict__ ticket) {
    const Params& P = *Pp;
    const SpeciesDev& S = P.sp[sp];
    __shared__ bool last;
    ull n = *S.n;
    if (n > S.cap) n = S.cap;
    double a[NSTAT] = {0, 0, 0, 0, 0, 0, 0, 0};
    const ull stride = (ull)gridDim.x * blockDim.x;
    for (ull i0 = (ull)blockIdx.x * blockDim.x + threadIdx.x; i0 < n; i0 += 2 * stride) {
        pair2 v[2][4];
        bool act[2];
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const ull i = i0 + u * stride < n ? i0 + u * stride : i0;
            const PT_GLOBAL pair2* r = (const PT_GLOBAL pair2*)&PF(S.f[0], i);
#pragma unroll
            for (int q = 0; q < 4; q++) v[u][q] = r[q];
            act[u] = S.active[i] && (u == 0 || i != i0);
        }
#pragma unroll
        for (int u = 0; u < 2; u++) {
            if (!act[u]) continue;
            const V3 x{v[u][0].x, v[u][0].y, v[u][1].x}, p{v[u][1].y, v[u][2].x, v[u][2].y};
            const double w = v[u][3].x, E = kinenergy(sp, p);
            a[0] += 1.0;
            a[1] += w;
            a[2] += w * E;
            a[3] += w * x.x;
            a[4] += w * x.y;
            a[5] += w * x.z;
            a[6] += w * dot3(x, x);
            a[7] = fmax(a[7], E);
        }
    }
    const double mine = stat_reduce(a);
    if (threadIdx.x < NSTAT) agent_store(&part[blockIdx.x * NSTAT + threadIdx.x], mine);
    wait_vmem();
    __syncthreads();
    if (threadIdx.x == 0)
        last = __hip_atomic_fetch_add(ticket, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x - 1;
    __syncthreads();
    if (!last) return;
    double t[NSTAT] = {0, 0, 0, 0, 0, 0, 0, 0};
    for (int b = threadIdx.x; b < (int)gridDim.x; b += blockDim.x)
        for (int q = 0; q < NSTAT; q++) {
            const double v = agent_load(&part[b * NSTAT + q]);
            t[q] = q == NSTAT - 1 ? fmax(t[q], v) : t[q] + v;
        }
    const double sum = stat_reduce(t);
    if (threadIdx.x < NSTAT) to_host(&P.report->stat[threadIdx.x], sum);
    if (threadIdx.x == 0) *ticket = 0;
}

// per-swarm sums over active particles: count, w, w*E and max E of each swarm.  Each workgroup
// has a run of consecutive slots, and each lane adds up its particles in registers as long as
// they belong to one swarm (they mostly do: swarms are laid out one after the other), then
// once into LDS (up to SWARM_LDS swarms; beyond that into global memory directly), and the
// workgroup adds what it found to the output.  (With an LDS atomic per particle the 64 lanes of
// a wave met on one address four times over.)
// out[4*i + 3] holds max E as the bit pattern of a non-negative double (ordered like the value).
constexpr int SWARM_LDS = 1024;
// With `host` (pinned memory) the last workgroup copies the sums there and clears `out` for the
// next call; the workgroups then add into `copies` arrays by turns, since atomics on one
// address, from eight XCDs, are done one after the other.  A call for 2 x 10^6 particles in 64
// swarms took 109 us with 2048 workgroups on one array, 77 with 512, 48 with 512 on 8 arrays
// (reading the records once takes 33 us); fewer than 128 workgroups use one array.
constexpr int SWARM_COPIES = 8;
__global__ void __launch_bounds__(256) k_swarm_stats(const Params* __restrict__ Pp, int sp, int nswarm,
                                                     double* __restrict__ sums, int copies,
                                                     double* __restrict__ host, ull* __restrict__ ticket) {
    double* const out = sums + (size_t)(blockIdx.x % copies) * 4 * nswarm;
    __shared__ bool last;
    __shared__ double acc[3 * SWARM_LDS];
    __shared__ ull emax[SWARM_LDS];
    const Params& P = *Pp;
    const SpeciesDev& S = P.sp[sp];
    const bool local = nswarm <= SWARM_LDS;
    if (local) {
        for (int q = threadIdx.x; q < 3 * nswarm; q += blockDim.x) acc[q] = 0.0;
        for (int q = threadIdx.x; q < nswarm; q += blockDim.x) emax[q] = 0ull;
        __syncthreads();
    }
    ull n = *S.n;
    if (n > S.cap) n = S.cap;
    const ull per = (n + gridDim.x - 1) / gridDim.x;
    const ull beg = (ull)blockIdx.x * per, end = beg + per < n ? beg + per : n;
    int cur = -1;
    double c0 = 0.0, c1 = 0.0, c2 = 0.0, c3 = 0.0;
    auto leave = [&]() {
        if (cur < 0) return;
        const ull eb = (ull)__double_as_longlong(c3);
        if (local) {
            atomicAdd(&acc[3 * cur], c0);
            atomicAdd(&acc[3 * cur + 1], c1);
            atomicAdd(&acc[3 * cur + 2], c2);
            atomicMax(&emax[cur], eb);
        } else {
            atomicAdd(&out[4 * cur], c0);
            atomicAdd(&out[4 * cur + 1], c1);
            atomicAdd(&out[4 * cur + 2], c2);
            atomicMax((ull*)&out[4 * cur + 3], eb);
        }
        c0 = c1 = c2 = c3 = 0.0;
    };
    for (ull i = beg + threadIdx.x; i < end; i += blockDim.x) {
        const PT_GLOBAL pair2* r = (const PT_GLOBAL pair2*)&PF(S.f[0], i);
        const pair2 v1 = r[1], v2 = r[2], v3 = r[3];
        const int sw = S.swarm[i];
        if (!S.active[i] || sw < 0 || sw >= nswarm) continue;
        if (sw != cur) {
            leave();
            cur = sw;
        }
        const double E = kinenergy(sp, V3{v1.y, v2.x, v2.y});
        c0 += 1.0;
        c1 += v3.x;
        c2 += v3.x * E;
        c3 = fmax(c3, E > 0.0 ? E : 0.0);
    }
    // the lanes of a wave that ends in one swarm are added up first
    const int lead = __builtin_amdgcn_readfirstlane(cur);
    if (__ballot(cur != lead) == 0) {
        for (int off = 32; off > 0; off >>= 1) {
            c0 += __shfl_down(c0, off, 64);
            c1 += __shfl_down(c1, off, 64);
            c2 += __shfl_down(c2, off, 64);
            c3 = fmax(c3, __shfl_down(c3, off, 64));
        }
        if ((threadIdx.x & 63) != 0) cur = -1;
    }
    leave();
    if (local) {
        __syncthreads();
        for (int q = threadIdx.x; q < nswarm; q += blockDim.x) {
            if (acc[3 * q] == 0.0) continue;
            atomicAdd(&out[4 * q], acc[3 * q]);
            atomicAdd(&out[4 * q + 1], acc[3 * q + 1]);
            atomicAdd(&out[4 * q + 2], acc[3 * q + 2]);
            atomicMax((ull*)&out[4 * q + 3], emax[q]);
        }
    }
    if (!host) return;
    wait_vmem();
    __syncthreads();
    if (threadIdx.x == 0)
        last = __hip_atomic_fetch_add(ticket, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x - 1;
    __syncthreads();
    if (!last) return;
    for (int q = threadIdx.x; q < 4 * nswarm; q += blockDim.x) {
        double u[SWARM_COPIES];
#pragma unroll
        for (int k = 0; k < SWARM_COPIES; k++) u[k] = k < copies ? agent_load(&sums[(size_t)k * 4 * nswarm + q]) : 0.0;
        double v = 0.0;
#pragma unroll
        for (int k = 0; k < SWARM_COPIES; k++) {
            v = (q & 3) == 3 ? fmax(v, u[k]) : v + u[k];
            if (k < copies) agent_store(&sums[(size_t)k * 4 * nswarm + q], 0.0);
        }
        to_host(&host[q], v);
    }
    if (threadIdx.x == 0) *ticket = 0;
}

// p[0..n) = 0 (a kernel, not a memset, so that it can also be captured in a graph)
__global__ void __launch_bounds__(256) k_zero_doubles(double* __restrict__ p, int n) {
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q < n) p[q] = 0.0;
}

// ------------------------------------------------------------------ debug kernels
__global__ void k_dbg_philox(const uint32_t* ctr, uint32_t k0, uint32_t k1, uint32_t* out, ull n) {
    ull i = (ull)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    uint32_t a = ctr[4 * i], b = ctr[4 * i + 1], c = ctr[4 * i + 2], d = ctr[4 * i + 3];
    philox10(a, b, c, d, k0, k1);
    out[4 * i] = a;
    out[4 * i + 1] = b;
    out[4 * i + 2] = c;
    out[4 * i + 3] = d;
}

__global__ void k_dbg_uniforms(uint64_t seed, uint64_t uid, uint32_t step, double* out, ull n) {
    if (blockIdx.x != 0 || threadIdx.x != 0) return;
    PhiloxStream g;
    g.init(seed, uid, step);
    for (ull i = 0; i < n; i++) out[i] = g.next();
}

__global__ void __launch_bounds__(256) k_dbg_select(const Params* __restrict__ Pp, int sp, ull n,
                                                    const double* E, const double* u,
                                                    const int32_t* swarm, int32_t* interval,
                                                    int32_t* proc, double* rbound) {
    __shared__ Shared sh;
    const Params& P = *Pp;
    stage(P, sh);
    ull i = (ull)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const SpLite& L = sh.sp[sp];
    int sw = swarm ? swarm[i] : 0;
    if (sw < 0 || sw >= P.nswarm) sw = 0;
    bool oob = false;
    double r = setr(L, E[i], sw, oob);
    double t1, t2;
    bool o;
    int iv = precheb(E[i], L.k, L.xmax, L.ixmax, L.two_k1, t1, t2, o);
    double xi = u[i] * r;
    int sel = select_process(as_lds(pt_lds) + L.rate_off + iv * L.nprocs * 3, L.nprocs, t1, t2, xi);
    if (sel >= L.nprocs) sel = -1;
    interval[i] = o ? -1 : iv;
    proc[i] = sel;
    rbound[i] = r;
}

__global__ void __launch_bounds__(256) k_dbg_push(const Params* __restrict__ Pp, int sp, ull n,
                                                  double* f0, double* f1, double* f2, double* f3,
                                                  double* f4, double* f5, double* f7,
                                                  const double* dt) {
    const Params& P = *Pp;
    ull i = (ull)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    V3 x{f0[i], f1[i], f2[i]}, p{f3[i], f4[i], f5[i]};
    double t = f7[i];
    push(sp, P.fields[0], x, p, t, dt[i], P.forcing_off);
    f0[i] = x.x;
    f1[i] = x.y;
    f2[i] = x.z;
    f3[i] = p.x;
    f4[i] = p.y;
    f5[i] = p.z;
    f7[i] = t;
}

// collide() with injected uniforms through the same sample_event / finish_event as the step
__global__ void __launch_bounds__(256) k_dbg_collide(const Params* __restrict__ Pp, int sp, int proc,
                                                     ull n, const double* in, const uint64_t* uid,
                                                     const double* u, int stride, uint32_t step,
                                                     int32_t* okind, int32_t* odraws, double* ost,
                                                     int32_t* osp, uint64_t* ouid) {
    const Params& P = *Pp;
    ull i = (ull)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double* st = in + i * PT_NFIELDS;
    V3 x{st[0], st[1], st[2]}, p{st[3], st[4], st[5]};
    double w = st[6], t = st[7];
    InjectedStream g;
    g.u = u + i * (ull)stride;
    g.n = stride;
    g.pos = 0;
    g.draw = 0;
    g.ran_out = false;
    double E = kinenergy(sp, p);
    double pn = norm3(p);
    Ev e;
    sample_event(P.tab[sp].procs[proc], sp, p, pn, E, P.sb, P.pe, g, e);
    V3 m0, m1;
    double s0, s1;
    bool drop1;
    finish_event(p, pn, e, g, m0, m1, s0, s1, nullptr, nullptr, -1.0, drop1);
    int kind = e.keep ? (e.ne == 1 ? 1 : 2) : (e.ne == 1 ? 3 : 4);
    okind[i] = g.ran_out ? -2 : (e.err ? -1 - 16 * e.err : kind);
    odraws[i] = (int32_t)g.draw;
    double* o = ost + i * 3 * PT_NFIELDS;
    for (int q = 0; q < 3 * PT_NFIELDS; q++) o[q] = 0.0;
    for (int q = 0; q < 3; q++) {
        osp[i * 3 + q] = -1;
        ouid[i * 3 + q] = 0;
    }
    // slot 0: the surviving primary; slots 1, 2: new particles in creation order
    V3 mom[2] = {m0, m1};
    double ss[2] = {s0, s1};
    int sps[2] = {e.sp0, e.sp1};
    int slot = 1;
    for (int q = 0; q < e.ne; q++) {
        int d = (q == 0 && e.keep) ? 0 : slot++;
        double v[PT_NFIELDS] = {x.x, x.y, x.z, mom[q].x, mom[q].y, mom[q].z, w, t, ss[q], 0.0};
        for (int f = 0; f < PT_NFIELDS; f++) o[d * PT_NFIELDS + f] = v[f];
        osp[i * 3 + d] = sps[q];
        ouid[i * 3 + d] = d == 0 ? uid[i] : child_uid(P.seed, uid[i], step, g.draw, d - 1);
    }
}

// ================================================================== host side
struct DevBuf {
    void* p = nullptr;
    size_t bytes = 0;
};

struct Span {
    hipEvent_t a, b;
    int kind;
};

constexpr int MAX_KV = 12;  // kernel variants with a residency entry

struct pt_ctx {
    pt_config cfg{};
    int device = 0;
    hipStream_t stream = nullptr;
    Params hp{};          // host copy of the parameters
    Params* dp = nullptr;  // device copy
    Report* report = nullptr;  // pinned: what kernels report
    bool dirty = true;
    std::vector<void*> allocs;
    char* slab = nullptr;  // block that small allocations are cut from
    size_t slab_used = 0;
    // per species
    ull* dn = nullptr;  // [3] counters
    ull hn[PT_NSPECIES] = {0, 0, 0};  // host view of the counts: exact while counts_known
    bool counts_known = true;
    // tables
    double* drate[PT_NSPECIES] = {nullptr, nullptr, nullptr};
    double* drb[PT_NSPECIES] = {nullptr, nullptr, nullptr};
    int L[PT_NSPECIES] = {0, 0, 0};
    int kint[PT_NSPECIES] = {0, 0, 0};
    double* dsb_le[MAX_SB] = {};
    double* dsb_data[MAX_SB] = {};
    Field* dfields = nullptr;
    std::vector<Field> hfields;
    // compaction: the kernels' arguments (scratch arrays included) and their grid
    Compaction cmp{};
    int cmp_blocks = 1;
    // a copy of the state at the start of a run's window (see run_window), kept from one
    // window to the next, given back when another allocation needs the room, and freed with
    // the context
    char* saved = nullptr;
    size_t saved_bytes = 0;
    bool saved_live = false;  // a window may yet be taken back
    double* stat_part = nullptr;
    // counters
    ull* dcounts = nullptr;
    ull* dflags = nullptr;
    ull* dwork = nullptr;
    ull* drange = nullptr;
    double* dtally = nullptr;
    double* ddose = nullptr;
    uint32_t step = 0;
    double last_t = 0.0;      // final time of the step launched last
    double lowest_rate = 0.0; // of an electron's collisions, over the intervals above the cut
    uint64_t next_uid = 0;
    int grid = 0;         // workgroups of the grid-stride utility kernels
    int ncu = 0;          // compute units
    int lds_bytes = 0;
    Clock* dclock = nullptr;
    pt_launch launch{256, 1, 8, 0, 1u << PT_PROC_SB, 2, 0};
    int resident[MAX_KV][3] = {};  // resident workgroups per CU: kernel variant x block 128/256/512 (0: no room)
    int resident_wide = 0;         // and of the wide history pass
    int tail_block = 512;          // threads of the one-workgroup passes
    bool queues = false;      // work and collision queues allocated
    int resident_lds = -1;        // LDS size the residency was computed for
    double* noalloc = nullptr;    // this device's copy of the allocation-free scratch array
    double* swarm_part = nullptr;  // per-swarm sums (zero between calls), and their copy in
    double* swarm_host = nullptr;  // pinned memory (behind the report)
    // learned samplers
    struct Learned {
        float* params = nullptr;  // FP32 parameters (device)
        uint16_t* wimg = nullptr;  // BF16 image used by the step
        float* bimg = nullptr;
        bool trained = false;
        bool on = false;
        double tcut = 1e4 * EV;
        double emin = 0.0, emax = 0.0;  // energy range the network is used in (its gated range)
    } learn[NLEARN];
    int sb_z[MAX_SB] = {0, 0, 0, 0};
    pt_wall_record* dwall = nullptr;  // wall records
    ull* dwall_n = nullptr;
    ull wall_cap = 0;
    std::vector<double> sb_le[MAX_SB];   // host copies of the Seltzer-Berger energy grids
    std::vector<double> sb_thr[MAX_SB];  // and of their cell thresholds (pt_sb_thresholds)
    double* dsb_thr[MAX_SB] = {};
    // captured runs: one graph per (steps, compaction) shape
    hipGraphExec_t gexec[2] = {nullptr, nullptr};
    int gsteps[2] = {0, 0};
    pt_launch glaunch[2] = {};
    int glds[2] = {0, 0};
    uint64_t ggen[2] = {0, 0};  // params_gen at capture
    uint64_t params_gen = 0;    // bumped by every upload of changed parameters
    // for pt_debug_choices
    int main_block = 0, main_grid = 0;
    int64_t late_windows = 0, windows_back = 0;
    bool profile = false;
    hipEvent_t ev[8] = {};
    std::vector<hipEvent_t> evq;  // event pool of the profiling spans
    size_t evq_used = 0;
    std::vector<Span> spans;      // recorded, not yet read
    double adv_ms = 0.0, tail_ms = 0.0, cmp_ms = 0.0, graph_ms = 0.0;
    ull adv_launches = 0;
    std::string err;
};

static int fail(pt_ctx* c, int code, const char* fmt, ...) {
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof(buf), fmt, ap);
    va_end(ap);
    if (c) c->err = buf;
    return code;
}

#define HIPCHK(c, call)                                                                     \
    do {                                                                                    \
        hipError_t e_ = (call);                                                             \
        if (e_ != hipSuccess)                                                               \
            return fail((c), PT_E_HIP, "%s failed: %s (%s:%d)", #call, hipGetErrorString(e_), \
                        __FILE__, __LINE__);                                                \
    } while (0)

// ---- the allocation-free entry point's scratch array (pt_swarm_stats_noalloc)
// The per-swarm sums of k_swarm_stats accumulate here instead of in a buffer the library
// allocates: a file-scope device array of fixed size, one copy on every GPU the library
// runs on, held until the process ends.  In host code `noalloc_sums` only names the
// symbol; its address on each device comes from hipGetSymbolAddress, called once per device
// with that device current (pt_create), and only that address is passed to kernels and
// copies.
constexpr int NOALLOC_SWARMS = 4096;  // 4 doubles per swarm: 128 KiB per device
static __device__ __align__(256) double noalloc_sums[4 * NOALLOC_SWARMS];
constexpr int NOALLOC_DEVICES = 64;
static double* g_noalloc[NOALLOC_DEVICES] = {};
static std::mutex g_noalloc_mu;

static int noalloc_scratch(pt_ctx* c) {
    if (c->device < 0 || c->device >= NOALLOC_DEVICES)
        return fail(c, PT_E_ARG, "device ordinal %d beyond %d", c->device, NOALLOC_DEVICES - 1);
    std::lock_guard<std::mutex> lock(g_noalloc_mu);
    if (!g_noalloc[c->device]) {
        void* p = nullptr;
        hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(noalloc_sums));
        if (e != hipSuccess || !p)
            return fail(c, PT_E_HIP, "hipGetSymbolAddress of the scratch array failed: %s", hipGetErrorString(e));
        g_noalloc[c->device] = (double*)p;
    }
    c->noalloc = g_noalloc[c->device];
    return PT_OK;
}

// device memory; a window's copy of the state (see run_window) gives way to it
static hipError_t dev_malloc(pt_ctx* c, void** p, size_t bytes) {
    hipError_t e = hipMalloc(p, bytes ? bytes : 8);
    if (e != hipSuccess && c->saved && !c->saved_live) {
        (void)hipGetLastError();
        (void)hipFree(c->saved);  // (waits for the work that uses it)
        c->saved = nullptr;
        c->saved_bytes = 0;
        e = hipMalloc(p, bytes ? bytes : 8);
    }
    if (e != hipSuccess) {
        (void)hipGetLastError();  // reported here: a later launch's check must not find it
        *p = nullptr;
    }
    return e;
}

// device memory of its own, freed with the context
static int dalloc_own(pt_ctx* c, void** p, size_t bytes) {
    hipError_t e = dev_malloc(c, p, bytes);
    if (e != hipSuccess) return fail(c, PT_E_NOMEM, "hipMalloc(%zu) failed: %s", bytes, hipGetErrorString(e));
    c->allocs.push_back(*p);
    return PT_OK;
}

// device memory, the small pieces from a zeroed block (a context has some forty of them, and
// each hipMalloc or clearing takes several us)
static int dalloc(pt_ctx* c, void** p, size_t bytes) {
    constexpr size_t BLOCK = 1 << 20, SMALL = 1 << 16;
    if (bytes > SMALL) return dalloc_own(c, p, bytes);
    const size_t need = std::max<size_t>(256, (bytes + 255) & ~(size_t)255);
    if (!c->slab || c->slab_used + need > BLOCK) {
        int rc = dalloc_own(c, (void**)&c->slab, BLOCK);
        if (rc) return rc;
        c->slab_used = 0;
        HIPCHK(c, hipMemsetAsync(c->slab, 0, BLOCK, c->stream));
    }
    *p = c->slab + c->slab_used;
    c->slab_used += need;
    return PT_OK;
}

static int sync_params(pt_ctx* c) {
    if (!c->dirty) return PT_OK;
    // LDS layout: the math table, then the rate tables
    int off = MATH_DOUBLES;
    c->hp.rb_in_lds = c->cfg.nswarm <= 1 ? 1 : 0;
    for (int s = 0; s < PT_NSPECIES; s++) {
        c->hp.lds_rate_off[s] = off;
        if (c->hp.tab[s].valid) off += (c->hp.tab[s].k + 1) * c->hp.tab[s].nprocs * 3 + SCAN_PAD;
        c->hp.lds_rb_off[s] = off;
        if (c->hp.tab[s].valid && c->hp.rb_in_lds) off += (c->hp.tab[s].k + 1) * 3;
        c->hp.lds_proc_off[s] = off;
        if (c->hp.tab[s].valid) off += c->hp.tab[s].nprocs * (int)(sizeof(DevProc) / sizeof(double));
    }
    // several swarms with homogeneous fields: their E and B vectors in LDS (one swarm's
    // field is staged in the static block)
    bool hom = c->cfg.nswarm <= MAX_LDS_FIELDS;
    for (const Field& F : c->hfields)
        hom = hom && F.e.kind == PT_FIELD_HOMOGENEOUS && F.b.kind == PT_FIELD_HOMOGENEOUS && !F.cl.on;
    c->hp.field_lds = hom ? 1 : 0;
    // no magnetic field anywhere and E without -0 components: the force is qE exactly
    bool nob = true;
    for (const Field& F : c->hfields) {
        const bool bzero = F.b.kind == PT_FIELD_NONE ||
                           (F.b.kind == PT_FIELD_HOMOGENEOUS && F.b.v[0] == 0.0 && F.b.v[1] == 0.0 && F.b.v[2] == 0.0);
        bool eok = F.e.kind == PT_FIELD_NONE || F.e.kind == PT_FIELD_HOMOGENEOUS;
        if (F.e.kind == PT_FIELD_HOMOGENEOUS)
            for (int d = 0; d < 3; d++) eok = eok && !(F.e.v[d] == 0.0 && std::signbit(F.e.v[d]));
        nob = nob && bzero && eok;
    }
    // homogeneous electric fields along z only
    bool along = hom;
    for (const Field& F : c->hfields) along = along && F.e.v[0] == 0.0 && F.e.v[1] == 0.0;
    c->hp.forcing_off = (c->hp.forcing_off & ~(OFF_NO_B | OFF_E_Z)) | (nob ? OFF_NO_B : 0u) | (along ? OFF_E_Z : 0u);
    c->hp.lds_field_off = off;
    if (hom) off += field_doubles(c->hp.forcing_off) * c->cfg.nswarm;
    c->hp.lds_dose_off = off;  // (zeros in the image)
    if (c->hp.dose_bins > 0 && c->hp.dose_bins <= DOSE_LDS) off += c->hp.dose_bins + 2;
    off = (off + 1) & ~1;
    c->hp.lds_doubles = off;
    c->lds_bytes = off * (int)sizeof(double);
    c->hp.lds_coop_off = (c->lds_bytes + 15) & ~15;
    HIPCHK(c, hipMemcpyAsync(c->dp, &c->hp, sizeof(Params), hipMemcpyHostToDevice, c->stream));
    hipLaunchKernelGGL(k_build_image, dim3(IMAGE_BLOCKS), dim3(256), 0, c->stream, c->dp);
    HIPCHK(c, hipGetLastError());
    c->dirty = false;
    // a captured step bakes in host-side choices made from these parameters (the kernel
    // variant for a wall, the LDS sizes, the queues): graphs captured before are stale
    c->params_gen++;
    return PT_OK;
}

// the counts that a finished kernel has reported
static void take_counts(pt_ctx* c) {
    for (int s = 0; s < PT_NSPECIES; s++) c->hn[s] = std::min<ull>(c->report->n[s], c->cfg.capacity[s]);
    c->counts_known = true;
}

// counts and flags as they are now
static int read_state(pt_ctx* c) {
    hipLaunchKernelGGL(k_report, dim3(1), dim3(64), 0, c->stream, c->dp);
    HIPCHK(c, hipGetLastError());
    HIPCHK(c, hipStreamSynchronize(c->stream));
    take_counts(c);
    return PT_OK;
}

static int read_counts(pt_ctx* c) { return c->counts_known ? PT_OK : read_state(c); }

template <class T>
struct Scratch {
    T* p = nullptr;
    ~Scratch() {
        if (p) (void)hipFree(p);
    }
};

template <class T>
static int dscratch(pt_ctx* c, Scratch<T>& s, size_t count) {
    if (dev_malloc(c, (void**)&s.p, sizeof(T) * count) != hipSuccess)
        return fail(c, PT_E_NOMEM, "scratch allocation of %zu bytes failed", sizeof(T) * count);
    return PT_OK;
}

// kernel variants: history pass over the step's slots, first collision round, later
// collision rounds, history pass over the work queues, sampling round
enum {
    KV_RANGE_FULL = 0, KV_RANGE_EVENT = 1, KV_QUEUE_EVENT = 2, KV_QUEUE_FULL = 3, KV_SAMPLE = 4, KV_RANGE_WALL = 5,
    // the same push/select kernels with the learned samplers evaluated in place
    KV_RANGE_FULL_MLP = 6, KV_RANGE_EVENT_MLP = 7, KV_QUEUE_EVENT_MLP = 8, KV_QUEUE_FULL_MLP = 9, NKV = 10
};
// The history pass of a population that fills the GPU several times over: workgroups of 768
// threads, three waves per SIMD instead of two (168 registers; a lane then reads its species'
// constants, its force and its rate bounds from LDS each time).  The pass is bound by
// instruction issue, and three waves hide more of one another's branches and LDS reads:
// 24 steps of 10^7 electrons 44.9 -> 35.1 ms (42.3 in small workgroups with the second push
// round), 48 of 10^6 10.7 -> 9.1, 16 of 1.2 x 10^8 in 256 swarms 333 -> 255.
// With few electrons per lane the launch is as long as its longest lanes' collisions, and a
// wave that shares its SIMD with two others takes 1.3 to 1.5 times as long for them: 32 steps
// of n electrons took (two against three waves, ms) 3.15/3.54 for 3 x 10^5, 4.74/5.61 for
// 6 x 10^5, 5.77/5.68 for 8 x 10^5, 7.82/7.47 for 1.2 x 10^6 and 11.96/10.68 for 2 x 10^6, so
// the line lies at four electrons or positrons per lane.  Photons do not count (most only
// fly): a beam of 2 x 10^6 photons and 10^5 electrons takes 168 against 256 ms.
constexpr int WIDE = 768;
constexpr ull WIDE_PER_LANE = 4;
// (a launch of one step has no chains that long: from 1.5 per lane on, 8 such launches for
// 3 x 10^5 electrons 1.62 -> 1.57 ms, 4 x 10^5 2.12 -> 1.72, 6 x 10^5 2.75 -> 1.97; 2 x 10^5
// 1.32 -> 1.55)
constexpr ull WIDE_PER_LANE_2 = 3;  // half a lane's electrons
// the variant of a push/select kernel that evaluates learned samplers in place
static int with_mlp(int v, bool mlp) { return mlp && v <= KV_QUEUE_FULL ? KV_RANGE_FULL_MLP + v : v; }
static_assert(NKV <= MAX_KV, "residency table too small for the kernel variants");

template <int BS>
static const void* kernel_variant(int v) {
    switch (v) {
        case KV_RANGE_FULL: return (const void*)k_advance<BS, SRC_RANGE, false>;
        case KV_RANGE_EVENT: return (const void*)k_advance<BS, SRC_RANGE, true>;
        case KV_QUEUE_EVENT: return (const void*)k_advance<BS, SRC_QUEUE, true>;
        case KV_QUEUE_FULL: return (const void*)k_advance<BS, SRC_QUEUE, false>;
        case KV_RANGE_WALL: return (const void*)k_advance<BS, SRC_RANGE, false, true>;
        case KV_RANGE_FULL_MLP: return (const void*)k_advance<BS, SRC_RANGE, false, false, true>;
        case KV_RANGE_EVENT_MLP: return (const void*)k_advance<BS, SRC_RANGE, true, false, true>;
        case KV_QUEUE_EVENT_MLP: return (const void*)k_advance<BS, SRC_QUEUE, true, false, true>;
        case KV_QUEUE_FULL_MLP: return (const void*)k_advance<BS, SRC_QUEUE, false, false, true>;
        default: return (const void*)k_sample<BS>;
    }
}

static const void* kernel_of(int v, int bs) {
    if (bs == WIDE) return (const void*)k_advance<WIDE, SRC_RANGE, false>;
    return bs == 128 ? kernel_variant<128>(v) : bs == 512 ? kernel_variant<512>(v) : kernel_variant<256>(v);
}

extern "C" {

int pt_abi_version(void) { return PT_ABI_VERSION; }

const char* pt_last_error(const pt_ctx* ctx) { return ctx ? ctx->err.c_str() : pt::host_last_error(); }

void pt_destroy(pt_ctx* c) {
    if (!c) return;
    (void)hipSetDevice(c->device);
    if (c->stream) (void)hipStreamSynchronize(c->stream);
    for (auto& g : c->gexec)
        if (g) (void)hipGraphExecDestroy(g);
    for (void* p : c->allocs) (void)hipFree(p);
    if (c->saved) (void)hipFree(c->saved);
    if (c->report) (void)hipHostFree(c->report);
    for (auto& e : c->ev)
        if (e) (void)hipEventDestroy(e);
    for (auto& e : c->evq)
        if (e) (void)hipEventDestroy(e);
    if (c->stream) (void)hipStreamDestroy(c->stream);
    delete c;
}

int pt_create(const pt_config* cfg, pt_ctx** out) {
    if (!cfg || !out) return PT_E_ARG;
    *out = nullptr;
    pt_ctx* c = new (std::nothrow) pt_ctx();
    if (!c) return PT_E_NOMEM;
    c->cfg = *cfg;
    if (c->cfg.nswarm < 1) c->cfg.nswarm = 1;
    int ndev = 0;
    // failures that return no context leave their message for pt_last_error(NULL)
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) {
        int rc = fail(c, PT_E_NOT_BUILT, "no HIP device available");
        host_set_error(c->err.c_str());
        delete c;
        return rc;
    }
    for (int s = 0; s < PT_NSPECIES; s++) {
        if (c->cfg.capacity[s] >= (1ull << 31)) {
            int rc = fail(c, PT_E_ARG, "capacity of species %d exceeds 2^31 - 1", s);
            host_set_error(c->err.c_str());
            pt_destroy(c);
            return rc;
        }
    }
    c->device = cfg->device;
    int rc = PT_OK;
#define TRY(x)             \
    do {                   \
        rc = (x);          \
        if (rc != PT_OK) { \
            *out = c;      \
            return rc;     \
        }                  \
    } while (0)
    if (hipSetDevice(c->device) != hipSuccess) TRY(fail(c, PT_E_HIP, "hipSetDevice(%d) failed", c->device));
    if (hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess)
        TRY(fail(c, PT_E_HIP, "hipStreamCreate failed"));
    for (auto& e : c->ev)
        if (hipEventCreate(&e) != hipSuccess) TRY(fail(c, PT_E_HIP, "hipEventCreate failed"));
    const size_t pinned = sizeof(Report) + sizeof(double) * 4 * (size_t)c->cfg.nswarm;
    if (hipHostMalloc((void**)&c->report, pinned, hipHostMallocDefault) != hipSuccess) {
        (void)hipGetLastError();
        c->report = nullptr;
        TRY(fail(c, PT_E_NOMEM, "pinned host memory allocation of %zu bytes failed", pinned));
    }
    c->swarm_host = (double*)(c->report + 1);
    Params& P = c->hp;
    memset(&P, 0, sizeof(P));
    memset(c->report, 0, sizeof(Report));
    P.report = c->report;
    TRY(dalloc(c, (void**)&c->dn, sizeof(ull) * PT_NSPECIES));
    for (int s = 0; s < PT_NSPECIES; s++) {
        SpeciesDev& S = P.sp[s];
        ull cap = c->cfg.capacity[s];
        S.cap = cap;
        S.tracked = c->cfg.tracked[s];
        S.n = c->dn + s;
        // one allocation: the records (slot i's field k at f[0][i * PT_NFIELDS + k]), then the
        // columns
        const size_t size[7] = {sizeof(double) * PT_NFIELDS, sizeof(uint64_t), sizeof(int32_t), sizeof(double),
                                sizeof(uint32_t), 1, 1};
        size_t off[8] = {0};
        for (int q = 0; q < 7; q++) off[q + 1] = off[q] + ((size[q] * std::max<ull>(cap, 1) + 255) & ~(size_t)255);
        char* base = nullptr;
        TRY(dalloc(c, (void**)&base, off[7]));
        S.f[0] = (double*)base;
        for (int f = 1; f < PT_NFIELDS; f++) S.f[f] = S.f[0] + f;
        S.uid = (uint64_t*)(base + off[1]);
        S.swarm = (int32_t*)(base + off[2]);
        S.trem = (double*)(base + off[3]);
        S.draw = (uint32_t*)(base + off[4]);
        S.active = (uint8_t*)(base + off[5]);
        S.evp = (uint8_t*)(base + off[6]);
        HIPCHK(c, hipMemsetAsync(S.active, 0, cap ? cap : 1, c->stream));
    }
    HIPCHK(c, hipMemsetAsync(c->dn, 0, sizeof(ull) * PT_NSPECIES, c->stream));
    TRY(dalloc(c, (void**)&c->dcounts, sizeof(ull) * PT_NSPECIES * NCOUNT));
    TRY(dalloc(c, (void**)&c->dflags, sizeof(ull) * NFLAGS));
    TRY(dalloc(c, (void**)&c->dwork, sizeof(ull) * NWORK));
    TRY(dalloc(c, (void**)&c->drange, sizeof(ull) * 2 * PT_NSPECIES));
    TRY(dalloc(c, (void**)&c->dclock, sizeof(Clock)));
    TRY(dalloc(c, (void**)&P.q.cnt, sizeof(ull) * NQCNT));
    HIPCHK(c, hipMemsetAsync(P.q.cnt, 0, sizeof(ull) * NQCNT, c->stream));
    for (int s = 0; s < PT_NSPECIES; s++)
        for (int k = 0; k < 16; k++) P.q.kq[s][k] = -1;
    HIPCHK(c, hipMemsetAsync(c->dclock, 0, sizeof(Clock), c->stream));
    HIPCHK(c, hipMemsetAsync(c->dcounts, 0, sizeof(ull) * PT_NSPECIES * NCOUNT, c->stream));
    HIPCHK(c, hipMemsetAsync(c->dflags, 0, sizeof(ull) * NFLAGS, c->stream));
    HIPCHK(c, hipMemsetAsync(c->dwork, 0, sizeof(ull) * NWORK, c->stream));
    HIPCHK(c, hipMemsetAsync(c->drange, 0, sizeof(ull) * 2 * PT_NSPECIES, c->stream));
    int bins = std::max(0, c->cfg.tally_bins);
    TRY(dalloc(c, (void**)&c->dtally, sizeof(double) * PT_NSPECIES * (bins + 2)));
    HIPCHK(c, hipMemsetAsync(c->dtally, 0, sizeof(double) * PT_NSPECIES * (bins + 2), c->stream));
    P.tally = c->dtally;
    P.tally_bins = bins;
    P.tally_tracked = c->cfg.tally_tracked ? 1 : 0;
    P.dose_bins = std::max(0, c->cfg.dose_bins);
    TRY(dalloc(c, (void**)&c->ddose, sizeof(double) * (P.dose_bins + 3)));
    HIPCHK(c, hipMemsetAsync(c->ddose, 0, sizeof(double) * (P.dose_bins + 3), c->stream));
    P.dose = c->ddose;
    P.dose_zlo = c->cfg.dose_zlo;
    P.dose_zhi = c->cfg.dose_zhi > c->cfg.dose_zlo ? c->cfg.dose_zhi : c->cfg.dose_zlo + 1.0;
    P.tally_lo = c->cfg.tally_lo > 0 ? c->cfg.tally_lo : 1e3 * EV;
    P.tally_hi = c->cfg.tally_hi > P.tally_lo ? c->cfg.tally_hi : 1e7 * EV;
    // fields
    c->hfields.assign(c->cfg.nswarm, Field{});
    TRY(dalloc(c, (void**)&c->dfields, sizeof(Field) * c->cfg.nswarm));
    HIPCHK(c, hipMemcpyAsync(c->dfields, c->hfields.data(), sizeof(Field) * c->cfg.nswarm,
                             hipMemcpyHostToDevice, c->stream));
    P.fields = c->dfields;
    P.nswarm = c->cfg.nswarm;
    P.seed = c->cfg.seed;
    P.counts = c->dcounts;
    P.flags = c->dflags;
    P.work = c->dwork;
    P.range = c->drange;
    P.clock = c->dclock;
    P.defer_mask = c->launch.defer_mask;
    // compaction scratch
    size_t most = 1;
    for (int s = 0; s < PT_NSPECIES; s++) {
        const size_t cap = c->cfg.capacity[s], chunks = (cap + CH - 1) / CH + 1;
        c->cmp.sp[s] = P.sp[s];
        unsigned** part[3] = {&c->cmp.cnt[s], &c->cmp.hole[s], &c->cmp.tail[s]};
        const size_t words = (chunks + 63) & ~(size_t)63;
        unsigned* base = nullptr;
        TRY(dalloc(c, (void**)&base, 3 * sizeof(unsigned) * words));
        for (int q = 0; q < 3; q++) *part[q] = base + q * words;
        // the lists of positions lie in the column of times left, which is in use only within a
        // step of collision rounds
        c->cmp.hpos[s] = (unsigned*)P.sp[s].trem;
        c->cmp.tpos[s] = c->cmp.hpos[s] + cap / 2 + 1;
        most = std::max(most, chunks);
    }
    TRY(dalloc(c, (void**)&c->cmp.info, sizeof(ull) * 4 * PT_NSPECIES));
    HIPCHK(c, hipMemsetAsync(c->cmp.info, 0, sizeof(ull) * 4 * PT_NSPECIES, c->stream));
    c->cmp.work = c->dwork;
    c->cmp.report = c->report;
    c->cmp_blocks = (int)std::min<size_t>(most, 512);
    TRY(dalloc(c, (void**)&c->stat_part, sizeof(double) * NSTAT * STAT_BLOCKS + sizeof(ull)));
    HIPCHK(c, hipMemsetAsync(c->stat_part + NSTAT * STAT_BLOCKS, 0, sizeof(ull), c->stream));
    TRY(dalloc(c, (void**)&c->dp, sizeof(Params)));
    TRY(dalloc(c, (void**)&P.image, IMAGE_BYTES));
    hipDeviceProp_t prop;
    HIPCHK(c, hipGetDeviceProperties(&prop, c->device));
    c->ncu = prop.multiProcessorCount;
    TRY(noalloc_scratch(c));
    c->grid = prop.multiProcessorCount * 8;
    c->dirty = true;
    TRY(sync_params(c));
    HIPCHK(c, hipStreamSynchronize(c->stream));
#undef TRY
    *out = c;
    return PT_OK;
}

int pt_upload_table(pt_ctx* c, int sp, const pt_table_desc* t) {
    if (!c) return PT_E_ARG;
    if (sp < 0 || sp >= PT_NSPECIES || !t) return fail(c, PT_E_ARG, "bad species or table");
    if (t->order != 3) return fail(c, PT_E_ARG, "Chebyshev order must be 3 (got %d)", t->order);
    if (t->nprocs < 0 || t->nprocs > MAX_PROCS) return fail(c, PT_E_ARG, "nprocs %d out of [0, %d]", t->nprocs, MAX_PROCS);
    if (t->nintervals < 1 || t->nintervals >= MAX_INTERVALS) return fail(c, PT_E_ARG, "nintervals out of range");
    int nsw = t->nswarm < 1 ? 1 : t->nswarm;
    if (nsw != 1 && nsw != c->cfg.nswarm) return fail(c, PT_E_ARG, "table nswarm %d != context nswarm %d", nsw, c->cfg.nswarm);
    if (!t->rate || !t->ratebound || (t->nprocs > 0 && !t->procs)) return fail(c, PT_E_ARG, "null table arrays");
    // every process descriptor is checked before anything of the table is written, so a
    // rejected table leaves the previous one in place
    int nkinds = 0;
    bool kind_seen[16] = {};
    for (int j = 0; j < t->nprocs; j++) {
        const pt_proc_desc& s = t->procs[j];
        if (s.kind < PT_PROC_ELASTIC || s.kind > PT_PROC_KN_COMPTON)
            return fail(c, PT_E_ARG, "process %d: unknown kind %d", j, s.kind);
        if ((s.kind == PT_PROC_SB && (s.slot < 0 || s.slot >= MAX_SB)) ||
            (s.kind == PT_PROC_PHOTOELECTRIC && (s.slot < 0 || s.slot >= MAX_PE)))
            return fail(c, PT_E_ARG, "process %d: data slot %d out of range", j, s.slot);
        if (s.kind == PT_PROC_RBEB && !(s.B > 0)) return fail(c, PT_E_ARG, "process %d: RBEB needs B > 0", j);
        if (s.kind == PT_PROC_ELASTIC && !(s.c[0] > 0))
            return fail(c, PT_E_ARG, "process %d: elastic needs the screening radius c[0]", j);
        if (s.kind == PT_PROC_BETHE_HEITLER && !(s.c[0] > 0))
            return fail(c, PT_E_ARG, "process %d: Bethe-Heitler needs c[0] = Z^(1/3)", j);
        if (!kind_seen[s.kind]) {
            kind_seen[s.kind] = true;
            nkinds++;
        }
    }
    if (nkinds > NKQ) return fail(c, PT_E_ARG, "more than %d sampler kinds in one table", NKQ);
    HIPCHK(c, hipSetDevice(c->device));
    int k = t->nintervals;
    size_t nr = (size_t)(k + 1) * t->nprocs * 3, nb = (size_t)(k + 1) * 3 * c->cfg.nswarm;
    if (!c->drate[sp] || c->L[sp] != t->nprocs || c->kint[sp] != k) {
        int rc = dalloc(c, (void**)&c->drate[sp], sizeof(double) * (nr ? nr : 1));
        if (rc) return rc;
        rc = dalloc(c, (void**)&c->drb[sp], sizeof(double) * nb);
        if (rc) return rc;
        c->L[sp] = t->nprocs;
        c->kint[sp] = k;
    }
    HIPCHK(c, hipMemcpyAsync(c->drate[sp], t->rate, sizeof(double) * nr, hipMemcpyHostToDevice, c->stream));
    if (nsw == 1) {
        for (int q = 0; q < c->cfg.nswarm; q++)
            HIPCHK(c, hipMemcpyAsync(c->drb[sp] + (size_t)q * (k + 1) * 3, t->ratebound,
                                     sizeof(double) * (k + 1) * 3, hipMemcpyHostToDevice, c->stream));
    } else {
        HIPCHK(c, hipMemcpyAsync(c->drb[sp], t->ratebound, sizeof(double) * nb, hipMemcpyHostToDevice, c->stream));
    }
    DevTable& D = c->hp.tab[sp];
    D.nprocs = t->nprocs;
    D.k = k;
    D.nswarm = c->cfg.nswarm;
    D.valid = 1;
    D.xmax = t->xmax;
    D.cut = t->energy_cut;
    D.rate = c->drate[sp];
    D.ratebound = c->drb[sp];
    for (int j = 0; j < t->nprocs; j++) {
        const pt_proc_desc& s = t->procs[j];
        DevProc& d = D.procs[j];
        d.kind = s.kind;
        d.Z = s.Z;
        d.slot = s.slot;
        d.N = s.N;
        d.B = s.B;
        d.U = s.U;
        d.tcut = s.tcut;
        d.zf = s.zf;
        for (int q = 0; q < 4; q++) d.c[q] = s.c[q];
        if (d.kind == PT_PROC_RBEB) {
            // the orbital's terms of rbeb_setup: B / mc^2, log(2 B / mc^2), 1 / B
            d.c[0] = d.B / MC2;
            d.c[1] = std::log(2.0 * d.c[0]);
            d.c[2] = 1.0 / d.B;
        }
    }
    if (sp == PT_ELECTRON) {
        c->lowest_rate = 0.0;
        for (int i = 1; i <= k; i++) {
            if (std::ldexp(t->xmax, i - k - 1) < t->energy_cut) continue;  // (the interval's lower end)
            double rate = 0.0;  // the mean over the interval
            for (int j = 0; j < t->nprocs; j++) rate += t->rate[((size_t)i * t->nprocs + j) * 3];
            if (c->lowest_rate == 0.0 || rate < c->lowest_rate) c->lowest_rate = rate;
        }
    }
    // one collision queue per sampler kind present in the table
    Queues& Q = c->hp.q;
    for (int k = 0; k < 16; k++) Q.kq[sp][k] = -1;
    Q.nkq[sp] = 0;
    for (int j = 0; j < t->nprocs; j++) {
        int kd = t->procs[j].kind;
        if (Q.kq[sp][kd] >= 0) continue;
        Q.qkind[sp][Q.nkq[sp]] = (int8_t)kd;
        Q.kq[sp][kd] = (int8_t)Q.nkq[sp]++;
    }
    c->queues = false;  // allocate the new kinds' queues before the next collision round
    c->dirty = true;
    int rc = sync_params(c);
    if (rc) return rc;
    HIPCHK(c, hipStreamSynchronize(c->stream));
    return PT_OK;
}

int pt_upload_sb(pt_ctx* c, int slot, int Z, int ne, int ncum, const double* le, const double* data) {
    if (!c) return PT_E_ARG;
    if (slot < 0 || slot >= MAX_SB || ne < 2 || ncum < 2 || !le || !data)
        return fail(c, PT_E_ARG, "bad SB upload arguments");
    std::vector<double> thr(ne);
    if (pt_sb_thresholds(le, ne, thr.data()) != PT_OK) return fail(c, PT_E_ARG, "%s", pt::host_last_error());
    HIPCHK(c, hipSetDevice(c->device));
    int rc = dalloc(c, (void**)&c->dsb_le[slot], sizeof(double) * ne);
    if (rc) return rc;
    rc = dalloc(c, (void**)&c->dsb_thr[slot], sizeof(double) * ne);
    if (rc) return rc;
    rc = dalloc(c, (void**)&c->dsb_data[slot], sizeof(double) * (size_t)ne * ncum);
    if (rc) return rc;
    HIPCHK(c, hipMemcpyAsync(c->dsb_le[slot], le, sizeof(double) * ne, hipMemcpyHostToDevice, c->stream));
    HIPCHK(c, hipMemcpyAsync(c->dsb_thr[slot], thr.data(), sizeof(double) * ne, hipMemcpyHostToDevice, c->stream));
    HIPCHK(c, hipMemcpyAsync(c->dsb_data[slot], data, sizeof(double) * (size_t)ne * ncum, hipMemcpyHostToDevice, c->stream));
    c->hp.sb[slot].ne = ne;
    c->hp.sb[slot].ncum = ncum;
    c->hp.sb[slot].log_energy = c->dsb_le[slot];
    c->hp.sb[slot].thr = c->dsb_thr[slot];
    c->hp.sb[slot].data = c->dsb_data[slot];
    c->sb_z[slot] = Z;
    c->sb_le[slot].assign(le, le + ne);
    c->sb_thr[slot] = thr;
    c->dirty = true;
    rc = sync_params(c);
    if (rc) return rc;
    HIPCHK(c, hipStreamSynchronize(c->stream));
    return PT_OK;
}

int pt_upload_pe(pt_ctx* c, int slot, int Z, int nshell, const double* binding) {
    if (!c) return PT_E_ARG;
    if (slot < 0 || slot >= MAX_PE || nshell < 1 || nshell > MAX_SHELLS || !binding)
        return fail(c, PT_E_ARG, "bad photoelectric upload arguments");
    c->hp.pe[slot].nshell = nshell;
    for (int q = 0; q < nshell; q++) c->hp.pe[slot].binding[q] = binding[q];
    (void)Z;
    c->dirty = true;
    return sync_params(c);
}

int pt_set_field(pt_ctx* c, int swarm, const pt_field_desc* f) {
    if (!c) return PT_E_ARG;
    if (swarm < 0 || swarm >= c->cfg.nswarm || !f) return fail(c, PT_E_ARG, "bad swarm %d", swarm);
    Field& F = c->hfields[swarm];
    const pt_field_fn* src[2] = {&f->e, &f->b};
    FieldFn* dst[2] = {&F.e, &F.b};
    for (int q = 0; q < 2; q++) {
        dst[q]->kind = src[q]->kind;
        for (int d = 0; d < 3; d++) {
            dst[q]->v[d] = src[q]->v[d];
            dst[q]->v2[d] = src[q]->v2[d];
        }
        dst[q]->z1 = src[q]->z1;
        dst[q]->z2 = src[q]->z2;
        dst[q]->sx = src[q]->sx;
        dst[q]->sy = src[q]->sy;
        dst[q]->sz = src[q]->sz;
        dst[q]->ez0 = src[q]->ez0;
    }
    HIPCHK(c, hipSetDevice(c->device));
    HIPCHK(c, hipMemcpyAsync(c->dfields + swarm, &F, sizeof(Field), hipMemcpyHostToDevice, c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    c->dirty = true;  // the choice of the fields' LDS form may change
    return sync_params(c);
}

int pt_count(pt_ctx* c, int sp, uint64_t* n) {
    if (!c || sp < 0 || sp >= PT_NSPECIES || !n) return c ? fail(c, PT_E_ARG, "bad arguments") : PT_E_ARG;
    HIPCHK(c, hipSetDevice(c->device));
    int rc = read_counts(c);
    if (rc) return rc;
    *n = c->hn[sp];
    return PT_OK;
}

static int put_particles(pt_ctx* c, int sp, ull base, const double* const soa[PT_NFIELDS],
                         const uint8_t* active, const uint64_t* uid, const int32_t* swarm, size_t n) {
    SpeciesDev& S = c->hp.sp[sp];
    if (n == 0) return PT_OK;
    // the host's columns into records (absent fields are zero), one copy
    std::vector<double> rec((size_t)PT_NFIELDS * n, 0.0);
    for (int f = 0; f < PT_NFIELDS; f++)
        if (soa[f])
            for (size_t i = 0; i < n; i++) rec[i * PT_NFIELDS + f] = soa[f][i];
    std::vector<uint64_t> u;
    if (!uid) {
        u.resize(n);
        for (size_t i = 0; i < n; i++) u[i] = c->next_uid + i;
        c->next_uid += n;
        uid = u.data();
    }
    std::vector<int32_t> sw;
    if (!swarm) {
        sw.assign(n, 0);
        swarm = sw.data();
    }
    for (size_t i = 0; i < n; i++)
        if (swarm[i] < 0 || swarm[i] >= c->cfg.nswarm)
            return fail(c, PT_E_ARG, "particle %zu: swarm %d out of range", i, swarm[i]);
    std::vector<uint8_t> act;
    if (!active) {
        act.assign(n, 1);
        active = act.data();
    }
    // every copy is enqueued after the checks, and the host buffers outlive them (the
    // stream is synchronised before they go)
    if (n)
        HIPCHK(c, hipMemcpyAsync(S.f[0] + (size_t)base * PT_NFIELDS, rec.data(), sizeof(double) * rec.size(),
                                 hipMemcpyHostToDevice, c->stream));
    HIPCHK(c, hipMemcpyAsync(S.uid + base, uid, sizeof(uint64_t) * n, hipMemcpyHostToDevice, c->stream));
    HIPCHK(c, hipMemcpyAsync(S.swarm + base, swarm, sizeof(int32_t) * n, hipMemcpyHostToDevice, c->stream));
    HIPCHK(c, hipMemcpyAsync(S.active + base, active, n, hipMemcpyHostToDevice, c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    return PT_OK;
}

int pt_add_particles(pt_ctx* c, int sp, const double* const soa[PT_NFIELDS], const uint64_t* uid,
                     const int32_t* swarm, size_t n) {
    if (!c) return PT_E_ARG;
    if (sp < 0 || sp >= PT_NSPECIES || !soa) return fail(c, PT_E_ARG, "bad arguments");
    HIPCHK(c, hipSetDevice(c->device));
    int rc = read_counts(c);
    if (rc) return rc;
    if (c->hn[sp] + n > c->cfg.capacity[sp])
        return fail(c, PT_E_CAPACITY, "species %d: %llu + %zu particles exceed capacity %llu", sp,
                    (unsigned long long)c->hn[sp], n, (unsigned long long)c->cfg.capacity[sp]);
    rc = put_particles(c, sp, c->hn[sp], soa, nullptr, uid, swarm, n);
    if (rc) return rc;
    ull nn = c->hn[sp] + n;
    HIPCHK(c, hipMemcpyAsync(c->dn + sp, &nn, sizeof(ull), hipMemcpyHostToDevice, c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    c->hn[sp] = nn;
    return PT_OK;
}

int pt_set_particles(pt_ctx* c, int sp, const double* const soa[PT_NFIELDS], const uint8_t* active,
                     const uint64_t* uid, const int32_t* swarm, size_t n) {
    if (!c) return PT_E_ARG;
    if (sp < 0 || sp >= PT_NSPECIES || !soa) return fail(c, PT_E_ARG, "bad arguments");
    if (n > c->cfg.capacity[sp]) return fail(c, PT_E_CAPACITY, "%zu particles exceed capacity", n);
    HIPCHK(c, hipSetDevice(c->device));
    int rc = put_particles(c, sp, 0, soa, active, uid, swarm, n);
    if (rc) return rc;
    ull nn = n;
    HIPCHK(c, hipMemcpyAsync(c->dn + sp, &nn, sizeof(ull), hipMemcpyHostToDevice, c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    c->hn[sp] = nn;
    return PT_OK;
}

int pt_init_particles(pt_ctx* c, int sp, size_t n, double e1, double e2, int loguniform, int swarm,
                      uint64_t uid0, double t0) {
    if (!c) return PT_E_ARG;
    if (sp < 0 || sp >= PT_NSPECIES) return fail(c, PT_E_ARG, "bad species");
    if (swarm < 0 || swarm >= c->cfg.nswarm) return fail(c, PT_E_ARG, "bad swarm");
    if (!(e1 > 0) || (loguniform && !(e2 > 0))) return fail(c, PT_E_ARG, "energies must be positive");
    HIPCHK(c, hipSetDevice(c->device));
    int rc = read_counts(c);
    if (rc) return rc;
    if (c->hn[sp] + n > c->cfg.capacity[sp]) return fail(c, PT_E_CAPACITY, "initial particles exceed capacity");
    rc = sync_params(c);
    if (rc) return rc;
    if (n) {
        int blocks = (int)std::min<size_t>((n + 255) / 256, 65535);
        hipLaunchKernelGGL(k_init_particles, dim3(blocks), dim3(256), 0, c->stream, c->dp, sp,
                           (ull)c->hn[sp], (ull)n, e1, e2, loguniform, swarm, uid0, t0);
        HIPCHK(c, hipGetLastError());
    }
    ull nn = c->hn[sp] + n;
    HIPCHK(c, hipMemcpyAsync(c->dn + sp, &nn, sizeof(ull), hipMemcpyHostToDevice, c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    c->hn[sp] = nn;
    if (uid0 + n > c->next_uid) c->next_uid = uid0 + n;
    return PT_OK;
}

int pt_init_beam(pt_ctx* c, int sp, size_t n, double e, const double dir[3], int swarm, uint64_t uid0, double t0) {
    if (!c) return PT_E_ARG;
    if (sp < 0 || sp >= PT_NSPECIES || !dir) return fail(c, PT_E_ARG, "bad arguments");
    if (swarm < 0 || swarm >= c->cfg.nswarm) return fail(c, PT_E_ARG, "bad swarm");
    double nrm = std::sqrt(dir[0] * dir[0] + dir[1] * dir[1] + dir[2] * dir[2]);
    if (!(e > 0) || !(nrm > 0)) return fail(c, PT_E_ARG, "energy and direction must be nonzero");
    HIPCHK(c, hipSetDevice(c->device));
    int rc = read_counts(c);
    if (rc) return rc;
    if (c->hn[sp] + n > c->cfg.capacity[sp]) return fail(c, PT_E_CAPACITY, "beam particles exceed capacity");
    if ((rc = sync_params(c))) return rc;
    if (n) {
        int blocks = (int)std::min<size_t>((n + 255) / 256, 65535);
        hipLaunchKernelGGL(k_init_beam, dim3(blocks), dim3(256), 0, c->stream, c->dp, sp, (ull)c->hn[sp], (ull)n, e,
                           dir[0] / nrm, dir[1] / nrm, dir[2] / nrm, swarm, uid0, t0);
        HIPCHK(c, hipGetLastError());
    }
    ull nn = c->hn[sp] + n;
    HIPCHK(c, hipMemcpyAsync(c->dn + sp, &nn, sizeof(ull), hipMemcpyHostToDevice, c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    c->hn[sp] = nn;
    if (uid0 + n > c->next_uid) c->next_uid = uid0 + n;
    return PT_OK;
}

int pt_download(pt_ctx* c, int sp, double* const soa[PT_NFIELDS], uint8_t* active, uint64_t* uid,
                int32_t* swarm, size_t cap, size_t* n) {
    if (!c) return PT_E_ARG;
    if (sp < 0 || sp >= PT_NSPECIES) return fail(c, PT_E_ARG, "bad species");
    HIPCHK(c, hipSetDevice(c->device));
    int rc = read_counts(c);
    if (rc) return rc;
    size_t m = c->hn[sp];
    if (n) *n = m;
    if (m > cap) return fail(c, PT_E_CAPACITY, "host buffer of %zu too small for %zu particles", cap, m);
    SpeciesDev& S = c->hp.sp[sp];
    std::vector<double> rec;
    bool want = false;
    for (int f = 0; f < PT_NFIELDS && soa; f++) want = want || soa[f];
    if (m) {
        if (want) {
            rec.resize((size_t)PT_NFIELDS * m);
            HIPCHK(c, hipMemcpyAsync(rec.data(), S.f[0], sizeof(double) * rec.size(), hipMemcpyDeviceToHost, c->stream));
        }
        if (active) HIPCHK(c, hipMemcpyAsync(active, S.active, m, hipMemcpyDeviceToHost, c->stream));
        if (uid) HIPCHK(c, hipMemcpyAsync(uid, S.uid, sizeof(uint64_t) * m, hipMemcpyDeviceToHost, c->stream));
        if (swarm) HIPCHK(c, hipMemcpyAsync(swarm, S.swarm, sizeof(int32_t) * m, hipMemcpyDeviceToHost, c->stream));
    }
    HIPCHK(c, hipStreamSynchronize(c->stream));
    // records back into the host's columns
    if (m && want)
        for (int f = 0; f < PT_NFIELDS; f++)
            if (soa[f])
                for (size_t i = 0; i < m; i++) soa[f][i] = rec[i * PT_NFIELDS + f];
    return PT_OK;
}

static int require_tables(pt_ctx* c) {
    for (int s = 0; s < PT_NSPECIES; s++) {
        if (c->cfg.tracked[s] && !c->hp.tab[s].valid && c->cfg.capacity[s] > 0)
            return fail(c, PT_E_STATE, "species %d is tracked but has no collision table", s);
        const DevTable& tb = c->hp.tab[s];
        if (!tb.valid) continue;
        for (int j = 0; j < tb.nprocs; j++) {
            const DevProc& d = tb.procs[j];
            if (d.kind == PT_PROC_SB && (!c->hp.sb[d.slot].data || c->hp.sb[d.slot].ne < 2))
                return fail(c, PT_E_STATE, "species %d process %d: SB slot %d not uploaded", s, j, d.slot);
            if (d.kind == PT_PROC_PHOTOELECTRIC && c->hp.pe[d.slot].nshell < 1)
                return fail(c, PT_E_STATE, "species %d process %d: photoelectric slot %d not uploaded", s, j, d.slot);
        }
    }
    return PT_OK;
}

int pt_init(pt_ctx* c) {
    if (!c) return PT_E_ARG;
    HIPCHK(c, hipSetDevice(c->device));
    int rc = require_tables(c);
    if (rc) return rc;
    rc = sync_params(c);
    if (rc) return rc;
    if ((rc = read_counts(c))) return rc;
    for (int s = 0; s < PT_NSPECIES; s++) {
        if (!c->hp.tab[s].valid || c->hn[s] == 0) continue;
        hipLaunchKernelGGL(k_setr, dim3(c->grid), dim3(256), c->lds_bytes, c->stream, c->dp, s);
        HIPCHK(c, hipGetLastError());
    }
    HIPCHK(c, hipStreamSynchronize(c->stream));
    return PT_OK;
}

// ---- profiling spans: pairs of events on the context's stream, read lazily
enum { SPAN_ADV = 0, SPAN_TAIL = 1, SPAN_CMP = 2, SPAN_GRAPH = 3 };

static int drain_events(pt_ctx* c) {
    if (c->spans.empty()) return PT_OK;
    HIPCHK(c, hipEventSynchronize(c->spans.back().b));
    for (const Span& s : c->spans) {
        float a = 0;
        HIPCHK(c, hipEventElapsedTime(&a, s.a, s.b));
        if (s.kind == SPAN_ADV) {
            c->adv_ms += a;
            c->adv_launches++;
        } else if (s.kind == SPAN_TAIL) {
            c->tail_ms += a;
        } else if (s.kind == SPAN_CMP) {
            c->cmp_ms += a;
        } else {
            c->graph_ms += a;
        }
    }
    c->spans.clear();
    c->evq_used = 0;
    return PT_OK;
}

static int next_event(pt_ctx* c, hipEvent_t* e) {
    if (c->evq_used == c->evq.size()) {
        hipEvent_t ne;
        HIPCHK(c, hipEventCreate(&ne));
        c->evq.push_back(ne);
    }
    *e = c->evq[c->evq_used++];
    return PT_OK;
}

// record an event that opens (or, with `kind`, closes) a span
static int mark(pt_ctx* c, hipEvent_t* e) {
    int rc;
    if (c->evq_used + 2 > 4096 && (rc = drain_events(c))) return rc;
    if ((rc = next_event(c, e))) return rc;
    HIPCHK(c, hipEventRecord(*e, c->stream));
    return PT_OK;
}

// ---- launch shape
static int block_index(int bs) { return bs == 128 ? 0 : bs == 512 ? 2 : 1; }

static bool mlp_any(const pt_ctx* c) { return c->hp.mlp[0].on || c->hp.mlp[1].on; }

// a network in use whose kind the push/select passes of a collision round sample in place
// (not deferred to the sampling kernel): only then do those passes need the MLP variant
static bool mlp_in_rounds(const pt_ctx* c) {
    const uint32_t dm = c->launch.defer_mask;
    return (c->hp.mlp[LEARN_SB].on && !((dm >> PT_PROC_SB) & 1u)) ||
           (c->hp.mlp[LEARN_MOLLER].on && !((dm >> PT_PROC_MOLLER) & 1u));
}

// A workgroup of 256 threads has room for the largest tables; one of 512 may have none, and the
// kernel then runs with 256.  The runtime compares the dynamic LDS alone with a CU's: what
// passes that and does not fit with the static LDS faults in the launch, so that every launch
// beyond 256 threads goes by lds_fits.
static_assert(MAX_TABLE_BYTES + (256 / 64) * COOP_WAVE_BYTES + sizeof(Shared) + 1024 <= LDS_BYTES,
              "a workgroup of 256 threads takes every table that can be uploaded");
static int lds_fits(pt_ctx* c, const void* kernel, size_t dynamic, bool* fits) {
    hipFuncAttributes a;
    HIPCHK(c, hipFuncGetAttributes(&a, kernel));
    *fits = a.sharedSizeBytes + dynamic <= LDS_BYTES;
    return PT_OK;
}

// dynamic LDS of a kernel variant: the rate tables (and for the push/select kernels the
// per-wave RBEB job areas); the learned samplers' inference needs none
static size_t kernel_lds(const pt_ctx* c, int v, int bs) {
    if (v == KV_SAMPLE) return (size_t)c->lds_bytes;
    // the advance kernels: tables, then the per-wave RBEB job areas
    return (size_t)c->hp.lds_coop_off + (size_t)(bs / 64) * COOP_WAVE_BYTES;
}

// the one-workgroup passes over secondaries: plain, with walls, with learned samplers
static const void* tail_kernel(int q) {
    return q == 1 ? (const void*)k_tail<true, false> : q == 2 ? (const void*)k_tail<false, true>
                                                              : (const void*)k_tail<false, false>;
}
static size_t tail_lds(const pt_ctx* c, int bs) {
    return (size_t)c->hp.lds_coop_off + (size_t)(bs / 64) * COOP_WAVE_BYTES;
}

static int ensure_residency(pt_ctx* c) {
    const int key = 2 * c->lds_bytes + (mlp_any(c) ? 1 : 0);
    if (c->resident_lds == key) return PT_OK;
    const int bss[3] = {128, 256, 512};
    int rc;
    bool fits;
    for (int v = 0; v < NKV; v++)
        for (int bi = 0; bi < 3; bi++) {
            const void* f = kernel_of(v, bss[bi]);
            const size_t lds = kernel_lds(c, v, bss[bi]);
            int nb = 0;
            c->resident[v][bi] = 0;
            if ((rc = lds_fits(c, f, lds, &fits))) return rc;
            if (!fits) continue;
            HIPCHK(c, hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, f, bss[bi], lds));
            c->resident[v][bi] = std::max(nb, 1);
        }
    c->resident_wide = 0;
    if ((rc = lds_fits(c, kernel_of(KV_RANGE_FULL, WIDE), kernel_lds(c, KV_RANGE_FULL, WIDE), &fits))) return rc;
    if (fits &&
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&c->resident_wide, kernel_of(KV_RANGE_FULL, WIDE), WIDE,
                                                     kernel_lds(c, KV_RANGE_FULL, WIDE)) != hipSuccess) {
        (void)hipGetLastError();
        c->resident_wide = 0;
    }
    c->tail_block = 512;
    for (int q = 0; q < 3; q++) {
        if ((rc = lds_fits(c, tail_kernel(q), tail_lds(c, 512), &fits))) return rc;
        if (!fits) c->tail_block = 256;
    }
    c->resident_lds = key;
    return PT_OK;
}

// work and collision queues of the collision rounds (allocated on first use)
static int ensure_queues(pt_ctx* c) {
    if (c->queues) return PT_OK;
    Queues& Q = c->hp.q;
    for (int s = 0; s < PT_NSPECIES; s++) {
        const size_t cap = c->cfg.capacity[s];
        if (cap == 0) continue;
        for (int b = 0; b < 2; b++)
            if (!Q.work[s][b]) {
                int rc = dalloc(c, (void**)&Q.work[s][b], sizeof(uint32_t) * cap);
                if (rc) return rc;
            }
        for (int k = 0; k < Q.nkq[s]; k++)
            if (!Q.ev[s][k]) {
                int rc = dalloc(c, (void**)&Q.ev[s][k], sizeof(uint32_t) * cap);
                if (rc) return rc;
            }
    }
    c->queues = true;
    c->dirty = true;
    return sync_params(c);
}

// The shape of a history pass, by the numbers known last.
// SHAPE_WIDE: by electrons and positrons (see WIDE), unless the caller asked for small
// workgroups or the tables leave too little LDS.
// SHAPE_LONE: one wave per SIMD where that gives a lane at most one particle.  Such a launch
// is as long as its longest lane's chain of collisions, and a wave that shares its SIMD goes
// through that more slowly: 32 steps of n electrons took (two waves against one, ms)
// 1.78/1.62 for 2 x 10^4 and 1.90/1.78 for 6 x 10^4, one step a launch 1.20/1.00; 8 x 10^4
// electrons, with a second round for some lanes, 1.96/2.07.  Photons with few electrons are
// such a case too, as most photons only fly and what takes long are the chains of the
// electrons that a few set free.  From 4 photons per lane on (with 1.5, where their electrons
// crowd in half as many waves, 10 steps of 1 ns took 106/121 ms) to 16 whatever the step (16
// steps of 10^6 photons of 10 MeV: 0.76/0.68 of 1 ps, 2.4/2.3 of 10 ps, 38.1/38.1 of 100 ps, 8
// of 1 ns 867/821), and to 128 if a step has room for many collisions: where the photons mostly
// fly, the launch waits for memory and needs the waves.  Of 4 x 10^6 photons, 16 steps of 1 ps
// took 1.52/1.90, of 10 ps 3.6/3.8, of 100 ps 42.5/42.0, 8 of 300 ps 109/105, of 600 ps 403/364, of
// 1 ns 1033/942; of 8 x 10^6 2.5/3.5, 4.2/5.2, 45.6/45.0, 124/113, 437/391 and 1147/1025; of
// 1.6 x 10^7, beyond the line, 4.3/6.6, 6.5/9.3, 50.9/59.2, 138/130, 488/441 and 1262/1216; 3 steps of
// 10^8 114/164.  An electron collides 1.5 times a ps in air where its rate is lowest, so the
// line lies at 200 collisions a step, 130 ps.  (Photons of 100 keV, whose electrons stop
// early, gain less: 8 steps of 1 ns took 52.9/48.2 for 10^6, 64.1/65.0 for 4 x 10^6, 76/87 for
// 8 x 10^6.)
// Not in captured runs (`full`), which may grow without the host knowing, and not where the
// caller asked for workgroups of 512 threads, which are two waves per SIMD each.
enum { SHAPE_FULL = 0, SHAPE_WIDE = 1, SHAPE_LONE = 2 };
constexpr double BEAM_COLLISIONS = 200.0;
static int pass_shape(const pt_ctx* c, bool full, int steps = 0, double dt = 0.0) {
    const ull electrons = c->hn[PT_ELECTRON] + c->hn[PT_POSITRON];
    const ull line = (!full && steps == 1 ? WIDE_PER_LANE_2 : 2 * WIDE_PER_LANE) * WIDE * c->ncu / 2;
    if (c->launch.block >= 256 && c->resident_wide > 0 && electrons >= line) return SHAPE_WIDE;
    if (full || c->launch.grid_mult != 1 || c->launch.block > 256) return SHAPE_FULL;
    const ull lanes = 256ull * c->ncu, photons = c->hn[PT_PHOTON];
    const ull most = dt * c->lowest_rate >= BEAM_COLLISIONS ? 128 * lanes : 16 * lanes;
    const bool beam = photons >= 4 * lanes && photons <= most && electrons <= std::min(photons / 8, 4 * lanes);
    return beam || electrons + photons <= lanes ? SHAPE_LONE : SHAPE_FULL;
}

// full: launch every resident workgroup x grid_mult (captured runs and queue rounds, whose
// sizes the host does not know); otherwise at most what the last known population needs
static int launch_kernel_args(pt_ctx* c, int v, bool full, int steps = 0, double dt = 0.0) {
    void* args[] = {(void*)&c->dp};
    const int shape = v == KV_RANGE_FULL ? pass_shape(c, full, steps, dt) : SHAPE_FULL;
    const int asked = c->launch.block == 512 && !c->resident[v][block_index(512)] ? 256 : c->launch.block;
    const int bs = shape == SHAPE_WIDE ? WIDE : asked;
    const int per_cu = shape == SHAPE_WIDE ? c->resident_wide : c->resident[v][block_index(bs)];
    ull blocks = (ull)per_cu * c->ncu * std::max(1, c->launch.grid_mult);
    if (shape == SHAPE_LONE) blocks = std::min<ull>(blocks, (ull)c->ncu * (256 / bs));
    if (!full) {
        ull est = c->hn[0] + c->hn[1] + c->hn[2];
        blocks = std::min<ull>(blocks, std::max<ull>((ull)c->ncu, est / (ull)(bs / 64)));
    }
    if (steps > 0) {
        c->main_block = bs;
        c->main_grid = (int)std::max<ull>(blocks, 1);
    }
    HIPCHK(c, hipLaunchKernel(kernel_of(v, bs), dim3((unsigned)std::max<ull>(blocks, 1)), dim3(bs), args,
                              kernel_lds(c, v, bs), c->stream));
    return PT_OK;
}

// secondaries the waves' stacks could not take: whole-grid passes, then one workgroup for
// whatever the last pass created
static int launch_tail(pt_ctx* c) {
    int rc;
    const bool wall = c->hp.wall.on != 0, mlp = mlp_any(c);
    const int in_place = wall ? KV_RANGE_WALL : with_mlp(KV_RANGE_FULL, mlp);
    for (int q = 0; q < c->launch.tail_passes; q++)
        if ((rc = launch_kernel_args(c, in_place, true))) return rc;
    int passes = 100000;
    void* args[] = {(void*)&c->dp, (void*)&passes};
    HIPCHK(c, hipLaunchKernel(tail_kernel(wall ? 1 : mlp ? 2 : 0), dim3(1), dim3(c->tail_block), args,
                              tail_lds(c, c->tail_block), c->stream));
    return PT_OK;
}

// one step.  clocked: tfinal and the step index come from the device clock (captured
// runs); otherwise they are given and the host counts steps.
static int launch_step(pt_ctx* c, bool clocked, double tfinal, double dt, int nsub, bool tail = true) {
    c->counts_known = false;
    int rc = ensure_residency(c);
    if (rc) return rc;
    const int R = c->launch.rounds;
    const bool wall = c->hp.wall.on != 0;
    // learned samplers in use: every kernel that samples collisions in place evaluates them
    const bool mlp = mlp_any(c);
    if (wall && R > 0) return fail(c, PT_E_STATE, "a wall needs collision rounds = 0");
    if (wall && mlp) return fail(c, PT_E_STATE, "a wall needs the learned samplers off");
    if (R > 0 && (rc = ensure_queues(c))) return rc;
    hipLaunchKernelGGL(k_snapshot, dim3(1), dim3(64), 0, c->stream, c->dp, clocked ? 1 : 0, tfinal, dt, c->step,
                       nsub);
    HIPCHK(c, hipGetLastError());
    hipEvent_t e0 = nullptr, e1 = nullptr, e2 = nullptr;
    const bool prof = c->profile && !clocked;
    if (prof && (rc = mark(c, &e0))) return rc;
    const int in_place = wall ? KV_RANGE_WALL : with_mlp(KV_RANGE_FULL, mlp);
    if (R == 0) {
        if ((rc = launch_kernel_args(c, in_place, clocked, nsub, dt))) return rc;
    } else {
        const bool mlp_ev = mlp_in_rounds(c);
        if ((rc = launch_kernel_args(c, with_mlp(KV_RANGE_EVENT, mlp_ev), clocked))) return rc;
        for (int r = 1; r <= R; r++) {
            if ((rc = launch_kernel_args(c, KV_SAMPLE, true))) return rc;
            hipLaunchKernelGGL(k_rotate, dim3(1), dim3(64), 0, c->stream, c->dp);
            HIPCHK(c, hipGetLastError());
            if (r < R && (rc = launch_kernel_args(c, with_mlp(KV_QUEUE_EVENT, mlp_ev), true))) return rc;
        }
        if ((rc = launch_kernel_args(c, with_mlp(KV_QUEUE_FULL, mlp), true))) return rc;
    }
    if (prof && (rc = mark(c, &e1))) return rc;
    if (tail && (rc = launch_tail(c))) return rc;
    if (prof) {
        if ((rc = mark(c, &e2))) return rc;
        c->spans.push_back(Span{e0, e1, SPAN_ADV});
        c->spans.push_back(Span{e1, e2, SPAN_TAIL});
    }
    if (clocked) {
        hipLaunchKernelGGL(k_tick, dim3(1), dim3(64), 0, c->stream, c->dp);
        HIPCHK(c, hipGetLastError());
    } else {
        c->step += (uint32_t)nsub;
        c->last_t = tfinal + (nsub - 1) * dt;
    }
    return PT_OK;
}

// steps that one launch may advance: collision rounds queue particles between kernels and
// take one step at a time
static int steps_per_launch(const pt_ctx* c) { return c->launch.rounds > 0 ? 1 : MAX_SUB; }

// the flags that have been reported (read_state, or the end of a pass)
static int check_flags(pt_ctx* c, int64_t* out) {
    const ull* f = c->report->flags;
    if (out)
        for (int q = 0; q < NFLAGS; q++) out[q] = (int64_t)f[q];
    if (f[FLAG_CAPACITY]) return fail(c, PT_E_CAPACITY, "%llu particles did not fit in their population", f[FLAG_CAPACITY]);
    if (f[FLAG_SAMPLER]) return fail(c, PT_E_SAMPLER, "%llu sampler domain failures", f[FLAG_SAMPLER]);
    if (f[FLAG_RANGE]) return fail(c, PT_E_TABLE_RANGE, "%llu energies above the table range", f[FLAG_RANGE]);
    if (f[FLAG_TAIL]) return fail(c, PT_E_STATE, "secondary passes did not finish within the pass limit");
    if (f[FLAG_RATEBOUND]) return fail(c, PT_E_RATEBOUND, "rate bound underestimated %llu times: increase safety factor", f[FLAG_RATEBOUND]);
    return PT_OK;
}

int pt_check(pt_ctx* c, int64_t* flags) {
    if (!c) return PT_E_ARG;
    HIPCHK(c, hipSetDevice(c->device));
    int rc = read_state(c);
    if (rc) return rc;
    return check_flags(c, flags);
}

int pt_advance(pt_ctx* c, double tfinal) {
    if (!c) return PT_E_ARG;
    HIPCHK(c, hipSetDevice(c->device));
    int rc = require_tables(c);
    if (rc) return rc;
    rc = sync_params(c);
    if (rc) return rc;
    // the main pass reports counts, flags and whether it left secondaries to further passes:
    // only then are those launched
    rc = launch_step(c, false, tfinal, tfinal - c->last_t, 1, false);
    if (rc) return rc;
    HIPCHK(c, hipStreamSynchronize(c->stream));
    if (c->report->left) {
        if ((rc = launch_tail(c))) return rc;
        if ((rc = read_state(c))) return rc;
    } else {
        take_counts(c);
    }
    return check_flags(c, nullptr);
}

// compaction of a species (-1: of all), entirely on the device, so that it can be captured
static int compact_all(pt_ctx* c, int sp, bool timed, bool one = false) {
    hipEvent_t a = nullptr, b = nullptr;
    int rc;
    unsigned mask = 0;
    for (int s = 0; s < PT_NSPECIES; s++)
        if ((sp < 0 || s == sp) && c->cfg.capacity[s] > 0) mask |= 1u << s;
    c->counts_known = false;
    if (timed && (rc = mark(c, &a))) return rc;
    if (mask) {
        const dim3 grid(one ? 1 : c->cmp_blocks, PT_NSPECIES);
        hipLaunchKernelGGL(k_cmp_count, grid, dim3(256), 0, c->stream, c->cmp, mask);
        HIPCHK(c, hipGetLastError());
    }
    if (mask && !one) {
        const dim3 grid(c->cmp_blocks, PT_NSPECIES);
        hipLaunchKernelGGL(k_cmp_fill, grid, dim3(256), 0, c->stream, c->cmp, mask);
        HIPCHK(c, hipGetLastError());
        hipLaunchKernelGGL(k_cmp_move, grid, dim3(256), 0, c->stream, c->cmp, mask);
        HIPCHK(c, hipGetLastError());
    }
    if (timed) {
        if ((rc = mark(c, &b))) return rc;
        c->spans.push_back(Span{a, b, SPAN_CMP});
    }
    return PT_OK;
}

int pt_compact(pt_ctx* c, int sp) {
    if (!c) return PT_E_ARG;
    if (sp < -1 || sp >= PT_NSPECIES) return fail(c, PT_E_ARG, "bad species");
    HIPCHK(c, hipSetDevice(c->device));
    // counts known and small: one launch does it all (k_cmp_count)
    bool one = c->counts_known;
    for (int s = 0; s < PT_NSPECIES; s++) one = one && c->hn[s] <= (ull)CMP_SMALL * CH;
    int rc;
    if ((rc = read_counts(c))) return rc;
    if ((rc = compact_all(c, sp, c->profile, one))) return rc;
    HIPCHK(c, hipStreamSynchronize(c->stream));
    // (of a species left out the count is as before)
    for (int s = 0; s < PT_NSPECIES; s++)
        if (sp >= 0 && s != sp) c->report->n[s] = c->hn[s];
    take_counts(c);
    return PT_OK;
}

// Steps [q, end) of a run from time t, in launches of up to steps_per_launch steps, with a
// compaction after the steps `every` divides (0: never).  `late`: compaction may wait until
// the last of those steps; before it, it runs once per launch.
static int run_steps(pt_ctx* c, double& t, double dt, int q, int end, int every, bool late) {
    const int last = every > 0 ? end - end % every : 0;  // the last compaction of the range
    int rc;
    while (q < end) {
        int k = std::min(end - q, steps_per_launch(c));
        if (every > 0 && late) k = q < last ? std::min(k, last - q) : k;
        else if (every > 0) k = std::min(k, every - q % every);
        if ((rc = launch_step(c, false, t + dt, dt, k))) return rc;
        for (int i = 0; i < k; i++) t += dt;
        q += k;
        if (every > 0 && (late ? q <= last : q % every == 0) && (rc = compact_all(c, -1, c->profile))) return rc;
    }
    return PT_OK;
}

// The state (particles, counters, tallies) copied aside, or back.
constexpr ull SAVE_MAX = 1ull << 21;  // particles of all species: their 93 bytes make 195 MB
static int save_state(pt_ctx* c, const ull n[PT_NSPECIES], bool back) {
    Copies cp{};
    void* live[MAX_COPIES];
    size_t at[MAX_COPIES], off = 0;  // places in the copy, 16-byte aligned
    auto add = [&](void* p, size_t bytes) {
        if (!bytes) return;
        live[cp.n] = p;
        at[cp.n] = off;
        cp.bytes[cp.n++] = bytes;
        off += (bytes + 15) & ~(size_t)15;
    };
    ull all = 0;
    for (int s = 0; s < PT_NSPECIES; s++) {
        const SpeciesDev& S = c->hp.sp[s];
        all += n[s];
        add(S.f[0], sizeof(double) * PT_NFIELDS * n[s]);
        add(S.active, n[s]);
        add(S.uid, sizeof(uint64_t) * n[s]);
        add(S.swarm, sizeof(int32_t) * n[s]);
    }
    add(c->dn, sizeof(ull) * PT_NSPECIES);
    add(c->dcounts, sizeof(ull) * PT_NSPECIES * NCOUNT);
    add(c->dflags, sizeof(ull) * NFLAGS);
    add(c->dwork, sizeof(ull) * NWORK);
    add(c->dtally, sizeof(double) * PT_NSPECIES * (c->hp.tally_bins + 2));
    add(c->ddose, sizeof(double) * (c->hp.dose_bins + 3));
    if (c->saved_bytes < off) {
        // room for half as many particles again, within the bound
        const size_t room = off + 93 * (size_t)std::min<ull>(std::max<ull>(all / 2, 4096), SAVE_MAX - all);
        if (c->saved) {
            HIPCHK(c, hipFree(c->saved));
            c->saved = nullptr;
            c->saved_bytes = 0;
        }
        if (dev_malloc(c, (void**)&c->saved, room) != hipSuccess)
            return fail(c, PT_E_NOMEM, "no room for a copy of %zu bytes", room);
        c->saved_bytes = room;
    }
    for (int q = 0; q < cp.n; q++) {
        cp.dst[q] = back ? live[q] : c->saved + at[q];
        cp.src[q] = back ? c->saved + at[q] : live[q];
    }
    hipLaunchKernelGGL(k_copy_ranges, dim3(c->grid), dim3(256), 0, c->stream, cp);
    HIPCHK(c, hipGetLastError());
    return PT_OK;
}

// Steps [q, end) of a run up to its next check.  Compaction never changes a particle, only
// which slots are free, so a run that asks for it more often than a launch has steps
// (compact_every 1 is the reference's droplow! of each step) can have it once per launch, unless
// a population reaches its capacity because of the slots that are not free yet.  The state is
// therefore copied aside first (a few us for the populations that gain by it, up to SAVE_MAX
// particles that fill no more than half their slots); if anything did not fit, the window is
// taken back and run with the compactions it asked for, so that it fails only where it did.
// 200 steps of 10^4 electrons with compaction in each: 33.8 -> 10.6 ms.
static int run_window(pt_ctx* c, double& t, double dt, int q, int end, int every) {
    const ull all = c->hn[0] + c->hn[1] + c->hn[2];
    bool late = every > 0 && every < steps_per_launch(c) && end - end % every > q + every && !c->hp.wall.on &&
                all <= SAVE_MAX;
    for (int s = 0; s < PT_NSPECIES; s++) late = late && 2 * c->hn[s] <= c->cfg.capacity[s];
    int rc;
    ull n[PT_NSPECIES] = {c->hn[0], c->hn[1], c->hn[2]};
    if (late && save_state(c, n, false) != PT_OK) late = false;  // no room for the copy
    if (late) c->late_windows++;
    c->saved_live = late;
    struct Release {
        bool& live;
        ~Release() { live = false; }
    } release{c->saved_live};
    const double t1 = t;
    const uint32_t step1 = c->step;
    if ((rc = run_steps(c, t, dt, q, end, every, late))) return rc;
    if ((rc = read_state(c))) return rc;
    if (!late) return check_flags(c, nullptr);
    rc = check_flags(c, nullptr);
    if (rc != PT_E_CAPACITY) return rc;
    if ((rc = save_state(c, n, true))) return rc;
    c->windows_back++;
    t = t1;
    c->step = step1;
    if ((rc = run_steps(c, t, dt, q, end, every, false))) return rc;
    if ((rc = read_state(c))) return rc;
    return check_flags(c, nullptr);
}

int pt_run(pt_ctx* c, double t0, double dt, int nsteps, int compact_every, int check_every) {
    if (!c) return PT_E_ARG;
    HIPCHK(c, hipSetDevice(c->device));
    int rc = require_tables(c);
    if (rc) return rc;
    rc = sync_params(c);
    if (rc) return rc;
    if (check_every < 1) check_every = 1;
    double t = t0;
    for (int q = 0; q < nsteps;) {
        const int end = std::min(nsteps, q + check_every - q % check_every);
        if (!c->counts_known && (rc = read_counts(c))) return rc;
        if ((rc = run_window(c, t, dt, q, end, compact_every))) return rc;
        q = end;
    }
    return PT_OK;
}

static int apply_launch(pt_ctx* c, const pt_launch& l) {
    c->launch = l;
    if (c->hp.defer_mask != l.defer_mask) {
        c->hp.defer_mask = l.defer_mask;
        c->dirty = true;
    }
    return sync_params(c);
}

int pt_set_launch(pt_ctx* c, const pt_launch* l) {
    if (!c) return PT_E_ARG;
    if (!l || (l->block != 128 && l->block != 256 && l->block != 512) || l->grid_mult < 1 ||
        l->grid_mult > 16 || l->compact_every < 1 || l->rounds < 0 || l->rounds > 8 || l->tail_passes < 0 ||
        l->tail_passes > 16)
        return fail(c, PT_E_ARG,
                    "launch: block must be 128, 256 or 512, grid_mult in 1..16, compact_every >= 1, rounds in 0..8, "
                    "tail_passes in 0..16");
    return apply_launch(c, *l);
}

int pt_get_launch(pt_ctx* c, pt_launch* l) {
    if (!c || !l) return PT_E_ARG;
    *l = c->launch;
    return PT_OK;
}

static bool same_launch(const pt_launch& a, const pt_launch& b) {
    return a.block == b.block && a.grid_mult == b.grid_mult && a.compact_every == b.compact_every &&
           a.rounds == b.rounds && a.defer_mask == b.defer_mask && a.tail_passes == b.tail_passes;
}

// capture `steps` clocked steps (+ one compaction of every species if `compact`)
static int capture(pt_ctx* c, int which, int steps, bool compact) {
    if (c->gexec[which]) {
        HIPCHK(c, hipGraphExecDestroy(c->gexec[which]));
        c->gexec[which] = nullptr;
    }
    int rc = ensure_residency(c);
    if (rc) return rc;
    if (c->launch.rounds > 0 && (rc = ensure_queues(c))) return rc;
    if ((rc = ensure_residency(c))) return rc;
    HIPCHK(c, hipStreamBeginCapture(c->stream, hipStreamCaptureModeThreadLocal));
    int lrc = PT_OK;
    for (int q = 0; q < steps && lrc == PT_OK;) {
        const int k = std::min(steps - q, steps_per_launch(c));
        lrc = launch_step(c, true, 0.0, 0.0, k);
        q += k;
    }
    if (lrc == PT_OK && compact) lrc = compact_all(c, -1, false);
    hipGraph_t g = nullptr;
    hipError_t e = hipStreamEndCapture(c->stream, &g);
    if (lrc) {
        if (g) (void)hipGraphDestroy(g);
        return lrc;
    }
    if (e != hipSuccess) return fail(c, PT_E_HIP, "hipStreamEndCapture failed: %s", hipGetErrorString(e));
    e = hipGraphInstantiate(&c->gexec[which], g, nullptr, nullptr, 0);
    (void)hipGraphDestroy(g);
    if (e != hipSuccess) return fail(c, PT_E_HIP, "hipGraphInstantiate failed: %s", hipGetErrorString(e));
    c->gsteps[which] = steps;
    c->glaunch[which] = c->launch;
    c->glds[which] = 4 * c->lds_bytes + (mlp_any(c) ? 1 : 0) + 2 * pass_shape(c, true);
    c->ggen[which] = c->params_gen;
    return PT_OK;
}

// a captured graph of `steps` steps that still matches the context: same launch, same LDS
// layout and no parameter upload since its capture
static bool graph_current(const pt_ctx* c, int which, int steps) {
    return c->gexec[which] && c->gsteps[which] == steps && same_launch(c->glaunch[which], c->launch) &&
           c->glds[which] == 4 * c->lds_bytes + (mlp_any(c) ? 1 : 0) + 2 * pass_shape(c, true) &&
           c->ggen[which] == c->params_gen;
}

static int replay(pt_ctx* c, int which) {
    hipEvent_t a = nullptr, b = nullptr;
    int rc;
    if (c->profile && (rc = mark(c, &a))) return rc;
    HIPCHK(c, hipGraphLaunch(c->gexec[which], c->stream));
    if (c->profile) {
        if ((rc = mark(c, &b))) return rc;
        c->spans.push_back(Span{a, b, SPAN_GRAPH});
    }
    return PT_OK;
}

int pt_run_graph(pt_ctx* c, double t0, double dt, int nsteps, int check_every) {
    if (!c) return PT_E_ARG;
    if (nsteps < 0) return fail(c, PT_E_ARG, "nsteps < 0");
    HIPCHK(c, hipSetDevice(c->device));
    int rc = require_tables(c);
    if (rc) return rc;
    if (c->hp.wall.on && c->launch.rounds > 0) return fail(c, PT_E_STATE, "a wall needs collision rounds = 0");
    if (c->hp.wall.on && mlp_any(c)) return fail(c, PT_E_STATE, "a wall needs the learned samplers off");
    // the queues of collision rounds (a table upload may have added sampler kinds) are in
    // place and their pointers uploaded before any graph is replayed or captured
    if (c->launch.rounds > 0 && (rc = ensure_queues(c))) return rc;
    rc = sync_params(c);
    if (rc) return rc;
    if (check_every < 1) check_every = 1;
    const int ce = c->launch.compact_every;
    const int full = nsteps / ce, rem = nsteps % ce;
    if (full > 0 && !graph_current(c, 0, ce)) {
        if ((rc = capture(c, 0, ce, true))) return rc;
    }
    if (rem > 0 && !graph_current(c, 1, rem)) {
        if ((rc = capture(c, 1, rem, false))) return rc;
    }
    Clock ck{};
    ck.t = t0;
    ck.dt = dt;
    ck.tfinal = t0;
    ck.step = c->step;
    HIPCHK(c, hipMemcpyAsync(c->dclock, &ck, sizeof(Clock), hipMemcpyHostToDevice, c->stream));
    c->counts_known = false;
    int done = 0, since = 0;
    for (int k = 0; k < full; k++) {
        if ((rc = replay(c, 0))) return rc;
        done += ce;
        since += ce;
        if (since >= check_every && done < nsteps) {
            since = 0;
            if ((rc = read_state(c))) return rc;
            if ((rc = check_flags(c, nullptr))) {
                c->step += (uint32_t)done;
                return rc;
            }
            // (the population may have come to need the other shape)
            if (k + 1 < full && !graph_current(c, 0, ce) && (rc = capture(c, 0, ce, true))) {
                c->step += (uint32_t)done;
                return rc;
            }
        }
    }
    if (rem > 0 && (rc = replay(c, 1))) return rc;
    c->step += (uint32_t)nsteps;
    if ((rc = read_state(c))) return rc;
    return check_flags(c, nullptr);
}

// particle-steps done so far (device work counter)
static int psteps_now(pt_ctx* c, ull* v) {
    ull w[NWORK];
    HIPCHK(c, hipMemcpyAsync(w, c->dwork, sizeof(w), hipMemcpyDeviceToHost, c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    *v = w[W_PSTEPS];
    return PT_OK;
}

int pt_autotune(pt_ctx* c, double t0, double dt, int trial_steps, pt_tune_trial* trials, int max_trials,
                int* ntrials, pt_launch* best, double* t_end) {
    if (!c) return PT_E_ARG;
    if (trial_steps < 1) return fail(c, PT_E_ARG, "trial_steps must be >= 1");
    HIPCHK(c, hipSetDevice(c->device));
    int rc = require_tables(c);
    if (rc) return rc;
    if ((rc = sync_params(c))) return rc;
    const bool prof = c->profile;
    c->profile = false;
    double t = t0;
    int nt = 0;
    hipEvent_t a = c->ev[0], b = c->ev[1];
    // one timed window: `steps` steps from t with compaction every `ce` (0: none)
    auto window = [&](int steps, int ce, double* rate) -> int {
        int r2;
        if ((r2 = compact_all(c, -1, false))) return r2;
        if ((r2 = read_counts(c))) return r2;
        ull p0, p1;
        if ((r2 = psteps_now(c, &p0))) return r2;
        HIPCHK(c, hipEventRecord(a, c->stream));
        for (int q = 0; q < steps;) {
            int k = std::min(steps - q, steps_per_launch(c));
            if (ce > 0) k = std::min(k, ce - q % ce);
            if ((r2 = launch_step(c, false, t + dt, dt, k))) return r2;
            for (int i = 0; i < k; i++) t += dt;
            q += k;
            if (ce > 0 && q % ce == 0 && (r2 = compact_all(c, -1, false))) return r2;
        }
        HIPCHK(c, hipEventRecord(b, c->stream));
        HIPCHK(c, hipEventSynchronize(b));
        float ms = 0;
        HIPCHK(c, hipEventElapsedTime(&ms, a, b));
        if ((r2 = psteps_now(c, &p1))) return r2;
        if ((r2 = read_state(c))) return r2;
        if ((r2 = check_flags(c, nullptr))) return r2;
        *rate = ms > 0 ? (double)(p1 - p0) / (ms * 1e-3) : 0.0;
        return PT_OK;
    };
    pt_launch keep = c->launch, top = c->launch;
    // collision rounds, with the current shape
    {
        const int rounds[4] = {0, 2, 3, 4};
        double best_rate = -1.0;
        for (int k = 0; k < 4 && rc == PT_OK; k++) {
            c->launch.rounds = rounds[k];
            double r = 0;
            rc = window(trial_steps, 0, &r);
            if (rc) break;
            if (trials && nt < max_trials) trials[nt] = pt_tune_trial{c->launch, r};
            nt++;
            if (r > best_rate) {
                best_rate = r;
                top = c->launch;
            }
        }
        c->launch = top;
    }
    // (a block that leads to the launches of a smaller one, as 512 does to those of 256 for a
    // large population, is not chosen over it: what differs is noise)
    double top_rate = -1.0;
    const int blocks[3] = {128, 256, 512}, mults[3] = {1, 2, 4};
    std::vector<std::pair<int, int>> shapes;
    for (int bi = 0; bi < 3 && rc == PT_OK; bi++)
        for (int mi = 0; mi < 3 && rc == PT_OK; mi++) {
            c->launch.block = blocks[bi];
            c->launch.grid_mult = mults[mi];
            double r = 0;
            rc = window(trial_steps, 0, &r);
            if (rc) break;
            if (trials && nt < max_trials) trials[nt] = pt_tune_trial{c->launch, r};
            nt++;
            const std::pair<int, int> shape{c->main_block, c->main_grid};
            const bool seen = c->launch.rounds == 0 && std::find(shapes.begin(), shapes.end(), shape) != shapes.end();
            shapes.push_back(shape);
            if (r > top_rate && !seen) {
                top_rate = r;
                top = c->launch;
            }
        }
    if (rc == PT_OK) {
        c->launch = top;
        const int cad[5] = {1, 2, 4, 8, 16};
        double best_rate = -1.0;
        for (int k = 0; k < 5 && rc == PT_OK; k++) {
            double r = 0;
            rc = window(16, cad[k], &r);
            if (rc) break;
            pt_launch l = top;
            l.compact_every = cad[k];
            if (trials && nt < max_trials) trials[nt] = pt_tune_trial{l, r};
            nt++;
            if (r > best_rate) {
                best_rate = r;
                top.compact_every = cad[k];
            }
        }
    }
    c->profile = prof;
    if (rc) {
        c->launch = keep;
        if (t_end) *t_end = t;
        if (ntrials) *ntrials = nt;
        return rc;
    }
    c->launch = top;
    if (best) *best = top;
    if (t_end) *t_end = t;
    if (ntrials) *ntrials = nt;
    return read_counts(c);
}

int pt_stats(pt_ctx* c, int sp, pt_pop_stats* out) {
    if (!c) return PT_E_ARG;
    if (sp < 0 || sp >= PT_NSPECIES || !out) return fail(c, PT_E_ARG, "bad arguments");
    HIPCHK(c, hipSetDevice(c->device));
    int rc = sync_params(c);
    if (rc) return rc;
    rc = read_counts(c);
    if (rc) return rc;
    const int blocks = (int)std::min<ull>(STAT_BLOCKS, std::max<ull>(1, (c->hn[sp] + 511) / 512));
    hipLaunchKernelGGL(k_stats, dim3(blocks), dim3(256), 0, c->stream, c->dp, sp, c->stat_part,
                       (ull*)(c->stat_part + NSTAT * STAT_BLOCKS));
    HIPCHK(c, hipGetLastError());
    HIPCHK(c, hipStreamSynchronize(c->stream));
    const double* a = c->report->stat;
    out->n = c->hn[sp];
    out->nactive = (uint64_t)a[0];
    out->weight = a[1];
    out->mean_energy = a[1] > 0 ? a[2] / a[1] : 0.0;
    for (int d = 0; d < 3; d++) out->centroid[d] = a[1] > 0 ? a[3 + d] / a[1] : 0.0;
    double xm2 = (out->centroid[0] * out->centroid[0] + out->centroid[1] * out->centroid[1]) +
                 out->centroid[2] * out->centroid[2];
    out->spread = a[1] > 0 ? std::sqrt(std::fabs(a[6] / a[1] - xm2)) : 0.0;
    out->max_energy = a[7];
    return PT_OK;
}

int pt_swarm_stats(pt_ctx* c, int sp, int nswarm, double* out) {
    if (!c) return PT_E_ARG;
    if (sp < 0 || sp >= PT_NSPECIES || !out || nswarm < 1 || nswarm > c->cfg.nswarm)
        return fail(c, PT_E_ARG, "bad arguments (nswarm must be in 1..%d)", c->cfg.nswarm);
    HIPCHK(c, hipSetDevice(c->device));
    int rc = sync_params(c);
    if (rc) return rc;
    const size_t bytes = sizeof(double) * 4 * (size_t)c->cfg.nswarm;
    const int most = c->cfg.nswarm <= SWARM_LDS ? SWARM_COPIES : 1;
    if (!c->swarm_part) {
        if ((rc = dalloc(c, (void**)&c->swarm_part, most * bytes))) return rc;
        HIPCHK(c, hipMemsetAsync(c->swarm_part, 0, most * bytes, c->stream));
    }
    rc = read_counts(c);
    if (rc) return rc;
    int blocks = (int)std::min<ull>(2 * c->ncu, std::max<ull>(1, (c->hn[sp] + 255) / 256));
    const int copies = blocks >= 16 * most ? most : 1;
    hipLaunchKernelGGL(k_swarm_stats, dim3(blocks), dim3(256), 0, c->stream, c->dp, sp, nswarm, c->swarm_part, copies,
                       c->swarm_host, (ull*)(c->stat_part + NSTAT * STAT_BLOCKS));
    HIPCHK(c, hipGetLastError());
    HIPCHK(c, hipStreamSynchronize(c->stream));
    memcpy(out, c->swarm_host, sizeof(double) * 4 * (size_t)nswarm);
    return PT_OK;
}

int pt_swarm_stats_noalloc(pt_ctx* c, int sp, int nswarm, double* out) {
    if (!c) return PT_E_ARG;
    if (sp < 0 || sp >= PT_NSPECIES || !out || nswarm < 1 || nswarm > c->cfg.nswarm)
        return fail(c, PT_E_ARG, "bad arguments (nswarm must be in 1..%d)", c->cfg.nswarm);
    if (nswarm > NOALLOC_SWARMS)
        return fail(c, PT_E_ARG, "pt_swarm_stats_noalloc: %d swarms exceed its maximum of %d", nswarm, NOALLOC_SWARMS);
    if (!c->noalloc) return fail(c, PT_E_STATE, "no scratch array on device %d", c->device);
    HIPCHK(c, hipSetDevice(c->device));
    int rc = sync_params(c);
    if (rc) return rc;
    if ((rc = read_counts(c))) return rc;
    // the array keeps the last call's sums: clear this call's part with a kernel
    const int n4 = 4 * nswarm;
    hipLaunchKernelGGL(k_zero_doubles, dim3((n4 + 255) / 256), dim3(256), 0, c->stream, c->noalloc, n4);
    HIPCHK(c, hipGetLastError());
    int blocks = (int)std::min<ull>(2 * c->ncu, std::max<ull>(1, (c->hn[sp] + 255) / 256));
    hipLaunchKernelGGL(k_swarm_stats, dim3(blocks), dim3(256), 0, c->stream, c->dp, sp, nswarm, c->noalloc, 1,
                       (double*)nullptr, (ull*)nullptr);
    HIPCHK(c, hipGetLastError());
    HIPCHK(c, hipMemcpyAsync(out, c->noalloc, sizeof(double) * (size_t)n4, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    return PT_OK;
}

int pt_collision_counts(pt_ctx* c, int sp, int64_t* out, int nmax, int reset) {
    if (!c) return PT_E_ARG;
    if (sp < 0 || sp >= PT_NSPECIES || !out || nmax < 1) return fail(c, PT_E_ARG, "bad arguments");
    HIPCHK(c, hipSetDevice(c->device));
    ull h[NCOUNT];
    HIPCHK(c, hipMemcpyAsync(h, c->dcounts + sp * NCOUNT, sizeof(h), hipMemcpyDeviceToHost, c->stream));
    if (reset) HIPCHK(c, hipMemsetAsync(c->dcounts + sp * NCOUNT, 0, sizeof(h), c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    for (int q = 0; q < std::min(nmax, NCOUNT); q++) out[q] = (int64_t)h[q];
    return PT_OK;
}

int pt_dose_read(pt_ctx* c, double* hist, int nbins, double* under, double* over, double* total, int reset) {
    if (!c) return PT_E_ARG;
    HIPCHK(c, hipSetDevice(c->device));
    const int b = c->hp.dose_bins;
    std::vector<double> h(b + 3);
    HIPCHK(c, hipMemcpyAsync(h.data(), c->ddose, sizeof(double) * (b + 3), hipMemcpyDeviceToHost, c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    if (hist)
        for (int q = 0; q < std::min(b, nbins); q++) hist[q] = h[q];
    if (under) *under = h[b];
    if (over) *over = h[b + 1];
    if (total) {
        double sum = 0.0;
        for (int q = 0; q < b + 2; q++) sum += h[q];
        *total = sum;
    }
    if (reset) {
        HIPCHK(c, hipMemsetAsync(c->ddose, 0, sizeof(double) * (b + 3), c->stream));
        HIPCHK(c, hipStreamSynchronize(c->stream));
    }
    return PT_OK;
}

int pt_tally_read(pt_ctx* c, int sp, double* hist, int nbins, double* count, double* weight) {
    if (!c) return PT_E_ARG;
    if (sp < 0 || sp >= PT_NSPECIES) return fail(c, PT_E_ARG, "bad species");
    HIPCHK(c, hipSetDevice(c->device));
    int b = c->hp.tally_bins;
    std::vector<double> h(b + 2);
    HIPCHK(c, hipMemcpyAsync(h.data(), c->dtally + (size_t)sp * (b + 2), sizeof(double) * (b + 2), hipMemcpyDeviceToHost, c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    if (hist)
        for (int q = 0; q < std::min(b, nbins); q++) hist[q] = h[q];
    if (count) *count = h[b];
    if (weight) *weight = h[b + 1];
    return PT_OK;
}

int pt_work_read(pt_ctx* c, pt_work* out, int reset) {
    if (!c) return PT_E_ARG;
    if (!out) return fail(c, PT_E_ARG, "null output");
    HIPCHK(c, hipSetDevice(c->device));
    int rc = drain_events(c);
    if (rc) return rc;
    ull w[NWORK];
    HIPCHK(c, hipMemcpyAsync(w, c->dwork, sizeof(w), hipMemcpyDeviceToHost, c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    memset(out, 0, sizeof(*out));
    out->particle_steps = w[W_PSTEPS];
    out->secondaries = w[W_SECONDARIES];
    out->moved = w[W_MOVED];
    out->events = w[W_EVENTS];
    out->tail_particles = w[W_TAIL];
    out->steps = c->step;
    out->advance_ms = c->adv_ms;
    out->advance_launches = c->adv_launches;
    out->tail_ms = c->tail_ms;
    out->compact_ms = c->cmp_ms;
    out->main_secondaries = w[W_MAIN_SEC];
    out->graph_ms = c->graph_ms;
    if (reset) {
        HIPCHK(c, hipMemsetAsync(c->dwork, 0, sizeof(w), c->stream));
        HIPCHK(c, hipStreamSynchronize(c->stream));
        c->adv_ms = c->tail_ms = c->cmp_ms = c->graph_ms = 0.0;
        c->adv_launches = 0;
    }
    return PT_OK;
}

int pt_profile_enable(pt_ctx* c, int on) {
    if (!c) return PT_E_ARG;
    c->profile = on != 0;
    return PT_OK;
}

int pt_set_step(pt_ctx* c, uint32_t step) {
    if (!c) return PT_E_ARG;
    c->step = step;
    return PT_OK;
}

int pt_get_step(pt_ctx* c, uint32_t* step) {
    if (!c || !step) return PT_E_ARG;
    *step = c->step;
    return PT_OK;
}

int pt_synchronize(pt_ctx* c) {
    if (!c) return PT_E_ARG;
    HIPCHK(c, hipSetDevice(c->device));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    return PT_OK;
}

// ---- test hooks

#define SCRATCH(c, var, T, count)                                                             \
    Scratch<T> var;                                                                           \
    do {                                                                                      \
        if (dev_malloc((c), (void**)&var.p, sizeof(T) * (count)) != hipSuccess)               \
            return fail((c), PT_E_NOMEM, "scratch allocation failed");                        \
    } while (0)

int pt_debug_philox(pt_ctx* c, const uint32_t* ctr, const uint32_t key[2], uint32_t* out, size_t n) {
    if (!c) return PT_E_ARG;
    if (!ctr || !key || !out) return fail(c, PT_E_ARG, "null argument");
    HIPCHK(c, hipSetDevice(c->device));
    SCRATCH(c, dc, uint32_t, 4 * n);
    SCRATCH(c, dout, uint32_t, 4 * n);
    HIPCHK(c, hipMemcpy(dc.p, ctr, sizeof(uint32_t) * 4 * n, hipMemcpyHostToDevice));
    if (n) {
        hipLaunchKernelGGL(k_dbg_philox, dim3((n + 255) / 256), dim3(256), 0, c->stream, dc.p, key[0], key[1], dout.p, (ull)n);
        HIPCHK(c, hipGetLastError());
    }
    HIPCHK(c, hipStreamSynchronize(c->stream));
    HIPCHK(c, hipMemcpy(out, dout.p, sizeof(uint32_t) * 4 * n, hipMemcpyDeviceToHost));
    return PT_OK;
}

int pt_debug_choices(pt_ctx* c, int64_t out[4]) {
    if (!c) return PT_E_ARG;
    if (!out) return fail(c, PT_E_ARG, "bad arguments");
    const int64_t v[4] = {c->main_block, c->main_grid, c->late_windows, c->windows_back};
    for (int q = 0; q < 4; q++) out[q] = v[q];
    return PT_OK;
}

int pt_debug_uniforms(pt_ctx* c, uint64_t uid, uint32_t step, double* out, size_t n) {
    if (!c) return PT_E_ARG;
    if (!out) return fail(c, PT_E_ARG, "null argument");
    HIPCHK(c, hipSetDevice(c->device));
    SCRATCH(c, d, double, n);
    hipLaunchKernelGGL(k_dbg_uniforms, dim3(1), dim3(64), 0, c->stream, c->cfg.seed, uid, step, d.p, (ull)n);
    HIPCHK(c, hipGetLastError());
    HIPCHK(c, hipStreamSynchronize(c->stream));
    HIPCHK(c, hipMemcpy(out, d.p, sizeof(double) * n, hipMemcpyDeviceToHost));
    return PT_OK;
}

int pt_debug_select(pt_ctx* c, int sp, size_t n, const double* E, const double* u, const int32_t* swarm,
                    int32_t* interval, int32_t* proc, double* rbound) {
    if (!c) return PT_E_ARG;
    if (sp < 0 || sp >= PT_NSPECIES || !E || !u || !interval || !proc || !rbound)
        return fail(c, PT_E_ARG, "bad arguments");
    if (!c->hp.tab[sp].valid) return fail(c, PT_E_STATE, "no table for species %d", sp);
    HIPCHK(c, hipSetDevice(c->device));
    int rc = sync_params(c);
    if (rc) return rc;
    SCRATCH(c, dE, double, n);
    SCRATCH(c, du, double, n);
    SCRATCH(c, dsw, int32_t, n);
    SCRATCH(c, di, int32_t, n);
    SCRATCH(c, dp, int32_t, n);
    SCRATCH(c, dr, double, n);
    HIPCHK(c, hipMemcpy(dE.p, E, sizeof(double) * n, hipMemcpyHostToDevice));
    HIPCHK(c, hipMemcpy(du.p, u, sizeof(double) * n, hipMemcpyHostToDevice));
    if (swarm) HIPCHK(c, hipMemcpy(dsw.p, swarm, sizeof(int32_t) * n, hipMemcpyHostToDevice));
    if (n) {
        hipLaunchKernelGGL(k_dbg_select, dim3((n + 255) / 256), dim3(256), c->lds_bytes, c->stream, c->dp, sp,
                           (ull)n, dE.p, du.p, swarm ? dsw.p : nullptr, di.p, dp.p, dr.p);
        HIPCHK(c, hipGetLastError());
    }
    HIPCHK(c, hipStreamSynchronize(c->stream));
    HIPCHK(c, hipMemcpy(interval, di.p, sizeof(int32_t) * n, hipMemcpyDeviceToHost));
    HIPCHK(c, hipMemcpy(proc, dp.p, sizeof(int32_t) * n, hipMemcpyDeviceToHost));
    HIPCHK(c, hipMemcpy(rbound, dr.p, sizeof(double) * n, hipMemcpyDeviceToHost));
    return PT_OK;
}

int pt_debug_push(pt_ctx* c, int sp, size_t n, double* const soa[PT_NFIELDS], const double* dt) {
    if (!c) return PT_E_ARG;
    if (sp < 0 || sp >= PT_NSPECIES || !soa || !dt) return fail(c, PT_E_ARG, "bad arguments");
    const int fi[7] = {PT_X, PT_Y, PT_Z, PT_PX, PT_PY, PT_PZ, PT_T};
    for (int q = 0; q < 7; q++)
        if (!soa[fi[q]]) return fail(c, PT_E_ARG, "push needs x, p and t");
    HIPCHK(c, hipSetDevice(c->device));
    int rc = sync_params(c);
    if (rc) return rc;
    SCRATCH(c, buf, double, 8 * n);
    for (int q = 0; q < 7; q++)
        HIPCHK(c, hipMemcpy(buf.p + (size_t)q * n, soa[fi[q]], sizeof(double) * n, hipMemcpyHostToDevice));
    HIPCHK(c, hipMemcpy(buf.p + 7 * n, dt, sizeof(double) * n, hipMemcpyHostToDevice));
    if (n) {
        double* b = buf.p;
        hipLaunchKernelGGL(k_dbg_push, dim3((n + 255) / 256), dim3(256), 0, c->stream, c->dp, sp, (ull)n, b,
                           b + n, b + 2 * n, b + 3 * n, b + 4 * n, b + 5 * n, b + 6 * n, b + 7 * n);
        HIPCHK(c, hipGetLastError());
    }
    HIPCHK(c, hipStreamSynchronize(c->stream));
    for (int q = 0; q < 7; q++)
        HIPCHK(c, hipMemcpy(soa[fi[q]], buf.p + (size_t)q * n, sizeof(double) * n, hipMemcpyDeviceToHost));
    return PT_OK;
}

int pt_debug_collide(pt_ctx* c, int sp, int proc, size_t n, const double* const soa[PT_NFIELDS],
                     const uint64_t* uid, const double* u, int stride, int32_t* out_kind, int32_t* out_draws,
                     double* out_states, int32_t* out_species, uint64_t* out_uid) {
    if (!c) return PT_E_ARG;
    if (sp < 0 || sp >= PT_NSPECIES || !soa || !uid || !u || stride < 1 || !out_kind || !out_draws ||
        !out_states || !out_species || !out_uid)
        return fail(c, PT_E_ARG, "bad arguments");
    if (!c->hp.tab[sp].valid || proc < 0 || proc >= c->hp.tab[sp].nprocs)
        return fail(c, PT_E_ARG, "process %d not in the table of species %d", proc, sp);
    for (int f = 0; f < 8; f++)
        if (!soa[f]) return fail(c, PT_E_ARG, "collide needs x, p, w, t");
    HIPCHK(c, hipSetDevice(c->device));
    int rc = require_tables(c);
    if (rc) return rc;
    rc = sync_params(c);
    if (rc) return rc;
    std::vector<double> in(n * PT_NFIELDS, 0.0);
    for (size_t i = 0; i < n; i++)
        for (int f = 0; f < 8; f++) in[i * PT_NFIELDS + f] = soa[f][i];
    SCRATCH(c, din, double, n * PT_NFIELDS);
    SCRATCH(c, duid, uint64_t, n);
    SCRATCH(c, du, double, n * (size_t)stride);
    SCRATCH(c, dk, int32_t, n);
    SCRATCH(c, dd, int32_t, n);
    SCRATCH(c, dst, double, n * 3 * PT_NFIELDS);
    SCRATCH(c, dsp, int32_t, n * 3);
    SCRATCH(c, dou, uint64_t, n * 3);
    HIPCHK(c, hipMemcpy(din.p, in.data(), sizeof(double) * n * PT_NFIELDS, hipMemcpyHostToDevice));
    HIPCHK(c, hipMemcpy(duid.p, uid, sizeof(uint64_t) * n, hipMemcpyHostToDevice));
    HIPCHK(c, hipMemcpy(du.p, u, sizeof(double) * n * stride, hipMemcpyHostToDevice));
    if (n) {
        hipLaunchKernelGGL(k_dbg_collide, dim3((n + 255) / 256), dim3(256), 0, c->stream, c->dp, sp, proc, (ull)n,
                           din.p, duid.p, du.p, stride, c->step, dk.p, dd.p, dst.p, dsp.p, dou.p);
        HIPCHK(c, hipGetLastError());
    }
    HIPCHK(c, hipStreamSynchronize(c->stream));
    HIPCHK(c, hipMemcpy(out_kind, dk.p, sizeof(int32_t) * n, hipMemcpyDeviceToHost));
    HIPCHK(c, hipMemcpy(out_draws, dd.p, sizeof(int32_t) * n, hipMemcpyDeviceToHost));
    HIPCHK(c, hipMemcpy(out_states, dst.p, sizeof(double) * n * 3 * PT_NFIELDS, hipMemcpyDeviceToHost));
    HIPCHK(c, hipMemcpy(out_species, dsp.p, sizeof(int32_t) * n * 3, hipMemcpyDeviceToHost));
    HIPCHK(c, hipMemcpy(out_uid, dou.p, sizeof(uint64_t) * n * 3, hipMemcpyDeviceToHost));
    return PT_OK;
}

// ---- learned samplers
int pt_learn_nparams(void) { return MLP_NPARAM; }

int pt_learn_defaults(int which, pt_learn_config* cfg) {
    if (!cfg || which < 0 || which >= NLEARN) return PT_E_ARG;
    memset(cfg, 0, sizeof(*cfg));
    cfg->nenergies = 8192;
    cfg->samples_per_row = 4096;
    cfg->quantiles = 256;
    cfg->batch = 16384;
    cfg->steps = 20000;
    cfg->ks_samples = 400000;
    cfg->ks_energies = 16;
    cfg->lr = 2e-3;
    cfg->tcut = 1e4 * EV;
    cfg->emin = which == LEARN_SB ? 4e4 * EV : 2.05 * cfg->tcut;
    cfg->emax = 1e8 * EV;
    cfg->ks_gate = 0.01;
    cfg->seed = 0x5EED1234ull;
    return PT_OK;
}

static const int LEARN_Z[3] = {7, 8, 18};

// buffers of one training batch
struct MlpBatch {
    Scratch<float> X, Tg, Z1, H1, Z2, H2, Z3, H3, Yz, Y, dY, dA, dB, part, lpart;
    int B = 0, ns = 0, nlb = 0;
};

static int mlp_batch_alloc(pt_ctx* c, MlpBatch& b, int B) {
    b.B = B;
    b.ns = (B + MLP_SLICE - 1) / MLP_SLICE;
    b.nlb = (B + 255) / 256;
    const size_t h = (size_t)B * MLP_H;
    int rc;
    if ((rc = dscratch(c, b.X, (size_t)B * MLP_IN)) || (rc = dscratch(c, b.Tg, 2 * (size_t)B)) ||
        (rc = dscratch(c, b.Z1, h)) || (rc = dscratch(c, b.H1, h)) || (rc = dscratch(c, b.Z2, h)) ||
        (rc = dscratch(c, b.H2, h)) || (rc = dscratch(c, b.Z3, h)) || (rc = dscratch(c, b.H3, h)) ||
        (rc = dscratch(c, b.Yz, 2 * (size_t)B)) || (rc = dscratch(c, b.Y, 2 * (size_t)B)) ||
        (rc = dscratch(c, b.dY, 2 * (size_t)B)) || (rc = dscratch(c, b.dA, h)) || (rc = dscratch(c, b.dB, h)) ||
        (rc = dscratch(c, b.part, (size_t)b.ns * MLP_H * (MLP_H + 1))) || (rc = dscratch(c, b.lpart, b.nlb)))
        return rc;
    return PT_OK;
}

static unsigned nblk(ull n, int bs) { return (unsigned)std::max<ull>(1, (n + bs - 1) / bs); }

// one forward and backward pass on the batch in b.X / b.Tg: gradient g (device), batch loss
// partials in b.lpart
static void gemm_launch(hipStream_t st, const MlpGemm& g, int slices) {
    hipLaunchKernelGGL(k_mlp_gemm, dim3((unsigned)((g.M + 31) / 32), (unsigned)((g.N + 31) / 32), (unsigned)slices),
                       dim3(64), 0, st, g);
}

// Z = X W^T + bias, H = gelu(Z) or Z, on the matrix cores (X: B x nin, W: nout x nin)
static void gemm_fwd(hipStream_t st, const float* X, int nin, const float* W, const float* bias, int nout, int B,
                     int act, float* Z, float* H) {
    MlpGemm g{};
    g.A = X;
    g.sam = nin;
    g.sak = 1;
    g.B = W;
    g.sbk = 1;
    g.sbn = nin;
    g.M = B;
    g.N = nout;
    g.K = nin;
    g.ones = -1;
    g.klen = nin;
    g.epi = GEMM_FWD;
    g.act = act;
    g.bias = bias;
    g.C = Z;
    g.C2 = H;
    g.ldc = nout;
    gemm_launch(st, g, 1);
}

static int mlp_fb(pt_ctx* c, MlpBatch& b, const float* P, float w0, float w1, float* g) {
    const int B = b.B;
    hipStream_t st = c->stream;
    gemm_fwd(st, b.X.p, MLP_IN, P + P_W1, P + P_B1, MLP_H, B, 1, b.Z1.p, b.H1.p);
    gemm_fwd(st, b.H1.p, MLP_H, P + P_W2, P + P_B2, MLP_H, B, 1, b.Z2.p, b.H2.p);
    gemm_fwd(st, b.H2.p, MLP_H, P + P_W3, P + P_B3, MLP_H, B, 1, b.Z3.p, b.H3.p);
    gemm_fwd(st, b.H3.p, MLP_H, P + P_W4, P + P_B4, MLP_OUT, B, 0, b.Yz.p, b.Y.p);
    hipLaunchKernelGGL(k_mlp_loss, dim3(b.nlb), dim3(256), 0, st, b.Y.p, b.Tg.p, w0, w1, B, b.dY.p, b.lpart.p);
    struct L {
        const float* dz;
        const float* in;
        int nin, nout, pw, pb;
        float* dnext;  // gradient of the layer's input (null for the first layer)
        const float* W;
        const float* zprev;
    } layers[4] = {
        {b.dY.p, b.H3.p, MLP_H, MLP_OUT, P_W4, P_B4, b.dA.p, P + P_W4, b.Z3.p},
        {b.dA.p, b.H2.p, MLP_H, MLP_H, P_W3, P_B3, b.dB.p, P + P_W3, b.Z2.p},
        {b.dB.p, b.H1.p, MLP_H, MLP_H, P_W2, P_B2, b.dA.p, P + P_W2, b.Z1.p},
        {b.dA.p, b.X.p, MLP_IN, MLP_H, P_W1, P_B1, nullptr, P + P_W1, nullptr},
    };
    for (const L& l : layers) {
        const int m = l.nout * (l.nin + 1);
        // weight and bias gradients per batch slice: part[z][o][i] = sum over the slice of
        // dZ[b][o] in[b][i] (i == nin: 1), then summed over slices in slice order
        MlpGemm gw{};
        gw.A = l.dz;
        gw.sam = 1;
        gw.sak = l.nout;
        gw.B = l.in;
        gw.sbk = l.nin;
        gw.sbn = 1;
        gw.M = l.nout;
        gw.N = l.nin + 1;
        gw.K = B;
        gw.ones = l.nin;
        gw.klen = MLP_SLICE;
        gw.epi = GEMM_PART;
        gw.C = b.part.p;
        gw.ldc = l.nin + 1;
        gemm_launch(st, gw, b.ns);
        hipLaunchKernelGGL(k_mlp_reduce, dim3(nblk(m, 256)), dim3(256), 0, st, b.part.p, b.ns, l.nin, l.nout, l.pw, l.pb, g);
        if (l.dnext) {
            // gradient of the layer's input through the previous layer's GELU:
            // dnext[b][i] = gelu'(zprev[b][i]) sum_o dZ[b][o] W[o][i]
            MlpGemm gd{};
            gd.A = l.dz;
            gd.sam = l.nout;
            gd.sak = 1;
            gd.B = l.W;
            gd.sbk = l.nin;
            gd.sbn = 1;
            gd.M = B;
            gd.N = l.nin;
            gd.K = l.nout;
            gd.ones = -1;
            gd.klen = l.nout;
            gd.epi = GEMM_DATA;
            gd.Zp = l.zprev;
            gd.C = l.dnext;
            gd.ldc = l.nin;
            gemm_launch(st, gd, 1);
        }
    }
    HIPCHK(c, hipGetLastError());
    return PT_OK;
}

// Xavier-uniform weights over the inputs in use, zero biases (host, seeded)
static void mlp_init(std::vector<float>& p, uint64_t seed) {
    p.assign(MLP_NPARAM, 0.0f);
    uint64_t st = seed ^ 0x9E3779B97F4A7C15ull;
    auto uni = [&]() {
        st ^= st << 13;
        st ^= st >> 7;
        st ^= st << 17;
        return (double)(st >> 11) * (1.0 / 9007199254740992.0);
    };
    struct {
        int off, nout, nin, fan_in;
    } ls[4] = {{P_W1, MLP_H, MLP_IN, 7}, {P_W2, MLP_H, MLP_H, MLP_H}, {P_W3, MLP_H, MLP_H, MLP_H}, {P_W4, MLP_OUT, MLP_H, MLP_H}};
    for (auto& l : ls) {
        double a = std::sqrt(6.0 / (l.fan_in + l.nout));
        for (int o = 0; o < l.nout; o++)
            for (int i = 0; i < l.nin; i++) p[l.off + o * l.nin + i] = (float)((2.0 * uni() - 1.0) * a);
    }
}

static int mlp_image(pt_ctx* c, const float* params, uint16_t* w, float* b) {
    hipLaunchKernelGGL(k_mlp_image, dim3(nblk(MLP_H * MLP_H, 256)), dim3(256), 0, c->stream, params, w, b);
    HIPCHK(c, hipGetLastError());
    return PT_OK;
}

static int learn_buffers(pt_ctx* c, int which) {
    pt_ctx::Learned& L = c->learn[which];
    int rc;
    if (!L.params && (rc = dalloc(c, (void**)&L.params, sizeof(float) * MLP_NPARAM))) return rc;
    if (!L.wimg && (rc = dalloc(c, (void**)&L.wimg, sizeof(uint16_t) * I_NW))) return rc;
    if (!L.bimg && (rc = dalloc(c, (void**)&L.bimg, sizeof(float) * I_NB))) return rc;
    return PT_OK;
}

static int set_learn_on(pt_ctx* c, int which, bool on) {
    pt_ctx::Learned& L = c->learn[which];
    L.on = on;
    c->hp.mlp[which].w = L.wimg;
    c->hp.mlp[which].b = L.bimg;
    c->hp.mlp[which].emin = L.emin;
    c->hp.mlp[which].emax = L.emax;
    c->hp.mlp[which].on = on ? 1 : 0;
    c->dirty = true;
    return sync_params(c);
}

// rows of (energy, Z): slot of the Seltzer-Berger data of each target
static int learn_rows(pt_ctx* c, int which, int per_z, double emin, double emax, double offset,
                      std::vector<double>& T, std::vector<int32_t>& Z, std::vector<int32_t>& slot) {
    T.clear();
    Z.clear();
    slot.clear();
    for (int zi = 0; zi < 3; zi++) {
        int sl = 0;
        if (which == LEARN_SB) {
            sl = -1;
            for (int q = 0; q < MAX_SB; q++)
                if (c->sb_z[q] == LEARN_Z[zi] && c->hp.sb[q].data) sl = q;
            if (sl < 0) return fail(c, PT_E_STATE, "no Seltzer-Berger data uploaded for Z = %d", LEARN_Z[zi]);
        }
        for (int m = 0; m < per_z; m++) {
            double f = (m + offset) / per_z;
            T.push_back(std::exp(std::log(emin) + f * (std::log(emax) - std::log(emin))));
            Z.push_back(LEARN_Z[zi]);
            slot.push_back(sl);
        }
    }
    return PT_OK;
}

// exact samples (K per row) of the rows, transformed: o0, o1 (device)
static int learn_exact(pt_ctx* c, int which, const std::vector<double>& T, const std::vector<int32_t>& slot, int K,
                       uint64_t seed, double tcut, Scratch<float>& o0, Scratch<float>& o1, float* ms = nullptr) {
    const size_t R = T.size();
    Scratch<double> dT;
    Scratch<int32_t> ds;
    int rc;
    if ((rc = dscratch(c, dT, R)) || (rc = dscratch(c, ds, R)) || (rc = dscratch(c, o0, R * (size_t)K)) ||
        (rc = dscratch(c, o1, R * (size_t)K)))
        return rc;
    HIPCHK(c, hipMemcpyAsync(dT.p, T.data(), sizeof(double) * R, hipMemcpyHostToDevice, c->stream));
    HIPCHK(c, hipMemcpyAsync(ds.p, slot.data(), sizeof(int32_t) * R, hipMemcpyHostToDevice, c->stream));
    if ((rc = sync_params(c))) return rc;
    if (ms) HIPCHK(c, hipEventRecord(c->ev[5], c->stream));
    hipLaunchKernelGGL(k_mlp_gen, dim3(c->grid), dim3(256), 0, c->stream, c->dp, which, dT.p, ds.p, (int)R, K, seed, tcut,
                       o0.p, o1.p);
    HIPCHK(c, hipGetLastError());
    if (ms) HIPCHK(c, hipEventRecord(c->ev[6], c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    if (ms) HIPCHK(c, hipEventElapsedTime(ms, c->ev[5], c->ev[6]));
    return PT_OK;
}

// network outputs for `reps` samples at each row (device Y, 2 per sample)
static int learn_infer(pt_ctx* c, int which, const uint16_t* wimg, const float* bimg, const std::vector<double>& T,
                       const std::vector<int32_t>& Z, const std::vector<int32_t>& slot, int reps, uint64_t seed,
                       Scratch<float>& Y, float* ms = nullptr) {
    const size_t R = T.size(), n = R * (size_t)reps;
    Scratch<double> dT;
    Scratch<int32_t> dZ, ds;
    Scratch<float> X;
    int rc;
    if ((rc = dscratch(c, dT, R)) || (rc = dscratch(c, dZ, R)) || (rc = dscratch(c, ds, R)) ||
        (rc = dscratch(c, X, n * MLP_IN)) || (rc = dscratch(c, Y, 2 * n)))
        return rc;
    HIPCHK(c, hipMemcpyAsync(dT.p, T.data(), sizeof(double) * R, hipMemcpyHostToDevice, c->stream));
    HIPCHK(c, hipMemcpyAsync(dZ.p, Z.data(), sizeof(int32_t) * R, hipMemcpyHostToDevice, c->stream));
    HIPCHK(c, hipMemcpyAsync(ds.p, slot.data(), sizeof(int32_t) * R, hipMemcpyHostToDevice, c->stream));
    if ((rc = sync_params(c))) return rc;
    if (ms) HIPCHK(c, hipEventRecord(c->ev[5], c->stream));
    hipLaunchKernelGGL(k_mlp_features, dim3(c->grid), dim3(256), 0, c->stream, c->dp, which, dT.p, dZ.p, ds.p, (ull)R,
                       reps, seed, X.p);
    hipLaunchKernelGGL(k_mlp_infer, dim3(c->grid), dim3(256), 0, c->stream, which, wimg, bimg, X.p, (int)n, Y.p);
    HIPCHK(c, hipGetLastError());
    if (ms) HIPCHK(c, hipEventRecord(c->ev[6], c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    if (ms) HIPCHK(c, hipEventElapsedTime(ms, c->ev[5], c->ev[6]));
    return PT_OK;
}

// the clamps the step applies to the outputs
static void learn_clamp(int which, float& y0, float& y1) {
    if (which == LEARN_SB) {
        y0 = std::min(y0, 0.0f);
        y1 = std::min(y1, 0.6931472f);
    } else {
        y0 = std::min(std::max(y0, 0.0f), 1.0f);
        y1 = 0.0f;
    }
}

static double ks2(std::vector<float>& a, std::vector<float>& b) {
    std::sort(a.begin(), a.end());
    std::sort(b.begin(), b.end());
    size_t i = 0, j = 0;
    double d = 0.0;
    while (i < a.size() && j < b.size()) {
        float v = std::min(a[i], b[j]);
        while (i < a.size() && a[i] <= v) i++;
        while (j < b.size() && b[j] <= v) j++;
        d = std::max(d, std::fabs((double)i / a.size() - (double)j / b.size()));
    }
    return d;
}

int pt_learn_train(pt_ctx* c, int which, const pt_learn_config* cfg, pt_learn_report* rep) {
    if (!c) return PT_E_ARG;
    if (which < 0 || which >= NLEARN || !cfg) return fail(c, PT_E_ARG, "bad learned-sampler arguments");
    const int M = cfg->nenergies, K = cfg->samples_per_row, Kq = cfg->quantiles, B = cfg->batch;
    if (M < 1 || K < 2 || K > 4096 || (K & (K - 1)) || Kq < 2 || Kq > K || B < 256 || cfg->steps < 1 ||
        cfg->ks_samples < 100 || cfg->ks_energies < 1 || !(cfg->emin > 0) || !(cfg->emax > cfg->emin) ||
        (which == LEARN_MOLLER && !(cfg->emin > 2.0 * cfg->tcut)))
        return fail(c, PT_E_ARG, "bad learned-sampler configuration");
    HIPCHK(c, hipSetDevice(c->device));
    int rc;
    if ((rc = learn_buffers(c, which))) return rc;
    pt_ctx::Learned& Ln = c->learn[which];
    Ln.tcut = cfg->tcut;
    Ln.emin = cfg->emin;
    Ln.emax = cfg->emax;
    pt_learn_report r{};
    // 1. training set: exact samples -> per-row quantiles
    std::vector<double> T;
    std::vector<int32_t> Z, slot;
    // the training energies reach a little beyond the gated range, so that the range's
    // edges are not the network's edges
    const double tlo = which == LEARN_MOLLER ? std::max(cfg->emin / 1.25, 2.0 * cfg->tcut * 1.0001) : cfg->emin / 1.25;
    if ((rc = learn_rows(c, which, M, tlo, cfg->emax * 1.25, 0.5, T, Z, slot))) return rc;
    const int R = (int)T.size();
    Scratch<float> Q0, Q1, rowx;
    if ((rc = dscratch(c, Q0, (size_t)R * Kq)) || (rc = dscratch(c, Q1, (size_t)R * Kq)) ||
        (rc = dscratch(c, rowx, (size_t)R * 5)))
        return rc;
    HIPCHK(c, hipEventRecord(c->ev[0], c->stream));
    {
        Scratch<float> o0, o1;
        if ((rc = learn_exact(c, which, T, slot, K, cfg->seed, cfg->tcut, o0, o1))) return rc;
        hipLaunchKernelGGL(k_mlp_sort_rows, dim3(R), dim3(1024), 0, c->stream, o0.p, K);
        hipLaunchKernelGGL(k_mlp_sort_rows, dim3(R), dim3(1024), 0, c->stream, o1.p, K);
        hipLaunchKernelGGL(k_mlp_quantiles, dim3(c->grid), dim3(256), 0, c->stream, o0.p, R, K, Kq, Q0.p);
        hipLaunchKernelGGL(k_mlp_quantiles, dim3(c->grid), dim3(256), 0, c->stream, o1.p, R, K, Kq, Q1.p);
        HIPCHK(c, hipGetLastError());
        HIPCHK(c, hipStreamSynchronize(c->stream));
    }
    HIPCHK(c, hipEventRecord(c->ev[1], c->stream));
    std::vector<float> hx((size_t)R * 5);
    for (int q = 0; q < R; q++) {
        float x[MLP_IN];
        double ph = 0.0;
        if (which == LEARN_SB) {
            const std::vector<double>& le = c->sb_le[slot[q]];
            ph = sb_phase(le.data(), c->sb_thr[slot[q]].data(), (int)le.size(), T[q]);
        }
        mlp_features(T[q] / EV, Z[q], 0.5, 0.5, ph, x);
        for (int k = 0; k < 4; k++) hx[(size_t)q * 5 + k] = x[k];
        hx[(size_t)q * 5 + 4] = x[6];
    }
    HIPCHK(c, hipMemcpyAsync(rowx.p, hx.data(), sizeof(float) * hx.size(), hipMemcpyHostToDevice, c->stream));
    r.samples = (int64_t)R * K;
    // 2. training
    std::vector<float> p0;
    mlp_init(p0, cfg->seed);
    HIPCHK(c, hipMemcpyAsync(Ln.params, p0.data(), sizeof(float) * MLP_NPARAM, hipMemcpyHostToDevice, c->stream));
    MlpBatch b;
    if ((rc = mlp_batch_alloc(c, b, B))) return rc;
    Scratch<float> g, m, v, lossv;
    if ((rc = dscratch(c, g, MLP_NPARAM)) || (rc = dscratch(c, m, MLP_NPARAM)) || (rc = dscratch(c, v, MLP_NPARAM)) ||
        (rc = dscratch(c, lossv, (size_t)cfg->steps)))
        return rc;
    Scratch<uint32_t> stepc;  // the step counter the training kernels read
    if ((rc = dscratch(c, stepc, 1))) return rc;
    HIPCHK(c, hipMemsetAsync(m.p, 0, sizeof(float) * MLP_NPARAM, c->stream));
    HIPCHK(c, hipMemsetAsync(v.p, 0, sizeof(float) * MLP_NPARAM, c->stream));
    HIPCHK(c, hipMemsetAsync(stepc.p, 0, sizeof(uint32_t), c->stream));
    const float w0 = 1.0f, w1 = which == LEARN_SB ? 1.0f : 0.0f;
    // one Adam step: batch, forward/backward, loss, update, counter (21 kernels)
    auto adam_step = [&]() -> int {
        hipLaunchKernelGGL(k_mlp_batch, dim3(nblk(B, 256)), dim3(256), 0, c->stream, which, Q0.p, Q1.p, rowx.p, R, Kq, B,
                           cfg->seed ^ 0xBA7C4ull, (const uint32_t*)stepc.p, b.X.p, b.Tg.p);
        int frc = mlp_fb(c, b, Ln.params, w0, w1, g.p);
        if (frc) return frc;
        hipLaunchKernelGGL(k_mlp_sum, dim3(1), dim3(256), 0, c->stream, b.lpart.p, b.nlb, lossv.p,
                           (const uint32_t*)stepc.p);
        hipLaunchKernelGGL(k_mlp_adam, dim3(nblk(MLP_NPARAM, 256)), dim3(256), 0, c->stream, Ln.params, g.p, m.p, v.p,
                           MLP_NPARAM, cfg->lr, cfg->steps, (const uint32_t*)stepc.p, 0.9f, 0.999f, 1e-8f);
        hipLaunchKernelGGL(k_mlp_tick, dim3(1), dim3(64), 0, c->stream, stepc.p);
        HIPCHK(c, hipGetLastError());
        return PT_OK;
    };
    for (int it = 0; it < cfg->steps; it++)
        if ((rc = adam_step())) return rc;
    HIPCHK(c, hipEventRecord(c->ev[2], c->stream));
    std::vector<float> hl(cfg->steps);
    HIPCHK(c, hipMemcpyAsync(hl.data(), lossv.p, sizeof(float) * hl.size(), hipMemcpyDeviceToHost, c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    const int nav = std::min(100, cfg->steps);
    for (int q = 0; q < nav; q++) {
        r.loss_first += hl[q] / nav;
        r.loss_last += hl[cfg->steps - 1 - q] / nav;
    }
    if ((rc = mlp_image(c, Ln.params, Ln.wimg, Ln.bimg))) return rc;
    Ln.trained = true;
    // 3. KS gate on held-out energies: rejection sampler vs network
    HIPCHK(c, hipEventRecord(c->ev[3], c->stream));
    std::vector<double> T2;
    std::vector<int32_t> Z2, slot2;
    if ((rc = learn_rows(c, which, cfg->ks_energies, cfg->emin, cfg->emax, 0.37, T2, Z2, slot2))) return rc;
    const int n = cfg->ks_samples;
    const size_t R2 = T2.size();
    std::vector<float> e0(R2 * (size_t)n), e1(R2 * (size_t)n), y(2 * R2 * (size_t)n);
    {
        Scratch<float> o0, o1, Y;
        if ((rc = learn_exact(c, which, T2, slot2, n, cfg->seed ^ 0x4B5ull, cfg->tcut, o0, o1))) return rc;
        if ((rc = learn_infer(c, which, Ln.wimg, Ln.bimg, T2, Z2, slot2, n, cfg->seed ^ 0x1F3ull, Y))) return rc;
        HIPCHK(c, hipMemcpy(e0.data(), o0.p, sizeof(float) * e0.size(), hipMemcpyDeviceToHost));
        HIPCHK(c, hipMemcpy(e1.data(), o1.p, sizeof(float) * e1.size(), hipMemcpyDeviceToHost));
        HIPCHK(c, hipMemcpy(y.data(), Y.p, sizeof(float) * y.size(), hipMemcpyDeviceToHost));
    }
    double ksmax = 0.0, kssum = 0.0;
    const int nout = which == LEARN_SB ? 2 : 1;
    const int nks = (int)R2 * nout;
    // the two-sample KS statistic of every (energy, target, output), on host threads (each
    // sorts 2 x ks_samples values); summed in a fixed order afterwards
    std::vector<double> ksv((size_t)nks, 0.0);
    {
        const int nth = (int)std::max(1u, std::min(16u, std::thread::hardware_concurrency()));
        auto work = [&](int first, int stride) {
            for (int k = first; k < nks; k += stride) {
                const size_t row = (size_t)(k / nout);
                const int o = k % nout;
                std::vector<float> a(n), bb(n);
                for (int q = 0; q < n; q++) {
                    size_t s = row * n + q;
                    a[q] = o == 0 ? e0[s] : e1[s];
                    float y0 = y[2 * s], y1 = y[2 * s + 1];
                    learn_clamp(which, y0, y1);
                    bb[q] = o == 0 ? y0 : y1;
                }
                ksv[(size_t)k] = ks2(a, bb);
            }
        };
        std::vector<std::thread> pool;
        try {
            for (int t = 1; t < nth; t++) pool.emplace_back(work, t, nth);
        } catch (...) {
            // no threads to spare: this thread does the rest
            for (auto& th : pool) th.join();
            pool.clear();
        }
        if (pool.empty()) {
            work(0, 1);
        } else {
            work(0, nth);
            for (auto& th : pool) th.join();
        }
    }
    for (int k = 0; k < nks; k++) {
        ksmax = std::max(ksmax, ksv[(size_t)k]);
        kssum += ksv[(size_t)k];
    }
    HIPCHK(c, hipEventRecord(c->ev[4], c->stream));
    HIPCHK(c, hipEventSynchronize(c->ev[4]));
    float ms = 0;
    HIPCHK(c, hipEventElapsedTime(&ms, c->ev[0], c->ev[1]));
    r.gen_ms = ms;
    HIPCHK(c, hipEventElapsedTime(&ms, c->ev[1], c->ev[2]));
    r.train_ms = ms;
    HIPCHK(c, hipEventElapsedTime(&ms, c->ev[3], c->ev[4]));
    r.eval_ms = ms;
    r.ks_max = ksmax;
    r.ks_mean = kssum / std::max(nks, 1);
    r.ks_noise = 1.36 * std::sqrt(2.0 / n);
    r.nparams = MLP_H * (which == LEARN_SB ? 7 : 6) + MLP_H + 2 * (MLP_H * MLP_H + MLP_H) + (which == LEARN_SB ? 2 : 1) * (MLP_H + 1);
    r.installed = ksmax <= cfg->ks_gate ? 1 : 0;
    if ((rc = set_learn_on(c, which, r.installed != 0))) return rc;
    c->resident_lds = -1;
    if (rep) *rep = r;
    return PT_OK;
}

int pt_learn_enable(pt_ctx* c, int which, int on) {
    if (!c) return PT_E_ARG;
    if (which < 0 || which >= NLEARN) return fail(c, PT_E_ARG, "bad learned sampler %d", which);
    if (on && !c->learn[which].trained) return fail(c, PT_E_STATE, "learned sampler %d is not trained", which);
    HIPCHK(c, hipSetDevice(c->device));
    c->resident_lds = -1;
    return set_learn_on(c, which, on != 0);
}

int pt_learn_params(pt_ctx* c, int which, float* params, int n, int set) {
    if (!c) return PT_E_ARG;
    if (which < 0 || which >= NLEARN || !params || n != MLP_NPARAM) return fail(c, PT_E_ARG, "bad arguments");
    HIPCHK(c, hipSetDevice(c->device));
    int rc = learn_buffers(c, which);
    if (rc) return rc;
    pt_ctx::Learned& L = c->learn[which];
    if (!set) {
        if (!L.trained) return fail(c, PT_E_STATE, "learned sampler %d has no parameters", which);
        HIPCHK(c, hipMemcpy(params, L.params, sizeof(float) * MLP_NPARAM, hipMemcpyDeviceToHost));
        return PT_OK;
    }
    HIPCHK(c, hipMemcpyAsync(L.params, params, sizeof(float) * MLP_NPARAM, hipMemcpyHostToDevice, c->stream));
    if ((rc = mlp_image(c, L.params, L.wimg, L.bimg))) return rc;
    HIPCHK(c, hipStreamSynchronize(c->stream));
    L.trained = true;
    c->resident_lds = -1;
    return set_learn_on(c, which, false);
}

int pt_learn_install(pt_ctx* c, int which, const float* params, int n, double emin, double emax) {
    if (!c) return PT_E_ARG;
    if (!(emin > 0.0 && emax > emin)) return fail(c, PT_E_ARG, "energy range must satisfy 0 < emin < emax");
    int rc = pt_learn_params(c, which, (float*)params, n, 1);
    if (rc) return rc;
    c->learn[which].emin = emin;
    c->learn[which].emax = emax;
    c->resident_lds = -1;
    return set_learn_on(c, which, true);
}

int pt_learn_sample(pt_ctx* c, int which, int learned, const double* T, const int32_t* Z, size_t n, uint64_t seed,
                    double* out) {
    if (!c) return PT_E_ARG;
    if (which < 0 || which >= NLEARN || !T || !Z || !out) return fail(c, PT_E_ARG, "bad arguments");
    if (learned && !c->learn[which].trained) return fail(c, PT_E_STATE, "learned sampler %d is not trained", which);
    HIPCHK(c, hipSetDevice(c->device));
    if (n == 0) return PT_OK;
    std::vector<double> Tv(T, T + n);
    std::vector<int32_t> Zv(Z, Z + n), slot(n, 0);
    for (size_t q = 0; q < n; q++) {
        if (which == LEARN_SB) {
            slot[q] = -1;
            for (int s = 0; s < MAX_SB; s++)
                if (c->sb_z[s] == Z[q] && c->hp.sb[s].data) slot[q] = s;
            if (slot[q] < 0) return fail(c, PT_E_STATE, "no Seltzer-Berger data uploaded for Z = %d", Z[q]);
        } else if (!(T[q] > 2.0 * c->learn[which].tcut)) {
            return fail(c, PT_E_ARG, "Moller energy %g J not above 2 tcut", T[q]);
        }
    }
    std::vector<float> y(2 * n);
    int rc;
    if (learned) {
        Scratch<float> Y;
        const pt_ctx::Learned& L = c->learn[which];
        if ((rc = learn_infer(c, which, L.wimg, L.bimg, Tv, Zv, slot, 1, seed, Y))) return rc;
        HIPCHK(c, hipMemcpy(y.data(), Y.p, sizeof(float) * 2 * n, hipMemcpyDeviceToHost));
        for (size_t q = 0; q < n; q++) learn_clamp(which, y[2 * q], y[2 * q + 1]);
    } else {
        Scratch<float> o0, o1;
        if ((rc = learn_exact(c, which, Tv, slot, 1, seed, c->learn[which].tcut, o0, o1))) return rc;
        std::vector<float> a(n), b(n);
        HIPCHK(c, hipMemcpy(a.data(), o0.p, sizeof(float) * n, hipMemcpyDeviceToHost));
        HIPCHK(c, hipMemcpy(b.data(), o1.p, sizeof(float) * n, hipMemcpyDeviceToHost));
        for (size_t q = 0; q < n; q++) {
            y[2 * q] = a[q];
            y[2 * q + 1] = b[q];
        }
    }
    for (size_t q = 0; q < 2 * n; q++) out[q] = y[q];
    return PT_OK;
}

int pt_learn_throughput(pt_ctx* c, int which, int learned, const double* T, const int32_t* Z, size_t nrows,
                        int per_row, uint64_t seed, double* samples_per_s) {
    if (!c) return PT_E_ARG;
    if (which < 0 || which >= NLEARN || !T || !Z || !samples_per_s || nrows == 0 || per_row < 1 ||
        nrows * (size_t)per_row > (1ull << 26))
        return fail(c, PT_E_ARG, "bad arguments (at most 2^26 samples)");
    if (learned && !c->learn[which].trained) return fail(c, PT_E_STATE, "learned sampler %d is not trained", which);
    HIPCHK(c, hipSetDevice(c->device));
    std::vector<double> Tv(T, T + nrows);
    std::vector<int32_t> Zv(Z, Z + nrows), slot(nrows, 0);
    for (size_t q = 0; q < nrows; q++) {
        if (which == LEARN_SB) {
            slot[q] = -1;
            for (int s = 0; s < MAX_SB; s++)
                if (c->sb_z[s] == Z[q] && c->hp.sb[s].data) slot[q] = s;
            if (slot[q] < 0) return fail(c, PT_E_STATE, "no Seltzer-Berger data uploaded for Z = %d", Z[q]);
        } else if (!(T[q] > 2.0 * c->learn[which].tcut)) {
            return fail(c, PT_E_ARG, "Moller energy %g J not above 2 tcut", T[q]);
        }
    }
    float ms = 0.0f;
    int rc;
    if (learned) {
        Scratch<float> Y;
        const pt_ctx::Learned& L = c->learn[which];
        if ((rc = learn_infer(c, which, L.wimg, L.bimg, Tv, Zv, slot, per_row, seed, Y, &ms))) return rc;
    } else {
        Scratch<float> o0, o1;
        if ((rc = learn_exact(c, which, Tv, slot, per_row, seed, c->learn[which].tcut, o0, o1, &ms))) return rc;
    }
    *samples_per_s = ms > 0.0f ? (double)nrows * per_row / (ms * 1e-3) : 0.0;
    return PT_OK;
}

int pt_debug_mlp_grad(pt_ctx* c, const float* params, const float* X, const float* Y, int B, float w0, float w1,
                      float* grad, float* loss) {
    if (!c) return PT_E_ARG;
    if (!params || !X || !Y || !grad || !loss || B < 1) return fail(c, PT_E_ARG, "bad arguments");
    HIPCHK(c, hipSetDevice(c->device));
    MlpBatch b;
    Scratch<float> P, g;
    int rc;
    if ((rc = mlp_batch_alloc(c, b, B)) || (rc = dscratch(c, P, MLP_NPARAM)) || (rc = dscratch(c, g, MLP_NPARAM)))
        return rc;
    HIPCHK(c, hipMemcpy(P.p, params, sizeof(float) * MLP_NPARAM, hipMemcpyHostToDevice));
    HIPCHK(c, hipMemcpy(b.X.p, X, sizeof(float) * (size_t)B * MLP_IN, hipMemcpyHostToDevice));
    HIPCHK(c, hipMemcpy(b.Tg.p, Y, sizeof(float) * 2 * (size_t)B, hipMemcpyHostToDevice));
    if ((rc = mlp_fb(c, b, P.p, w0, w1, g.p))) return rc;
    HIPCHK(c, hipStreamSynchronize(c->stream));
    std::vector<float> lp(b.nlb);
    HIPCHK(c, hipMemcpy(lp.data(), b.lpart.p, sizeof(float) * lp.size(), hipMemcpyDeviceToHost));
    HIPCHK(c, hipMemcpy(grad, g.p, sizeof(float) * MLP_NPARAM, hipMemcpyDeviceToHost));
    double s = 0.0;
    for (float v : lp) s += v;
    *loss = (float)s;
    return PT_OK;
}

int pt_debug_mlp_infer(pt_ctx* c, const float* params, const float* X, int n, float* Y) {
    if (!c) return PT_E_ARG;
    if (!params || !X || !Y || n < 1) return fail(c, PT_E_ARG, "bad arguments");
    HIPCHK(c, hipSetDevice(c->device));
    Scratch<float> P, bimg, dX, dY;
    Scratch<uint16_t> wimg;
    int rc;
    if ((rc = dscratch(c, P, MLP_NPARAM)) || (rc = dscratch(c, wimg, I_NW)) || (rc = dscratch(c, bimg, I_NB)) ||
        (rc = dscratch(c, dX, (size_t)n * MLP_IN)) || (rc = dscratch(c, dY, 2 * (size_t)n)))
        return rc;
    HIPCHK(c, hipMemcpy(P.p, params, sizeof(float) * MLP_NPARAM, hipMemcpyHostToDevice));
    HIPCHK(c, hipMemcpy(dX.p, X, sizeof(float) * (size_t)n * MLP_IN, hipMemcpyHostToDevice));
    if ((rc = mlp_image(c, P.p, wimg.p, bimg.p))) return rc;
    hipLaunchKernelGGL(k_mlp_infer, dim3(nblk(n, 256)), dim3(256), 0, c->stream, -1, wimg.p, bimg.p, dX.p, n, dY.p);
    HIPCHK(c, hipGetLastError());
    HIPCHK(c, hipStreamSynchronize(c->stream));
    HIPCHK(c, hipMemcpy(Y, dY.p, sizeof(float) * 2 * (size_t)n, hipMemcpyDeviceToHost));
    return PT_OK;
}


int pt_set_wall(pt_ctx* c, int sp, int coord, double v, int drop, size_t capacity) {
    if (!c) return PT_E_ARG;
    if (sp < 0 || sp >= PT_NSPECIES || coord < -1 || coord > 2) return fail(c, PT_E_ARG, "bad wall arguments");
    HIPCHK(c, hipSetDevice(c->device));
    if (coord >= 0 && capacity > c->wall_cap) {
        int rc;
        if ((rc = dalloc(c, (void**)&c->dwall, sizeof(pt_wall_record) * capacity))) return rc;
        if (!c->dwall_n) {
            if ((rc = dalloc(c, (void**)&c->dwall_n, sizeof(ull)))) return rc;
            HIPCHK(c, hipMemsetAsync(c->dwall_n, 0, sizeof(ull), c->stream));
        }
        c->wall_cap = capacity;
    }
    WallDev& W = c->hp.wall;
    W.coord[sp] = coord;
    W.v[sp] = v;
    W.drop[sp] = drop ? 1 : 0;
    W.rec = c->dwall;
    W.n = c->dwall_n;
    W.cap = c->wall_cap;
    W.on = 0;
    for (int q = 0; q < PT_NSPECIES; q++)
        if (W.coord[q] >= 0) W.on = 1;
    if (W.on && !c->dwall) return fail(c, PT_E_ARG, "a wall needs a record capacity");
    c->dirty = true;
    int rc = sync_params(c);
    if (rc) return rc;
    HIPCHK(c, hipStreamSynchronize(c->stream));
    return PT_OK;
}

int pt_wall_read(pt_ctx* c, pt_wall_record* out, size_t cap, size_t* n, int reset) {
    if (!c) return PT_E_ARG;
    HIPCHK(c, hipSetDevice(c->device));
    ull m = 0;
    if (c->dwall_n) {
        HIPCHK(c, hipMemcpyAsync(&m, c->dwall_n, sizeof(ull), hipMemcpyDeviceToHost, c->stream));
        HIPCHK(c, hipStreamSynchronize(c->stream));
    }
    if (n) *n = (size_t)m;
    size_t k = (size_t)std::min<ull>(m, c->wall_cap);
    if (out && k) {
        if (k > cap) return fail(c, PT_E_CAPACITY, "host buffer of %zu too small for %zu wall records", cap, k);
        HIPCHK(c, hipMemcpy(out, c->dwall, sizeof(pt_wall_record) * k, hipMemcpyDeviceToHost));
    }
    if (reset && c->dwall_n) {
        HIPCHK(c, hipMemsetAsync(c->dwall_n, 0, sizeof(ull), c->stream));
        HIPCHK(c, hipStreamSynchronize(c->stream));
    }
    return PT_OK;
}

// roulette! / split! with a constant factor (v == NULL) or one value per slot in use
static int roulette_split(pt_ctx* c, bool split, int sp, double f, const double* v, size_t n) {
    HIPCHK(c, hipSetDevice(c->device));
    int rc = sync_params(c);
    if (rc) return rc;
    if ((rc = read_counts(c))) return rc;
    if (v && n != c->hn[sp])
        return fail(c, PT_E_ARG, "%zu values given for %llu slots in use", n, (unsigned long long)c->hn[sp]);
    if (v)
        for (size_t i = 0; i < n; i++)
            if (split ? !(v[i] >= 0.0 && v[i] <= 100.0) : !(v[i] > 0.0 && v[i] <= 1.0))
                return fail(c, PT_E_ARG, "slot %zu: %s %g out of range", i, split ? "mean" : "probability", v[i]);
    Scratch<double> dv;
    if (v && n) {
        if ((rc = dscratch(c, dv, n))) return rc;
        HIPCHK(c, hipMemcpyAsync(dv.p, v, sizeof(double) * n, hipMemcpyHostToDevice, c->stream));
    }
    c->counts_known = false;
    if (c->hn[sp]) {
        int blocks = (int)std::min<ull>((ull)c->grid, (c->hn[sp] + 255) / 256);
        if (split)
            hipLaunchKernelGGL(k_split, dim3(blocks), dim3(256), 0, c->stream, c->dp, sp, f, (const double*)dv.p, c->step,
                               (ull)c->hn[sp]);
        else
            hipLaunchKernelGGL(k_roulette, dim3(blocks), dim3(256), 0, c->stream, c->dp, sp, f, (const double*)dv.p,
                               c->step, (ull)c->hn[sp]);
        HIPCHK(c, hipGetLastError());
    }
    if ((rc = read_state(c))) return rc;
    return check_flags(c, nullptr);
}

int pt_roulette(pt_ctx* c, int sp, double q) {
    if (!c) return PT_E_ARG;
    if (sp < 0 || sp >= PT_NSPECIES || !(q > 0.0) || q > 1.0) return fail(c, PT_E_ARG, "bad roulette arguments");
    return roulette_split(c, false, sp, q, nullptr, 0);
}

int pt_split(pt_ctx* c, int sp, double f) {
    if (!c) return PT_E_ARG;
    if (sp < 0 || sp >= PT_NSPECIES || !(f >= 0.0) || f > 100.0) return fail(c, PT_E_ARG, "bad split arguments");
    return roulette_split(c, true, sp, f, nullptr, 0);
}

int pt_roulette_each(pt_ctx* c, int sp, const double* q, size_t n) {
    if (!c) return PT_E_ARG;
    if (sp < 0 || sp >= PT_NSPECIES || (n && !q)) return fail(c, PT_E_ARG, "bad roulette arguments");
    return roulette_split(c, false, sp, 1.0, q, n);
}

int pt_split_each(pt_ctx* c, int sp, const double* f, size_t n) {
    if (!c) return PT_E_ARG;
    if (sp < 0 || sp >= PT_NSPECIES || (n && !f)) return fail(c, PT_E_ARG, "bad split arguments");
    return roulette_split(c, true, sp, 0.0, f, n);
}


int pt_set_forcing(pt_ctx* c, uint32_t field_species, uint32_t loss_species, uint32_t push_species) {
    if (!c) return PT_E_ARG;
    const uint32_t all = (1u << PT_NSPECIES) - 1u;
    if ((field_species | loss_species | push_species) & ~all)
        return fail(c, PT_E_ARG, "species masks have bits beyond the %d species", PT_NSPECIES);
    HIPCHK(c, hipSetDevice(c->device));
    uint32_t off = 0;
    for (int s = 0; s < PT_NSPECIES; s++) {
        if (!((field_species >> s) & 1u)) off |= off_em(s);
        if (!((loss_species >> s) & 1u)) off |= off_cl(s);
        if (!((push_species >> s) & 1u)) off |= off_push(s);
    }
    c->hp.forcing_off = off;
    c->dirty = true;
    int rc = sync_params(c);
    if (rc) return rc;
    HIPCHK(c, hipStreamSynchronize(c->stream));
    return PT_OK;
}

int pt_set_continuum_loss(pt_ctx* c, int nintervals, int order, double xmax, const double* electron,
                          const double* positron) {
    if (!c) return PT_E_ARG;
    HIPCHK(c, hipSetDevice(c->device));
    const bool on = electron && positron;
    if (on && (nintervals < 1 || nintervals >= MAX_INTERVALS || order < 1 || order > 16 || !(xmax > 0)))
        return fail(c, PT_E_ARG, "bad continuum-loss table (k in 1..%d, order in 1..16, xmax > 0)", MAX_INTERVALS - 1);
    ContLoss cl{};
    if (on) {
        const size_t m = (size_t)(nintervals + 1) * order;
        double* d[2] = {nullptr, nullptr};
        for (int q = 0; q < 2; q++) {
            int rc = dalloc(c, (void**)&d[q], sizeof(double) * m);
            if (rc) return rc;
            HIPCHK(c, hipMemcpyAsync(d[q], q == 0 ? electron : positron, sizeof(double) * m, hipMemcpyHostToDevice,
                                     c->stream));
        }
        cl.c[0] = d[0];
        cl.c[1] = d[1];
        cl.xmax = xmax;
        cl.ixmax = 1.0 / xmax;
        cl.k = nintervals;
        cl.order = order;
        cl.on = 1;
    }
    for (auto& F : c->hfields) F.cl = cl;
    HIPCHK(c, hipMemcpyAsync(c->dfields, c->hfields.data(), sizeof(Field) * c->hfields.size(), hipMemcpyHostToDevice,
                             c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    c->dirty = true;  // the choice of the fields' LDS form may change
    return sync_params(c);
}

}  // extern "C"

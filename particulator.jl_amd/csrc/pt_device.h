// pt_device.h -- device code of the null-collision step: constants, the uid-keyed Philox
// stream, kinematics, the binary-interval Chebyshev rate tables, the RK2 push and every
// collision sampler.  Compiled for gfx950 with -ffp-contract=off: the arithmetic follows
// the reference's Julia evaluation order (a*b*c == (a*b)*c, x^2 == x*x, x^3 == x*x*x,
// left-fold sums), so selection, indices and pushes are bit-identical to a CPU
// restatement of the same code; transcendental functions come from the ROCm device
// library.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/particulator_hip.h"
#include "pt_consts.h"
#include "pt_math.h"

namespace pt {

// Explicit address spaces for pointers held in structs (the compiler cannot trace them to
// their allocation): a generic pointer becomes a flat access, whose wait covers both the
// LDS and the global counters.
#define PT_LDS __attribute__((address_space(3)))
#define PT_GLOBAL __attribute__((address_space(1)))
template <typename T>
__device__ __forceinline__ const PT_LDS T* as_lds(const T* p) {
    return (const PT_LDS T*)p;
}
template <typename T>
__device__ __forceinline__ const PT_GLOBAL T* as_global(const T* p) {
    return (const PT_GLOBAL T*)p;
}
// atomicAdd on a counter in global memory, issued as a global (not flat) atomic
__device__ __forceinline__ unsigned long long global_add(unsigned long long* p, unsigned long long v) {
    return __hip_atomic_fetch_add((unsigned long long PT_GLOBAL*)p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// the table of pt_math.h: in global memory, and staged at the start of the step kernels' dynamic
// LDS
static __device__ const double g_math[MATH_DOUBLES] = {PT_MATH_TABLE};
extern __shared__ __attribute__((aligned(16))) double pt_lds[];

constexpr int MAX_PROCS = 24;
constexpr int MAX_INTERVALS = 64;
constexpr int MAX_SHELLS = 8;
constexpr int MAX_SB = 4;
constexpr int MAX_PE = 4;
// at most this many swarms keep their (homogeneous) fields in LDS: 48 B each, 12 KB in all,
// which keeps two 256-thread step workgroups per CU
constexpr int MAX_LDS_FIELDS = 256;
// Hard limits that bound every loop of a particle's step: uniforms drawn and loop
// iterations.  Reaching one sets the sampler error flag and ends the particle's step.
constexpr uint32_t DRAW_LIMIT = 1u << 24;
constexpr uint32_t ITER_LIMIT = 1u << 22;

// ---------------------------------------------------------------- device tables
struct DevProc {
    int kind, Z, slot, N;
    double B, U, tcut, zf;
    double c[4];
};

struct DevTable {
    int nprocs, k, nswarm, valid;
    double xmax, cut;
    const double* rate;       // [(k+1)][L][3]
    const double* ratebound;  // [nswarm][(k+1)][3]
    DevProc procs[MAX_PROCS];
};

struct DevSB {
    int ne, ncum;
    const double* log_energy;  // [ne]
    const double* thr;         // [ne]: smallest T with log(T) > log_energy[j] (pt_sb_thresholds)
    const double* data;        // [ne][ncum]
};

// searchsortedfirst(log_energy, log(T)) (1-based, src/seltzer.jl:104) from the thresholds:
// log_energy[j] < log(T) exactly when T >= thr[j], so the cell is found by comparisons of T
// alone and equals the host libm's on every input
__host__ __device__ inline int sb_cell(const double* thr, int ne, double T) {
    int lo = 0, hi = ne;  // number of thresholds <= T
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (thr[mid] <= T) lo = mid + 1;
        else hi = mid;
    }
    return lo + 1;
}

struct DevPE {
    int nshell;
    double binding[MAX_SHELLS];
};

struct FieldFn {
    int kind, pad;
    double v[3], v2[3];
    double z1, z2, sx, sy, sz, ez0;
};
// ChebContinuumLoss (src/continuum.jl:21-59): friction -f(E) p/|p| on e- and e+, f a
// Chebyshev expansion of `order` terms on BinaryIntervals(k, xmax); coefficients per species
// [(k+1)][order] (the reference's (order, k+1) column-major)
struct ContLoss {
    const double* c[2];  // electron, positron
    double xmax, ixmax;  // ixmax = 1 / xmax
    int k, order, on, pad;
};

struct Field {
    FieldFn e, b;
    ContLoss cl;  // CombinedForcing(field, continuum loss) when on
};

// Restrictions of the forcing and the pusher as RestrictedForcing / RestrictedPusher /
// NullPusher make them (src/pusher.jl:27-34, :66-76), one word for the context (bit s of
// each 3-bit group: species s): bits 0-2, the electromagnetic force is zero for the species;
// bits 3-5, the continuum loss is; bits 6-8, the species is not pushed and only its time
// advances.  Zero: no restriction.  The step reads it once per kernel.
__host__ __device__ constexpr uint32_t off_em(int sp) { return 1u << sp; }
__host__ __device__ constexpr uint32_t off_cl(int sp) { return 8u << sp; }
__host__ __device__ constexpr uint32_t off_push(int sp) { return 64u << sp; }
// Set by the library, not a restriction: every swarm's B is zero and its E homogeneous (or
// absent) with no component -0.0.  Then each component of v x B is +0 or -0, and E + v x B
// equals E bit for bit, so the electromagnetic force is qE.
constexpr uint32_t OFF_NO_B = 1u << 9;
// Set by the library: every swarm's E is homogeneous and along z.
constexpr uint32_t OFF_E_Z = 1u << 10;

// ---------------------------------------------------------------- Philox4x32-10
// Salmon et al., SC'11: multipliers 0xD2511F53, 0xCD9E8D57; key increments 0x9E3779B9,
// 0xBB67AE85; ten rounds.  The key is the same for every lane of a wave (it is always the
// context's seed, or a kernel argument): read from the first active lane, the key schedule
// runs on the scalar unit, and each round costs four vector instructions (two 32x32->64
// products, two three-input XORs).
__device__ __forceinline__ void philox10(uint32_t& c0, uint32_t& c1, uint32_t& c2, uint32_t& c3,
                                         uint32_t k0, uint32_t k1) {
    k0 = __builtin_amdgcn_readfirstlane(k0);
    k1 = __builtin_amdgcn_readfirstlane(k1);
#pragma unroll
    for (int r = 0; r < 10; r++) {
        if (r) {
            k0 += 0x9E3779B9u;
            k1 += 0xBB67AE85u;
        }
        // one 32x32->64 product per word (a single v_mad_u64_u32) instead of separate
        // high and low multiplies
        const uint64_t m0 = (uint64_t)0xD2511F53u * c0, m1 = (uint64_t)0xCD9E8D57u * c2;
        uint32_t hi0 = (uint32_t)(m0 >> 32), lo0 = (uint32_t)m0;
        uint32_t hi1 = (uint32_t)(m1 >> 32), lo1 = (uint32_t)m1;
        // a ^ b ^ c in one v_bitop3_b32 (truth table 0x96)
        uint32_t n0 = __builtin_amdgcn_bitop3_b32(hi1, c1, k0, 0x96);
        uint32_t n2 = __builtin_amdgcn_bitop3_b32(hi0, c3, k1, 0x96);
        c0 = n0;
        c1 = lo1;
        c2 = n2;
        c3 = lo0;
    }
}

// 64 random bits -> (0,1): with m the top 52 bits, (m + 1/2) 2^-52.  Built from bits: the
// double 1 + m 2^-52 (exponent of 1, mantissa m) minus (1 - 2^-53) is (2m + 1) 2^-53, which
// has 53 significant bits, so the subtraction is exact and the value is (m + 1/2) 2^-52 bit
// for bit, in four instructions instead of two conversions, a scaling and two additions.
__device__ __forceinline__ double u01(uint32_t lo, uint32_t hi) {
    const uint32_t mlo = __builtin_amdgcn_alignbit(hi, lo, 12);  // bits 12..43 of (hi:lo)
    const uint32_t mhi = (hi >> 12) | 0x3FF00000u;
    return __hiloint2double((int)mhi, (int)mlo) - (1.0 - 0x1p-53);
}

// uniform stream of one particle in one step: counter (uid, step, draw/2), key = seed
struct PhiloxStream {
    uint32_t k0, k1, u0, u1, step;
    uint32_t draw;
    uint32_t cblk;
    double c0, c1;
    __device__ const PT_GLOBAL double* tab() const { return as_global(g_math); }
    __device__ bool exhausted() const { return draw >= DRAW_LIMIT; }
    __device__ void init(uint64_t seed, uint64_t uid, uint32_t st) {
        k0 = (uint32_t)seed;
        k1 = (uint32_t)(seed >> 32);
        u0 = (uint32_t)uid;
        u1 = (uint32_t)(uid >> 32);
        step = st;
        draw = 0;
        cblk = 0;
    }
    __device__ uint64_t uid() const { return (uint64_t)u1 << 32 | u0; }
    // the same particle's stream of another step
    __device__ __forceinline__ void restart(uint32_t st) {
        step = st;
        draw = 0;
        cblk = 0;
    }
    // Invariant: when `draw` is odd, the block holding draw - 1 (and draw) is cached.  next()
    // keeps it by itself; skip() and resume() compute the block when they leave `draw` odd.
    __device__ __forceinline__ void fill(uint32_t blk) {
        uint32_t a = u0, b = u1, c = step, e = blk;
        philox10(a, b, c, e, k0, k1);
        c0 = u01(a, b);
        c1 = u01(c, e);
        cblk = blk + 1;
    }
    // continue the stream at draw d0 (a particle resumed by another kernel)
    __device__ __forceinline__ void resume(uint32_t d0) {
        draw = d0;
        if (d0 & 1) fill(d0 >> 1);
    }
    // advance past one draw whose value is not needed
    __device__ __forceinline__ void skip() {
        const uint32_t d = draw++;
        if (!(d & 1) && cblk != (d >> 1) + 1) fill(d >> 1);
    }
    __device__ __forceinline__ double next() {
        uint32_t d = draw++;
        uint32_t blk = d >> 1;
        if (cblk != blk + 1) fill(blk);
        return (d & 1) ? c1 : c0;
    }
    // the next k = 1 or 2 uniforms (b is set when k == 2), as k next() calls return them,
    // with at most one Philox block computed, at one place
    __device__ __forceinline__ void next12(int k, double& a, double& b) {
        const uint32_t d = draw;
        draw = d + (uint32_t)k;
        const double first = c1;  // draw d when d is odd (the invariant)
        const uint32_t need = (d + (uint32_t)k - 1u) >> 1;
        if (cblk != need + 1) fill(need);
        a = (d & 1) ? first : c0;
        b = (d & 1) ? c0 : c1;
    }
    // the next two uniforms, as two next() calls return them, with at most one Philox block
    // computed at one place: in a rejection loop every lane needs its block at the same
    // instruction, instead of half of the lanes at each of two draw sites
    __device__ __forceinline__ void next2(double& a, double& b) {
        const uint32_t d = draw;
        draw = d + 2;
        const double first = c1;  // draw d when d is odd (the invariant)
        const uint32_t need = (d + 1) >> 1;
        if (cblk != need + 1) fill(need);
        a = (d & 1) ? first : c0;
        b = (d & 1) ? c0 : c1;
    }
};

// the stream in the step kernels, where the math table is in LDS
struct StepStream : PhiloxStream {
    __device__ const PT_LDS double* tab() const { return as_lds(pt_lds); }
};

// injected uniforms (test hook): consumed in order, 0.5 once exhausted
struct InjectedStream {
    const double* u;
    int n, pos;
    uint32_t draw;
    bool ran_out;
    __device__ const PT_GLOBAL double* tab() const { return as_global(g_math); }
    __device__ bool exhausted() const { return ran_out; }
    __device__ __forceinline__ void skip() { (void)next(); }
    __device__ __forceinline__ double next() {
        draw++;
        if (pos >= n) {
            ran_out = true;
            return 0.5;
        }
        return u[pos++];
    }
    __device__ __forceinline__ void next2(double& a, double& b) {
        a = next();
        b = next();
    }
    __device__ __forceinline__ void next12(int k, double& a, double& b) {
        a = next();
        b = k == 2 ? next() : 0.0;
    }
};

// uid of the k-th particle created by the event that ended at draw `draw` of the stream
// (uid, step): a Philox counter with the top bit of word 3 set (never a uniform draw)
__device__ __forceinline__ uint64_t child_uid(uint64_t seed, uint64_t uid, uint32_t step,
                                              uint32_t draw, int k) {
    uint32_t a = (uint32_t)uid, b = (uint32_t)(uid >> 32), c = step;
    uint32_t e = 0x80000000u | ((draw & 0x3FFFFFFFu) << 1) | (uint32_t)(k & 1);
    philox10(a, b, c, e, (uint32_t)seed, (uint32_t)(seed >> 32));
    return ((uint64_t)b << 32) | a;
}

// -log(u) of a draw: a stream's are in (0, 1), an injected one may be zero
template <class G>
__device__ __forceinline__ double neg_log(double u, G& g) {
    return -log_tab(u, g.tab());
}
__device__ __forceinline__ double neg_log(double u, InjectedStream& g) {
    return u == 0.0 ? __builtin_inf() : -log_tab(u, g.tab());
}

template <class G>
__device__ __forceinline__ double nextcoll(G& g) {  // src/util.jl:17
    return neg_log(g.next(), g);
}

// ---------------------------------------------------------------- kinematics
struct V3 {
    double x, y, z;
};
__device__ __forceinline__ double dot3(const V3& a, const V3& b) {
    return (a.x * b.x + a.y * b.y) + a.z * b.z;
}
__device__ __forceinline__ double norm3(const V3& a) { return qsqrt(dot3(a, a)); }

// a / b for a constant b with inv = 1/b correctly rounded: the product a * inv is within an
// ulp of a/b, the remainder a - q b is exact in one FMA, and one more FMA rounds the quotient
// correctly (Markstein, IBM J. Res. Dev. 34 (1990) 111-119), so the result is a / b bit for
// bit (normal operands; NaN and infinity pass through) in three operations instead of a
// full division
__device__ __forceinline__ double div_const(double a, double b, double inv) {
    const double q = a * inv;
    const double r = fma(-q, b, a);
    return (r == 0.0 || r != r) ? q : fma(r, inv, q);
}

// the same for finite operands, without the test of the remainder
__device__ __forceinline__ double div_const_fin(double a, double b, double inv) {
    const double q = a * inv;
    return fma(fma(-q, b, a), inv, q);
}

// src/electron.jl:53, src/photon.jl:52.  Photons and electrons of a wave share the root.
__device__ __forceinline__ double kinenergy(int sp, const V3& p) {
    const double pp = dot3(p, p);
    const bool ph = sp == PT_PHOTON;
    const double q = qsqrt(ph ? pp : MC2 * MC2 + C2 * pp);
    return ph ? q * C : q - MC2;
}
// src/electron.jl:51
__device__ __forceinline__ double mom_from_kin(int sp, double kin) {
    if (sp == PT_PHOTON) return kin / C;
    double a = kin + MC2;
    return sqrt(a * a - MC2 * MC2) / C;
}
// src/electron.jl:54-56, src/photon.jl:47: p c / |p|, or p / (m gamma)
__device__ __forceinline__ V3 velocity(int sp, const V3& p) {
    constexpr double MC2SQ = MC2 * MC2;
    const double pp = dot3(p, p);
    const bool ph = sp == PT_PHOTON;
    const double q = qsqrt(ph ? pp : 1.0 + div_const_fin(C2 * pp, MC2SQ, 1.0 / MC2SQ));
    const double f = qdiv(ph ? C : 1.0, ph ? q : ME * q);
    return V3{p.x * f, p.y * f, p.z * f};
}

// ---------------------------------------------------------------- Chebyshev
// precheb, src/cheby.jl:127-143 (+ chebval :57-81).  The index is clamped to [0, k]
// (the reference reads out of bounds above xmax); `oob` reports it.
// two_k1 = 2^(k+1).
__device__ __forceinline__ int precheb(double x, int k, double xmax, double ixmax, double two_k1, double& t1,
                                       double& t2, bool& oob) {
    // x / xmax (ixmax = 1 / xmax) and its frexp
    const double x1 = div_fixup(div_const_fin(x, xmax, ixmax), xmax, x);
    const double s = frexp_mant(x1);
    int i = (x1 == 0.0) ? 0 : frexp_exp(x1) + k;
    // 4 s - 3, or 2^(k+1) x1 - 1 in the lowest interval (the products are exact)
    const bool low = i <= 0;
    const double xi = fma(low ? two_k1 : 4.0, low ? x1 : s, low ? -1.0 : -3.0);
    i = low ? 0 : i;
    t1 = xi;
    t2 = 2.0 * xi * xi - 1.0;
    oob = i > k;
    return i > k ? k : i;
}

// sum(ntuple(k -> c[k]*t[k], Val(3))), src/collision_table.jl:91,105
template <typename Ptr>
__device__ __forceinline__ double cheb3(Ptr c, double t1, double t2) {
    return (c[0] * 1.0 + c[1] * t1) + c[2] * t2;
}

// ---------------------------------------------------------------- turn, sphere
// turn, src/util.jl:40-57.  Where the reference yields NaN, 1 - cos^2 < 0 (rounding) is
// clamped to 0 and an exactly axial direction (s == 0) uses the axis-aligned rotation.
__device__ __forceinline__ V3 turn(const V3& u, double cost, double phi, double n) {
    double nrm = norm3(u);
    double m0 = u.x / nrm, m1 = u.y / nrm, m2 = u.z / nrm;
    double sp, cp;
    sincos(phi, &sp, &cp);
    double q = 1.0 - cost * cost;
    double sint = sqrt(q > 0.0 ? q : 0.0);
    double qs = 1.0 - m2 * m2;
    double s = sqrt(qs > 0.0 ? qs : 0.0);
    double x, y, z;
    if (s > 0.0) {
        double bx = m0 * m2 * cp + (-m1) * sp;
        double by = m1 * m2 * cp + m0 * sp;
        x = sint * bx / s + m0 * cost;
        y = sint * by / s + m1 * cost;
        z = -s * sint * cp + m2 * cost;
    } else {
        x = sint * cp;
        y = sint * sp;
        z = m2 * cost;
    }
    return V3{n * x, n * y, n * z};
}

// randsphere, src/util.jl:4-12
template <class G>
__device__ __forceinline__ V3 randsphere(G& g) {
    double phi = TWO_PI * g.next();
    double sp, cp;
    sincos(phi, &sp, &cp);
    double u = 2.0 * g.next() - 1.0;
    double v = sqrt(1.0 - u * u);
    return V3{v * cp, v * sp, u};
}

// ---------------------------------------------------------------- samplers
// sample_modified_tsai_cos_theta, src/util.jl:143-159
template <class G>
__device__ __forceinline__ double sample_tsai(double T, G& g) {
    double umax = 2.0 * (1.0 + T / (ME * C2));
    const double a1 = 1.6, a2 = 1.6 / 3.0, border = 0.25;
    double u;
    for (;;) {
        double r1 = g.next();
        double r2 = g.next();
        double uu = -log(r1 * r2);
        u = border > g.next() ? uu * a1 : uu * a2;
        if (u <= umax || g.exhausted()) break;
    }
    return 1.0 - 2.0 * (u * u) / (umax * umax);
}

// sample_rel_sr, src/relativistic_coulomb.jl:35-51
template <class G>
__device__ __forceinline__ double sample_rel_sr(double alpha, double beta, G& g) {
    double x;
    for (;;) {
        double u, z;
        g.next2(u, z);
        x = qdiv(alpha * u, alpha + 1.0 - u);
        if (z < 1.0 - beta * beta * x || g.exhausted()) break;
    }
    return 1.0 - 2.0 * x;
}

// rbeb_sample / _rbeb_sample, src/rbeb.jl:156-196, in three parts: the constants of the
// rejection loop, one trip (uniforms u, z), and the loop.  A trip is a function of the two
// uniforms alone, so the wave can also run the trips of its particles in parallel.
struct RbebSetup {
    double t, A, Cc, M, pbn, ratio, iratio;
};
// The orbital's own terms come with the process (set when the table is uploaded): pr.c[0] =
// b' = B / mc^2, pr.c[1] = log(2 b'), pr.c[2] = 1 / B.  T / mc^2 and T / B are exact
// divisions by constants (div_const).
template <class T_>
__device__ __forceinline__ RbebSetup rbeb_setup(double T, double B, double c0, double c1, double c2, T_ tab) {
    RbebSetup s;
    const double t1 = div_const_fin(T, MC2, 1.0 / MC2);
    const Recip g2((1.0 + t1) * (1.0 + t1));
    const double bt2 = 1.0 - g2.inverse();
    const double b1 = c0;
    s.t = div_const_fin(T, B, c2);
    s.A = g2(qdiv(-(1.0 + 2.0 * t1), s.t + 1.0));
    s.Cc = (log_tab(qdiv(bt2, 1.0 - bt2), tab) - bt2) - c1;
    s.M = g2(b1 * b1);
    s.pbn = 2.0 * 1.0 + 2.0 * s.Cc + (s.t + 1.0) * (s.t + 1.0) * 1.0 * s.M / 4.0;
    s.ratio = qdiv_any(s.t + 1.0, s.t - 1.0);
    s.iratio = qdiv_any(1.0, s.ratio);
    return s;
}
// One trip: w (exact) and whether it is accepted.  The reference's 1/(1+w)^k and
// 1/(t-w)^k come from 1/(1+w) = (ratio - u) / ratio and one reciprocal (two divisions
// instead of eight): the acceptance terms are within a few ulps of the reference's, so
// only a z * pb within ~1e-15 of p0 could be decided otherwise.
__device__ __forceinline__ bool rbeb_trip(const RbebSetup& s, double u, double z, double& w) {
    const double den = s.ratio - u;
    w = qdiv(u, den);
    double tw = s.t - w;
    double ra = den * s.iratio, rt = Recip(tw).inverse();
    double ra2 = ra * ra, rt2 = rt * rt;
    double pb = s.pbn * ra2;
    double g1 = ra + rt;
    double g2 = ra2 + rt2;
    double g3 = ra2 * ra + rt2 * rt;
    double p0 = s.A * g1 + 1.0 * (g2 + s.M) + s.Cc * g3;
    return z * pb < p0;
}
template <class G>
__device__ __forceinline__ double rbeb_sample(double T, const DevProc& pr, G& g) {
    const RbebSetup s = rbeb_setup(T, pr.B, pr.c[0], pr.c[1], pr.c[2], g.tab());
    double w;
    for (;;) {
        double u, z;
        g.next2(u, z);
        if (rbeb_trip(s, u, z, w) || g.exhausted()) break;
    }
    return pr.B * w;
}

// sample_secondary_energy(::Moller), src/moller.jl:64-87
template <class G>
__device__ __forceinline__ double moller_sample(double tcut, double eng, G& g) {
    double e0 = tcut / eng;
    double gm = 1.0 + eng / MC2;
    double pre = 4.0 / (9.0 * (gm * gm) - 10.0 * gm + 5.0);
    double ca = (gm - 1.0) * (gm - 1.0);
    double cb = 2.0 * (gm * gm) + 2.0 * gm - 1.0;
    double cc = gm * gm;
    double eps;
    for (;;) {
        double r, z;
        g.next2(r, z);
        eps = e0 / (1.0 - r + 2.0 * e0 * r);
        double om = 1.0 - eps;
        double gg = pre * (ca * (eps * eps) - cb * (eps / om) + cc / (om * om));
        if (z < gg || g.exhausted()) break;
    }
    return eps * eng;
}

// bhaba_bs, src/bhaba.jl:84-91
__device__ __forceinline__ void bhabha_bs(double y, double& B1, double& B2, double& B3,
                                          double& B4) {
    double q = 1.0 - 2.0 * y;
    B1 = 2.0 - y * y;
    B2 = q * (3.0 + y * y);
    B3 = q * q + q * q * q;
    B4 = q * q * q;
}

// sample_secondary_energy(::Bhaba), src/bhaba.jl:55-81
template <class G>
__device__ __forceinline__ double bhabha_sample(double tcut, double eng, G& g) {
    double e0 = tcut / eng;
    double gm = 1.0 + eng / MC2;
    double y = 1.0 / (gm + 1.0);
    double B0 = gm * gm / (gm * gm - 1.0);
    double B1, B2, B3, B4;
    bhabha_bs(y, B1, B2, B3, B4);
    double g2 = (((B0 + B1 * e0) + B2 * (e0 * e0)) + B3 * (e0 * e0 * e0)) + B4 * pow(e0, 4.0);
    double eps;
    for (;;) {
        double r, z;
        g.next2(r, z);
        eps = e0 / (1.0 - r + e0 * r);
        double g1 = (((B0 + B1 * eps) + B2 * (eps * eps)) + B3 * (eps * eps * eps)) +
                    B4 * pow(eps, 4.0);
        double gg = g1 / g2;
        if (z < gg || g.exhausted()) break;
    }
    return eps * eng;
}

// searchsortedfirst(LinRange(0,1,ncum), x): first i (1-based) with (i-1)/(ncum-1) >= x
__device__ __forceinline__ int pcum_first(double x, int ncum) {
    double d = (double)(ncum - 1);
    int i = (int)(x * d) + 1;
    if (i < 1) i = 1;
    if (i > ncum) i = ncum;
    while (i > 1 && (double)(i - 2) / d >= x) i--;
    while (i < ncum && (double)(i - 1) / d < x) i++;
    return i;
}

// sample_secondary_energy(::SeltzerBerger), src/seltzer.jl:97-122.  Returns k/T, or a
// negative value where the reference indexes out of bounds.
template <class G>
__device__ __forceinline__ double sb_sample(const DevSB& sb, double T, G& g) {
    double x = g.next();
    double y = log(T);
    int ncum = sb.ncum;
    double d = (double)(ncum - 1);
    int i2 = pcum_first(x, ncum), i1 = i2 - 1;
    int j2 = sb_cell(sb.thr, sb.ne, T), j1 = j2 - 1;
    if (i1 < 1 || j1 < 1 || j2 > sb.ne) return -1.0;
    double x1 = (double)(i1 - 1) / d, x2 = (double)(i2 - 1) / d;
    double y1 = sb.log_energy[j1 - 1], y2 = sb.log_energy[j2 - 1];
    const double* c1 = sb.data + (size_t)(j1 - 1) * ncum;
    const double* c2 = sb.data + (size_t)(j2 - 1) * ncum;
    double A = (x2 - x1) * (y2 - y1);
    double S = c1[i1 - 1] * (x2 - x) * (y2 - y) + c2[i1 - 1] * (x - x1) * (y2 - y);
    S = S + c1[i2 - 1] * (x2 - x) * (y - y1);
    S = S + c2[i2 - 1] * (x - x1) * (y - y1);
    return exp(S / A);
}

// Position of log T inside its cell of the Seltzer-Berger energy grid, in (0, 1]: the cell
// sb_sample interpolates in (the same search).  Its interpolation swaps the energy corners
// (src/seltzer.jl:116-119), so the sampled distribution jumps at every grid node; a learned
// sampler gets this phase as an input to follow those jumps.
__host__ __device__ inline double sb_phase(const double* log_energy, const double* thr, int ne, double T) {
    double y = log(T);
    const int lo = sb_cell(thr, ne, T) - 1;
    if (lo < 1 || lo >= ne) return 0.0;
    double y1 = log_energy[lo - 1], y2 = log_energy[lo];
    return (y - y1) / (y2 - y1);
}

// sample_secondary_energy_and_cos_theta(::Compton), src/compton.jl:119-144
template <class G>
__device__ __forceinline__ void compton_sample(double eng, G& g, double& E1, double& cost) {
    double e0 = MC2 / (MC2 + 2.0 * eng);
    double a1 = -log(e0);
    double a2 = (1.0 - e0 * e0) / 2.0;
    double thr = a1 / (a1 + a2);
    double t, eps;
    for (;;) {
        if (g.next() < thr) eps = exp(-g.next() * a1);
        else eps = sqrt(e0 * e0 + (1.0 - e0 * e0) * g.next());
        t = MC2 * (1.0 - eps) / (eps * eng);
        double gg = 1.0 - eps / (1.0 + eps * eps) * t * (2.0 - t);
        if (g.next() < gg || g.exhausted()) break;
    }
    cost = 1.0 - t;
    E1 = eps * eng;
}

// sample_electron_cos_theta(::PhotoElectric), src/photo_electric.jl:78-99
template <class G>
__device__ __forceinline__ double sauter_sample(double ee, G& g) {
    double gm = 1.0 + ee / MC2;
    double b = sqrt(1.0 - 1.0 / (gm * gm));
    double A = 1.0 / b - 1.0;
    double k2 = b * gm * (gm - 1.0) * (gm - 2.0) / 2.0;
    double g0 = 2.0 * (1.0 / A + k2);
    double A2 = (A + 2.0) * (A + 2.0);
    double nu;
    for (;;) {
        double xi = g.next();
        nu = 2.0 * A / (A2 - 4.0 * xi) * (2.0 * xi + (A + 2.0) * sqrt(xi));
        double xi1 = g.next();
        double gn = (2.0 - nu) * (1.0 / (A + nu) + k2);
        if (xi1 * g0 < gn || g.exhausted()) break;
    }
    return 1.0 - nu;
}

// _screen_function1/2, src/bethe_heitler.jl:175-193
__device__ __forceinline__ double screen1(double d) {
    return d > 1.4 ? 42.038 - 8.29 * log(d + 0.958) : 42.184 - d * (7.444 - 1.623 * d);
}
__device__ __forceinline__ double screen2(double d) {
    return d > 1.4 ? 42.038 - 8.29 * log(d + 0.958) : 41.326 - d * (5.848 - 0.902 * d);
}
__device__ __forceinline__ double jmax(double a, double b) {
    if (a != a || b != b) return a + b;  // NaN propagates as in Julia's max
    return a > b ? a : b;
}

// sample_secondary_energy(::BetheHeitler), src/bethe_heitler.jl:85-146.  cz = Z^(1/3),
// fz_lo = 8 log(Z)/3, fz_hi = fz_lo + 8 fc (precomputed by the host).  Returns the
// reference's (ekin, pkin).
template <class G>
__device__ __forceinline__ void bh_sample(double cz, double fz_lo, double fz_hi, double eng, G& g,
                          double& ekin, double& pkin) {
    double e0 = MC2 / eng;
    double eps;
    if (eng < 2e6 * EV) {
        eps = e0 + (0.5 - e0) * g.next();
    } else {
        double d0 = 136.0 * e0 / cz;
        double FZ = eng > 50e6 * EV ? fz_hi : fz_lo;
        double dmin = 4.0 * d0;
        double dmax = exp((42.24 - FZ) / 8.368) - 0.952;
        double ep = (1.0 - sqrt(1.0 - dmin / dmax)) / 2.0;
        double emin = e0 > ep ? e0 : ep;
        double erange = 0.5 - emin;
        double F10 = screen1(dmin) - FZ, F20 = screen2(dmin) - FZ;
        double NF1 = jmax(F10 * (erange * erange), 0.0);
        double NF2 = jmax(1.5 * F20, 0.0);
        double NC = NF1 / (NF1 + NF2);
        for (;;) {
            bool acc;
            if (NC > g.next()) {
                eps = 0.5 - erange * pow(g.next(), 1.0 / 3.0);
                double d = d0 / (eps * (1.0 - eps));
                acc = g.next() < (screen1(d) - FZ) / F10;
            } else {
                eps = emin + erange * g.next();
                double d = d0 / (eps * (1.0 - eps));
                acc = g.next() < (screen2(d) - FZ) / F20;
            }
            if (acc || g.exhausted()) break;
        }
    }
    double etot, ptot;
    if (g.next() < 0.5) {  // rand(Bool), src/bethe_heitler.jl:133
        etot = (1.0 - eps) * eng;
        ptot = eps * eng;
    } else {
        ptot = (1.0 - eps) * eng;
        etot = eps * eng;
    }
    ekin = jmax(0.0, etot - MC2);
    pkin = jmax(0.0, ptot - MC2);
}

// sample_secondary_energy_fraction(::PositronAnihilation), src/anihilation.jl:39-59
template <class G>
__device__ __forceinline__ double annih_sample(double eng, G& g) {
    double gm = 1.0 + eng / MC2;
    double sq = sqrt((gm - 1.0) / (gm + 1.0));
    double emax = (1.0 + sq) / 2.0, emin = (1.0 - sq) / 2.0;
    double ratio = emax / emin;
    double den = (gm + 1.0) * (gm + 1.0);
    double eps;
    for (;;) {
        double r, z;
        g.next2(r, z);
        eps = emin * pow(ratio, r);
        double gg = 1.0 - eps + (2.0 * gm * eps - 1.0) / (eps * den);
        if (z < gg || g.exhausted()) break;
    }
    return eps;
}

// ---------------------------------------------------------------- fields and push
template <class FF>
__device__ __forceinline__ V3 field_eval(const FF& f, const V3& x) {
    switch (f.kind) {
    case PT_FIELD_HOMOGENEOUS:
        return V3{f.v[0], f.v[1], f.v[2]};
    case PT_FIELD_DOUBLELAYER:
        if (f.z1 < x.z && x.z < f.z2) return V3{f.v[0], f.v[1], f.v[2]};
        return V3{0.0, 0.0, 0.0};
    case PT_FIELD_STEP:
        if (x.z < f.z1) return V3{f.v[0], f.v[1], f.v[2]};
        return V3{f.v2[0], f.v2[1], f.v2[2]};
    case PT_FIELD_CONFINED: {
        double g = exp(-(x.x * x.x / (2.0 * (f.sx * f.sx)) + x.y * x.y / (2.0 * (f.sy * f.sy)) +
                         x.z * x.z / (2.0 * (f.sz * f.sz))));
        return V3{-(f.ez0 * g * x.x * x.z) / (f.sx * f.sx), -(f.ez0 * g * x.y * x.z) / (f.sy * f.sy),
                  f.ez0 * g - (f.ez0 * g * (x.z * x.z)) / (f.sz * f.sz)};
    }
    default:
        return V3{0.0, 0.0, 0.0};
    }
}

// The fields of a population whose swarms all have homogeneous E and B and no continuum
// loss, one swarm's six values (E then B) in LDS: the same force as the general form, read
// without a vector memory load
struct HomFieldFn {
    const PT_LDS double* v;
};
__device__ __forceinline__ V3 field_eval(const HomFieldFn& f, const V3&) { return V3{f.v[0], f.v[1], f.v[2]}; }
struct NoLoss {
    static constexpr int on = 0, k = 0, order = 1;
    static constexpr double xmax = 1.0, ixmax = 1.0;
    const double* c[2];
};
struct HomField {
    HomFieldFn e, b;
    NoLoss cl;
};

// force(::ElectromagneticField, s), src/field.jl:62-68
// chebeval with `order` terms (src/cheby.jl:55-81, :111-143): T_j = (2 xi) T_{j-1} - T_{j-2},
// summed left to right; the interval index is clamped to [0, k]
template <typename Ptr>
__device__ __forceinline__ double chebeval_n(Ptr c, int k, int order, double xmax, double ixmax, double x) {
    double t1, t2;
    bool oob;
    int i = precheb(x, k, xmax, ixmax, ldexp(1.0, k + 1), t1, t2, oob);
    Ptr a = c + (size_t)i * order;
    double tm2 = 1.0, tm1 = t1;
    double acc = a[0] * 1.0;
    if (order > 1) acc = acc + a[1] * t1;
    for (int j = 2; j < order; j++) {
        double tj = 2.0 * t1 * tm1 - tm2;
        acc = acc + a[j] * tj;
        tm2 = tm1;
        tm1 = tj;
    }
    return acc;
}

template <class FT>
__device__ __forceinline__ V3 force(int sp, const FT& f, const V3& x, const V3& p, const V3& v, uint32_t off) {
    if (sp == PT_PHOTON) return V3{0.0, 0.0, 0.0};
    V3 F{0.0, 0.0, 0.0};
    if (!(off & off_em(sp))) {
        V3 e = field_eval(f.e, x);
        double q = (sp == PT_ELECTRON ? -1.0 : 1.0) * QE;
        if (off & OFF_NO_B) {
            F = V3{q * e.x, q * e.y, q * e.z};
        } else {
            V3 b = field_eval(f.b, x);
            double cx = v.y * b.z - v.z * b.y;
            double cy = v.z * b.x - v.x * b.z;
            double cz = v.x * b.y - v.y * b.x;
            F = V3{q * (e.x + cx), q * (e.y + cy), q * (e.z + cz)};
        }
    }
    if (f.cl.on && !(off & off_cl(sp))) {
        // CombinedForcing(field, ContinuumLoss): the sum of the forces (src/pusher.jl:14-23);
        // the loss term is p * (-f / |p|) (src/continuum.jl:17-20)
        double fc = chebeval_n(as_global(f.cl.c[sp == PT_ELECTRON ? 0 : 1]), f.cl.k, f.cl.order, f.cl.xmax,
                                f.cl.ixmax, kinenergy(sp, p));
        double sc = -fc / norm3(p);
        F = V3{F.x + p.x * sc, F.y + p.y * sc, F.z + p.z * sc};
    }
    return F;
}

// advance_particle(::RK2Pusher, y, dt), src/pusher.jl:41-63: what a push by dt adds to the
// position and the momentum
template <class FT>
__device__ __forceinline__ void push_delta(int sp, const FT& f, const V3& x, const V3& p, double dt, uint32_t off,
                                           V3& dx, V3& dp) {
    V3 v1 = velocity(sp, p);
    V3 f1 = force(sp, f, x, p, v1, off);
    double dt2 = 2.0 * dt;
    constexpr double THIRD = 1.0 / 3.0;
    V3 x2{x.x + div_const_fin(dt2 * v1.x, 3.0, THIRD), x.y + div_const_fin(dt2 * v1.y, 3.0, THIRD),
          x.z + div_const_fin(dt2 * v1.z, 3.0, THIRD)};
    V3 p2{p.x + div_const_fin(dt2 * f1.x, 3.0, THIRD), p.y + div_const_fin(dt2 * f1.y, 3.0, THIRD),
          p.z + div_const_fin(dt2 * f1.z, 3.0, THIRD)};
    V3 v2 = velocity(sp, p2);
    V3 f2 = force(sp, f, x2, p2, v2, off);
    // dt (v1 / 4 + 3 v2 / 4): the quarters are exact and are taken out of the sum
    const double q = dt * 0.25;
    dx = V3{q * (v1.x + 3.0 * v2.x), q * (v1.y + 3.0 * v2.y), q * (v1.z + 3.0 * v2.z)};
    dp = V3{q * (f1.x + 3.0 * f2.x), q * (f1.y + 3.0 * f2.y), q * (f1.z + 3.0 * f2.z)};
}

// the same for a force F that does not depend on position, momentum or time; `along`: F is
// along z (the other components are zero, and adding a zero changes nothing)
__device__ __forceinline__ void push_uniform(int sp, const V3& F, bool along, const V3& p, double dt, V3& dx, V3& dp) {
    const V3 v1 = velocity(sp, p);
    const double dt2 = 2.0 * dt, q = dt * 0.25;
    constexpr double THIRD = 1.0 / 3.0;
    V3 p2 = p;
    dp = V3{0.0, 0.0, q * (F.z + 3.0 * F.z)};
    p2.z = p.z + div_const_fin(dt2 * F.z, 3.0, THIRD);
    if (!along) {
        p2.x = p.x + div_const_fin(dt2 * F.x, 3.0, THIRD);
        p2.y = p.y + div_const_fin(dt2 * F.y, 3.0, THIRD);
        dp.x = q * (F.x + 3.0 * F.x);
        dp.y = q * (F.y + 3.0 * F.y);
    }
    const V3 v2 = velocity(sp, p2);
    dx = V3{q * (v1.x + 3.0 * v2.x), q * (v1.y + 3.0 * v2.y), q * (v1.z + 3.0 * v2.z)};
}

// the push itself; a species the pusher is restricted away from (RestrictedPusher,
// NullPusher, src/pusher.jl:66-76) only has its time advanced
template <class FT>
__device__ __forceinline__ void push(int sp, const FT& f, V3& x, V3& p, double& t, double dt, uint32_t off) {
    if (!(off & off_push(sp))) {
        V3 dx, dp;
        push_delta(sp, f, x, p, dt, off, dx, dp);
        x = V3{x.x + dx.x, x.y + dx.y, x.z + dx.z};
        p = V3{p.x + dp.x, p.y + dp.y, p.z + dp.z};
    }
    t = t + dt;
}

// ---------------------------------------------------------------- collide
// One real collision, split in two parts so that lanes of a wave that sample different
// processes still share the expensive arithmetic:
//   sample_event: the process-specific draws (energy sharing, polar angles, azimuth) in
//                 the reference's order, producing at most two rotations of the primary's
//                 momentum, turn A = (cA, phi, nA) and turn B = (cB, sgnB*phi, nB);
//   finish_event: both rotations (`turn`, src/util.jl:40-57, sharing the primary's
//                 direction and sincos(phi)) and the constructors' s = nextcoll() draws.
// Every outgoing particle takes turn A, turn B or p - (turn A), listed in constructor order
// (which is the order of the s draws).  The primary either survives as entry 0 (`keep`)
// or is removed (ReplaceParticle*Outcome, src/collisions.jl:112-133).
enum { SRC_A = 0, SRC_B = 1, SRC_PMA = 2 };

struct Ev {
    double cA, nA, cB, nB, phi;
    double dep;  // energy left at the collision point (binding energy)
    double eB;   // kinetic energy of the particle taking turn B when it is known, else -1
    int nturn, sgnB, keep, ne;
    int src0, src1, sp0, sp1;
    int err;
};

template <class G>
__device__ __forceinline__ void sample_event(const DevProc& pr, int sp, const V3& p, double pnorm,
                                             double eng, const DevSB* sbs, const DevPE* pes, G& g,
                                             Ev& e, double dropcut = -1.0) {
    e.err = 0;
    e.nturn = 1;
    e.sgnB = 1;
    e.cB = 0.0;
    e.nB = 0.0;
    e.dep = 0.0;
    e.eB = -1.0;
    e.src1 = SRC_A;
    e.sp1 = sp;
    switch (pr.kind) {
    case PT_PROC_ELASTIC: {  // src/relativistic_coulomb.jl:10-23
        e.phi = TWO_PI * g.next();
        V3 v = velocity(sp, p);
        double beta = div_const(norm3(v), C, 1.0 / C);  // exact: |v| / c
        double a = pr.c[0];
        double al = qdiv(HBAR * HBAR, 4.0 * dot3(p, p) * (a * a));
        e.cA = sample_rel_sr(al, beta, g);
        e.nA = pnorm;
        e.keep = 1;
        e.ne = 1;
        e.src0 = SRC_A;
        e.sp0 = sp;
        break;
    }
    case PT_PROC_RBEB:  // src/rbeb.jl:54-80
    case PT_PROC_MOLLER:  // src/moller.jl:13-37
    case PT_PROC_BHABHA: {  // src/bhaba.jl:9-33
        double E0 = eng, E1, E2;
        if (pr.kind == PT_PROC_RBEB) {
            E2 = rbeb_sample(E0, pr, g);
            E1 = E0 - E2 - pr.B;
            e.dep = pr.B;
            if (!(E2 < E1)) e.err = 1;
        } else {
            E2 = pr.kind == PT_PROC_MOLLER ? moller_sample(pr.tcut, eng, g) : bhabha_sample(pr.tcut, eng, g);
            E1 = E0 - E2;
        }
        e.phi = TWO_PI * g.next();
        // Lehtinen 1999 angles; those of a secondary the caller drops unseen (E2 < dropcut,
        // see finish_event) are not needed
        e.nA = div_const(qsqrt(E1 * E1 + 2.0 * MC2 * E1), C, 1.0 / C);
        e.eB = E2;
        e.cA = qsqrt(qdiv(E1 * (E0 + 2.0 * MC2), E0 * (E1 + 2.0 * MC2)));
        if (!(E2 < dropcut)) {
            e.nB = div_const(qsqrt(E2 * E2 + 2.0 * MC2 * E2), C, 1.0 / C);
            e.cB = qsqrt(qdiv(E2 * (E0 + 2.0 * MC2), E0 * (E2 + 2.0 * MC2)));
        }
        e.nturn = 2;
        e.sgnB = -1;
        e.keep = 1;
        e.ne = 2;
        e.src0 = SRC_A;
        e.sp0 = sp;
        e.src1 = SRC_B;
        e.sp1 = PT_ELECTRON;
        break;
    }
    case PT_PROC_SB: {  // src/seltzer.jl:67-90
        double kf = sb_sample(sbs[pr.slot], eng, g);
        if (kf < 0.0) e.err = 4;
        double k = eng * kf;
        if (!(k < eng)) e.err = 2;
        e.nA = k / C;
        e.cA = sample_tsai(eng, g);
        e.phi = TWO_PI * g.next();
        e.keep = 1;
        e.ne = 2;
        e.src0 = SRC_PMA;
        e.sp0 = PT_ELECTRON;
        e.src1 = SRC_A;
        e.sp1 = PT_PHOTON;
        break;
    }
    case PT_PROC_COMPTON:
    case PT_PROC_KN_COMPTON: {  // src/compton.jl:9-28
        double E1, cost;
        compton_sample(eng, g, E1, cost);
        e.cA = cost;
        e.phi = TWO_PI * g.next();
        e.nA = E1 / C;
        e.keep = 1;
        e.ne = 2;
        e.src0 = SRC_A;
        e.sp0 = PT_PHOTON;
        e.src1 = SRC_PMA;
        e.sp1 = PT_ELECTRON;
        break;
    }
    case PT_PROC_PHOTOELECTRIC: {  // src/photo_electric.jl:38-52, :60-76
        const DevPE& pe = pes[pr.slot];
        double b = pe.binding[0];
        for (int q = 0; q < pe.nshell; q++) {
            b = pe.binding[q];
            if (eng > b) break;
        }
        if (!(eng > b)) e.err = 3;
        double ee = eng - b;
        e.dep = b;
        e.cA = sauter_sample(ee, g);
        e.phi = TWO_PI * g.next();
        e.nA = mom_from_kin(PT_ELECTRON, ee);
        e.keep = 0;
        e.ne = 1;
        e.src0 = SRC_A;
        e.sp0 = PT_ELECTRON;
        break;
    }
    case PT_PROC_BETHE_HEITLER: {  // src/bethe_heitler.jl:5-25 (names swapped as there)
        double pkin, ekin;
        bh_sample(pr.c[0], pr.c[1], pr.c[2], eng, g, pkin, ekin);
        e.phi = TWO_PI * g.next();
        e.cA = sample_tsai(ekin, g);
        e.nA = mom_from_kin(PT_ELECTRON, ekin);
        e.cB = sample_tsai(pkin, g);
        e.nB = mom_from_kin(PT_POSITRON, pkin);
        e.nturn = 2;
        e.sgnB = 1;
        e.keep = 0;
        e.ne = 2;
        e.src0 = SRC_A;
        e.sp0 = PT_ELECTRON;
        e.src1 = SRC_B;
        e.sp1 = PT_POSITRON;
        break;
    }
    case PT_PROC_ANNIHILATION: {  // src/anihilation.jl:6-23, :61-67
        double eps = annih_sample(eng, g);
        double gm = 1.0 + eng / MC2;
        e.cA = (eps * (gm + 1.0) - 1.0) / (eps * sqrt(gm * gm - 1.0));
        e.phi = TWO_PI * g.next();
        double etot = eng + 2.0 * MC2;
        e.nA = eps * etot / C;
        e.keep = 0;
        e.ne = 2;
        e.src0 = SRC_A;
        e.sp0 = PT_PHOTON;
        e.src1 = SRC_PMA;
        e.sp1 = PT_PHOTON;
        break;
    }
    default:
        e.err = 5;
        e.phi = 0.0;
        e.cA = 1.0;
        e.nA = pnorm;
        e.keep = 1;
        e.ne = 1;
        e.src0 = SRC_A;
        e.sp0 = sp;
        break;
    }
}

// The collision of a bremsstrahlung or Moller process from the outputs of its learned
// sampler (y0, y1: see pt_mlp.h) instead of the rejection samplers; the kinematics and the
// remaining draws (azimuth, constructors) are those of sample_event.
template <class G>
__device__ __forceinline__ void learned_event(const DevProc& pr, int sp, double eng, float y0, float y1, G& g, Ev& e) {
    e.err = 0;
    e.dep = 0.0;
    e.eB = -1.0;
    e.nturn = 1;
    e.sgnB = 1;
    e.cB = 0.0;
    e.nB = 0.0;
    e.src1 = SRC_A;
    e.sp1 = sp;
    if (pr.kind == PT_PROC_SB) {
        double kf = exp((double)(y0 < 0.0f ? y0 : 0.0f));
        double k = eng * kf;
        double omc = exp((double)(y1 < 0.6931472f ? y1 : 0.6931472f));
        double cost = 1.0 - omc;
        e.nA = k / C;
        e.cA = cost < -1.0 ? -1.0 : cost;
        e.phi = TWO_PI * g.next();
        e.keep = 1;
        e.ne = 2;
        e.src0 = SRC_PMA;
        e.sp0 = PT_ELECTRON;
        e.src1 = SRC_A;
        e.sp1 = PT_PHOTON;
        if (!(k < eng)) e.err = 2;
    } else {  // Moller
        double E0 = eng;
        double e0 = pr.tcut / E0;
        double y = y0 < 0.0f ? 0.0 : (y0 > 1.0f ? 1.0 : (double)y0);
        double eps = e0 * exp(y * log(0.5 / e0));
        double E2 = eps * E0, E1 = E0 - E2;
        e.phi = TWO_PI * g.next();
        e.nA = sqrt(E1 * E1 + 2.0 * MC2 * E1) / C;
        e.nB = sqrt(E2 * E2 + 2.0 * MC2 * E2) / C;
        e.eB = E2;
        e.cA = sqrt(E1 * (E0 + 2.0 * MC2) / (E0 * (E1 + 2.0 * MC2)));
        e.cB = sqrt(E2 * (E0 + 2.0 * MC2) / (E0 * (E2 + 2.0 * MC2)));
        e.nturn = 2;
        e.sgnB = -1;
        e.keep = 1;
        e.ne = 2;
        e.src0 = SRC_A;
        e.sp0 = sp;
        e.src1 = SRC_B;
        e.sp1 = PT_ELECTRON;
    }
}

// turn (src/util.jl:40-57) of p by turn A and, if requested, turn B; momenta of the
// outgoing entries and the constructors' s draws (src/electron.jl:32, src/photon.jl:30).
// cut[sp] / tracked[sp] (NULL: every s is computed) tell which new particles add_particle!
// drops (at or below the cut, or not tracked): their s is never read, so its draw only
// advances the stream.
// dropcut > 0: entry 1 taking turn B with a known energy below dropcut is dropped by the
// caller without looking at it (no deposit is kept): its turn is not computed, m1 = 0 and
// drop1 is set; dropcut sits far enough below the cut that the exact test would drop it too.
template <class G>
__device__ __forceinline__ void finish_event(const V3& p, double pnorm, const Ev& e, G& g, V3& m0,
                                             V3& m1, double& s0, double& s1, const double* cut,
                                             const int* tracked, double dropcut, bool& drop1) {
    drop1 = e.ne == 2 && e.src1 == SRC_B && e.eB >= 0.0 && e.eB < dropcut;
    const Recip rp(pnorm);
    const double u0 = rp(p.x), u1 = rp(p.y), u2 = rp(p.z);
    double sp, cp;
    sincos_turn(e.phi, sp, cp, g.tab());
    double qs = 1.0 - u2 * u2;
    const double s = qsqrt(qs > 0.0 ? qs : 0.0);
    const Recip rs(s);  // used where s > 0
    V3 pa, pb;
    {
        double q = 1.0 - e.cA * e.cA;
        const double st = qsqrt(q > 0.0 ? q : 0.0);
        double x, y, z;
        if (s > 0.0) {
            double bx = u0 * u2 * cp + (-u1) * sp;
            double by = u1 * u2 * cp + u0 * sp;
            x = rs(st * bx) + u0 * e.cA;
            y = rs(st * by) + u1 * e.cA;
            z = -s * st * cp + u2 * e.cA;
        } else {
            x = st * cp;
            y = st * sp;
            z = u2 * e.cA;
        }
        pa = V3{e.nA * x, e.nA * y, e.nA * z};
    }
    if (e.nturn == 2 && !drop1) {
        double spb = e.sgnB > 0 ? sp : -sp;
        double q = 1.0 - e.cB * e.cB;
        const double st = qsqrt(q > 0.0 ? q : 0.0);
        double x, y, z;
        if (s > 0.0) {
            double bx = u0 * u2 * cp + (-u1) * spb;
            double by = u1 * u2 * cp + u0 * spb;
            x = rs(st * bx) + u0 * e.cB;
            y = rs(st * by) + u1 * e.cB;
            z = -s * st * cp + u2 * e.cB;
        } else {
            x = st * cp;
            y = st * spb;
            z = u2 * e.cB;
        }
        pb = V3{e.nB * x, e.nB * y, e.nB * z};
    } else {
        pb = V3{0.0, 0.0, 0.0};
    }
    V3 pma{p.x - pa.x, p.y - pa.y, p.z - pa.z};
    // chosen component by component: a choice between whole vectors selects between their
    // addresses, which can leave them in scratch memory
    auto pick = [](int src, double a, double b, double c) { return src == SRC_A ? a : (src == SRC_B ? b : c); };
    m0 = V3{pick(e.src0, pa.x, pb.x, pma.x), pick(e.src0, pa.y, pb.y, pma.y), pick(e.src0, pa.z, pb.z, pma.z)};
    m1 = V3{pick(e.src1, pa.x, pb.x, pma.x), pick(e.src1, pa.y, pb.y, pma.y), pick(e.src1, pa.z, pb.z, pma.z)};
    auto stored = [&](int spk, const V3& m) {
        return !cut || (tracked[spk] && kinenergy(spk, m) > cut[spk]);
    };
    const bool need0 = e.keep || stored(e.sp0, m0);
    const bool need1 = e.ne == 2 && !drop1 && stored(e.sp1, m1);
    double q0, q1;
    g.next12(e.ne == 2 ? 2 : 1, q0, q1);  // both draws at one place
    s0 = need0 ? neg_log(q0, g) : 0.0;  // nextcoll(), src/util.jl:17
    s1 = need1 ? neg_log(q1, g) : 0.0;
}

// What the common event needs of its process record, in registers.
struct ProcVals {
    int kind;
    double B, c0;
};

// The two common collisions of electrons (and elastic ones of positrons) from selection to
// momentum, for lanes of both kinds at once: `el`, elastic scattering (src/
// relativistic_coulomb.jl:10-23), or an ionisation whose rejection loop has run and left a
// secondary of energy E2 (src/rbeb.jl:54-80).  Operations and their order are those of
// sample_event and finish_event (bit for bit: collision rounds sample these kinds there), but
// each lane selects its operands and a wave runs every root, division, sine and logarithm
// once for both kinds; the azimuth, the first trial of the elastic rejection loop and the
// constructors' draws come from the two blocks that follow in the stream, computed at two
// places instead of up to four.  `drop`: there is no secondary to return.  False: the
// secondary's energy is not below the primary's.
//   elastic: g = sqrt(1 + c^2 p.p / (mc^2)^2), v = p / (m g), beta = |v| / c
//   ionisation: n = sqrt(E1^2 + 2 mc^2 E1) / c, cos = sqrt(E1 (E0 + 2 mc^2) / (E0 (E1 + 2 mc^2)))
__device__ __forceinline__ bool common_event(bool el, const ProcVals& pv, const V3& p, double E0, double E2, bool drop,
                                             StepStream& g, V3& m0, V3& m1, double& s0, double& s1) {
    constexpr double MC2SQ = MC2 * MC2;
    // the stream: q0, q1, q2, q3 are its next four draws
    const uint32_t d = g.draw, blk = (d + 1) >> 1;
    const bool odd = (d & 1) != 0;
    const double half = g.c1;
    g.fill(blk);
    const double a0 = g.c0, a1 = g.c1;
    double b0 = 0.0, b1 = 0.0;
    if (el || !drop) {
        g.fill(blk + 1);
        b0 = g.c0;
        b1 = g.c1;
    }
    const double q0 = odd ? half : a0, q1 = odd ? a0 : a1, q2 = odd ? a1 : b0, q3 = odd ? b0 : b1;
    const double phi = TWO_PI * q0;
    // energies and angles
    const double pp = dot3(p, p), pn = qsqrt(pp);
    const double E1 = E0 - E2 - pv.B;
    const double r1 = qsqrt(el ? 1.0 + div_const_fin(C2 * pp, MC2SQ, 1.0 / MC2SQ) : E1 * E1 + 2.0 * MC2 * E1);
    const double q = qdiv(el ? 1.0 : E1 * (E0 + 2.0 * MC2), el ? ME * r1 : E0 * (E1 + 2.0 * MC2));
    const V3 v{p.x * q, p.y * q, p.z * q};
    const double r2 = qsqrt(el ? dot3(v, v) : q);
    const double n = div_const_fin(el ? r2 : r1, C, 1.0 / C);
    double cA = r2, u0 = q1;  // u0: the draw of s
    uint32_t used = 3;
    if (el) {
        // sample_rel_sr (src/relativistic_coulomb.jl:35-51), the first trial here
        const double al = qdiv(HBAR * HBAR, 4.0 * pp * (pv.c0 * pv.c0));
        const double xs = qdiv(al * q1, al + 1.0 - q1);
        cA = 1.0 - 2.0 * xs;
        used = 4;
        u0 = q3;
        if (!(q2 < 1.0 - n * n * xs)) {
            // rejected: the loop goes on from the draw after this trial
            g.draw = d + 3;
            cA = sample_rel_sr(al, n, g);
            u0 = g.next();
            used = g.draw - d;
        }
    }
    g.draw = d + used;
    const double nA = el ? pn : n;
    // turn (src/util.jl:40-57)
    const Recip rp(pn);
    const double w0 = rp(p.x), w1 = rp(p.y), w2 = rp(p.z);
    double sp, cp;
    sincos_turn(phi, sp, cp, g.tab());
    const double qs = 1.0 - w2 * w2;
    const double s = qsqrt(qs > 0.0 ? qs : 0.0);
    const Recip rs(s);  // used where s > 0
    {
        const double qa = 1.0 - cA * cA;
        const double st = qsqrt(qa > 0.0 ? qa : 0.0);
        const double bx = w0 * w2 * cp + (-w1) * sp;
        const double by = w1 * w2 * cp + w0 * sp;
        const bool tilted = s > 0.0;
        const double x = tilted ? rs(st * bx) + w0 * cA : st * cp;
        const double y = tilted ? rs(st * by) + w1 * cA : st * sp;
        const double z = tilted ? -s * st * cp + w2 * cA : w2 * cA;
        m0 = V3{nA * x, nA * y, nA * z};
    }
    s0 = -log_tab(u0, g.tab());  // nextcoll(), src/util.jl:17
    if (!drop) {
        const double nB = div_const_fin(qsqrt(E2 * E2 + 2.0 * MC2 * E2), C, 1.0 / C);
        const double cB = qsqrt(qdiv(E2 * (E0 + 2.0 * MC2), E0 * (E2 + 2.0 * MC2)));
        const double spb = -sp;
        const double qb = 1.0 - cB * cB;
        const double st = qsqrt(qb > 0.0 ? qb : 0.0);
        const double bx = w0 * w2 * cp + (-w1) * spb;
        const double by = w1 * w2 * cp + w0 * spb;
        const bool tilted = s > 0.0;
        const double x = tilted ? rs(st * bx) + w0 * cB : st * cp;
        const double y = tilted ? rs(st * by) + w1 * cB : st * spb;
        const double z = tilted ? -s * st * cp + w2 * cB : w2 * cB;
        m1 = V3{nB * x, nB * y, nB * z};
        s1 = -log_tab(q2, g.tab());
    }
    return el || E2 < E1;
}

}  // namespace pt

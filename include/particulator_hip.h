/*
 * particulator_hip.h -- C ABI of the MI355X (gfx950) null-collision Monte Carlo step.
 *
 * The library advances electron / photon / positron populations in applied E/B fields:
 * relativistic RK2 push, null-collision selection from a binary-interval Chebyshev rate
 * table, per-process secondary sampling, append of secondaries and compaction of the
 * populations.  Host code (Julia `ccall`, Python `ctypes`, C/C++) owns table building and
 * the run loop; the library owns device memory.
 *
 * Conventions: every entry point returns PT_OK (0) or a negative pt_status; the message of
 * the last failure is pt_last_error(ctx).  No C++ exception crosses this boundary.  A
 * context is used from one host thread at a time.  Calls are ordered on the context's HIP
 * stream and complete before they return unless noted.  Units are SI (J, s, m, kg m/s).
 *
 * Each entry point names the reference function (Particulator.jl, file:line) whose role
 * it takes over.
 */
#ifndef PARTICULATOR_HIP_H
#define PARTICULATOR_HIP_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define PT_ABI_VERSION 1

/* particle species: the MultiPopulation order of the reference scripts
 * (scripts/swarm.jl:68-71) */
enum pt_species { PT_ELECTRON = 0, PT_PHOTON = 1, PT_POSITRON = 2, PT_NSPECIES = 3 };

/* collision processes (the `collide` methods of src/rbeb.jl, src/moller.jl, src/seltzer.jl,
 * src/relativistic_coulomb.jl, src/compton.jl, src/photo_electric.jl,
 * src/bethe_heitler.jl, src/bhaba.jl, src/anihilation.jl) */
enum pt_proc_kind {
    PT_PROC_NULL = 0,
    PT_PROC_ELASTIC = 1,        /* RelativisticCoulomb(Z) */
    PT_PROC_SB = 2,             /* SeltzerBerger(Z) */
    PT_PROC_RBEB = 3,           /* RBEB(B, U, N) */
    PT_PROC_MOLLER = 4,         /* Moller(Z, tcut) */
    PT_PROC_COMPTON = 5,        /* Compton(Z) */
    PT_PROC_PHOTOELECTRIC = 6,  /* PhotoElectric(Z) */
    PT_PROC_BETHE_HEITLER = 7,  /* BetheHeitler(Z) */
    PT_PROC_BHABHA = 8,         /* Bhaba(Z, tcut) */
    PT_PROC_ANNIHILATION = 9,   /* PositronAnihilation(Z) */
    PT_PROC_KN_COMPTON = 10     /* KleinNishinaCompton(Z) */
};

/* field functors, src/field.jl:4-52 */
enum pt_field_kind {
    PT_FIELD_NONE = 0, PT_FIELD_HOMOGENEOUS = 1, PT_FIELD_DOUBLELAYER = 2,
    PT_FIELD_STEP = 3, PT_FIELD_CONFINED = 4
};

enum pt_status {
    PT_OK = 0,
    PT_E_ARG = -1,          /* invalid argument */
    PT_E_HIP = -2,          /* HIP runtime error */
    PT_E_CAPACITY = -3,     /* a population reached its capacity (src/population.jl:107) */
    PT_E_RATEBOUND = -4,    /* rate bound underestimated (src/collisions.jl:186) */
    PT_E_STATE = -5,        /* call out of order (e.g. no table uploaded) */
    PT_E_NOMEM = -6,        /* device allocation failed */
    PT_E_TABLE_RANGE = -7,  /* energy above the table's xmax (src/cheby.jl:127-143) */
    PT_E_SAMPLER = -8,      /* a sampler's domain assertion failed (e.g. src/seltzer.jl:73) */
    PT_E_NOT_BUILT = -9     /* operation needs a GPU */
};

/* structure-of-arrays field order of a particle state (src/electron.jl:13-26) */
enum pt_field_index {
    PT_X = 0, PT_Y = 1, PT_Z = 2, PT_PX = 3, PT_PY = 4, PT_PZ = 5,
    PT_W = 6, PT_T = 7, PT_S = 8, PT_R = 9, PT_NFIELDS = 10
};

typedef struct pt_ctx pt_ctx;

/* a state recorded by a wall (WallCallback, src/callback.jl:146-184) */
typedef struct {
    double x[3], p[3], w, t;
    uint64_t uid;
    int32_t species, swarm;
} pt_wall_record;

/* One process of a collision table, in table order (the `proc` tuple of
 * ChebyshevCollisionTable, src/collision_table.jl:63-75). */
typedef struct {
    int32_t kind;      /* pt_proc_kind */
    int32_t Z;         /* target atomic number */
    int32_t slot;      /* SB or photoelectric data slot (pt_upload_sb / pt_upload_pe) */
    int32_t N;         /* RBEB occupation number */
    double B, U;       /* RBEB binding and kinetic energy of the orbital (J) */
    double tcut;       /* Moller / Bhabha secondary-energy cut (J) */
    double zf;         /* Z as a real number (annihilation accepts an effective Z) */
    double c[4];       /* per-process constants computed by the host with libm:
                          ELASTIC: c[0] = 1.3413 * Z^(-1/3) * a_0 (screening radius);
                          BETHE_HEITLER: c[0] = Z^(1/3), c[1] = 8 log(Z)/3,
                          c[2] = c[1] + 8 fc, c[3] unused (src/bethe_heitler.jl:97-100,
                          _fc :153-161) */
} pt_proc_desc;

/* ChebyshevCollisionTable (src/collision_table.jl:63-106) of one species */
typedef struct {
    int32_t nprocs;      /* L */
    int32_t order;       /* Chebyshev order, must be 3 */
    int32_t nintervals;  /* k (intervals 0..k), must be <= 63 */
    int32_t nswarm;      /* rate bounds given per swarm (>= 1) */
    double xmax;         /* BinaryIntervals root (J) */
    double energy_cut;   /* Population energy_cut (J) */
    const double* rate;      /* [(k+1)][L][order], the reference's column-major (order, L, k+1) */
    const double* ratebound; /* [nswarm][(k+1)][order] */
    const pt_proc_desc* procs;
} pt_table_desc;

typedef struct {
    int32_t kind;        /* pt_field_kind */
    int32_t pad;
    double v[3];         /* HOMOGENEOUS, DOUBLELAYER value; STEP value below z */
    double v2[3];        /* STEP value above z */
    double z1, z2;       /* DOUBLELAYER bounds; STEP: z = z1 */
    double sx, sy, sz, ez0; /* CONFINED */
} pt_field_fn;

/* ElectromagneticField(e, b), src/field.jl:54-70 */
typedef struct {
    pt_field_fn e, b;
} pt_field_desc;

typedef struct {
    uint64_t capacity[PT_NSPECIES]; /* slots per species (Population max_particles) */
    uint64_t seed;                  /* Philox key */
    int32_t tracked[PT_NSPECIES];   /* 0: particles of this species are tallied at birth,
                                       not stored */
    int32_t nswarm;                 /* independent swarms (fields, rate bounds) */
    int32_t device;                 /* HIP device ordinal */
    int32_t tally_bins;             /* log-spaced energy bins of the birth tallies */
    double tally_lo, tally_hi;      /* tally energy range (J) */
    int32_t dose_bins;              /* depth-dose bins in z (0: no dose tally) */
    int32_t tally_tracked;          /* 1: births of tracked species are tallied too */
    double dose_zlo, dose_zhi;      /* depth-dose range (m) */
} pt_config;

/* population statistics (src/population.jl:89-223) */
typedef struct {
    uint64_t n;              /* slots in use (nparticles) */
    uint64_t nactive;        /* nactives */
    double weight;           /* weight */
    double mean_energy;      /* meanenergy (J) */
    double centroid[3];      /* spread()[1] */
    double spread;           /* spread()[2] */
    double max_energy;       /* maxenergy over active particles */
} pt_pop_stats;

/* counters of the algorithmic work done (for throughput and roofline figures) */
typedef struct {
    uint64_t particle_steps;     /* active particles at step start, summed over steps */
    uint64_t secondaries;        /* particles appended to a population */
    uint64_t moved;              /* particles moved by the compactions that ran (pt_run) */
    uint64_t events;             /* real + null collision events */
    uint64_t steps;
    uint64_t tail_particles;     /* secondaries advanced within their birth step */
    double advance_ms;           /* summed duration of the main advance kernel */
    uint64_t advance_launches;
    double tail_ms;
    double compact_ms;
    uint64_t main_secondaries;   /* particles appended by the main advance kernel */
    double graph_ms;             /* summed duration of graph replays (pt_run_graph) */
} pt_work;

/* ---- lifecycle ---------------------------------------------------------------- */
int pt_abi_version(void);
/* Population(...) constructors + MultiPopulation (src/population.jl:34-44,
 * src/mixed_population.jl:4-12): allocates capacity[s] slots per species. */
int pt_create(const pt_config* cfg, pt_ctx** out);
void pt_destroy(pt_ctx* ctx);
/* the last failure of ctx; with NULL, of the last context-free call on this thread */
const char* pt_last_error(const pt_ctx* ctx);

/* ---- tables and fields ------------------------------------------------------------ */
/* Upload a ChebyshevCollisionTable built by collision_table_from_processes
 * (src/collision_table.jl:115-149) for one species. */
int pt_upload_table(pt_ctx* ctx, int species, const pt_table_desc* table);
/* SeltzerBerger sampling data (src/seltzer.jl:9-49): log_energy[ne],
 * data[ne][ncum] = log(k/T) at pcum = LinRange(0,1,ncum) for each primary energy. */
int pt_upload_sb(pt_ctx* ctx, int slot, int Z, int ne, int ncum, const double* log_energy,
                 const double* data);
/* PhotoElectric binding energies (src/photo_electric.jl:17, :60-76), K shell first. */
int pt_upload_pe(pt_ctx* ctx, int slot, int Z, int nshell, const double* binding);
/* pusher forcing ElectromagneticField (src/field.jl:54-70) of one swarm */
int pt_set_field(pt_ctx* ctx, int swarm, const pt_field_desc* field);

/* ChebContinuumLoss(ContinuumLoss(nel, I, Tcut), Tmax, n) (src/continuum.jl:6-59) added to
 * the forcing of every swarm as CombinedForcing(field, loss) (src/pusher.jl:14-23):
 * electron[] and positron[] are the fits' `ec` and `pc` ((order, k+1) column-major, i.e.
 * [(k+1)][order]) on BinaryIntervals(nintervals, xmax).  NULL arrays remove the loss. */
int pt_set_continuum_loss(pt_ctx* ctx, int nintervals, int order, double xmax, const double* electron,
                          const double* positron);

/* Restrictions of the forcing and the pusher (bit s of a mask: species s; all swarms):
 * field_species: the species the electromagnetic force acts on, and loss_species: those the
 * continuum loss acts on (RestrictedForcing{T}(f) acts only on T, src/pusher.jl:27-34;
 * NullForcing acts on none, :11); push_species: the species that are pushed, the others
 * keep x and p and only advance t (RestrictedPusher{T}, NullPusher, :66-76).  The default
 * is 7, 7, 7 (no restriction). */
int pt_set_forcing(pt_ctx* ctx, uint32_t field_species, uint32_t loss_species, uint32_t push_species);

/* ---- table building on the host (no context, no device) -----------------------------
 * The init-time half of the tables: totalcs of every process kind, collision_table_from_
 * processes (src/collision_table.jl:115-149) with chebfit (src/cheby.jl:211-227),
 * compratebound (src/collision_table.jl:152-167) and the process order (:137-146), and the
 * Seltzer-Berger inverse CDFs (src/seltzer.jl:9-64, :163-192).  The outputs are the arrays
 * pt_upload_table and pt_upload_sb take, so a caller can hand the library raw processes.
 * On failure pt_last_error(NULL) returns the message (per host thread). */
typedef struct {
    int32_t kind;          /* pt_proc_kind */
    int32_t Z;             /* atomic number of the target */
    int32_t N;             /* RBEB: electrons in the orbital */
    int32_t ntab;          /* SB: points of tab_x / tab_y; PHOTOELECTRIC: Sandia intervals */
    double coef;           /* target density (m^-3): rate = coef * speed * totalcs */
    double B, U;           /* RBEB: binding and mean kinetic energy of the orbital (J) */
    double tcut;           /* MOLLER, BHABHA: smallest secondary energy (J) */
    const double* tab_x;   /* SB: log of the tabulated primary energies (log J);
                              PHOTOELECTRIC: left edges of the Sandia intervals (J) */
    const double* tab_y;   /* SB: total cross sections (m^2) at tab_x (pt_sb_build);
                              PHOTOELECTRIC: ntab rows of 4 coefficients (m^2 J^i, i = 1..4) */
} pt_process;

/* totalcs(process, E) at n kinetic energies (J), in m^2 (the reference's totalcs methods:
 * src/relativistic_coulomb.jl:58, src/rbeb.jl:117, src/moller.jl:40, src/bhaba.jl:35,
 * src/anihilation.jl:25, src/compton.jl:34,59, src/bethe_heitler.jl:28,
 * src/photo_electric.jl:54, src/seltzer.jl:217) */
int pt_totalcs(const pt_process* proc, const double* eng, size_t n, double* out);
/* the pt_proc_desc of a process in a table, with the host-computed constants */
int pt_process_desc(const pt_process* proc, int slot, pt_proc_desc* out);
/* SeltzerBerger(Z) from its G4 data file (a RawG4Physics2DVector, src/util.jl:165-190):
 * nx photon fractions k/T, ny values log(T / energy_scale) and values[ny][nx].  Fills
 * log_energy[ny] (log J), tcs[ny] (m^2) and data[ny][ncum], the inverse CDF of log(k/T)
 * at ncum evenly spaced probabilities with k between gamma_min and gamma_max (J). */
int pt_sb_build(int Z, const double* kfrac, int nx, const double* logT, int ny, const double* values,
                int ncum, double gamma_min, double gamma_max, double energy_scale,
                double* log_energy, double* tcs, double* data);
/* The primary-energy cell of sample_secondary_energy (src/seltzer.jl:97-106): there
 * j2 = searchsortedfirst(log_energy, log(T)).  thr[j] receives the smallest double T with
 * log(T) > log_energy[j] (this host's libm log), so that j2 = 1 + #{j : T >= thr[j]}: the
 * device finds the cell by comparisons alone, with the same result as the host's log on
 * every input, and pt_upload_sb stores these thresholds beside the table. */
int pt_sb_thresholds(const double* log_energy, int ne, double* thr);
/* collision_table_from_processes(procs, species, Fdt; safety, nintervals, order,
 * max_energy) with one rate bound per impulse fdt[s] (Fdt = e E_s dt of swarm s).  Fills
 * rate[(nintervals+1)][nprocs][order] in table order, ratebound[nswarm][nintervals+1][order],
 * perm[nprocs] (table position -> index into procs) and keys[nprocs] (sort keys, table
 * order); any output may be NULL. */
int pt_table_build(const pt_process* procs, int nprocs, int species, const double* fdt, int nswarm,
                   double safety, int nintervals, int order, double max_energy, double* rate,
                   double* ratebound, int32_t* perm, double* keys);

/* ---- particles --------------------------------------------------------------------- */
/* Append particles (the initial states given to Population(), src/population.jl:34-44).
 * soa[f] points to n values of field f (pt_field_index); uid and swarm may be NULL
 * (uids then continue from the context's counter, swarm 0). */
int pt_add_particles(pt_ctx* ctx, int species, const double* const soa[PT_NFIELDS],
                     const uint64_t* uid, const int32_t* swarm, size_t n);
/* Generate n particles on the device: kinetic energy e1 (or log-uniform in [e1, e2]),
 * isotropic direction (randsphere, src/util.jl:4-12), x = 0, w = 1, t = t0,
 * s = nextcoll(); uid = uid0 + i. */
int pt_init_particles(pt_ctx* ctx, int species, size_t n, double e1, double e2,
                      int loguniform, int swarm, uint64_t uid0, double t0);
/* Generate n particles of kinetic energy e at the origin moving along dir (a pencil beam,
 * the initial photons of scripts/beam.jl:52-60): w = 1, t = t0, s = nextcoll(),
 * uid = uid0 + i. */
int pt_init_beam(pt_ctx* ctx, int species, size_t n, double e, const double dir[3], int swarm,
                 uint64_t uid0, double t0);
/* Copy a population back (eachparticle, src/population.jl:81).  soa entries may be NULL. */
int pt_download(pt_ctx* ctx, int species, double* const soa[PT_NFIELDS], uint8_t* active,
                uint64_t* uid, int32_t* swarm, size_t cap, size_t* n);
/* Replace the state of a population with n particles (used for checkpoint restore). */
int pt_set_particles(pt_ctx* ctx, int species, const double* const soa[PT_NFIELDS],
                     const uint8_t* active, const uint64_t* uid, const int32_t* swarm,
                     size_t n);
int pt_count(pt_ctx* ctx, int species, uint64_t* n);

/* ---- the step ------------------------------------------------------------------------ */
/* init! (src/mixed_population.jl:20-35): r = ratebound(E) of every active particle. */
int pt_init(pt_ctx* ctx);
/* One time step: advance! (src/mixed_population.jl:38-47: advance_init!, advance1!
 * passes, do_one_collision!, collide, apply!, setr!) followed by the deactivation half of
 * droplow! (src/population.jl:273-284).  Slots are freed by pt_compact.  The step index
 * of the random streams advances by one. */
int pt_advance(pt_ctx* ctx, double tfinal);
/* `nsteps` calls of pt_advance at t0 + dt, t0 + 2dt, ..., with pt_compact every
 * `compact_every` steps (0: never) and error checks every `check_every` steps.
 * Up to 16 steps run in one launch; where several compactions fall among the steps of a
 * launch, one at its end may stand for them.  The particles are the same, and a population
 * fails to fit only where it would with every compaction in its place; but the slots that
 * particles have (their order in pt_download) and pt_work.moved follow the compactions that
 * ran.  The context keeps a copy of the state for that (of at most 2^21 particles that fill no
 * more than half their slots: up to 195 MB, and the tallies) and runs the steps since the
 * last check again, compacting as asked, if something did not fit. */
int pt_run(pt_ctx* ctx, double t0, double dt, int nsteps, int compact_every, int check_every);
/* repack! (src/population.jl:229-259): fill holes below the active count with active
 * particles from the end (not order preserving, as in the reference). */
int pt_compact(pt_ctx* ctx, int species);
/* ---- device callbacks ---------------------------------------------------------------- */
/* WallCallback{P}(coord, v, drop) (src/callback.jl:146-184) for one species: a particle
 * crossing x[coord] = v upwards during a push is recorded as lincomb(new, old, w)
 * (src/electron.jl:127-132; the positron method's field error, src/positron.jl:51, does
 * not arise here) and dropped if `drop`.  coord = -1 removes the wall.  Records beyond
 * `capacity` are counted but not stored.  Needs collision rounds = 0. */
int pt_set_wall(pt_ctx* ctx, int species, int coord, double v, int drop, size_t capacity);
/* copy the wall records (n: how many crossings were recorded, possibly > cap) */
int pt_wall_read(pt_ctx* ctx, pt_wall_record* out, size_t cap, size_t* n, int reset);
/* roulette!(q, popl) with a constant survival probability (src/population.jl:291-309, the
 * RouletteCallback of src/callback.jl:210-226): streams keyed by uid and step */
int pt_roulette(pt_ctx* ctx, int species, double q);
/* split!(f, popl) with a constant mean (src/population.jl:316-330, the SplitCallback of
 * src/callback.jl:231-247): weights / (1 + f), Poisson(f) copies with new uids */
int pt_split(pt_ctx* ctx, int species, double f);
/* roulette!(f, popl) / split!(f, popl) with a function of the particle (src/population.jl:
 * 291-330): the caller evaluates f (roulette: of the kinetic energy, split: of the state) for
 * each of the n slots in use (n = pt_count; inactive slots are ignored) and passes the
 * values; survival, weights and copies are then drawn on the device as in pt_roulette /
 * pt_split, without moving the population through the host. */
int pt_roulette_each(pt_ctx* ctx, int species, const double* q, size_t n);
int pt_split_each(pt_ctx* ctx, int species, const double* f, size_t n);

/* ---- launch shape, captured runs, autotuning ---------------------------------------
 * The particle results do not depend on any of these: every random stream is keyed by
 * (seed, particle uid, step), so launch shape and compaction cadence change only where a
 * particle sits in its population, not its history. */
typedef struct {
    int32_t block;          /* threads per workgroup of the advance kernel: 128, 256 or 512 (with 256
                               and 512, large populations run in workgroups of 768) */
    int32_t grid_mult;      /* workgroups launched = resident workgroups x grid_mult (1..16) */
    int32_t compact_every;  /* steps between compactions in pt_run_graph (>= 1) */
    int32_t rounds;         /* collision rounds per step (0..8): the push/select kernels queue
                               real collisions of the kinds in defer_mask per sampler kind
                               and sampling kernels apply them, `rounds` times, before a
                               pass that samples every kind in place finishes the step;
                               0: every collision is sampled in place */
    uint32_t defer_mask;    /* bit k set: collisions of pt_proc_kind k go through the
                               sampling kernels in collision rounds */
    int32_t tail_passes;    /* whole-grid passes over the secondaries a step's lanes could
                               not advance themselves (the advance1! passes,
                               src/mixed_population.jl:43-46), before one workgroup
                               finishes the rest (0..16) */
    int32_t pad;
} pt_launch;
/* No reference counterpart (the reference's @batch threads split the loop statically,
 * src/mixed_population.jl:61). */
int pt_set_launch(pt_ctx* ctx, const pt_launch* launch);
int pt_get_launch(pt_ctx* ctx, pt_launch* launch);
/* run! (src/run.jl:1-29) with a fixed dt and no host callbacks: compact_every steps
 * (snapshot, advance, secondary passes, clock tick) and one compaction are captured as a
 * hipGraph and replayed; the step clock lives on the device (tfinal = t + dt, t = tfinal),
 * so the times are those of pt_run.  Steps left over (nsteps not a multiple of
 * compact_every) run as a shorter graph without compaction.  Errors are checked every
 * check_every steps (rounded up to whole replays). */
int pt_run_graph(pt_ctx* ctx, double t0, double dt, int nsteps, int check_every);
typedef struct {
    pt_launch launch;
    double rate;            /* particle-steps/s measured over the trial */
} pt_tune_trial;
/* Autotuner (no reference counterpart): times trial_steps steps of the live run for each
 * number of collision rounds (0/2/3/4), then for each kernel shape (block 128/256/512 x
 * grid_mult 1/2/4) with the fastest rounds, then 16 steps for each compaction cadence
 * 1/2/4/8/16 with the fastest shape, and sets the fastest as the context's launch.  The trial steps advance the run from t0 by dt; *t_end is the time
 * reached.  trials[] receives up to max_trials measurements. */
int pt_autotune(pt_ctx* ctx, double t0, double dt, int trial_steps, pt_tune_trial* trials,
                int max_trials, int* ntrials, pt_launch* best, double* t_end);
/* nactives / weight / meanenergy per swarm (src/population.jl:89-223 applied to each of
 * the independent populations the reference scripts run, scripts/swarm.jl:63-99):
 * out[4*i + 0..3] = active count, weight, sum of w*E (J), max E (J) of swarm i. */
int pt_swarm_stats(pt_ctx* ctx, int species, int nswarm, double* out);
/* No counterpart in the reference.  pt_swarm_stats for callers that cannot allocate device
 * memory (code under graph capture, tight serving loops, hosts that forbid allocation): it
 * calls no hipMalloc/hipFree; its per-swarm sums live in a fixed device array of the
 * library (4096 swarms at most, 128 KiB per GPU, held until the process ends; larger
 * nswarm is rejected with PT_E_ARG).  Same output as pt_swarm_stats (sums to rounding:
 * floating atomics).  Calls on one GPU share that array: calls that overlap on one GPU
 * (from several host threads or contexts) race. */
int pt_swarm_stats_noalloc(pt_ctx* ctx, int species, int nswarm, double* out);

/* population statistics (src/population.jl:89-223) over active particles */
int pt_stats(pt_ctx* ctx, int species, pt_pop_stats* out);
/* CollisionCounter (src/callback.jl:118-141): out[0] null events, out[1+j] process j in
 * table order; nmax entries at most.  reset != 0 clears the counters afterwards. */
int pt_collision_counts(pt_ctx* ctx, int species, int64_t* out, int nmax, int reset);
/* depth-dose tally (build-defined deposition; the reference has none): the kinetic energy
 * of particles dropped below the cut (droplow!, src/population.jl:273-284) and of
 * secondaries born below it (add_particle!, src/population.jl:105), and the binding energy
 * of ionisation (src/rbeb.jl:68) and photoabsorption (src/photo_electric.jl:45), in
 * weight x J, binned in z; under / over hold what fell outside [dose_zlo, dose_zhi) */
int pt_dose_read(pt_ctx* ctx, double* hist, int nbins, double* under, double* over, double* total, int reset);
/* birth tallies of an untracked species: weight histogram over tally bins, count, weight */
int pt_tally_read(pt_ctx* ctx, int species, double* hist, int nbins, double* count,
                  double* weight);
/* work counters and (if profiling is on) kernel durations measured with HIP events on
 * the context's stream */
int pt_work_read(pt_ctx* ctx, pt_work* out, int reset);
int pt_profile_enable(pt_ctx* ctx, int on);
/* step index of the random streams (Philox counter word 2) */
int pt_set_step(pt_ctx* ctx, uint32_t step);
int pt_get_step(pt_ctx* ctx, uint32_t* step);
/* error flags accumulated on the device: flags[0] rate-bound violations, [1] particles
 * lost to a full population, [2] energies above the table range, [3] sampler domain
 * failures, [4] secondary passes left unfinished.  flags may be NULL (5 entries).
 * Returns the status of the first nonzero flag. */
int pt_check(pt_ctx* ctx, int64_t* flags);
int pt_synchronize(pt_ctx* ctx);

/* ---- learned samplers (no reference counterpart) ------------------------------------
 * Small MLP inverse-CDF samplers replace the rejection samplers of bremsstrahlung
 * (SeltzerBerger photon energy k/T and modified-Tsai cos theta, src/seltzer.jl:67-122,
 * src/util.jl:143-159) and of Moller (secondary energy fraction, src/moller.jl:64-87).
 * Inputs (log10 T, one-hot target Z in {7, 8, 18}, two uniforms) -> 3 hidden layers x 64,
 * GELU -> outputs (log(k/T), log(1 - cos theta)) or (log(eps/eps0) / log(0.5/eps0)).
 * Trained on the device in FP32 on quantiles of samples the step's own samplers draw;
 * evaluated with BF16 weights on the matrix cores (FP32 accumulation) wherever the step
 * samples a collision of the kind: in place by the push/select kernels (the wave's
 * collisions of one kind go through the network together) and by the sampling kernel of
 * collision rounds. */
enum pt_learned { PT_LEARN_SB = 0, PT_LEARN_MOLLER = 1 };

typedef struct {
    int32_t nenergies;        /* training energies per target Z (log-spaced) */
    int32_t samples_per_row;  /* exact samples per (energy, Z), a power of two <= 4096 */
    int32_t quantiles;        /* quantile levels kept per (energy, Z) */
    int32_t batch;            /* training batch */
    int32_t steps;            /* Adam steps (cosine-decayed learning rate) */
    int32_t ks_samples;       /* held-out samples per (energy, Z) of the KS gate */
    int32_t ks_energies;      /* held-out energies per Z */
    int32_t pad;
    double lr;                /* initial learning rate */
    double emin, emax;        /* energy range of the KS gate (J), and the range in which the
                                 step uses the network (the rejection sampler elsewhere);
                                 training covers [emin / 1.25, 1.25 emax] (Moller: above
                                 2 tcut) */
    double tcut;              /* Moller secondary-energy cut (J) */
    double ks_gate;           /* the network is used when the held-out KS <= ks_gate */
    uint64_t seed;
} pt_learn_config;

typedef struct {
    double loss_first;        /* mean batch loss of the first 100 steps (squared quantile
                                 errors weighted by the inverse squared quantile slope) */
    double loss_last;         /* mean batch loss of the last 100 steps */
    double ks_max;            /* held-out two-sample KS, max over (energy, Z, output) */
    double ks_mean;
    double ks_noise;          /* 95% KS noise floor of the held-out comparison */
    double gen_ms, train_ms, eval_ms;
    int64_t samples;          /* exact samples drawn for the training set */
    int32_t installed;        /* 1: ks_max <= ks_gate and the network is enabled */
    int32_t nparams;          /* parameters of the network (inputs in use) */
} pt_learn_report;

/* fill a config with the defaults for `which` */
int pt_learn_defaults(int which, pt_learn_config* cfg);
/* generate the training set, train, build the BF16 image and check it against the KS gate:
 * enabled if it passes, otherwise the rejection sampler stays in use (fallback) */
int pt_learn_train(pt_ctx* ctx, int which, const pt_learn_config* cfg, pt_learn_report* rep);
/* use (on = 1) or stop using (0) a trained network */
int pt_learn_enable(pt_ctx* ctx, int which, int on);
/* read (set = 0) or load (set = 1) the FP32 parameters (n = pt_learn_nparams()); loading
 * rebuilds the BF16 image and leaves the network disabled */
int pt_learn_nparams(void);
int pt_learn_params(pt_ctx* ctx, int which, float* params, int n, int set);
/* load a network trained in another context (pt_learn_params, set = 0, there) whose KS gate
 * passed for energies in [emin, emax] (J), and use it in that range: a sweep of many
 * contexts in the same material trains each sampler once */
int pt_learn_install(pt_ctx* ctx, int which, const float* params, int n, double emin, double emax);
/* n samples at energies T[i] (J) on targets Z[i]: the network's outputs (learned = 1,
 * clamped as the step clamps them) or the same transforms of the rejection samplers'
 * draws (learned = 0); out[2i], out[2i+1] */
int pt_learn_sample(pt_ctx* ctx, int which, int learned, const double* T, const int32_t* Z, size_t n,
                    uint64_t seed, double* out);
/* samples per second of a sampler on the device, measured with HIP events around its
 * kernels: the network (learned = 1: input features from the stream, then the matrix-core
 * inference) or the exact rejection sampler (learned = 0), per_row samples at each of the
 * nrows energies T[i] (J) on targets Z[i] (at most 2^26 samples) */
int pt_learn_throughput(pt_ctx* ctx, int which, int learned, const double* T, const int32_t* Z, size_t nrows,
                        int per_row, uint64_t seed, double* samples_per_s);

/* ---- test hooks: same device code as the step, on explicit inputs ------------------ */
/* Philox4x32-10 on the device: out[4i..4i+3] for counters ctr[4i..] and key. */
int pt_debug_philox(pt_ctx* ctx, const uint32_t* ctr, const uint32_t key[2], uint32_t* out,
                    size_t n);
/* the uniforms a particle stream (uid, step) yields: out[0..n) */
int pt_debug_uniforms(pt_ctx* ctx, uint64_t uid, uint32_t step, double* out, size_t n);
/* selection of do_one_collision! (src/collisions.jl:153-186) for n particles of a species:
 * interval index, selected process (-1 null) and the rate bound ratebound(E). */
int pt_debug_select(pt_ctx* ctx, int species, size_t n, const double* energy,
                    const double* u, const int32_t* swarm, int32_t* interval,
                    int32_t* proc, double* rbound);
/* one RK2 push (src/pusher.jl:41-63) of n states (soa in/out) by dt[i] in swarm 0 field */
int pt_debug_push(pt_ctx* ctx, int species, size_t n, double* const soa[PT_NFIELDS],
                  const double* dt);
/* collide() of process `proc` (table order) for n particles with injected uniforms
 * u[i*stride ..]: out_kind[i] outcome kind, out_draws[i] uniforms consumed,
 * out_states[(i*3+q)*PT_NFIELDS + f] the up to 3 resulting states (primary, new, new),
 * out_species[i*3+q], out_uid[i*3+q]. */
int pt_debug_collide(pt_ctx* ctx, int species, int proc, size_t n,
                     const double* const soa[PT_NFIELDS], const uint64_t* uid,
                     const double* u, int stride, int32_t* out_kind, int32_t* out_draws,
                     double* out_states, int32_t* out_species, uint64_t* out_uid);

/* what the library chose by itself: out[0], out[1] threads and number of workgroups of the last
 * main pass launched or captured with every collision in place, out[2] windows of pt_run that
 * compacted late, out[3] how many of those were taken back and repeated */
int pt_debug_choices(pt_ctx* ctx, int64_t out[4]);

/* one forward/backward pass of the training kernels on a batch: loss and the gradient of
 * the FP32 parameters (X: B x 16 inputs, Y: B x 2 targets, output weights w0, w1) */
int pt_debug_mlp_grad(pt_ctx* ctx, const float* params, const float* X, const float* Y, int B, float w0,
                      float w1, float* grad, float* loss);
/* matrix-core BF16 inference of the network with parameters `params` on n input rows */
int pt_debug_mlp_infer(pt_ctx* ctx, const float* params, const float* X, int n, float* Y);

#ifdef __cplusplus
}
#endif
#endif

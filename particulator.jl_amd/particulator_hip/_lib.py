"""ctypes binding of libparticulator_hip.so (include/particulator_hip.h).

The library is built in-tree by build.py (hipcc for gfx950).  Loading it never falls back
to anything else: if the shared object is missing, `lib()` raises.
"""
import ctypes as C
import os

HERE = os.path.dirname(os.path.abspath(__file__))
LIBNAME = "libparticulator_hip.so"
LIBPATH = os.path.join(HERE, LIBNAME)

PT_ELECTRON, PT_PHOTON, PT_POSITRON = 0, 1, 2
NSPECIES = 3
(PROC_NULL, PROC_ELASTIC, PROC_SB, PROC_RBEB, PROC_MOLLER, PROC_COMPTON, PROC_PHOTOELECTRIC,
 PROC_BETHE_HEITLER, PROC_BHABHA, PROC_ANNIHILATION, PROC_KN_COMPTON) = range(11)
FIELD_NONE, FIELD_HOMOGENEOUS, FIELD_DOUBLELAYER, FIELD_STEP, FIELD_CONFINED = range(5)
NFIELDS = 10
FIELD_NAMES = ("x", "y", "z", "px", "py", "pz", "w", "t", "s", "r")

STATUS = {
    0: "PT_OK", -1: "PT_E_ARG", -2: "PT_E_HIP", -3: "PT_E_CAPACITY", -4: "PT_E_RATEBOUND",
    -5: "PT_E_STATE", -6: "PT_E_NOMEM", -7: "PT_E_TABLE_RANGE", -8: "PT_E_SAMPLER",
    -9: "PT_E_NOT_BUILT",
}


class PTError(RuntimeError):
    def __init__(self, code, msg):
        super().__init__("%s (%d): %s" % (STATUS.get(code, "?"), code, msg))
        self.code = code


class ProcDesc(C.Structure):
    _fields_ = [("kind", C.c_int32), ("Z", C.c_int32), ("slot", C.c_int32), ("N", C.c_int32),
                ("B", C.c_double), ("U", C.c_double), ("tcut", C.c_double), ("zf", C.c_double),
                ("c", C.c_double * 4)]


class Process(C.Structure):
    """pt_process: a raw process for the host table builder"""
    _fields_ = [("kind", C.c_int32), ("Z", C.c_int32), ("N", C.c_int32), ("ntab", C.c_int32),
                ("coef", C.c_double), ("B", C.c_double), ("U", C.c_double), ("tcut", C.c_double),
                ("tab_x", C.POINTER(C.c_double)), ("tab_y", C.POINTER(C.c_double))]


class TableDesc(C.Structure):
    _fields_ = [("nprocs", C.c_int32), ("order", C.c_int32), ("nintervals", C.c_int32),
                ("nswarm", C.c_int32), ("xmax", C.c_double), ("energy_cut", C.c_double),
                ("rate", C.POINTER(C.c_double)), ("ratebound", C.POINTER(C.c_double)),
                ("procs", C.POINTER(ProcDesc))]


class FieldFn(C.Structure):
    _fields_ = [("kind", C.c_int32), ("pad", C.c_int32), ("v", C.c_double * 3),
                ("v2", C.c_double * 3), ("z1", C.c_double), ("z2", C.c_double),
                ("sx", C.c_double), ("sy", C.c_double), ("sz", C.c_double), ("ez0", C.c_double)]


class FieldDesc(C.Structure):
    _fields_ = [("e", FieldFn), ("b", FieldFn)]


class Config(C.Structure):
    _fields_ = [("capacity", C.c_uint64 * 3), ("seed", C.c_uint64), ("tracked", C.c_int32 * 3),
                ("nswarm", C.c_int32), ("device", C.c_int32), ("tally_bins", C.c_int32),
                ("tally_lo", C.c_double), ("tally_hi", C.c_double), ("dose_bins", C.c_int32),
                ("tally_tracked", C.c_int32), ("dose_zlo", C.c_double), ("dose_zhi", C.c_double)]


class PopStats(C.Structure):
    _fields_ = [("n", C.c_uint64), ("nactive", C.c_uint64), ("weight", C.c_double),
                ("mean_energy", C.c_double), ("centroid", C.c_double * 3),
                ("spread", C.c_double), ("max_energy", C.c_double)]


class Work(C.Structure):
    _fields_ = [("particle_steps", C.c_uint64), ("secondaries", C.c_uint64),
                ("moved", C.c_uint64), ("events", C.c_uint64), ("steps", C.c_uint64),
                ("tail_particles", C.c_uint64), ("advance_ms", C.c_double),
                ("advance_launches", C.c_uint64), ("tail_ms", C.c_double),
                ("compact_ms", C.c_double), ("main_secondaries", C.c_uint64),
                ("graph_ms", C.c_double)]


class Launch(C.Structure):
    _fields_ = [("block", C.c_int32), ("grid_mult", C.c_int32), ("compact_every", C.c_int32),
                ("rounds", C.c_int32), ("defer_mask", C.c_uint32), ("tail_passes", C.c_int32),
                ("pad", C.c_int32)]


class LearnConfig(C.Structure):
    _fields_ = [("nenergies", C.c_int32), ("samples_per_row", C.c_int32), ("quantiles", C.c_int32),
                ("batch", C.c_int32), ("steps", C.c_int32), ("ks_samples", C.c_int32),
                ("ks_energies", C.c_int32), ("pad", C.c_int32), ("lr", C.c_double), ("emin", C.c_double),
                ("emax", C.c_double), ("tcut", C.c_double), ("ks_gate", C.c_double), ("seed", C.c_uint64)]


class LearnReport(C.Structure):
    _fields_ = [("loss_first", C.c_double), ("loss_last", C.c_double), ("ks_max", C.c_double),
                ("ks_mean", C.c_double), ("ks_noise", C.c_double), ("gen_ms", C.c_double),
                ("train_ms", C.c_double), ("eval_ms", C.c_double), ("samples", C.c_int64),
                ("installed", C.c_int32), ("nparams", C.c_int32)]


class WallRecord(C.Structure):
    _fields_ = [("x", C.c_double * 3), ("p", C.c_double * 3), ("w", C.c_double), ("t", C.c_double),
                ("uid", C.c_uint64), ("species", C.c_int32), ("swarm", C.c_int32)]


class TuneTrial(C.Structure):
    _fields_ = [("launch", Launch), ("rate", C.c_double)]


DP = C.POINTER(C.c_double)
FP = C.POINTER(C.c_float)
SOA = DP * NFIELDS
VP = C.c_void_p

# name -> (restype, argtypes); the C ABI declared in include/particulator_hip.h
SIGNATURES = {
    "pt_abi_version": (C.c_int, []),
    "pt_create": (C.c_int, [C.POINTER(Config), C.POINTER(VP)]),
    "pt_destroy": (None, [VP]),
    "pt_last_error": (C.c_char_p, [VP]),
    "pt_upload_table": (C.c_int, [VP, C.c_int, C.POINTER(TableDesc)]),
    "pt_totalcs": (C.c_int, [C.POINTER(Process), DP, C.c_size_t, DP]),
    "pt_process_desc": (C.c_int, [C.POINTER(Process), C.c_int, C.POINTER(ProcDesc)]),
    "pt_sb_build": (C.c_int, [C.c_int, DP, C.c_int, DP, C.c_int, DP, C.c_int, C.c_double, C.c_double,
                              C.c_double, DP, DP, DP]),
    "pt_sb_thresholds": (C.c_int, [DP, C.c_int, DP]),
    "pt_table_build": (C.c_int, [C.POINTER(Process), C.c_int, C.c_int, DP, C.c_int, C.c_double, C.c_int,
                                 C.c_int, C.c_double, DP, DP, C.POINTER(C.c_int32), DP]),
    "pt_upload_sb": (C.c_int, [VP, C.c_int, C.c_int, C.c_int, C.c_int, DP, DP]),
    "pt_upload_pe": (C.c_int, [VP, C.c_int, C.c_int, C.c_int, DP]),
    "pt_set_field": (C.c_int, [VP, C.c_int, C.POINTER(FieldDesc)]),
    "pt_set_continuum_loss": (C.c_int, [VP, C.c_int, C.c_int, C.c_double, DP, DP]),
    "pt_set_forcing": (C.c_int, [VP, C.c_uint32, C.c_uint32, C.c_uint32]),
    "pt_add_particles": (C.c_int, [VP, C.c_int, SOA, C.POINTER(C.c_uint64),
                                   C.POINTER(C.c_int32), C.c_size_t]),
    "pt_init_particles": (C.c_int, [VP, C.c_int, C.c_size_t, C.c_double, C.c_double, C.c_int,
                                    C.c_int, C.c_uint64, C.c_double]),
    "pt_init_beam": (C.c_int, [VP, C.c_int, C.c_size_t, C.c_double, DP, C.c_int, C.c_uint64, C.c_double]),
    "pt_download": (C.c_int, [VP, C.c_int, SOA, C.POINTER(C.c_uint8), C.POINTER(C.c_uint64),
                              C.POINTER(C.c_int32), C.c_size_t, C.POINTER(C.c_size_t)]),
    "pt_set_particles": (C.c_int, [VP, C.c_int, SOA, C.POINTER(C.c_uint8),
                                   C.POINTER(C.c_uint64), C.POINTER(C.c_int32), C.c_size_t]),
    "pt_count": (C.c_int, [VP, C.c_int, C.POINTER(C.c_uint64)]),
    "pt_init": (C.c_int, [VP]),
    "pt_advance": (C.c_int, [VP, C.c_double]),
    "pt_run": (C.c_int, [VP, C.c_double, C.c_double, C.c_int, C.c_int, C.c_int]),
    "pt_compact": (C.c_int, [VP, C.c_int]),
    "pt_stats": (C.c_int, [VP, C.c_int, C.POINTER(PopStats)]),
    "pt_set_launch": (C.c_int, [VP, C.POINTER(Launch)]),
    "pt_get_launch": (C.c_int, [VP, C.POINTER(Launch)]),
    "pt_run_graph": (C.c_int, [VP, C.c_double, C.c_double, C.c_int, C.c_int]),
    "pt_autotune": (C.c_int, [VP, C.c_double, C.c_double, C.c_int, C.POINTER(TuneTrial), C.c_int,
                              C.POINTER(C.c_int), C.POINTER(Launch), DP]),
    "pt_swarm_stats": (C.c_int, [VP, C.c_int, C.c_int, DP]),
    "pt_swarm_stats_noalloc": (C.c_int, [VP, C.c_int, C.c_int, DP]),
    "pt_set_wall": (C.c_int, [VP, C.c_int, C.c_int, C.c_double, C.c_int, C.c_size_t]),
    "pt_wall_read": (C.c_int, [VP, C.c_void_p, C.c_size_t, C.POINTER(C.c_size_t), C.c_int]),
    "pt_roulette": (C.c_int, [VP, C.c_int, C.c_double]),
    "pt_split": (C.c_int, [VP, C.c_int, C.c_double]),
    "pt_roulette_each": (C.c_int, [VP, C.c_int, DP, C.c_size_t]),
    "pt_split_each": (C.c_int, [VP, C.c_int, DP, C.c_size_t]),
    "pt_learn_defaults": (C.c_int, [C.c_int, C.POINTER(LearnConfig)]),
    "pt_learn_train": (C.c_int, [VP, C.c_int, C.POINTER(LearnConfig), C.POINTER(LearnReport)]),
    "pt_learn_enable": (C.c_int, [VP, C.c_int, C.c_int]),
    "pt_learn_nparams": (C.c_int, []),
    "pt_learn_params": (C.c_int, [VP, C.c_int, FP, C.c_int, C.c_int]),
    "pt_learn_install": (C.c_int, [VP, C.c_int, FP, C.c_int, C.c_double, C.c_double]),
    "pt_learn_throughput": (C.c_int, [VP, C.c_int, C.c_int, DP, C.POINTER(C.c_int32), C.c_size_t, C.c_int,
                                      C.c_uint64, DP]),
    "pt_learn_sample": (C.c_int, [VP, C.c_int, C.c_int, DP, C.POINTER(C.c_int32), C.c_size_t, C.c_uint64, DP]),
    "pt_debug_mlp_grad": (C.c_int, [VP, FP, FP, FP, C.c_int, C.c_float, C.c_float, FP, FP]),
    "pt_debug_mlp_infer": (C.c_int, [VP, FP, FP, C.c_int, FP]),
    "pt_collision_counts": (C.c_int, [VP, C.c_int, C.POINTER(C.c_int64), C.c_int, C.c_int]),
    "pt_tally_read": (C.c_int, [VP, C.c_int, DP, C.c_int, DP, DP]),
    "pt_dose_read": (C.c_int, [VP, DP, C.c_int, DP, DP, DP, C.c_int]),
    "pt_work_read": (C.c_int, [VP, C.POINTER(Work), C.c_int]),
    "pt_profile_enable": (C.c_int, [VP, C.c_int]),
    "pt_set_step": (C.c_int, [VP, C.c_uint32]),
    "pt_get_step": (C.c_int, [VP, C.POINTER(C.c_uint32)]),
    "pt_check": (C.c_int, [VP, C.POINTER(C.c_int64)]),
    "pt_synchronize": (C.c_int, [VP]),
    "pt_debug_philox": (C.c_int, [VP, C.POINTER(C.c_uint32), C.POINTER(C.c_uint32),
                                  C.POINTER(C.c_uint32), C.c_size_t]),
    "pt_debug_choices": (C.c_int, [VP, C.POINTER(C.c_int64)]),
    "pt_debug_uniforms": (C.c_int, [VP, C.c_uint64, C.c_uint32, DP, C.c_size_t]),
    "pt_debug_select": (C.c_int, [VP, C.c_int, C.c_size_t, DP, DP, C.POINTER(C.c_int32),
                                  C.POINTER(C.c_int32), C.POINTER(C.c_int32), DP]),
    "pt_debug_push": (C.c_int, [VP, C.c_int, C.c_size_t, SOA, DP]),
    "pt_debug_collide": (C.c_int, [VP, C.c_int, C.c_int, C.c_size_t, SOA, C.POINTER(C.c_uint64),
                                   DP, C.c_int, C.POINTER(C.c_int32), C.POINTER(C.c_int32), DP,
                                   C.POINTER(C.c_int32), C.POINTER(C.c_uint64)]),
}

_lib = None


def lib():
    """Load the HIP library; raise if it has not been built (there is no fallback)."""
    global _lib
    if _lib is None:
        if not os.path.exists(LIBPATH):
            raise PTError(-9, "%s is not built; run particulator_hip.build.build()" % LIBPATH)
        L = C.CDLL(LIBPATH)
        for name, (res, args) in SIGNATURES.items():
            f = getattr(L, name)
            f.restype = res
            f.argtypes = args
        _lib = L
    return _lib


def check(ctx, rc):
    if rc != 0:
        msg = lib().pt_last_error(ctx).decode()
        raise PTError(rc, msg)
    return rc

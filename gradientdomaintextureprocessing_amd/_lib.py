"""ctypes binding of libgdtp.so (the C ABI declared in include/gdtp.h)."""
import ctypes
import hashlib
import os

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(_HERE, "libgdtp.so")
CSRC = os.path.join(_HERE, "csrc")


def source_hash():
    """SHA-256 (hex, first 16 digits) over the names and contents of the library's sources; the
    build embeds it (gdtp_build_id) so that a library older than its sources is refused."""
    h = hashlib.sha256()
    for name in sorted(os.listdir(CSRC)):
        if name.endswith((".h", ".cpp", ".hip")):
            h.update(name.encode())
            with open(os.path.join(CSRC, name), "rb") as fh:
                h.update(fh.read())
    return h.hexdigest()[:16]

c_int, c_double, c_void_p, c_char_p, c_size_t, c_ull = (ctypes.c_int, ctypes.c_double, ctypes.c_void_p, ctypes.c_char_p,
                                                         ctypes.c_size_t, ctypes.c_ulonglong)
P = ctypes.POINTER

# name -> (restype, argtypes)
SIGNATURES = {
    "gdtp_last_error": (c_char_p, []),
    "gdtp_build_id": (c_char_p, []),
    "gdtp_device_count": (c_int, [P(c_int)]),
    "gdtp_mesh_create": (c_int, [c_void_p, c_int, c_void_p, c_int, c_void_p, P(c_void_p)]),
    "gdtp_mesh_read_ply": (c_int, [c_char_p, P(c_void_p)]),
    "gdtp_mesh_create_cube": (c_int, [c_int, c_int, c_int, P(c_void_p)]),
    "gdtp_mesh_create_icosphere": (c_int, [c_int, c_int, c_int, c_double, c_ull, P(c_void_p)]),
    "gdtp_mesh_create_torus": (c_int, [c_int, c_int, c_int, c_int, c_double, c_double, c_double, c_ull, c_int, c_int, P(c_void_p)]),
    "gdtp_mesh_counts": (c_int, [c_void_p, P(c_int), P(c_int)]),
    "gdtp_mesh_read": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p]),
    "gdtp_mesh_destroy": (None, [c_void_p]),
    "gdtp_hierarchy_create": (c_int, [c_void_p, c_int, c_int, c_int, c_int, P(c_void_p)]),
    "gdtp_hierarchy_create_with_metric": (c_int, [c_void_p, c_int, c_int, c_int, c_void_p, P(c_void_p)]),
    "gdtp_hierarchy_level_info": (c_int, [c_void_p, c_int, c_void_p]),
    "gdtp_hierarchy_array_i32": (c_int, [c_void_p, c_int, c_char_p, c_void_p, P(c_size_t)]),
    "gdtp_hierarchy_array_f64": (c_int, [c_void_p, c_int, c_char_p, c_void_p, P(c_size_t)]),
    "gdtp_hierarchy_destroy": (None, [c_void_p]),
    "gdtp_system_create": (c_int, [c_void_p, c_double, c_double, c_int, P(c_void_p)]),
    "gdtp_system_update": (c_int, [c_void_p, c_double, c_double]),
    "gdtp_system_array_i32": (c_int, [c_void_p, c_int, c_char_p, c_void_p, P(c_size_t)]),
    "gdtp_system_array_f64": (c_int, [c_void_p, c_int, c_char_p, c_void_p, P(c_size_t)]),
    "gdtp_system_destroy": (None, [c_void_p]),
    "gdtp_vcycle": (c_int, [c_void_p, c_void_p, c_void_p, c_int, c_void_p]),
    "gdtp_relax": (c_int, [c_void_p, c_int, c_void_p, c_void_p, c_void_p, c_int, c_void_p]),
    "gdtp_band_sweep": (c_int, [c_void_p, c_int, c_void_p, c_void_p, c_void_p, c_int, c_void_p]),
    "gdtp_restrict": (c_int, [c_void_p, c_int, c_void_p, c_void_p, c_int, c_void_p]),
    "gdtp_prolong_add": (c_int, [c_void_p, c_int, c_void_p, c_void_p, c_int, c_void_p]),
    "gdtp_boundary_solve": (c_int, [c_void_p, c_int, c_void_p, c_void_p, c_int, c_void_p]),
    "gdtp_coarse_solve": (c_int, [c_void_p, c_void_p, c_void_p, c_int, c_void_p]),
    "gdtp_apply": (c_int, [c_void_p, c_int, c_void_p, c_void_p, c_int, c_void_p]),
    "gdtp_residual": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_void_p]),
    "gdtp_residual_norms": (c_int, [c_void_p, c_void_p, c_void_p, c_int, c_void_p, c_void_p, c_void_p]),
    "gdtp_residual_norms_noalloc": (c_int, [c_void_p, c_void_p, c_void_p, c_int, c_void_p, c_void_p, c_void_p]),
    "gdtp_weighted_residual_norms": (c_int, [c_void_p, c_void_p, c_void_p, c_int, c_void_p, c_void_p, c_void_p]),
    "gdtp_direct_solve": (c_int, [c_void_p, c_void_p, c_void_p, c_int, c_void_p, P(c_int), c_void_p]),
    "gdtp_solve_weighted": (c_int, [c_void_p, c_void_p, c_void_p, c_int, c_void_p, c_double, c_int, c_void_p, P(c_int), c_void_p]),
    "gdtp_geodesic_divergence": (c_int, [c_void_p, c_void_p, c_void_p, c_int, c_void_p]),
    "gdtp_solve": (c_int, [c_void_p, c_void_p, c_void_p, c_int, c_double, c_int, c_int, c_void_p, P(c_int), c_void_p]),
    "gdtp_solve_yielding": (c_int, [c_void_p, c_void_p, c_void_p, c_int, c_double, c_int, c_int, c_void_p, P(c_int), c_void_p, c_void_p,
                                    c_void_p]),
    "gdtp_mixed_configure": (c_int, [c_void_p, c_int, c_int, c_int, c_double, c_int]),
    "gdtp_mixed_cycles": (c_int, [c_void_p, c_int]),
    "gdtp_hierarchy_create_ex": (c_int, [c_void_p, c_int, c_int, c_int, c_int, c_void_p, c_int, P(c_void_p)]),
    "gdtp_modulation_create": (c_int, [c_void_p, c_void_p, c_int, P(c_void_p)]),
    "gdtp_modulated_stiffness": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p]),
    "gdtp_modulation_info": (c_int, [c_void_p, c_void_p]),
    "gdtp_modulation_array_f64": (c_int, [c_void_p, c_char_p, c_void_p, P(c_size_t)]),
    "gdtp_modulation_array_i32": (c_int, [c_void_p, c_char_p, c_void_p, P(c_size_t)]),
    "gdtp_modulation_destroy": (None, [c_void_p]),
    "gdtp_mixed_acceleration": (c_int, [c_void_p, c_int]),
    "gdtp_mixed_deep_sweep": (c_int, [c_void_p, c_int, c_int, c_void_p]),
    "gdtp_mixed_tile_shape": (c_int, [c_void_p, c_int, P(c_int)]),
    "gdtp_mixed_level_tile_shape": (c_int, [c_void_p, c_int, c_int, P(c_int)]),
    "gdtp_mixed_tile_shape_info": (c_int, [c_int, P(c_int), P(c_int), P(c_int), P(c_int)]),
    "gdtp_mixed_fuse_transfers": (c_int, [c_void_p, c_int]),
    "gdtp_system_memory": (c_int, [c_void_p, P(c_size_t), P(c_size_t)]),
}

_lib = None


class GdtpError(RuntimeError):
    def __init__(self, code, message):
        super().__init__(f"gdtp error {code}: {message}")
        self.code = code


def built_id():
    """The source identifier embedded in libgdtp.so, read from the file (the library is not loaded:
    a process that loaded a library keeps that copy even after the file is rebuilt)."""
    if not os.path.exists(LIB_PATH):
        return None
    with open(LIB_PATH, "rb") as fh:
        data = fh.read()
    at = data.find(b"gdtp-build-id:")
    return data[at + 14:at + 30].decode(errors="replace") if at >= 0 else None


def is_current():
    """True when libgdtp.so exists and was built from the sources in csrc/ as they are now."""
    return built_id() == source_hash()


def load():
    """Load libgdtp.so (fails loudly if the HIP library has not been built, or was built from
    other sources than those in csrc/)."""
    global _lib
    if _lib is not None:
        return _lib
    if not os.path.exists(LIB_PATH):
        raise ImportError(f"{LIB_PATH} is missing: run `python -m gradientdomaintextureprocessing_amd.build` first")
    # torch first: its HIP runtime then serves the library too (one runtime per process; a second
    # copy loaded before torch leaves torch without a visible GPU)
    import torch  # noqa: F401
    lib = ctypes.CDLL(LIB_PATH)
    lib.gdtp_build_id.restype = c_char_p
    built = lib.gdtp_build_id().decode()
    if built != source_hash():
        raise ImportError(f"{LIB_PATH} was built from other sources ({built}, sources now {source_hash()}): "
                          "run `python -m gradientdomaintextureprocessing_amd.build` again")
    for name, (res, args) in SIGNATURES.items():
        fn = getattr(lib, name)
        fn.restype = res
        fn.argtypes = args
    _lib = lib
    return lib


def check(rc):
    if rc != 0:
        raise GdtpError(rc, load().gdtp_last_error().decode())
    return rc

"""Python binding of the MI355X PatchMatch-MVS library (libhp3d_pm.so).

Thin ctypes layer over the C ABI declared in include/hp3d_pm.h and
include/hp3d_scene.h.  Nothing here computes: every solve runs in the HIP
kernels of csrc/.  If the library is not built, importing this package
raises, so no caller can silently fall back to a CPU path.

The directory name contains a hyphen; load it with load_package() from
__graft_entry__.py (or importlib) under the module name
``hemiphoto3d_private_amd``.
"""
import ctypes
import os
import subprocess

import numpy as np

HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(HERE, "libhp3d_pm.so")

MAX_SRC = 8
OK = 0
ERR_INVALID_ARG, ERR_OOM_BUDGET, ERR_DEVICE, ERR_CANCELLED = -1, -2, -3, -4
ERR_NOT_FOUND, ERR_UNSUPPORTED, ERR_IO, ERR_AGAIN = -5, -6, -7, -8
FMT_U8, FMT_F32 = 0, 1
STORE_F32, STORE_F16 = 0, 1
CTX_TIMING = 1
SCENE_PLANE, SCENE_SPHERE_GROUND, SCENE_SPHERE = 0, 1, 2

_f32p = ctypes.POINTER(ctypes.c_float)
_f64p = ctypes.POINTER(ctypes.c_double)
_u8p = ctypes.POINTER(ctypes.c_uint8)


class HP3DError(RuntimeError):
    def __init__(self, code, msg):
        super().__init__(f"hp3d error {code}: {msg}")
        self.code = code


class Opts(ctypes.Structure):
    _fields_ = [("device", ctypes.c_int), ("hbm_budget", ctypes.c_size_t),
                ("stream", ctypes.c_void_p), ("flags", ctypes.c_int)]


class SeedPoint(ctypes.Structure):
    _fields_ = [("x", ctypes.c_int), ("y", ctypes.c_int), ("depth", ctypes.c_float),
                ("normal", ctypes.c_float * 3)]


class ViewDesc(ctypes.Structure):
    _fields_ = [
        ("ref", ctypes.c_uint64), ("src", ctypes.c_uint64 * MAX_SRC), ("num_src", ctypes.c_int),
        ("K_ref_inv", ctypes.c_double * 9),
        ("A", (ctypes.c_double * 9) * MAX_SRC), ("b", (ctypes.c_double * 3) * MAX_SRC),
        ("depth_min", ctypes.c_float), ("depth_max", ctypes.c_float),
        ("radius", ctypes.c_int), ("stride", ctypes.c_int), ("iterations", ctypes.c_int),
        ("top_k", ctypes.c_int), ("seed", ctypes.c_uint64),
        ("init_depth", _f32p), ("init_normal", _f32p),
        ("seeds", ctypes.POINTER(SeedPoint)), ("num_seeds", ctypes.c_int),
        ("seed_radius", ctypes.c_int), ("first_iteration", ctypes.c_int),
    ]


class SfmCamera(ctypes.Structure):
    _fields_ = [("image_id", ctypes.c_int), ("is_registered", ctypes.c_int),
                ("K", ctypes.c_double * 9), ("R", ctypes.c_double * 9), ("t", ctypes.c_double * 3)]


class SfmPoint(ctypes.Structure):
    _fields_ = [("position", ctypes.c_double * 3), ("image_ids", ctypes.POINTER(ctypes.c_int)),
                ("num_image_ids", ctypes.c_int)]


class SourceView(ctypes.Structure):
    _fields_ = [("image_id", ctypes.c_int), ("score", ctypes.c_float),
                ("baseline_deg", ctypes.c_float)]


class ViewParams(ctypes.Structure):
    _fields_ = [("ref_image_id", ctypes.c_int), ("num_src", ctypes.c_int),
                ("src", SourceView * MAX_SRC), ("depth_min", ctypes.c_float),
                ("depth_max", ctypes.c_float)]


class ViewOut(ctypes.Structure):
    _fields_ = [("depth", _f32p), ("normal", _f32p), ("cost", _f32p), ("confidence", _f32p),
                ("on_device", ctypes.c_int)]


class BatchOpts(ctypes.Structure):
    _fields_ = [("variant", ctypes.c_int), ("use_graph", ctypes.c_int),
                ("persistent", ctypes.c_int), ("chunk", ctypes.c_int)]


NUM_VARIANTS = 6
JOB_QUEUED, JOB_RUNNING, JOB_DONE, JOB_FAILED, JOB_CANCELLED = 0, 1, 2, 3, 4


class ServerOpts(ctypes.Structure):
    _fields_ = [("device", ctypes.c_int), ("hbm_budget", ctypes.c_size_t),
                ("max_jobs", ctypes.c_int), ("radius", ctypes.c_int), ("stride", ctypes.c_int),
                ("store", ctypes.c_int), ("variant", ctypes.c_int)]


class JobDesc(ctypes.Structure):
    _fields_ = [("width", ctypes.c_int), ("height", ctypes.c_int), ("num_src", ctypes.c_int),
                ("ref", _u8p), ("src", _u8p * MAX_SRC),
                ("K_ref_inv", ctypes.c_double * 9),
                ("A", (ctypes.c_double * 9) * MAX_SRC), ("b", (ctypes.c_double * 3) * MAX_SRC),
                ("depth_min", ctypes.c_float), ("depth_max", ctypes.c_float),
                ("iterations", ctypes.c_int), ("top_k", ctypes.c_int), ("seed", ctypes.c_uint64),
                ("out_depth", _f32p), ("out_normal", _f32p), ("out_cost", _f32p),
                ("fail_at_step", ctypes.c_int), ("ref_image", ctypes.c_uint64),
                ("src_image", ctypes.c_uint64 * MAX_SRC), ("level", ctypes.c_int)]


class JobStatus(ctypes.Structure):
    _fields_ = [("state", ctypes.c_int), ("error", ctypes.c_int), ("t_submit", ctypes.c_double),
                ("t_admit", ctypes.c_double), ("t_done", ctypes.c_double), ("steps", ctypes.c_int)]


class ServerStats(ctypes.Structure):
    _fields_ = [("steps", ctypes.c_longlong), ("busy_ms", ctypes.c_double),
                ("wall_s", ctypes.c_double), ("submitted", ctypes.c_longlong),
                ("done", ctypes.c_longlong), ("failed", ctypes.c_longlong),
                ("cancelled", ctypes.c_longlong), ("rejected", ctypes.c_longlong),
                ("taps", ctypes.c_double), ("mpix_iters", ctypes.c_double),
                ("arena_bytes", ctypes.c_size_t), ("arena_peak", ctypes.c_size_t),
                ("max_active", ctypes.c_int), ("image_uploads", ctypes.c_longlong),
                ("image_reuses", ctypes.c_longlong), ("resident_images", ctypes.c_longlong),
                ("wait_ms", ctypes.c_double)]


class GeomView(ctypes.Structure):
    _fields_ = [("width", ctypes.c_int), ("height", ctypes.c_int), ("depth", _f32p),
                ("normal", _f32p), ("confidence", _f32p), ("K", ctypes.c_double * 9),
                ("R", ctypes.c_double * 9), ("t", ctypes.c_double * 3), ("num_src", ctypes.c_int),
                ("src", ctypes.c_int * MAX_SRC)]


class FuseView(ctypes.Structure):
    _fields_ = [("width", ctypes.c_int), ("height", ctypes.c_int), ("depth", _f32p),
                ("normal", _f32p), ("confidence", _f32p), ("color", _u8p),
                ("color_channels", ctypes.c_int), ("K", ctypes.c_double * 9),
                ("R", ctypes.c_double * 9), ("t", ctypes.c_double * 3)]


class Stats(ctypes.Structure):
    _fields_ = [("ms_total", ctypes.c_double), ("ms_init", ctypes.c_double),
                ("ms_cost", ctypes.c_double), ("ms_propagate", ctypes.c_double),
                ("n_propagate", ctypes.c_int), ("ms_finalize", ctypes.c_double),
                ("taps", ctypes.c_double), ("hbm_in_use", ctypes.c_size_t),
                ("hbm_budget", ctypes.c_size_t)]


class Scene(ctypes.Structure):
    _fields_ = [("kind", ctypes.c_int), ("seed", ctypes.c_uint64), ("octaves", ctypes.c_int),
                ("tex_freq", ctypes.c_double), ("plane_point", ctypes.c_double * 3),
                ("plane_normal", ctypes.c_double * 3), ("sphere_center", ctypes.c_double * 3),
                ("sphere_radius", ctypes.c_double), ("ground_y", ctypes.c_double),
                ("backdrop_z", ctypes.c_double)]


class Camera(ctypes.Structure):
    _fields_ = [("width", ctypes.c_int), ("height", ctypes.c_int), ("K", ctypes.c_double * 9),
                ("R", ctypes.c_double * 9), ("t", ctypes.c_double * 3)]


# Every exported symbol of the C ABI, with (restype, argtypes).
SIGNATURES = {
    "hp3d_pm_version": (ctypes.c_char_p, []),
    "hp3d_pm_create": (ctypes.c_int, [ctypes.POINTER(Opts), ctypes.POINTER(ctypes.c_void_p)]),
    "hp3d_pm_destroy": (ctypes.c_int, [ctypes.c_void_p]),
    "hp3d_pm_last_error": (ctypes.c_char_p, [ctypes.c_void_p]),
    "hp3d_pm_image_upload": (ctypes.c_int, [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_int,
                                            ctypes.c_int, ctypes.c_size_t, ctypes.c_int,
                                            ctypes.c_int, ctypes.POINTER(ctypes.c_uint64)]),
    "hp3d_pm_image_release": (ctypes.c_int, [ctypes.c_void_p, ctypes.c_uint64]),
    "hp3d_pm_image_info": (ctypes.c_int, [ctypes.c_void_p, ctypes.c_uint64,
                                          ctypes.POINTER(ctypes.c_int), ctypes.POINTER(ctypes.c_int),
                                          ctypes.POINTER(ctypes.c_int),
                                          ctypes.POINTER(ctypes.c_size_t)]),
    "hp3d_pm_compose": (ctypes.c_int, [_f64p] * 8),
    "hp3d_pm_invert3": (ctypes.c_int, [_f64p, _f64p]),
    "hp3d_pm_run_view": (ctypes.c_int, [ctypes.c_void_p, ctypes.POINTER(ViewDesc),
                                        ctypes.POINTER(ViewOut)]),
    "hp3d_pm_run_views": (ctypes.c_int, [ctypes.c_void_p, ctypes.POINTER(ViewDesc), ctypes.c_int,
                                         ctypes.POINTER(ViewOut)]),
    "hp3d_pm_run_view_noalloc": (ctypes.c_int, [ctypes.c_void_p, ctypes.POINTER(ViewDesc),
                                                ctypes.POINTER(ViewOut)]),
    "hp3d_pm_host_alloc": (ctypes.c_int, [ctypes.c_void_p, ctypes.c_size_t,
                                          ctypes.POINTER(ctypes.c_void_p)]),
    "hp3d_pm_host_free": (ctypes.c_int, [ctypes.c_void_p, ctypes.c_void_p]),
    "hp3d_pm_init_hypotheses": (ctypes.c_int, [ctypes.c_void_p, ctypes.POINTER(ViewDesc),
                                               _f32p, _f32p]),
    "hp3d_pm_cost_eval": (ctypes.c_int, [ctypes.c_void_p, ctypes.POINTER(ViewDesc), _f32p, _f32p,
                                         _f32p]),
    "hp3d_pm_get_stats": (ctypes.c_int, [ctypes.c_void_p, ctypes.POINTER(Stats)]),
    "hp3d_pm_batch_run": (ctypes.c_int, [ctypes.c_void_p, ctypes.POINTER(ViewDesc), ctypes.c_int,
                                         ctypes.POINTER(ViewOut), ctypes.POINTER(BatchOpts)]),
    "hp3d_pm_autotune": (ctypes.c_int, [ctypes.c_void_p, ctypes.POINTER(ViewDesc), ctypes.c_int,
                                        ctypes.POINTER(ctypes.c_int), _f32p]),
    "hp3d_pm_variant_info": (ctypes.c_int, [ctypes.c_int, ctypes.POINTER(ctypes.c_int),
                                            ctypes.POINTER(ctypes.c_int),
                                            ctypes.POINTER(ctypes.c_int)]),
    "hp3d_pm_tune_save": (ctypes.c_int, [ctypes.c_void_p, ctypes.c_char_p]),
    "hp3d_pm_tune_load": (ctypes.c_int, [ctypes.c_void_p, ctypes.c_char_p]),
    "hp3d_pm_geom_filter": (ctypes.c_int, [ctypes.c_void_p, ctypes.POINTER(GeomView), ctypes.c_int,
                                           ctypes.c_float, ctypes.c_float, ctypes.c_int,
                                           ctypes.POINTER(ctypes.c_int)]),
    "hp3d_pm_fuse": (ctypes.c_int, [ctypes.c_void_p, ctypes.POINTER(FuseView), ctypes.c_int,
                                    ctypes.c_float, _f32p, _f32p, _f32p, ctypes.c_size_t,
                                    ctypes.POINTER(ctypes.c_size_t)]),
    "hp3d_server_create": (ctypes.c_int, [ctypes.POINTER(ServerOpts),
                                          ctypes.POINTER(ctypes.c_void_p)]),
    "hp3d_server_submit": (ctypes.c_int, [ctypes.c_void_p, ctypes.POINTER(JobDesc),
                                          ctypes.POINTER(ctypes.c_uint64)]),
    "hp3d_server_poll": (ctypes.c_int, [ctypes.c_void_p, ctypes.c_uint64,
                                        ctypes.POINTER(JobStatus)]),
    "hp3d_server_wait": (ctypes.c_int, [ctypes.c_void_p, ctypes.c_uint64, ctypes.c_double,
                                        ctypes.POINTER(JobStatus)]),
    "hp3d_server_cancel": (ctypes.c_int, [ctypes.c_void_p, ctypes.c_uint64]),
    "hp3d_server_forget": (ctypes.c_int, [ctypes.c_void_p, ctypes.c_uint64]),
    "hp3d_server_get_stats": (ctypes.c_int, [ctypes.c_void_p, ctypes.POINTER(ServerStats)]),
    "hp3d_server_last_error": (ctypes.c_char_p, [ctypes.c_void_p]),
    "hp3d_server_image_add": (ctypes.c_int, [ctypes.c_void_p, _u8p, ctypes.c_int, ctypes.c_int,
                                             ctypes.c_size_t, ctypes.c_int,
                                             ctypes.POINTER(ctypes.c_uint64)]),
    "hp3d_server_image_remove": (ctypes.c_int, [ctypes.c_void_p, ctypes.c_uint64]),
    "hp3d_server_image_read": (ctypes.c_int, [ctypes.c_void_p, ctypes.c_uint64, ctypes.c_int,
                                              ctypes.POINTER(ctypes.c_int),
                                              ctypes.POINTER(ctypes.c_int), _f32p,
                                              ctypes.c_size_t]),
    "hp3d_server_destroy": (ctypes.c_int, [ctypes.c_void_p]),
    "hp3d_pm_device_alloc": (ctypes.c_int, [ctypes.c_void_p, ctypes.c_size_t,
                                            ctypes.POINTER(ctypes.c_void_p)]),
    "hp3d_pm_device_free": (ctypes.c_int, [ctypes.c_void_p, ctypes.c_void_p]),
    "hp3d_pm_device_copy": (ctypes.c_int, [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p,
                                           ctypes.c_size_t, ctypes.c_int]),
    "hp3d_select_source_views": (ctypes.c_int, [ctypes.POINTER(SfmCamera), ctypes.c_int,
                                                ctypes.POINTER(SfmPoint), ctypes.c_int,
                                                ctypes.c_int, ctypes.POINTER(ViewParams),
                                                ctypes.POINTER(ctypes.c_int)]),
    "hp3d_project_seed_points": (ctypes.c_int, [ctypes.POINTER(SfmCamera),
                                                ctypes.POINTER(SfmPoint), ctypes.c_int,
                                                ctypes.c_float, ctypes.c_float, ctypes.c_int,
                                                ctypes.c_int, ctypes.c_int,
                                                ctypes.POINTER(SeedPoint),
                                                ctypes.POINTER(ctypes.c_int)]),
    "hp3d_pfm_save": (ctypes.c_int, [ctypes.c_char_p, ctypes.c_int, ctypes.c_int, _f32p]),
    "hp3d_pfm_load": (ctypes.c_int, [ctypes.c_char_p, ctypes.POINTER(ctypes.c_int),
                                     ctypes.POINTER(ctypes.c_int), _f32p, ctypes.c_size_t]),
    "hp3d_pfm_save_ex": (ctypes.c_int, [ctypes.c_char_p, ctypes.c_int, ctypes.c_int,
                                        ctypes.c_int, _f32p]),
    "hp3d_pfm_load_ex": (ctypes.c_int, [ctypes.c_char_p, ctypes.POINTER(ctypes.c_int),
                                        ctypes.POINTER(ctypes.c_int),
                                        ctypes.POINTER(ctypes.c_int), _f32p, ctypes.c_size_t]),
    "hp3d_scene_render": (ctypes.c_int, [ctypes.POINTER(Scene), ctypes.POINTER(Camera),
                                         ctypes.c_double, ctypes.c_uint64, _u8p, _f32p, _f32p,
                                         ctypes.c_int]),
}


def build():
    """Compile the HIP kernels and host runtime into libhp3d_pm.so (in-tree)."""
    subprocess.check_call(["make", "-s", "-C", HERE, f"-j{min(8, os.cpu_count() or 1)}"])


_lib = None


def lib():
    global _lib
    if _lib is None:
        if not os.path.exists(LIB_PATH):
            raise ImportError(f"{LIB_PATH} is not built; run __graft_entry__.build() "
                              "(make -C hemiphoto3d-private_amd)")
        L = ctypes.CDLL(LIB_PATH)
        for name, (res, args) in SIGNATURES.items():
            fn = getattr(L, name)
            fn.restype = res
            fn.argtypes = args
        _lib = L
    return _lib


def _p(a, t):
    return a.ctypes.data_as(t)


def _check(code, ctx=None):
    if code != OK:
        msg = lib().hp3d_pm_last_error(ctx).decode() if ctx else ""
        raise HP3DError(code, msg)


# ---------------------------------------------------------------------------
# Host math
# ---------------------------------------------------------------------------
def invert3(M):
    M = np.ascontiguousarray(M, dtype=np.float64).reshape(9)
    out = np.zeros(9)
    _check(lib().hp3d_pm_invert3(_p(M, _f64p), _p(out, _f64p)))
    return out.reshape(3, 3)


def compose(K_ref, R_ref, t_ref, K_src, R_src, t_src):
    """FP64 plane-homography terms (A, b) of one source view."""
    args = [np.ascontiguousarray(a, dtype=np.float64).reshape(-1)
            for a in (K_ref, R_ref, t_ref, K_src, R_src, t_src)]
    A = np.zeros(9)
    b = np.zeros(3)
    _check(lib().hp3d_pm_compose(*[_p(a, _f64p) for a in args], _p(A, _f64p), _p(b, _f64p)))
    return A.reshape(3, 3), b


def pfm_save(path, depth):
    depth = np.ascontiguousarray(depth, dtype=np.float32)
    H, W = depth.shape
    _check(lib().hp3d_pfm_save(os.fsencode(path), W, H, _p(depth, _f32p)))


def pfm_save_ex(path, data):
    """(H, W) -> "Pf", (H, W, 3) -> "PF"."""
    data = np.ascontiguousarray(data, dtype=np.float32)
    H, W = data.shape[:2]
    C = 1 if data.ndim == 2 else data.shape[2]
    _check(lib().hp3d_pfm_save_ex(os.fsencode(path), W, H, C, _p(data, _f32p)))


def pfm_load_ex(path):
    W, H, C = ctypes.c_int(0), ctypes.c_int(0), ctypes.c_int(0)
    _check(lib().hp3d_pfm_load_ex(os.fsencode(path), ctypes.byref(W), ctypes.byref(H),
                                  ctypes.byref(C), None, 0))
    shape = (H.value, W.value) if C.value == 1 else (H.value, W.value, C.value)
    out = np.zeros(shape, dtype=np.float32)
    _check(lib().hp3d_pfm_load_ex(os.fsencode(path), ctypes.byref(W), ctypes.byref(H),
                                  ctypes.byref(C), _p(out, _f32p), out.size))
    return out


def pfm_load(path):
    W, H = ctypes.c_int(0), ctypes.c_int(0)
    _check(lib().hp3d_pfm_load(os.fsencode(path), ctypes.byref(W), ctypes.byref(H), None, 0))
    out = np.zeros((H.value, W.value), dtype=np.float32)
    _check(lib().hp3d_pfm_load(os.fsencode(path), ctypes.byref(W), ctypes.byref(H),
                               _p(out, _f32p), out.size))
    return out


def render(scene, camera, noise_sigma=0.0, noise_seed=0, threads=0, gt=True):
    """Render (image uint8 (H,W), gt_depth (H,W) or None, gt_normal (H,W,3) or None)."""
    H, W = camera.height, camera.width
    img = np.zeros((H, W), dtype=np.uint8)
    gd = np.zeros((H, W), dtype=np.float32) if gt else None
    gn = np.zeros((H, W, 3), dtype=np.float32) if gt else None
    rc = lib().hp3d_scene_render(ctypes.byref(scene), ctypes.byref(camera), float(noise_sigma),
                                 int(noise_seed), _p(img, _u8p),
                                 _p(gd, _f32p) if gt else None, _p(gn, _f32p) if gt else None,
                                 int(threads))
    if rc != 0:
        raise HP3DError(ERR_INVALID_ARG, "scene render failed")
    return img, gd, gn


# ---------------------------------------------------------------------------
# Device context
# ---------------------------------------------------------------------------
class Context:
    """One hp3d_pm_ctx: images, state buffers and a HIP stream on one device."""

    def __init__(self, device=0, hbm_budget=0, timing=False):
        o = Opts(device, hbm_budget, None, CTX_TIMING if timing else 0)
        h = ctypes.c_void_p()
        code = lib().hp3d_pm_create(ctypes.byref(o), ctypes.byref(h))
        if code != OK:
            raise HP3DError(code, "hp3d_pm_create failed (no usable HIP device?)")
        self.h = h

    def close(self):
        if self.h:
            lib().hp3d_pm_destroy(self.h)
            self.h = None

    def __enter__(self):
        return self

    def __exit__(self, *exc):
        self.close()

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass

    def last_error(self):
        return lib().hp3d_pm_last_error(self.h).decode()

    def upload(self, image, store=STORE_F32):
        """Upload an (H, W) uint8 DN image or float32 gray image in [0, 1]."""
        a = np.ascontiguousarray(image)
        if a.dtype == np.uint8:
            fmt = FMT_U8
        elif a.dtype == np.float32:
            fmt = FMT_F32
        else:
            raise TypeError("image must be uint8 or float32")
        H, W = a.shape
        out = ctypes.c_uint64(0)
        _check(lib().hp3d_pm_image_upload(self.h, a.ctypes.data, W, H, a.strides[0], fmt,
                                          store, ctypes.byref(out)), self.h)
        return out.value

    def release(self, img):
        _check(lib().hp3d_pm_image_release(self.h, img), self.h)

    def image_info(self, img):
        W, H, st, nb = ctypes.c_int(), ctypes.c_int(), ctypes.c_int(), ctypes.c_size_t()
        _check(lib().hp3d_pm_image_info(self.h, img, ctypes.byref(W), ctypes.byref(H),
                                        ctypes.byref(st), ctypes.byref(nb)), self.h)
        return W.value, H.value, st.value, nb.value

    def stats(self):
        s = Stats()
        _check(lib().hp3d_pm_get_stats(self.h, ctypes.byref(s)), self.h)
        return {f: getattr(s, f) for f, _ in Stats._fields_}

    def run_view(self, desc, shape, with_normal=True, with_cost=True, with_confidence=False):
        H, W = shape
        depth = np.empty((H, W), dtype=np.float32)
        normal = np.empty((H, W, 3), dtype=np.float32) if with_normal else None
        cost = np.empty((H, W), dtype=np.float32) if with_cost else None
        conf = np.empty((H, W), dtype=np.float32) if with_confidence else None
        out = ViewOut(_p(depth, _f32p), _p(normal, _f32p) if with_normal else None,
                      _p(cost, _f32p) if with_cost else None,
                      _p(conf, _f32p) if with_confidence else None, 0)
        _check(lib().hp3d_pm_run_view(self.h, ctypes.byref(desc), ctypes.byref(out)), self.h)
        res = {"depth": depth, "normal": normal, "cost": cost}
        if with_confidence:
            res["confidence"] = conf
        return res

    def host_array(self, shape, dtype=np.float32):
        """A numpy array in page-locked host memory owned by the context
        (hp3d_pm_host_alloc); valid until host_free or close."""
        dtype = np.dtype(dtype)
        nbytes = int(np.prod(shape)) * dtype.itemsize
        p = ctypes.c_void_p()
        _check(lib().hp3d_pm_host_alloc(self.h, max(nbytes, 1), ctypes.byref(p)), self.h)
        buf = (ctypes.c_char * max(nbytes, 1)).from_address(p.value)
        return np.frombuffer(buf, dtype=dtype, count=int(np.prod(shape))).reshape(shape)

    def host_free(self, arr):
        _check(lib().hp3d_pm_host_free(self.h, ctypes.c_void_p(arr.ctypes.data)), self.h)

    def host_outputs(self, shape, with_normal=True, with_cost=True, pinned=False):
        """Output arrays of one view: depth, normal and cost (pinned or pageable)."""
        H, W = shape
        mk = (lambda shp: self.host_array(shp)) if pinned else \
            (lambda shp: np.zeros(shp, dtype=np.float32))
        return {"depth": mk((H, W)), "normal": mk((H, W, 3)) if with_normal else None,
                "cost": mk((H, W)) if with_cost else None}

    def run_views(self, descs, outs):
        """Solve views back to back (hp3d_pm_run_views): each view's outputs
        download while the next view computes.  outs: dicts from
        host_outputs, filled in place; returns outs."""
        n = len(descs)
        darr = (ViewDesc * n)(*descs)
        oarr = (ViewOut * n)()
        for i, o in enumerate(outs):
            oarr[i] = ViewOut(_p(o["depth"], _f32p),
                              _p(o["normal"], _f32p) if o.get("normal") is not None else None,
                              _p(o["cost"], _f32p) if o.get("cost") is not None else None,
                              None, 0)
        _check(lib().hp3d_pm_run_views(self.h, darr, n, oarr), self.h)
        return outs

    def device_alloc(self, nbytes):
        """Device buffer owned by the context (counted against its HBM budget)."""
        p = ctypes.c_void_p()
        _check(lib().hp3d_pm_device_alloc(self.h, int(nbytes), ctypes.byref(p)), self.h)
        return p.value

    def device_free(self, ptr):
        _check(lib().hp3d_pm_device_free(self.h, ctypes.c_void_p(ptr)), self.h)

    def download(self, ptr, shape, dtype=np.float32):
        out = np.empty(shape, dtype=dtype)
        _check(lib().hp3d_pm_device_copy(self.h, out.ctypes.data, ctypes.c_void_p(ptr),
                                         out.nbytes, 1), self.h)
        return out

    def upload_bytes(self, ptr, array):
        a = np.ascontiguousarray(array)
        _check(lib().hp3d_pm_device_copy(self.h, ctypes.c_void_p(ptr), a.ctypes.data, a.nbytes, 0),
               self.h)

    def run_view_device(self, desc, depth_ptr, normal_ptr=0, cost_ptr=0):
        """Solve into caller-owned device buffers (raw device addresses)."""
        out = ViewOut(ctypes.cast(depth_ptr, _f32p), ctypes.cast(normal_ptr or None, _f32p),
                      ctypes.cast(cost_ptr or None, _f32p), None, 1)
        _check(lib().hp3d_pm_run_view(self.h, ctypes.byref(desc), ctypes.byref(out)), self.h)

    def batch_run(self, descs, shapes, variant=-1, use_graph=True, with_normal=True,
                  with_cost=True, persistent=False, chunk=0):
        """Solve many views in one graph launch (a graph of step launches, or
        one persistent kernel); returns one output dict per view."""
        n = len(descs)
        arr = (ViewDesc * n)(*descs)
        outs = (ViewOut * n)()
        res = []
        for j, (H, W) in enumerate(shapes):
            r = {"depth": np.empty((H, W), np.float32),
                 "normal": np.empty((H, W, 3), np.float32) if with_normal else None,
                 "cost": np.empty((H, W), np.float32) if with_cost else None}
            outs[j] = ViewOut(_p(r["depth"], _f32p),
                              _p(r["normal"], _f32p) if with_normal else None,
                              _p(r["cost"], _f32p) if with_cost else None, None, 0)
            res.append(r)
        o = BatchOpts(int(variant), 1 if use_graph else 0, 1 if persistent else 0, int(chunk))
        _check(lib().hp3d_pm_batch_run(self.h, arr, n, outs, ctypes.byref(o)), self.h)
        return res

    def batch_run_device(self, descs, out_ptrs, variant=-1, use_graph=True, persistent=False,
                         chunk=0):
        """Batch into caller device buffers: out_ptrs = [(depth, normal, cost)] per view."""
        n = len(descs)
        arr = (ViewDesc * n)(*descs)
        outs = (ViewOut * n)()
        for j, (dd, dn, dc) in enumerate(out_ptrs):
            outs[j] = ViewOut(ctypes.cast(dd, _f32p), ctypes.cast(dn or None, _f32p),
                              ctypes.cast(dc or None, _f32p), None, 1)
        o = BatchOpts(int(variant), 1 if use_graph else 0, 1 if persistent else 0, int(chunk))
        _check(lib().hp3d_pm_batch_run(self.h, arr, n, outs, ctypes.byref(o)), self.h)

    def geom_filter(self, maps, depth_tol=0.12, normal_tol_deg=180.0, min_consistent=2):
        """In-order, in-place geometric filter.  maps: list of dicts with keys
        depth (H,W) float32 (modified), normal (H,W,3), confidence (optional,
        modified), K, R, t, src (list of indices).  Returns retained counts."""
        n = len(maps)
        arr = (GeomView * n)()
        for i, m in enumerate(maps):
            for k in ("depth", "normal", "confidence"):
                if m.get(k) is not None:
                    assert m[k].dtype == np.float32 and m[k].flags.c_contiguous
            g = arr[i]
            g.height, g.width = m["depth"].shape
            g.depth = _p(m["depth"], _f32p)
            g.normal = _p(m["normal"], _f32p)
            g.confidence = _p(m["confidence"], _f32p) if m.get("confidence") is not None else None
            for j, val in enumerate(np.asarray(m["K"], np.float64).reshape(9)):
                g.K[j] = val
            for j, val in enumerate(np.asarray(m["R"], np.float64).reshape(9)):
                g.R[j] = val
            for j, val in enumerate(np.asarray(m["t"], np.float64).reshape(3)):
                g.t[j] = val
            g.num_src = len(m["src"])
            for j, s in enumerate(m["src"]):
                g.src[j] = int(s)
        ret = (ctypes.c_int * n)()
        _check(lib().hp3d_pm_geom_filter(self.h, arr, n, float(depth_tol), float(normal_tol_deg),
                                         int(min_consistent), ret), self.h)
        return list(ret)

    def fuse(self, maps, min_confidence=0.0, with_normals=True, with_colors=True):
        """Fuse depth maps into points.  maps: dicts with depth (H,W), optional
        normal (H,W,3), confidence (H,W), color (H,W) or (H,W,3) uint8, and
        K, R, t.  Returns (positions, normals, colors) as (N, 3) float32."""
        n = len(maps)
        arr = (FuseView * n)()
        keep = []
        for i, m in enumerate(maps):
            g = arr[i]
            d = np.ascontiguousarray(m["depth"], np.float32)
            keep.append(d)
            g.height, g.width = d.shape
            g.depth = _p(d, _f32p)
            for k, t in (("normal", np.float32), ("confidence", np.float32)):
                if m.get(k) is not None:
                    a = np.ascontiguousarray(m[k], t)
                    keep.append(a)
                    setattr(g, k, _p(a, _f32p))
            if m.get("color") is not None:
                c = np.ascontiguousarray(m["color"], np.uint8)
                keep.append(c)
                g.color = _p(c, _u8p)
                g.color_channels = 1 if c.ndim == 2 else c.shape[2]
            for name, cnt in (("K", 9), ("R", 9), ("t", 3)):
                for j, val in enumerate(np.asarray(m[name], np.float64).reshape(cnt)):
                    getattr(g, name)[j] = val
        cnt = ctypes.c_size_t(0)
        _check(lib().hp3d_pm_fuse(self.h, arr, n, float(min_confidence), None, None, None, 0,
                                  ctypes.byref(cnt)), self.h)
        N = cnt.value
        pos = np.empty((N, 3), np.float32)
        nrm = np.empty((N, 3), np.float32) if with_normals else None
        col = np.empty((N, 3), np.float32) if with_colors else None
        if N:
            _check(lib().hp3d_pm_fuse(self.h, arr, n, float(min_confidence), _p(pos, _f32p),
                                      _p(nrm, _f32p) if with_normals else None,
                                      _p(col, _f32p) if with_colors else None, N,
                                      ctypes.byref(cnt)), self.h)
        return pos, nrm, col

    def autotune(self, descs):
        n = len(descs)
        arr = (ViewDesc * n)(*descs)
        best = ctypes.c_int(-1)
        times = np.zeros(NUM_VARIANTS, np.float32)
        _check(lib().hp3d_pm_autotune(self.h, arr, n, ctypes.byref(best), _p(times, _f32p)),
               self.h)
        return best.value, times

    def tune_save(self, path):
        _check(lib().hp3d_pm_tune_save(self.h, os.fsencode(path)), self.h)

    def tune_load(self, path):
        _check(lib().hp3d_pm_tune_load(self.h, os.fsencode(path)), self.h)

    def init_hypotheses(self, desc, shape):
        H, W = shape
        depth = np.empty((H, W), dtype=np.float32)
        normal = np.empty((H, W, 3), dtype=np.float32)
        _check(lib().hp3d_pm_init_hypotheses(self.h, ctypes.byref(desc), _p(depth, _f32p),
                                             _p(normal, _f32p)), self.h)
        return depth, normal

    def cost_eval(self, desc, depth, normal):
        depth = np.ascontiguousarray(depth, dtype=np.float32)
        normal = np.ascontiguousarray(normal, dtype=np.float32)
        cost = np.empty(depth.shape, dtype=np.float32)
        _check(lib().hp3d_pm_cost_eval(self.h, ctypes.byref(desc), _p(depth, _f32p),
                                       _p(normal, _f32p), _p(cost, _f32p)), self.h)
        return cost


# ---------------------------------------------------------------------------
# Host view set-up (SfM cameras and points as plain arrays)
# ---------------------------------------------------------------------------
class SfM:
    """Cameras (K, R, t world->camera, registered flag; image id = index) and
    sparse points (position, observing image ids), packed for the C ABI."""

    def __init__(self, cameras, points):
        self.cams = (SfmCamera * max(1, len(cameras)))()
        for i, c in enumerate(cameras):
            cc = self.cams[i]
            cc.image_id = i
            cc.is_registered = int(c.get("registered", True))
            for name in ("K", "R", "t"):
                vals = np.asarray(c[name], np.float64).reshape(-1)
                for j, v in enumerate(vals):
                    getattr(cc, name)[j] = v
        self.n_cams = len(cameras)
        self.pts = (SfmPoint * max(1, len(points)))()
        self._ids = []
        for k, (pos, ids) in enumerate(points):
            ids = np.ascontiguousarray(ids, dtype=np.int32)
            self._ids.append(ids)
            p = self.pts[k]
            for j in range(3):
                p.position[j] = float(pos[j])
            p.image_ids = ids.ctypes.data_as(ctypes.POINTER(ctypes.c_int))
            p.num_image_ids = len(ids)
        self.n_pts = len(points)

    def select_source_views(self, num_sources=5):
        """selectSourceViews: list of dicts (ref_image_id, sources [(id, score, deg)],
        depth_min, depth_max), one per registered camera."""
        out = (ViewParams * max(1, self.n_cams))()
        n = ctypes.c_int(0)
        _check(lib().hp3d_select_source_views(self.cams, self.n_cams, self.pts, self.n_pts,
                                              int(num_sources), out, ctypes.byref(n)))
        res = []
        for i in range(n.value):
            v = out[i]
            res.append({"ref_image_id": v.ref_image_id,
                        "sources": [(v.src[s].image_id, v.src[s].score, v.src[s].baseline_deg)
                                    for s in range(v.num_src)],
                        "depth_min": v.depth_min, "depth_max": v.depth_max})
        return res

    def seed_points(self, ref_id, depth_min, depth_max, width, height, seed_radius=50):
        """SfM seeds of camera ref_id: ctypes array of SeedPoint (and its length)."""
        out = (SeedPoint * max(1, self.n_pts))()
        n = ctypes.c_int(0)
        _check(lib().hp3d_project_seed_points(ctypes.byref(self.cams[ref_id]), self.pts,
                                              self.n_pts, float(depth_min), float(depth_max),
                                              int(width), int(height), int(seed_radius), out,
                                              ctypes.byref(n)))
        return out, n.value


def make_desc(ref, srcs, K_ref_inv, A, b, depth_min, depth_max, radius=5, stride=1,
              iterations=0, top_k=3, seed=42, init=None, seeds=None, seed_radius=50,
              first_iteration=0):
    """Build a ViewDesc.  ref/srcs are image handles; A, b lists of FP64 terms.

    init: optional (depth (H,W), normal (H,W,3)) float32 host arrays replacing
    the random initialisation; the arrays are kept alive on the descriptor.
    """
    d = ViewDesc()
    d.ref = ref
    for i, s in enumerate(srcs):
        d.src[i] = s
    d.num_src = len(srcs)
    Ki = np.asarray(K_ref_inv, dtype=np.float64).reshape(9)
    for i in range(9):
        d.K_ref_inv[i] = Ki[i]
    for s in range(len(srcs)):
        a = np.asarray(A[s], dtype=np.float64).reshape(9)
        bb = np.asarray(b[s], dtype=np.float64).reshape(3)
        for i in range(9):
            d.A[s][i] = a[i]
        for i in range(3):
            d.b[s][i] = bb[i]
    d.depth_min, d.depth_max = float(depth_min), float(depth_max)
    d.radius, d.stride, d.iterations, d.top_k = int(radius), int(stride), int(iterations), int(top_k)
    d.seed = int(seed)
    d.first_iteration = int(first_iteration)
    if init is not None:
        idp = np.ascontiguousarray(init[0], dtype=np.float32)
        inn = np.ascontiguousarray(init[1], dtype=np.float32)
        d._keep = (idp, inn)
        d.init_depth = _p(idp, _f32p)
        d.init_normal = _p(inn, _f32p)
    if seeds is not None:
        arr, n = seeds
        d._keep_seeds = arr
        d.seeds = ctypes.cast(arr, ctypes.POINTER(SeedPoint))
        d.num_seeds = int(n)
        d.seed_radius = int(seed_radius)
    return d


# ---------------------------------------------------------------------------
# Serving form
# ---------------------------------------------------------------------------
class Server:
    """Continuous-batching request loop (hp3d_server_*): submit jobs at any time."""

    def __init__(self, hbm_budget, max_jobs=32, radius=5, stride=1, store=STORE_F16, device=0,
                 variant=-1):
        o = ServerOpts(device, int(hbm_budget), max_jobs, radius, stride, store, variant)
        h = ctypes.c_void_p()
        code = lib().hp3d_server_create(ctypes.byref(o), ctypes.byref(h))
        if code != OK:
            raise HP3DError(code, "hp3d_server_create failed")
        self.h = h
        self._jobs = {}

    def close(self):
        if self.h:
            lib().hp3d_server_destroy(self.h)
            self.h = None

    def __enter__(self):
        return self

    def __exit__(self, *exc):
        self.close()

    def image_add(self, image, levels=1):
        """Keep an (H, W) uint8 image resident (with `levels` pyramid levels);
        returns its handle for submit(ref=handle, srcs=[handles])."""
        a = np.ascontiguousarray(image, dtype=np.uint8)
        H, W = a.shape
        h = ctypes.c_uint64(0)
        code = lib().hp3d_server_image_add(self.h, _p(a, _u8p), W, H, W, int(levels),
                                           ctypes.byref(h))
        if code != OK:
            raise HP3DError(code, lib().hp3d_server_last_error(self.h).decode())
        return h.value

    def image_remove(self, handle):
        _check(lib().hp3d_server_image_remove(self.h, handle))

    def image_read(self, handle, level=0):
        """A resident image's pyramid level as DN values, (H_l, W_l) float32."""
        W, H = ctypes.c_int(), ctypes.c_int()
        _check(lib().hp3d_server_image_read(self.h, handle, level, ctypes.byref(W),
                                            ctypes.byref(H), None, 0))
        out = np.zeros((H.value, W.value), np.float32)
        _check(lib().hp3d_server_image_read(self.h, handle, level, ctypes.byref(W),
                                            ctypes.byref(H), _p(out, _f32p), out.size))
        return out

    def submit(self, ref, srcs, K_ref_inv, A, b, depth_min, depth_max, iterations, seed=42,
               top_k=3, with_normal=False, with_cost=True, fail_at_step=0, level=0, shape=None):
        """Queue one job; returns its id.  Output arrays are filled on completion.
        ref and each source: an (H, W) uint8 image, or the handle of a resident
        image (then shape = (H, W) at `level`)."""
        keep = []
        d = JobDesc()
        d.num_src = len(srcs)
        d.level = int(level)
        H = W = None
        for k, im in enumerate([ref] + list(srcs)):
            if isinstance(im, (int, np.integer)):
                if k == 0:
                    d.ref_image = int(im)
                else:
                    d.src_image[k - 1] = int(im)
                continue
            a = np.ascontiguousarray(im, dtype=np.uint8)
            keep.append(a)
            H, W = a.shape
            if k == 0:
                d.ref = _p(a, _u8p)
            else:
                d.src[k - 1] = _p(a, _u8p)
        if shape is not None:
            H, W = shape
        if H is None:
            raise ValueError("shape is needed when every image is resident")
        d.width, d.height = W, H
        for i, val in enumerate(np.asarray(K_ref_inv, dtype=np.float64).reshape(9)):
            d.K_ref_inv[i] = val
        for s in range(len(srcs)):
            for i, val in enumerate(np.asarray(A[s], dtype=np.float64).reshape(9)):
                d.A[s][i] = val
            for i, val in enumerate(np.asarray(b[s], dtype=np.float64).reshape(3)):
                d.b[s][i] = val
        d.depth_min, d.depth_max = float(depth_min), float(depth_max)
        d.iterations, d.top_k, d.seed = int(iterations), int(top_k), int(seed)
        out = {"depth": np.zeros((H, W), np.float32),
               "normal": np.zeros((H, W, 3), np.float32) if with_normal else None,
               "cost": np.zeros((H, W), np.float32) if with_cost else None}
        d.out_depth = _p(out["depth"], _f32p)
        d.out_normal = _p(out["normal"], _f32p) if with_normal else None
        d.out_cost = _p(out["cost"], _f32p) if with_cost else None
        d.fail_at_step = int(fail_at_step)
        jid = ctypes.c_uint64(0)
        code = lib().hp3d_server_submit(self.h, ctypes.byref(d), ctypes.byref(jid))
        if code != OK:
            raise HP3DError(code, lib().hp3d_server_last_error(self.h).decode())
        self._jobs[jid.value] = out
        return jid.value

    def submit_job(self, job, **kw):
        return self.submit(job.ref, job.srcs, job.Kinv, job.A, job.b, job.dmin, job.dmax,
                           kw.pop("iterations", job.iterations), seed=kw.pop("seed", job.seed),
                           top_k=job.top_k, **kw)

    @staticmethod
    def _status(st):
        return {f: getattr(st, f) for f, _ in JobStatus._fields_}

    def poll(self, jid):
        st = JobStatus()
        _check(lib().hp3d_server_poll(self.h, jid, ctypes.byref(st)))
        return self._status(st)

    def wait(self, jid, timeout=-1.0):
        st = JobStatus()
        code = lib().hp3d_server_wait(self.h, jid, float(timeout), ctypes.byref(st))
        if code == ERR_AGAIN:
            return None
        _check(code)
        return self._status(st)

    def result(self, jid):
        return self._jobs[jid]

    def forget(self, jid):
        """Drop a finished job (its record in the server and its output
        arrays here); HP3DError(ERR_AGAIN) while it is queued or running."""
        _check(lib().hp3d_server_forget(self.h, jid))
        self._jobs.pop(jid, None)

    def cancel(self, jid):
        _check(lib().hp3d_server_cancel(self.h, jid))

    def stats(self):
        s = ServerStats()
        _check(lib().hp3d_server_get_stats(self.h, ctypes.byref(s)))
        return {f: getattr(s, f) for f, _ in ServerStats._fields_}

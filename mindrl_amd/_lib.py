"""ctypes binding of libmrb.so (C ABI declared in include/mrb.h).

There is no fallback: if the library has not been built, or a call fails, an
exception is raised. Build with `python -m mindrl_amd.build`.
"""
import ctypes as C
import os

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(_HERE, "csrc", "libmrb.so")

MRB_OK, MRB_EINVAL, MRB_EHANDLE, MRB_EHIP, MRB_ESTATE, MRB_EDEVICE = 0, 1, 2, 3, 4, 5
DERR_INDEX, DERR_PRIORITY, DERR_TOTAL, DERR_UNFILLED, DERR_OVERLAP = 1, 2, 4, 8, 16
MAX_FIELDS = 16
ABI_VERSION = 4  # MRB_ABI_VERSION of include/mrb.h this binding was written against

_vp, _i64, _u64, _f32, _int = C.c_void_p, C.c_int64, C.c_uint64, C.c_float, C.c_int
_pvp = C.POINTER(C.c_void_p)
_pi64 = C.POINTER(C.c_int64)

# name -> argtypes; every function returns int except mrb_last_error
SIGNATURES = {
    "mrb_backend": [],
    "mrb_version": [],
    "mrb_set_option": [_i64, C.c_char_p, _i64],
    "mrb_field_layout": [_i64, _int, _pvp, _pi64],
    "mrb_urb_create": [_i64, _int, _pi64, _pi64],
    "mrb_urb_append": [_i64, _pvp, _i64, _vp],
    "mrb_urb_append_from": [_i64, _i64, _i64, _i64, _vp],
    "mrb_urb_get_item": [_i64, _i64, _pvp, _vp],
    "mrb_urb_gather": [_i64, _vp, _i64, _pvp, _vp],
    "mrb_urb_sample": [_i64, _i64, _vp, _pvp, _vp],
    "mrb_urb_seed": [_i64, _u64],
    "mrb_urb_state": [_i64, C.POINTER(C.c_int32), C.POINTER(C.c_int32)],
    "mrb_urb_reset": [_i64],
    "mrb_urb_check": [_i64, C.POINTER(C.c_uint32), _vp],
    "mrb_urb_field_ptr": [_i64, _int, _pvp],
    "mrb_urb_destroy": [_i64],
    "mrb_per_create": [_i64, _f32, _int, _pi64, _u64, _pi64],
    "mrb_per_push": [_i64, _pvp, _i64, _vp, _vp],
    "mrb_per_sample": [_i64, _i64, _f32, _vp, _vp, _vp, _pvp, _vp],
    "mrb_per_sample_many": [_i64, _i64, _i64, _f32, _vp, _vp, _vp, _pvp, _vp],
    "mrb_per_sample_next": [_i64, _i64, _f32, _vp, _int, _int, _vp, _vp, _pvp, _vp, _vp],
    "mrb_per_gather": [_i64, _vp, _i64, _pvp, _vp],
    "mrb_per_update": [_i64, _vp, _vp, _i64, _vp],
    "mrb_per_update_push": [_i64, _vp, _vp, _i64, _pvp, _i64, _vp, _vp],
    "mrb_per_update_push_sample": [_i64, _vp, _vp, _i64, _pvp, _i64, _vp, _i64, _f32, _vp, _vp, _vp, _pvp, _vp],
    "mrb_per_update_noalloc": [_i64, _vp, _vp, _i64, _vp],
    "mrb_per_export_tree": [_i64, _vp, _vp, _pi64, _vp],
    "mrb_per_state": [_i64, _pi64, _pi64, C.POINTER(C.c_float), _vp],
    "mrb_per_check": [_i64, C.POINTER(C.c_uint32), _vp],
    "mrb_per_field_ptr": [_i64, _int, _pvp],
    "mrb_per_destroy": [_i64],
    "mrb_res_create": [_i64, _int, _pi64, _u64, _pi64],
    "mrb_res_push": [_i64, _pvp, _i64, _vp],
    "mrb_res_sample": [_i64, _i64, _vp, _pvp, _vp],
    "mrb_res_state": [_i64, _pi64, _pi64],
    "mrb_res_field_ptr": [_i64, _int, _pvp],
    "mrb_res_destroy": [_i64],
    "mrb_urb_get_counters": [_i64, _pi64],
    "mrb_urb_set_counters": [_i64, _pi64],
    "mrb_per_get_counters": [_i64, _pi64],
    "mrb_per_set_counters": [_i64, _pi64],
    "mrb_res_get_counters": [_i64, _pi64],
    "mrb_res_set_counters": [_i64, _pi64],
    "mrb_per_load_leaves": [_i64, _vp, _i64, _f32, _vp],
    "mrb_bench_launch": [_int, _vp, _vp, _i64, _vp],
    "mrb_discounted_return": [_vp, _vp, _vp, _vp, _i64, _i64, _i64, _f32, _vp],
}

# the same for include/mrb_more.h
MORE_SIGNATURES = {
    "mrb_discounted_return_grad": [_vp, _vp, _vp, _vp, _i64, _i64, _i64, _f32, _vp],
    "mrb_stage": [_i64, _i64, _pvp, _vp],
    "mrb_host_settled": [_pvp, _int, _vp],
}

_lib = None
_native = None


class MrbError(RuntimeError):
    """A libmrb call returned a non-zero status."""

    def __init__(self, code, message):
        super().__init__("libmrb error %d: %s" % (code, message))
        self.code = code


def lib():
    """Loads libmrb.so once. Raises if it has not been built."""
    global _lib
    if _lib is not None:
        return _lib
    if not os.path.exists(LIB_PATH):
        raise RuntimeError(
            "libmrb.so is missing (%s): build the HIP library with `python -m mindrl_amd.build`; "
            "there is no CPU fallback" % LIB_PATH)
    L = C.CDLL(LIB_PATH)
    L.mrb_last_error.restype = C.c_char_p
    L.mrb_last_error.argtypes = []
    for name, args in list(SIGNATURES.items()) + list(MORE_SIGNATURES.items()):
        fn = getattr(L, name)
        fn.restype = C.c_int
        fn.argtypes = args
    if L.mrb_version() != ABI_VERSION:
        raise RuntimeError("libmrb.so reports ABI version %d, this binding expects %d: rebuild the library with "
                           "`python -m mindrl_amd.build`" % (L.mrb_version(), ABI_VERSION))
    _lib = L
    return L


def native():
    """The extension module mindrl_amd._native (the host side of the buffer classes' calls; csrc/native.cpp), loaded
    once. Raises if it has not been built."""
    global _native
    if _native is None:
        lib()  # the C ABI it calls
        try:
            from . import _native as module
        except ImportError as e:
            raise RuntimeError("the extension mindrl_amd._native does not load (%s): build it with `python -m "
                               "mindrl_amd.build`" % e)
        _native = module
    return _native


def check(rc):
    """Maps a status code to the exception the reference's runtime would raise."""
    if rc == MRB_OK:
        return
    msg = lib().mrb_last_error().decode("utf-8", "replace")
    if rc in (MRB_EINVAL, MRB_EHANDLE, MRB_ESTATE):
        raise ValueError("libmrb: " + msg)
    raise MrbError(rc, msg)


def set_option(handle, name, value):
    """Sets a launch option of one buffer (see mrb_set_option in include/mrb.h)."""
    check(lib().mrb_set_option(int(handle), name.encode(), int(value)))


_PTR_ARRAYS = {}


def ptr_array(pointers):
    n = len(pointers)
    kind = _PTR_ARRAYS.get(n)
    if kind is None:
        kind = _PTR_ARRAYS[n] = C.c_void_p * n
    return kind(*pointers)

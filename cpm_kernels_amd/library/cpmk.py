"""Binding of libcpmk_hip.so (include/cpmk.h): the launchers through native/call.cpp where it is built, all else through ctypes.

Replaces cpm_kernels/library/{cuda,cudart,cublaslt}.py of the reference: instead of a CUDA
driver launch (library/cuda.py:249-267) or a cuBLASLt call (library/cublaslt.py:113-150)
per kernel, every kernel has one ``extern "C"`` launcher.  A non-zero status raises
``RuntimeError`` like the reference's check*Status helpers (library/cudart.py:325-327).
"""
import ctypes
from .base import Lib, load_native

lib = Lib("cpmk_hip")

# the launchers (all return an int status), without their prefix, with their parameters: i int32_t or int, l int64_t, f float,
# p pointer
_LAUNCHERS = {
    "gemm_calc_scale": "iiippp", "gemm_calc_scale_transpose": "iiippp", "gemm_round": "iiipppp",
    "gemm_round_transpose": "iiipppp", "gemm_scale": "iiippppiip", "gemm_scale_x": "iiipppp",
    "gemm_scale_y": "iiipppp", "gemm_int8": "iiiiiiipppp", "gemm_int8_scale": "iiiiiiippppiipp",
    "gemm_quantize": "iiipppip", "gemm_quantize_pair": "lppplpppip", "gemm_quantize_cols": "iiipppip",
    "gemm_fp16": "iiiiiiipppp", "gemm_quantize_cols_ld": "iiippippipip", "gemm_quantize_pair_ld": "lppplpppiip",
    "gemm_backward_round_scale_ld": "iiipppipip", "gemm_int8_scale_one": "iiiiiiippppiipp",
    "transpose_i8_ld": "iiipipip", "gemm_int8_scale_sum": "iiiiippppp", "gemm_fp16_sum": "iiiiipppp",
    "gemm_int8_scale_parts": "iiiiippppp", "gemm_fp16_parts": "iiiiiipppp", "gemm_add_parts": "ilppp",
    "gemm_quantize_cols_rows": "iiipppipilpppp", "gemm_backward_quantize_both": "iiippippipipipp", "gemm_int8_scale_split": "iiiiiiippppiipipp", "gemm_fp16_split": "iiiiiiipppipp",
    "gemv_fp16": "iiipppp", "gemv_fp16_transpose": "iiipppp", "gemv_broadcast_mat_fp16": "iiipppp",
    "embedding_forward": "iiipppp", "embedding_step": "iipppp", "copy_data_to_kv": "iiippip",
    "gemv_calc_scale": "iippp", "gemv_round": "iipppp", "gemv_broadcast_mat_int8": "iiipppppp",
    "layernorm_forward": "iiippfip", "layernorm_forward_noalloc": "iiippfip", "layernorm_step": "iippfip",
    "layernorm_affine_forward": "iiippppfip", "layernorm_affine_forward_stats": "iiipppppfip",
    "layernorm_affine_backward": "iiippppppppp", "softmax_forward": "iiippp", "softmax_step_inplace": "iipp",
    "gelu_forward": "iippp", "position_embedding_init": "iipip", "position_embedding_forward": "iiiiipppip",
    "position_embedding_step": "iiiiipppip", "arith_ln_mul_add": "iiippppp", "arith_ln_mul": "iiipppp",
    "arith_element_add": "iipppp", "mask": "iiippfpp", "arith_global_scale": "lpfpp", "arith_element_mul": "iipppp",
    "arith_batch_add_forward": "iipppp", "arith_batch_add_backward": "ilppp", "arith_ln_add": "iiipppp",
    "arith_ln_div": "iiipppp", "arith_ln_sub_div": "iiippppp", "arith_ln_mul_backward": "iiipppp",
    "arith_ln_add_backward": "iiippp", "arith_batch_mul_add": "iippppp", "arith_batch_mul": "iipppp",
    "gelu_backward": "iipppp", "softmax_backward": "iiipppp", "layernorm_forward_v": "iiipppfp",
    "layernorm_forward_mv": "iiippppfp", "layernorm_backward_v": "iiippppp", "layernorm_backward_mv": "iiipppppp",
    "gemm_backward_round_scale": "iiippppip", "gemm_backward_scale_round": "iiippppip",
    "position_embedding_backward": "iiiiipppip", "embedding_backward_stage1": "iiippppppp",
    "embedding_backward_stage2": "iipppp", "embedding_order_ids": "ipppp", "embedding_backward_rows": "iipppppp", "embedding_backward_prepare": "iiiippppppp",
    "transpose": "iiippp", "transpose_i8": "iiippp", "array_add": "piip", "adjustify_logits": "iipfffpp",
    "copy_extend_buffer": "iiippp", "has_nan_inf": "lppp", "copy_pos_hidden": "iiiippp", "async_status": "",
    "selftest_exchange_timeout": "ip",
}
_CTYPES = {"i": ctypes.c_int32, "l": ctypes.c_int64, "f": ctypes.c_float, "p": ctypes.c_void_p}

EXPORTED_SYMBOLS = sorted(["cpmk_" + n for n in _LAUNCHERS] + [
    "cpmk_version", "cpmk_error_string", "cpmk_device_count", "cpmk_get_device",
    "cpmk_set_device", "cpmk_device_props", "cpmk_exchange_capture_slots_left", "cpmk_gemm_sum_groups", "cpmk_gemm_sum_groups_for", "cpmk_gemm_sum_krows_groups",
    "cpmk_gemm_sum_groups_timed",
    "cpmk_gemm_depth_parts", "cpmk_gemm_fp16_copy_pays",
])


@lib.bind("cpmk_error_string", [ctypes.c_int], ctypes.c_char_p)
def error_string(code: int) -> str:
    return lib.cpmk_error_string(code).decode()


@lib.bind("cpmk_version", [], ctypes.c_int)
def _version() -> int:
    return lib.cpmk_version()


def checkStatus(status: int) -> None:
    if status != 0:
        raise RuntimeError("HIP Error: %s" % error_string(status))


def _value(obj, size=None):
    """What an argument stands for that is no Python number: for a pointer its address (ctypes.c_void_p and what ctypes casts
    to it), else the value of a ctypes number of the parameter's own type (size 4 or 8: integers, 0: float)."""
    if size is None:
        return obj.value if isinstance(obj, ctypes.c_void_p) else ctypes.cast(obj, ctypes.c_void_p).value
    ctype = {0: ctypes.c_float, 4: ctypes.c_int32, 8: ctypes.c_int64}[size]
    if isinstance(obj, ctype):
        return obj.value
    raise TypeError("expected a number or a %s, got %s" % (ctype.__name__, type(obj).__name__))


# Beside the library there may be an extension module for this Python that calls the launchers at a third of ctypes' cost
# (native/call.cpp); without it (a library from elsewhere, another Python, a build without a C++ compiler) ctypes does it.
_native = load_native("_cpmk_call") if lib.loaded else None
_native_names = ()
if _native is not None:
    _native.init(lib.address("cpmk_error_string"), _value)
    _native_names = _native.names()


def _make(name, parameters):
    @lib.bind(name, [_CTYPES[c] for c in parameters], ctypes.c_int)
    def call(*args):
        checkStatus(getattr(lib, name)(*args))
    call.__name__ = name[len("cpmk_"):]
    call.__doc__ = "Launch %s (see include/cpmk.h)." % name
    if name in _native_names and hasattr(lib, name):
        return _native.bind(name, lib.address(name))
    return call


for _name, _parameters in _LAUNCHERS.items():
    globals()[_name] = _make("cpmk_" + _name, _parameters)


def check() -> None:
    """Raise ``RuntimeError`` if a kernel launched on the current device has failed while it ran (a
    team of workgroups whose partial results did not arrive in time: the outputs then hold NaN, or 0
    in int8 tensors), and clear the condition.  Blocks like a device-to-host copy, so it sees all work
    queued before it on the blocking streams; synchronise non-blocking streams first.  Until it is
    called, every other call into the library raises the same error (the reference raises pending
    failures from the status check of whichever call comes next, library/cudart.py:325-327)."""
    globals()["async_status"]()


@lib.bind("cpmk_exchange_capture_slots_left", [ctypes.POINTER(ctypes.c_int32)], ctypes.c_int)
def exchange_capture_slots_left() -> int:
    n = ctypes.c_int32(0)
    checkStatus(lib.cpmk_exchange_capture_slots_left(ctypes.byref(n)))
    return n.value


@lib.bind("cpmk_gemm_sum_groups", [ctypes.c_int32] * 3, ctypes.c_int32)
def gemm_sum_groups(m: int, n: int, batch: int) -> int:
    return lib.cpmk_gemm_sum_groups(m, n, batch)


@lib.bind("cpmk_gemm_sum_krows_groups", [ctypes.c_int32] * 4, ctypes.c_int32)
def gemm_sum_krows_groups(m: int, k: int, n: int, batch: int) -> int:
    return lib.cpmk_gemm_sum_krows_groups(m, k, n, batch)


@lib.bind("cpmk_gemm_sum_groups_for", [ctypes.c_int] + [ctypes.c_int32] * 4, ctypes.c_int32)
def gemm_sum_groups_for(kind: int, m: int, k: int, n: int, batch: int) -> int:
    return lib.cpmk_gemm_sum_groups_for(kind, m, k, n, batch)


@lib.bind("cpmk_gemm_sum_groups_timed", [ctypes.c_int] + [ctypes.c_int32] * 4, ctypes.c_int32)
def gemm_sum_groups_timed(kind: int, m: int, k: int, n: int, batch: int) -> int:
    return lib.cpmk_gemm_sum_groups_timed(kind, m, k, n, batch)


@lib.bind("cpmk_gemm_depth_parts", [ctypes.c_int] + [ctypes.c_int32] * 5 + [ctypes.c_int] * 2, ctypes.c_int32)
def gemm_depth_parts(f16: int, m: int, k: int, n: int, batchA: int, batchB: int, aT: int, bT: int) -> int:
    return lib.cpmk_gemm_depth_parts(f16, m, k, n, batchA, batchB, aT, bT)


@lib.bind("cpmk_gemm_fp16_copy_pays", [ctypes.c_int32] * 4 + [ctypes.c_int], ctypes.c_int)
def gemm_fp16_copy_pays(m: int, k: int, n: int, batch: int, bT: int) -> int:
    return lib.cpmk_gemm_fp16_copy_pays(m, k, n, batch, bT)


@lib.bind("cpmk_device_count", [ctypes.POINTER(ctypes.c_int)], ctypes.c_int)
def device_count() -> int:
    n = ctypes.c_int(0)
    checkStatus(lib.cpmk_device_count(ctypes.byref(n)))
    return n.value


@lib.bind("cpmk_get_device", [ctypes.POINTER(ctypes.c_int)], ctypes.c_int)
def get_device() -> int:
    d = ctypes.c_int(0)
    checkStatus(lib.cpmk_get_device(ctypes.byref(d)))
    return d.value


@lib.bind("cpmk_set_device", [ctypes.c_int], ctypes.c_int)
def set_device(device: int) -> None:
    checkStatus(lib.cpmk_set_device(device))


@lib.bind("cpmk_device_props", [ctypes.c_int, ctypes.c_char_p, ctypes.c_int] +
          [ctypes.POINTER(ctypes.c_int)] * 7 + [ctypes.POINTER(ctypes.c_uint64)], ctypes.c_int)
def device_props(device: int) -> dict:
    name = ctypes.create_string_buffer(64)
    ints = [ctypes.c_int(0) for _ in range(7)]
    mem = ctypes.c_uint64(0)
    checkStatus(lib.cpmk_device_props(device, name, 64, *[ctypes.byref(i) for i in ints],
                                      ctypes.byref(mem)))
    keys = ["compute_units", "lds_bytes", "wavefront", "clock_khz", "mem_clock_khz",
            "mem_bus_bits", "l2_bytes"]
    props = {k: v.value for k, v in zip(keys, ints)}
    props["name"] = name.value.decode()
    props["global_mem_bytes"] = mem.value
    return props


try:
    version = _version()
except RuntimeError:      # library not built / not loadable on this host
    version = 0

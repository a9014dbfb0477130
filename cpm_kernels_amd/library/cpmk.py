"""Binding of libcpmk_hip.so (include/cpmk.h): the launchers through native/call.cpp, the rest through ctypes.

Replaces cpm_kernels/library/{cuda,cudart,cublaslt}.py of the reference: instead of a CUDA
driver launch (library/cuda.py:249-267) or a cuBLASLt call (library/cublaslt.py:113-150)
per kernel, every kernel has one ``extern "C"`` launcher.  A non-zero status raises
``RuntimeError`` like the reference's check*Status helpers (library/cudart.py:325-327).
"""
import ctypes
from .base import Lib, load_native

lib = Lib("cpmk_hip")

# the launchers (all return an int status), without their prefix; native/call.cpp takes their argument types from include/cpmk.h
_LAUNCHERS = (
    "gemm_calc_scale", "gemm_calc_scale_transpose", "gemm_round", "gemm_round_transpose", "gemm_scale",
    "gemm_scale_x", "gemm_scale_y", "gemm_int8", "gemm_int8_scale", "gemm_quantize", "gemm_quantize_pair",
    "gemm_quantize_cols", "gemm_fp16", "gemm_quantize_cols_ld", "gemm_quantize_pair_ld",
    "gemm_backward_round_scale_ld", "gemm_int8_scale_one", "transpose_i8_ld", "gemm_int8_scale_sum", "gemm_fp16_sum",
    "gemm_int8_scale_parts", "gemm_fp16_parts", "gemm_add_parts",
    "gemv_fp16", "gemv_fp16_transpose", "gemv_broadcast_mat_fp16", "embedding_forward", "embedding_step",
    "copy_data_to_kv", "gemv_calc_scale", "gemv_round", "gemv_broadcast_mat_int8", "layernorm_forward",
    "layernorm_forward_noalloc", "layernorm_step", "layernorm_affine_forward", "layernorm_affine_forward_stats",
    "layernorm_affine_backward", "softmax_forward", "softmax_step_inplace", "gelu_forward", "position_embedding_init",
    "position_embedding_forward", "position_embedding_step", "arith_ln_mul_add", "arith_ln_mul", "arith_element_add",
    "mask", "arith_global_scale", "arith_element_mul", "arith_batch_add_forward", "arith_batch_add_backward",
    "arith_ln_add", "arith_ln_div", "arith_ln_sub_div", "arith_ln_mul_backward", "arith_ln_add_backward",
    "arith_batch_mul_add", "arith_batch_mul", "gelu_backward", "softmax_backward", "layernorm_forward_v",
    "layernorm_forward_mv", "layernorm_backward_v", "layernorm_backward_mv", "gemm_backward_round_scale",
    "gemm_backward_scale_round", "position_embedding_backward", "embedding_backward_stage1",
    "embedding_backward_stage2", "embedding_order_ids", "embedding_backward_rows", "transpose", "transpose_i8", "array_add",
    "adjustify_logits", "copy_extend_buffer", "has_nan_inf", "copy_pos_hidden", "async_status", "selftest_exchange_timeout",
)

EXPORTED_SYMBOLS = sorted(["cpmk_" + n for n in _LAUNCHERS] + [
    "cpmk_version", "cpmk_error_string", "cpmk_device_count", "cpmk_get_device",
    "cpmk_set_device", "cpmk_device_props", "cpmk_exchange_capture_slots_left", "cpmk_gemm_sum_groups", "cpmk_gemm_sum_groups_for",
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


_native = load_native("_cpmk_call") if lib.loaded else None
if _native is not None:
    _native.init(lib.address("cpmk_error_string"), _value)


def _make(name):
    address = lib.address(name)
    if address is not None and _native is not None:
        return _native.bind(name, address)

    def call(*args):
        if lib.loaded and _native is not None:
            raise AttributeError("%s: undefined symbol: %s" % (lib.path, name))
        raise RuntimeError("Library %s is not initialized" % ("_cpmk_call" if lib.loaded else "cpmk_hip"))
    call.__name__ = name[len("cpmk_"):]
    return call


for _name in _LAUNCHERS:
    globals()[_name] = _make("cpmk_" + _name)


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


@lib.bind("cpmk_gemm_sum_groups_for", [ctypes.c_int] + [ctypes.c_int32] * 4, ctypes.c_int32)
def gemm_sum_groups_for(kind: int, m: int, k: int, n: int, batch: int) -> int:
    return lib.cpmk_gemm_sum_groups_for(kind, m, k, n, batch)


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

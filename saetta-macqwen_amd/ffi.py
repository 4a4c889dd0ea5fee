"""ctypes binding of include/saetta_hip.h.  One function per exported symbol.

The calls that a program makes per chunk and per token go through an extension module instead (`calls`)."""
import ctypes
import importlib.machinery
import importlib.util
import os
import sysconfig

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.environ.get("SAETTA_HIP_LIB") or os.path.join(_HERE, "lib", "libsaetta_hip.so")
CALLS_PATH = os.path.join(_HERE, "lib", "_saetta_calls" + sysconfig.get_config_var("EXT_SUFFIX"))  # (of this Python)

# Every symbol include/saetta_hip.h declares; tests check the library exports each.
SYMBOLS = [
    "saetta_init", "saetta_last_error", "saetta_device_status", "saetta_token_params_set", "saetta_plan_begin",
    "saetta_plan_end", "saetta_plan_launches", "saetta_plan_run", "saetta_plan_free", "saetta_kv_quantize", "saetta_kv_dequantize", "saetta_kv_dequantize_f32", "saetta_to_half", "saetta_attn_prep_store", "saetta_deltanet_conv", "saetta_deltanet_step", "saetta_deltanet_conv_rows", "saetta_deltanet_rows", "saetta_deltanet_rows_ws", "saetta_deltanet_rows_workspace_bytes", "saetta_deltanet_token", "saetta_deltanet_rows_fused", "saetta_deltanet_fused_sync_bytes",
    "saetta_deltanet_token_sync", "saetta_deltanet_rows_fused_sync",
    "saetta_part_o_bytes", "saetta_part_ml_bytes", "saetta_attn_decode", "saetta_attn_decode_quant",
    "saetta_attn_rows", "saetta_attn_rows_quant", "saetta_static_scratch_bytes", "saetta_attn_decode_quant_static", "saetta_prefill_workspace_bytes", "saetta_attn_prefill", "saetta_attn_prefill_quant",
    "saetta_attn_gemm_workspace_bytes", "saetta_attn_gemm",
]

STAGE_PARTIAL, STAGE_REDUCE, STAGE_ALL, STAGE_NO_LOADERS = 1, 2, 3, 4


class TokenParamsC(ctypes.Structure):
    _fields_ = [("token", ctypes.c_uint32), ("position", ctypes.c_uint32), ("kv_len", ctypes.c_uint32),
                ("pad", ctypes.c_uint32)]


class KvQuantParamsC(ctypes.Structure):
    _fields_ = [("groups", ctypes.c_uint32), ("per_token", ctypes.c_uint32)]


class DecodeParamsC(ctypes.Structure):
    _fields_ = [("heads", ctypes.c_uint32), ("kv_heads", ctypes.c_uint32), ("capacity", ctypes.c_uint32),
                ("scale", ctypes.c_float)]


class RowsParamsC(ctypes.Structure):
    _fields_ = [("heads", ctypes.c_uint32), ("kv_heads", ctypes.c_uint32), ("capacity", ctypes.c_uint32),
                ("scale", ctypes.c_float), ("rows", ctypes.c_uint32), ("splits", ctypes.c_uint32)]


class FlashParamsC(ctypes.Structure):
    _fields_ = [("heads", ctypes.c_uint32), ("kv_heads", ctypes.c_uint32), ("pos", ctypes.c_uint32),
                ("tokens", ctypes.c_uint32), ("scale", ctypes.c_float)]


class QuantRowsC(ctypes.Structure):
    _fields_ = [("data", ctypes.c_void_p), ("scales", ctypes.c_void_p), ("biases", ctypes.c_void_p)]


class SaettaError(RuntimeError):
    """A non-zero return of the C ABI (the reference panics in these places)."""


class _Calls:
    """The extension module of csrc/calls.cpp, set up for this copy of the package: loaded when the package is imported if it
    can be, else when the first of its calls is made.  One that is built after the import does, and where there is none, or one
    that does not load, importing works and a call raises.  (It wants torch to be imported.)"""

    def _load(self):
        if not os.path.exists(CALLS_PATH):
            raise SaettaError(f"{CALLS_PATH} is missing: run __graft_entry__.build() (make -C csrc)")
        loader = importlib.machinery.ExtensionFileLoader("_saetta_calls", CALLS_PATH)
        try:
            module = importlib.util.module_from_spec(importlib.util.spec_from_file_location("_saetta_calls", CALLS_PATH, loader=loader))
            loader.exec_module(module)
        except ImportError as e:
            raise SaettaError(f"{CALLS_PATH} does not load (built for another Python or torch?): run __graft_entry__.build() (make -C csrc): {e}") from e
        module.setup(LIB_PATH, SaettaError, FlashParamsC)
        vars(self).update((k, v) for k, v in vars(module).items() if not k.startswith("__"))  # (found there from now on)

    def __getattr__(self, name):
        if name.startswith("__"):
            raise AttributeError(name)
        self._load()
        if name not in vars(self):
            raise AttributeError(name)
        return vars(self)[name]

    def ready(self):
        """Itself, loaded if it can be.  (At the import: loaded by the first call, with the GPU in use, it left everything that the
        program did in Python slower for good; recording 30 DeltaNet layers 240 -> 270 us.)"""
        try:
            self._load()
        except SaettaError:
            pass
        return self


calls = _Calls()

_lib = None


def lib():
    """Loads the library on first use; raises if it has not been built."""
    global _lib
    if _lib is None:
        if not os.path.exists(LIB_PATH):
            raise SaettaError(f"{LIB_PATH} is missing: run __graft_entry__.build() (make -C csrc)")
        l = ctypes.CDLL(LIB_PATH)
        vp, u32, i32, sz = ctypes.c_void_p, ctypes.c_uint32, ctypes.c_int, ctypes.c_size_t
        l.saetta_init.restype, l.saetta_init.argtypes = i32, []
        l.saetta_last_error.restype, l.saetta_last_error.argtypes = ctypes.c_char_p, []
        l.saetta_device_status.restype, l.saetta_device_status.argtypes = u32, [i32]
        l.saetta_token_params_set.restype = i32
        l.saetta_token_params_set.argtypes = [vp, vp, TokenParamsC]
        l.saetta_plan_begin.restype, l.saetta_plan_begin.argtypes = i32, []
        l.saetta_plan_end.restype, l.saetta_plan_end.argtypes = vp, []
        l.saetta_plan_launches.restype, l.saetta_plan_launches.argtypes = u32, [vp]
        l.saetta_plan_run.restype, l.saetta_plan_run.argtypes = i32, [vp, vp]
        l.saetta_plan_free.restype, l.saetta_plan_free.argtypes = None, [vp]
        l.saetta_kv_quantize.restype = i32
        l.saetta_kv_quantize.argtypes = [vp, i32, vp, QuantRowsC, KvQuantParamsC, vp, u32]
        l.saetta_kv_dequantize.restype = i32
        l.saetta_kv_dequantize.argtypes = [vp, i32, QuantRowsC, vp, KvQuantParamsC]
        l.saetta_kv_dequantize_f32.restype = i32
        l.saetta_kv_dequantize_f32.argtypes = [vp, i32, QuantRowsC, vp, KvQuantParamsC]
        l.saetta_to_half.restype, l.saetta_to_half.argtypes = i32, [vp, vp, vp, sz]
        l.saetta_deltanet_conv.restype = i32
        l.saetta_deltanet_conv.argtypes = [vp, vp, vp, vp, vp, ConvParamsC]
        l.saetta_deltanet_step.restype = i32
        l.saetta_deltanet_step.argtypes = [vp] * 12 + [StepParamsC]
        l.saetta_deltanet_token.restype = i32
        l.saetta_deltanet_token.argtypes = [vp] * 12 + [ConvParamsC, StepParamsC]
        l.saetta_deltanet_fused_sync_bytes.restype, l.saetta_deltanet_fused_sync_bytes.argtypes = sz, [u32]
        l.saetta_deltanet_token_sync.restype = i32
        l.saetta_deltanet_token_sync.argtypes = [vp] * 12 + [ConvParamsC, StepParamsC, vp]
        l.saetta_deltanet_rows_fused_sync.restype = i32
        l.saetta_deltanet_rows_fused_sync.argtypes = [vp] * 14 + [RowsFusedParamsC, vp]
        l.saetta_deltanet_rows_fused.restype = i32
        l.saetta_deltanet_rows_fused.argtypes = [vp] * 14 + [RowsFusedParamsC]
        l.saetta_deltanet_conv_rows.restype = i32
        l.saetta_deltanet_conv_rows.argtypes = [vp] * 6 + [ConvRowsParamsC]
        l.saetta_deltanet_rows.restype = i32
        l.saetta_deltanet_rows.argtypes = [vp] * 11 + [RowsStepParamsC]
        l.saetta_deltanet_rows_ws.restype = i32
        l.saetta_deltanet_rows_ws.argtypes = [vp] * 11 + [RowsStepParamsC, vp, ctypes.c_size_t]
        l.saetta_deltanet_rows_workspace_bytes.restype = ctypes.c_size_t
        l.saetta_deltanet_rows_workspace_bytes.argtypes = [RowsStepParamsC]
        l.saetta_attn_prep_store.restype = i32
        l.saetta_attn_prep_store.argtypes = [vp, i32, vp, vp, vp, vp, vp, vp, vp, vp, QuantRowsC, QuantRowsC, vp,
                                             PrepParamsC, u32, u32, vp]
        l.saetta_part_o_bytes.restype, l.saetta_part_o_bytes.argtypes = sz, [u32, u32, u32]
        l.saetta_part_ml_bytes.restype, l.saetta_part_ml_bytes.argtypes = sz, [u32, u32, u32]
        l.saetta_attn_decode.restype = i32
        l.saetta_attn_decode.argtypes = [vp, vp, vp, vp, vp, vp, vp, vp, DecodeParamsC, vp, u32]
        l.saetta_attn_decode_quant.restype = i32
        l.saetta_attn_decode_quant.argtypes = [vp, i32, vp, QuantRowsC, QuantRowsC, vp, vp, vp, vp,
                                               DecodeParamsC, vp, u32]
        l.saetta_static_scratch_bytes.restype, l.saetta_static_scratch_bytes.argtypes = sz, []
        l.saetta_attn_decode_quant_static.restype = i32
        l.saetta_attn_decode_quant_static.argtypes = [vp, i32, vp, QuantRowsC, QuantRowsC, vp, vp, DecodeParamsC, vp, u32]
        l.saetta_attn_rows.restype = i32
        l.saetta_attn_rows.argtypes = [vp, vp, vp, vp, vp, vp, vp, vp, RowsParamsC, vp, u32]
        l.saetta_attn_rows_quant.restype = i32
        l.saetta_attn_rows_quant.argtypes = [vp, i32, vp, QuantRowsC, QuantRowsC, vp, vp, vp, vp,
                                             RowsParamsC, vp, u32]
        l.saetta_attn_prefill.restype = i32
        l.saetta_attn_prefill.argtypes = [vp, vp, vp, vp, vp, vp, FlashParamsC, vp, ctypes.c_size_t]
        l.saetta_prefill_workspace_bytes.restype = ctypes.c_size_t
        l.saetta_prefill_workspace_bytes.argtypes = [ctypes.c_uint32, ctypes.c_uint32, ctypes.c_uint32]
        l.saetta_attn_prefill_quant.restype = i32
        l.saetta_attn_prefill_quant.argtypes = [vp, i32, vp, QuantRowsC, QuantRowsC, vp, vp, FlashParamsC, vp,
                                                ctypes.c_size_t]
        l.saetta_attn_gemm_workspace_bytes.restype = ctypes.c_size_t
        l.saetta_attn_gemm_workspace_bytes.argtypes = [ctypes.c_uint32] * 4
        l.saetta_attn_gemm.restype = i32
        l.saetta_attn_gemm.argtypes = [vp, i32, vp, QuantRowsC, QuantRowsC, vp, vp, FlashParamsC, u32, u32, vp,
                                       ctypes.c_size_t]
        _lib = l
    return _lib


class PrepParamsC(ctypes.Structure):
    _fields_ = [("heads", ctypes.c_uint32), ("kv_heads", ctypes.c_uint32), ("dim", ctypes.c_uint32),
                ("half_dims", ctypes.c_uint32), ("log2_theta", ctypes.c_float), ("eps", ctypes.c_float)]


class ConvParamsC(ctypes.Structure):
    _fields_ = [("channels", ctypes.c_uint32), ("kernel_size", ctypes.c_uint32)]


class StepParamsC(ctypes.Structure):
    _fields_ = [("k_heads", ctypes.c_uint32), ("v_heads", ctypes.c_uint32), ("v_dim", ctypes.c_uint32),
                ("eps", ctypes.c_float)]


class ConvRowsParamsC(ctypes.Structure):
    _fields_ = [("channels", ctypes.c_uint32), ("kernel_size", ctypes.c_uint32), ("tokens", ctypes.c_uint32),
                ("snapshots", ctypes.c_uint32)]


class RowsStepParamsC(ctypes.Structure):
    _fields_ = [("k_heads", ctypes.c_uint32), ("v_heads", ctypes.c_uint32), ("v_dim", ctypes.c_uint32),
                ("tokens", ctypes.c_uint32), ("eps", ctypes.c_float), ("snapshots", ctypes.c_uint32)]


class RowsFusedParamsC(ctypes.Structure):
    _fields_ = [("k_heads", ctypes.c_uint32), ("v_heads", ctypes.c_uint32), ("v_dim", ctypes.c_uint32),
                ("kernel_size", ctypes.c_uint32), ("eps", ctypes.c_float), ("rows", ctypes.c_uint32),
                ("snapshots", ctypes.c_uint32)]


def check(rc, what):
    if rc != 0:
        msg = lib().saetta_last_error().decode()
        raise SaettaError(f"{what}: {msg} (code {rc})")

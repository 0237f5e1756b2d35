"""Host-side mirror of the Lean entry points ``Tyr.GPU.GFX950.*`` for torch tensors.

Same names, argument meaning and error behaviour as the Lean declarations in
``tyr_amd/lean/Tyr/GPU/GFX950.lean`` (which bind ``lean_tyr_gpu_*`` in
``csrc/lean_shim.cpp``): outputs are freshly allocated and returned, every tensor argument
is checked the way the reference's generated launcher checks it
(Tyr/GPU/Codegen/Attribute.lean:334-336: device, contiguity, rank <= 4) and a failed
check or a negative status from the C ABI raises ``TyrGpuError`` -- the analogue of the
``IO.userError`` the Lean wrappers return.  torch is used for device memory and the
current stream only; all arithmetic happens in ``libtyr_hip.so``.
"""
from __future__ import annotations

import contextlib
import ctypes

import torch

from . import _lib


class TyrGpuError(RuntimeError):
    """Raised where the Lean wrapper would return ``IO.userError msg``."""


# Checks, allocation and the C ABI call of every entry point below are native code (csrc/torch_binding.cpp): in Python
# they took longer than most of the kernels they launch.
_n = _lib.load_binding(TyrGpuError)
_flash_attn_fwd, _flash_attn_bwd, _gqa_decode, _decode_rope_append = _n.flash_attn_fwd, _n.flash_attn_bwd, _n.gqa_decode, _n.decode_rope_append
_rope_fwd, _layernorm_residual, _copy, _matmul_bf16, _gemm_bf16 = _n.rope_fwd, _n.layernorm_residual, _n.copy, _n.matmul_bf16, _n.gemm_bf16
_gemm_fp8, _gemm_fp8_scaled, _mse_loss_grad, _sgd_step = _n.gemm_fp8, _n.gemm_fp8_scaled, _n.mse_loss_grad, _n.sgd_step


def library_path() -> str:
    return _lib.LIB_PATH


def _raise(rc: int, what: str) -> None:
    if rc != 0:
        msg = _lib.load().tyr_hip_strerror(rc).decode()
        raise TyrGpuError(f"{what}: {msg} (status {rc})")


@contextlib.contextmanager
def _launch_stream(stream):
    """Outputs and scratch come from torch's caching allocator, which ties a block to the stream that was
    current when it was allocated and may hand a freed block to the next allocation on that stream.  The kernels
    run on the caller's ``stream``; when that is not torch's current stream it is made current for the call, so the
    blocks belong to it and a scratch tensor dropped on return (its kernels still queued) can only be reused by
    work queued behind them.  ``stream`` may be a ``torch.cuda.Stream`` or a raw ``hipStream_t`` handle."""
    if not isinstance(stream, torch.cuda.Stream):
        stream = torch.cuda.ExternalStream(int(stream)) if int(stream) else torch.cuda.default_stream()
    with torch.cuda.stream(stream):
        yield


def _on_stream(stream, fn, *args):
    with _launch_stream(stream):
        return fn(*args)


def device_info(device: int = 0) -> dict:
    L = _lib.load()
    name = ctypes.create_string_buffer(64)
    cu, lds, clk = ctypes.c_int(), ctypes.c_int(), ctypes.c_int()
    hbm = ctypes.c_size_t()
    _raise(L.tyr_hip_device_info(device, name, 64, ctypes.byref(cu), ctypes.byref(lds), ctypes.byref(clk),
                                 ctypes.byref(hbm)), "device_info")
    return {"arch": name.value.decode(), "compute_units": cu.value, "lds_bytes_per_cu": lds.value,
            "clock_mhz": clk.value, "hbm_bytes": hbm.value}


def flash_attn_fwd(q, k, v, causal: bool = True, scale: float | None = None, window: int = 0, kv_lens=None,
                   key_mask=None, stream=None):
    """O, LSE = flashAttnFwd q k v causal scale.

    q bf16 [B,Hq,N,D]; k, v bf16 [B,Hkv,N,D] with Hq % Hkv == 0 (query head h reads kv head h / (Hq/Hkv));
    ``window`` > 0 (causal only) lets query i see keys (i - window, i]; ``kv_lens`` (int32 [B] on the device)
    masks the keys at or beyond each sequence's length; ``key_mask`` (bool / uint8 [B,N] on the device, nonzero =
    visible) hides any set of keys per sequence instead.  -> (bf16 [B,Hq,N,D], f32 [B,Hq,N])."""
    if stream is None:
        return _flash_attn_fwd(q, k, v, causal, scale, window, kv_lens, key_mask)
    return _on_stream(stream, _flash_attn_fwd, q, k, v, causal, scale, window, kv_lens, key_mask)


def flash_attn_bwd(q, k, v, o, lse, d_o, causal: bool = True, scale: float | None = None, window: int = 0,
                   kv_lens=None, key_mask=None, stream=None):
    """dQ, dK, dV = flashAttnBwd q k v o lse dO causal scale.

    q, o, d_o bf16 [B,Hq,N,D]; k, v bf16 [B,Hkv,N,D]; lse f32 [B,Hq,N]; o and lse as returned by
    flash_attn_fwd for the same q, k, v, causal, scale, window, kv_lens and key_mask.  Returns dQ [B,Hq,N,D] and
    dK, dV [B,Hkv,N,D] (summed over the query heads of each kv head), bf16."""
    if stream is None:
        return _flash_attn_bwd(q, k, v, o, lse, d_o, causal, scale, window, kv_lens, key_mask)
    return _on_stream(stream, _flash_attn_bwd, q, k, v, o, lse, d_o, causal, scale, window, kv_lens, key_mask)


def gqa_decode(q, k, v, scale: float | None = None, num_splits: int = 0, kv_len: int | None = None,
               kv_lens=None, window: int = 0, stream=None):
    """O, LSE = gqaDecode q k v scale numSplits.

    q bf16 [B,Hq,1,D]; k, v bf16 [B,Hkv,Lmax,D] (the preallocated cache); the first ``kv_len``
    rows (default all) of every (batch, kv head) are attended to.  ``kv_lens`` (int32 [B] on the device)
    gives every sequence its own length in [0, kv_len] (a length of 0 yields O = 0, LSE = -inf); ``window`` > 0 restricts each sequence to its last
    ``window`` rows.  -> (bf16 [B,Hq,1,D], f32 [B,Hq]).
    """
    if stream is None:
        return _gqa_decode(q, k, v, scale, num_splits, kv_len, kv_lens, window)
    return _on_stream(stream, _gqa_decode, q, k, v, scale, num_splits, kv_len, kv_lens, window)


def decode_rope_append(q, k_new, v_new, cos, sin, k_cache, v_cache, pos: int, stream=None):
    """qRot = decodeRopeAppend q kNew vNew cos sin kCache vCache pos.

    q bf16 [B,Hq,1,D] (or [B,1,Hq,D]); k_new, v_new bf16 [B,Hkv,1,D]; cos, sin f32 [1,D/2] (or [D/2]) for
    position ``pos``; caches bf16 [B,Hkv,maxLen,D], row ``pos`` of each is overwritten in place.  Returns the
    rotated q with q's shape."""
    if stream is None:
        return _decode_rope_append(q, k_new, v_new, cos, sin, k_cache, v_cache, pos)
    return _on_stream(stream, _decode_rope_append, q, k_new, v_new, cos, sin, k_cache, v_cache, pos)


def rope_fwd(x, cos, sin, stream=None):
    """y = applyRotaryEmb x cos sin.  x f32 or bf16 [B,S,H,D]; cos, sin f32 [S,D/2]."""
    if stream is None:
        return _rope_fwd(x, cos, sin)
    return _on_stream(stream, _rope_fwd, x, cos, sin)


def layernorm_residual(x, residual, weight, bias, eps: float = 1e-5, stream=None):
    """(out, outResid) = fusedLayerNormResidual x residual weight bias.  bf16; x, residual [..., d]; weight, bias [d]."""
    if stream is None:
        return _layernorm_residual(x, residual, weight, bias, eps)
    return _on_stream(stream, _layernorm_residual, x, residual, weight, bias, eps)


def copy(src, stream=None):
    """out = copy src (any dtype, contiguous)."""
    if stream is None:
        return _copy(src)
    return _on_stream(stream, _copy, src)


def matmul_bf16(a, b, trans_b: bool = False, stream=None):
    """C = matmul a b for operands of rank > 2 (`lean_torch_matmul`): a bf16 [..., M, K]; b bf16 [..., K, N] with
    the same leading extents, or a plain [K, N] matrix used for every batch entry (b is [..., N, K] / [N, K] with
    trans_b) -> bf16 [..., M, N]."""
    if stream is None:
        return _matmul_bf16(a, b, trans_b)
    return _on_stream(stream, _matmul_bf16, a, b, trans_b)


def gemm_bf16(a, b, trans_b: bool = False, stream=None):
    """C = gemmBf16 a b.  a bf16 [M,K]; b bf16 [K,N] (or [N,K] with trans_b) -> bf16 [M,N]."""
    if stream is None:
        return _gemm_bf16(a, b, trans_b)
    return _on_stream(stream, _gemm_bf16, a, b, trans_b)


def gemm_fp8(aq, bq, scale_a: float, scale_b: float, trans_b: bool = False, stream=None):
    """C = gemmFp8 aq bq scaleA scaleB.  aq e4m3 [M,K]; bq e4m3 [K,N] (or [N,K]) -> bf16 [M,N]."""
    if stream is None:
        return _gemm_fp8(aq, bq, scale_a, scale_b, trans_b)
    return _on_stream(stream, _gemm_fp8, aq, bq, scale_a, scale_b, trans_b)


def gemm_fp8_scaled(aq, bq, row_scale=None, col_scale=None, scale: float = 1.0, out_dtype=torch.float32,
                    trans_b: bool = False, stream=None):
    """C = gemmFp8Scaled aq bq rowScale colScale: out_dtype(scale * rowScale[m] * colScale[n] * (aq bq)[m, n]).

    The per-row / per-column dequantisation epilogue of `tkH100Fp8ScaledGemmFwd` (f32 out) and, with no scales and
    out_dtype = torch.float8_e4m3fn, the E4M3 epilogue of `tkH100Fp8E4M3GemmFwd`.  aq e4m3 [M,K]; bq e4m3 [K,N] (or
    [N,K] with trans_b); row_scale f32 [M], col_scale f32 [N] or None."""
    if stream is None:
        return _gemm_fp8_scaled(aq, bq, row_scale, col_scale, scale, out_dtype, trans_b)
    return _on_stream(stream, _gemm_fp8_scaled, aq, bq, row_scale, col_scale, scale, out_dtype, trans_b)


def mse_loss_grad(out, target, stream=None):
    """(loss, dO) = lossAndGradOut out target: loss = 0.5 mean((out - target)^2) as an f32 scalar tensor,
    dO = bf16((out - target) / numel).  out, target bf16, same shape, numel % 8 == 0."""
    if stream is None:
        return _mse_loss_grad(out, target)
    return _on_stream(stream, _mse_loss_grad, out, target)


def sgd_step(param, grad, lr: float, in_place: bool = False, stream=None):
    """(param', bf16 param') = sgdUpdate param grad lr: param' = param - f32(grad) * lr for an f32 master and a bf16
    gradient of the same shape, together with the bf16 cast the next step's kernels take.  ``in_place`` overwrites
    ``param`` instead of allocating."""
    if stream is None:
        return _sgd_step(param, grad, lr, in_place)
    return _on_stream(stream, _sgd_step, param, grad, lr, in_place)


def quantize_e4m3(x: torch.Tensor):
    """Per-tensor absmax quantisation used by the harness: s = absmax/448, xq = e4m3fn(x / s)."""
    s = float(x.abs().max()) / 448.0
    if s == 0.0:
        s = 1.0
    xq = (x.float() / s).clamp(-448.0, 448.0).to(torch.float8_e4m3fn)
    return xq, s

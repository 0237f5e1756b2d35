"""The work a program built on this framework spends its time in, as cases that can be timed and compared.

Six kinds, each one pass through the public entry points of ``tyr_amd``:

  attn_fwd   attention over a whole sequence (prefill, the forward of training)
  attn_bwd   its gradients, from what the forward left
  train      one attention train step: forward, loss and dO, backward, SGD on three f32 masters
  decode     one token: rotate q and k, append k and v to the cache, attend to the cache
  rows       the row-wise work between the products of a layer: residual + LayerNorm, rotary of q and k
  gemm       a projection, bf16 or e4m3, from one decoded token to a whole training batch

``mask`` of the attention kinds: "full", "causal", "lens" (causal, a batch padded to one length, lengths known),
"keys" (causal, the same batch padded on the left, given as a [B, N] key mask), "window" (causal, sliding window).
"""
from __future__ import annotations

import math

import torch

import tyr_amd

HEADS = ((4, 4), (8, 2), (16, 16), (16, 4), (32, 8), (32, 32))
MASKS = ("causal", "causal", "full", "lens", "keys", "window")


def listed():
    return [
        # a padded batch of prompts of ordinary, uneven length, grouped queries
        dict(name="prefill_padded", kind="attn_fwd", B=2, Hq=32, Hkv=8, N=1111, D=128, mask="lens", window=0),
        # the headline configuration: long sequences, full batch
        dict(name="attn_fwd_large", kind="attn_fwd", B=16, Hq=16, Hkv=16, N=4096, D=128, mask="causal", window=0),
        # fine-tuning on few ragged sequences: gradients with grouped queries
        dict(name="attn_bwd_grouped", kind="attn_bwd", B=1, Hq=32, Hkv=8, N=2000, D=128, mask="causal", window=0),
        # the train step of the reference's runner: one head, 128 tokens -- latency and launches
        dict(name="train_runner", kind="train", B=1, H=1, N=128, D=64, mask="full"),
        # the same step at the headline shape: forward, backward and 1.2 GB of element-wise work
        dict(name="train_large", kind="train", B=16, H=16, N=4096, D=128, mask="causal"),
        # interactive generation: one sequence, a short cache
        dict(name="decode_single", kind="decode", B=1, Hq=32, Hkv=8, L=1500, Lmax=2048, D=128, lens=False),
        # batched serving with a long cache (1 GiB of K and V)
        dict(name="decode_batch", kind="decode", B=32, Hq=32, Hkv=8, L=8192, Lmax=8192, D=128, lens=False),
        # row-wise work of one layer over a prompt batch
        dict(name="rows_prompt", kind="rows", B=2, S=1111, Hq=32, Hkv=8, D=128, d_model=4096),
        # projection of a batch of decoded tokens: the weights are what has to be read
        dict(name="gemm_bf16_decode", kind="gemm", dtype="bf16", batch=1, M=32, N=4096, K=4096, trans_b=True, out="bf16", scales="tensor"),
        # the square configuration
        dict(name="gemm_bf16_square", kind="gemm", dtype="bf16", batch=1, M=4096, N=4096, K=4096, trans_b=False, out="bf16", scales="tensor"),
        # a prompt chunk through a quantised projection with per-row and per-column scales
        dict(name="gemm_fp8_prompt", kind="gemm", dtype="fp8", batch=1, M=333, N=4096, K=4096, trans_b=True, out="bf16", scales="rowcol"),
        # the large quantised projection
        dict(name="gemm_fp8_large", kind="gemm", dtype="fp8", batch=1, M=8192, N=8192, K=8192, trans_b=False, out="bf16", scales="tensor"),
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("attn_fwd", "attn_bwd", "train", "decode", "rows", "gemm", "gemm"))
    while True:
        if kind in ("attn_fwd", "attn_bwd"):
            hq, hkv = rng.choice(HEADS)
            mask = rng.choice(MASKS)
            n = _log(rng, 64, 8192)
            c = dict(kind=kind, B=_log(rng, 1, 16), Hq=hq, Hkv=hkv, N=n, D=rng.choice((64, 128, 128)), mask=mask,
                     window=_log(rng, 64, max(64, n)) if mask == "window" else 0)
            if c["B"] * hq * n <= 1 << 20 and c["B"] * hq * n * n * (2 if mask == "full" else 1) <= 1 << 32:
                return c
        elif kind == "train":
            c = dict(kind=kind, B=_log(rng, 1, 16), H=rng.choice((1, 4, 8, 16)), N=_log(rng, 64, 4096), D=rng.choice((64, 128)),
                     mask=rng.choice(("causal", "full")))
            if c["B"] * c["H"] * c["N"] ** 2 * (2 if c["mask"] == "full" else 1) <= 1 << 31:
                return c
        elif kind == "decode":
            hq, hkv = rng.choice(HEADS)
            n = _log(rng, 64, 32768)
            c = dict(kind=kind, B=_log(rng, 1, 64), Hq=hq, Hkv=hkv, L=n, Lmax=n + rng.randrange(0, 1 + n // 2), D=rng.choice((64, 128, 128)),
                     lens=rng.random() < 0.5)
            if c["B"] * hkv * c["Lmax"] * c["D"] <= 32 * 8 * 8192 * 128:
                return c
        elif kind == "rows":
            hq, hkv = rng.choice(HEADS)
            d = rng.choice((64, 128, 128))
            c = dict(kind=kind, B=_log(rng, 1, 16), S=_log(rng, 1, 4096), Hq=hq, Hkv=hkv, D=d, d_model=min(8192, 8 * _log(rng, 64, 1024)))
            if c["B"] * c["S"] * (c["d_model"] + hq * d) <= 1 << 28:
                return c
        else:
            fp8 = rng.random() < 0.5
            step = 16 if fp8 else 8
            c = dict(kind=kind, dtype="fp8" if fp8 else "bf16", batch=1, M=_log(rng, 1, 8192), N=step * _log(rng, 256 // step, 8192 // step),
                     K=step * _log(rng, 256 // step, 8192 // step), trans_b=rng.random() < 0.5, out="bf16", scales="tensor")
            if fp8:
                c["scales"] = rng.choice(("tensor", "rowcol"))
                c["out"] = rng.choice(("bf16", "f32", "e4m3")) if c["scales"] == "rowcol" else "bf16"
            elif rng.random() < 0.25:
                c["batch"] = _log(rng, 2, 32)
            if c["batch"] * c["M"] * c["N"] * c["K"] <= 1 << (39 if fp8 else 38) and c["batch"] * c["M"] * max(c["N"], c["K"]) <= 1 << 26:
                return c


def _lengths(B, N):
    """Lengths of a padded batch: the longest fills it, the shortest half of it."""
    return [N - (i * (N // 2)) // max(1, B - 1) if B > 1 else N for i in range(B)]


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _normal(g, *shape, std=1.0, dtype=torch.bfloat16):
    x = torch.randn(*shape, generator=g, device="cuda")
    return (x * std if std != 1.0 else x).to(dtype)


def _rotary(S, D):
    ang = torch.outer(torch.arange(S, device="cuda", dtype=torch.float32),
                      10000.0 ** (-torch.arange(0, D, 2, device="cuda", dtype=torch.float32) / D))
    return torch.cos(ang).contiguous(), torch.sin(ang).contiguous()


def prepare(case, seed):
    g = _gen(seed)
    kind = case["kind"]
    st = dict(case=case)
    if kind in ("attn_fwd", "attn_bwd"):
        B, Hq, Hkv, N, D = (case[k] for k in ("B", "Hq", "Hkv", "N", "D"))
        st["q"] = _normal(g, B, Hq, N, D)
        st["k"], st["v"] = _normal(g, B, Hkv, N, D), _normal(g, B, Hkv, N, D)
        opt = dict(causal=case["mask"] != "full")
        # which sequence of the batch has which length follows the seed
        lens = torch.tensor(_lengths(B, N), dtype=torch.int32, device="cuda")[torch.randperm(B, generator=g, device="cuda")]
        if case["mask"] == "lens":
            opt["kv_lens"] = lens.contiguous()
        elif case["mask"] == "keys":
            opt["key_mask"] = (torch.arange(N, device="cuda")[None, :] >= N - lens[:, None]).contiguous()
        elif case["mask"] == "window":
            opt["window"] = case["window"]
        st["opt"] = opt
        if kind == "attn_bwd":
            st["o"], st["lse"] = tyr_amd.flash_attn_fwd(st["q"], st["k"], st["v"], **opt)
            st["d_o"] = _normal(g, B, Hq, N, D)
    elif kind == "train":
        shape = (case["B"], case["H"], case["N"], case["D"])
        clean = [_normal(g, *shape, dtype=torch.float32) for _ in range(3)]
        causal = case["mask"] == "causal"
        st["target"], _ = tyr_amd.flash_attn_fwd(*(t.to(torch.bfloat16) for t in clean), causal=causal)
        st["masters"] = [t + _normal(g, *shape, std=0.5, dtype=torch.float32) for t in clean]
        st["lows"] = [m.to(torch.bfloat16) for m in st["masters"]]
        st["causal"] = causal
    elif kind == "decode":
        B, Hq, Hkv, Lmax, D = (case[k] for k in ("B", "Hq", "Hkv", "Lmax", "D"))
        st["q"] = _normal(g, B, Hq, 1, D)
        st["kn"], st["vn"] = _normal(g, B, Hkv, 1, D), _normal(g, B, Hkv, 1, D)
        st["kc"], st["vc"] = _normal(g, B, Hkv, Lmax, D), _normal(g, B, Hkv, Lmax, D)
        cos, sin = _rotary(case["L"], D)
        st["cos"], st["sin"] = cos[-1:].contiguous(), sin[-1:].contiguous()
        st["lens"] = None
        if case["lens"]:
            st["lens"] = torch.tensor(_lengths(B, case["L"]), dtype=torch.int32, device="cuda")[
                torch.randperm(B, generator=g, device="cuda")].contiguous()
    elif kind == "rows":
        B, S, Hq, Hkv, D, d = (case[k] for k in ("B", "S", "Hq", "Hkv", "D", "d_model"))
        st["x"], st["res"] = _normal(g, B, S, d), _normal(g, B, S, d)
        st["w"], st["b"] = (1.0 + _normal(g, d, std=0.1, dtype=torch.float32)).to(torch.bfloat16), _normal(g, d, std=0.1)
        st["q"], st["k"] = _normal(g, B, S, Hq, D), _normal(g, B, S, Hkv, D)
        st["cos"], st["sin"] = _rotary(S, D)
    else:
        M, N, K, nb = (case[k] for k in ("M", "N", "K", "batch"))
        lead = (nb,) if nb > 1 else ()
        a = _normal(g, *lead, M, K)
        b = _normal(g, *lead, *((N, K) if case["trans_b"] else (K, N)), std=K ** -0.5)
        if case["dtype"] == "bf16":
            st["a"], st["b"] = a, b
        else:
            st["a"], st["sa"] = tyr_amd.quantize_e4m3(a)
            st["b"], st["sb"] = tyr_amd.quantize_e4m3(b)
            if case["scales"] == "rowcol":
                unit = 64.0 if case["out"] == "e4m3" else 1.0
                st["rs"] = (torch.rand(M, generator=g, device="cuda") + 0.5) * (st["sa"] * unit)
                st["cs"] = (torch.rand(N, generator=g, device="cuda") + 0.5) * st["sb"]
    return st


_OUT = {"bf16": torch.bfloat16, "f32": torch.float32, "e4m3": torch.float8_e4m3fn}


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "attn_fwd":
        return tyr_amd.flash_attn_fwd(st["q"], st["k"], st["v"], **st["opt"])
    if kind == "attn_bwd":
        return tyr_amd.flash_attn_bwd(st["q"], st["k"], st["v"], st["o"], st["lse"], st["d_o"], **st["opt"])
    if kind == "train":
        q, k, v = st["lows"]
        o, lse = tyr_amd.flash_attn_fwd(q, k, v, causal=st["causal"])
        loss, d_o = tyr_amd.mse_loss_grad(o, st["target"])
        grads = tyr_amd.flash_attn_bwd(q, k, v, o, lse, d_o, causal=st["causal"])
        return loss, grads, [tyr_amd.sgd_step(m, g, 200.0) for m, g in zip(st["masters"], grads)]
    if kind == "decode":
        qr = tyr_amd.decode_rope_append(st["q"], st["kn"], st["vn"], st["cos"], st["sin"], st["kc"], st["vc"], case["L"] - 1)
        o, lse = tyr_amd.gqa_decode(qr, st["kc"], st["vc"], kv_len=case["L"], kv_lens=st["lens"])
        return qr, o, lse, st["kc"], st["vc"]
    if kind == "rows":
        out, resid = tyr_amd.layernorm_residual(st["x"], st["res"], st["w"], st["b"])
        return out, resid, tyr_amd.rope_fwd(st["q"], st["cos"], st["sin"]), tyr_amd.rope_fwd(st["k"], st["cos"], st["sin"])
    if case["dtype"] == "bf16":
        if case["batch"] > 1:
            return tyr_amd.matmul_bf16(st["a"], st["b"], trans_b=case["trans_b"])
        return tyr_amd.gemm_bf16(st["a"], st["b"], trans_b=case["trans_b"])
    if case["scales"] == "tensor":
        return tyr_amd.gemm_fp8(st["a"], st["b"], st["sa"], st["sb"], trans_b=case["trans_b"])
    return tyr_amd.gemm_fp8_scaled(st["a"], st["b"], st["rs"], st["cs"], out_dtype=_OUT[case["out"]], trans_b=case["trans_b"])


def _pairs(case):
    """(query, key) pairs that see each other, over the whole batch, per head."""
    B, N, mask = case["B"], case["N"], case["mask"]
    if mask == "full":
        return B * N * N
    if mask == "window":
        w = min(case["window"], N)
        return B * (w * (w + 1) // 2 + (N - w) * w)
    if mask == "lens":
        return sum(n * (n + 1) // 2 + (N - n) * n for n in _lengths(B, N))
    if mask == "keys":
        return sum(n * (n + 1) // 2 for n in _lengths(B, N))
    return B * N * (N + 1) // 2


def work(case):
    kind = case["kind"]
    if kind in ("attn_fwd", "attn_bwd"):
        B, Hq, Hkv, N, D = (case[k] for k in ("B", "Hq", "Hkv", "N", "D"))
        q, kv, pairs = B * Hq * N, B * Hkv * N, _pairs(case) * Hq
        if kind == "attn_fwd":
            return {"bytes": 2 * D * (2 * q + 2 * kv) + 4 * q, "flops": 4 * D * pairs}
        return {"bytes": 2 * D * (4 * q + 4 * kv) + 4 * q, "flops": 10 * D * pairs}
    if kind == "train":
        n = case["B"] * case["H"] * case["N"] * case["D"]
        pairs = _pairs(case) * case["H"]
        # q, k, v, target and the masters in; gradients, new masters and their bf16 copies out
        return {"bytes": n * (4 * 2 + 3 * 4 + 3 * 2 + 3 * 4 + 3 * 2), "flops": 14 * case["D"] * pairs}
    if kind == "decode":
        B, Hq, Hkv, D = (case[k] for k in ("B", "Hq", "Hkv", "D"))
        rows = sum(_lengths(B, case["L"])) if case["lens"] else B * case["L"]
        return {"bytes": 2 * D * (2 * Hkv * rows + 3 * B * Hq + 4 * B * Hkv), "flops": 4 * D * Hq * rows}
    if kind == "rows":
        t = case["B"] * case["S"]
        heads = (case["Hq"] + case["Hkv"]) * case["D"]
        return {"bytes": 2 * t * (4 * case["d_model"] + 2 * heads) + 8 * case["S"] * case["D"], "flops": t * (10 * case["d_model"] + 3 * heads)}
    M, N, K, nb = (case[k] for k in ("M", "N", "K", "batch"))
    e_in = 2 if case["dtype"] == "bf16" else 1
    e_out = {"bf16": 2, "f32": 4, "e4m3": 1}[case["out"]]
    return {"bytes": nb * (e_in * (M * K + K * N) + e_out * M * N), "flops": 2 * nb * M * N * K}


def tolerance(case):
    if case["kind"] == "gemm":
        # f32 accumulation in another order, then one rounding: none to speak of, to bf16, or to 3 bits of mantissa
        # (bytes that sit on a rounding boundary may go either way)
        return {"f32": {"rel": 1e-4}, "bf16": {"rel": 5e-3}, "e4m3": {"rel": 1e-2, "max": 0.3}}[case["out"]]
    if case["kind"] == "rows":
        return {"rel": 5e-3}          # bf16 results of f32 row statistics
    return {"rel": 1e-2}              # bf16 probabilities and bf16 results

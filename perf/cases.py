"""The work that users of this framework have it do, as cases that can be timed and checked.

Layers and blocks of the supported models (SmolLM2, Qwen3, LLaMA-3.2 widths) through the C ABI of
include/ember_hip.h, as a foreign binding calls it, and through the C++ layer's trainer, as the
training and generation programs call it.  Everything is fp32.

A case is a dict of plain values; its "kind" says which path it takes:
  linear   one Linear over a batch of tokens, forward or backward
  mlp      RMSNorm -> SwiGLU MLP -> residual, forward and backward, all weight gradients
  attn     RMSNorm -> QKV -> (QK-Norm) RoPE -> causal GQA attention -> output projection ->
           residual, forward and backward, all weight gradients
  head     LM head + masked cross-entropy over the active rows, loss and both gradients
  optim    gradient-norm clip and AdamW over a model's parameter list
  block    Trainer.block_step: one checkpointed transformer block, host arrays in and out
  prefill  Trainer.forward of a prompt into a KV cache, last token's logits
  decode   Trainer.forward of one more token per sequence over a filled KV cache
"""
import ctypes as C
import math

import numpy as np
import torch
import torch.utils.checkpoint

from emberlm_amd import capi
from emberlm_amd import trainer as TR

F32 = torch.float32

# hidden, intermediate, heads, KV heads, head dim, QK-Norm, vocabulary, layers, RoPE theta, eps
WIDTHS = {
    "smollm2-135m": (576, 1536, 9, 3, 64, False, 49152, 30, 1e5, 1e-5),
    "smollm2-360m": (960, 2560, 15, 5, 64, False, 49152, 32, 1e5, 1e-5),
    "qwen3-0.6b": (1024, 3072, 16, 8, 128, True, 151936, 28, 1e6, 1e-6),
    "qwen3-1.7b": (2048, 6144, 16, 8, 128, True, 151936, 28, 1e6, 1e-6),
    "llama3.2-1b": (2048, 8192, 32, 8, 64, False, 128256, 16, 5e5, 1e-5),
}


def _mlp(tokens, hidden, inter):
    return {"kind": "mlp", "tokens": tokens, "hidden": hidden, "inter": inter}


def _attn(batch, seq, width):
    h, _, nh, nk, d, qk, _, _, theta, eps = WIDTHS[width]
    return {"kind": "attn", "batch": batch, "seq": seq, "hidden": h, "heads": nh, "kv_heads": nk,
            "head_dim": d, "qk_norm": qk, "theta": theta, "eps": eps}


def _head(tokens, hidden, vocab, active):
    return {"kind": "head", "tokens": tokens, "hidden": hidden, "vocab": vocab, "active": active}


def listed():
    return [
        # the smallest product of a fine-tuning step: one projection over one short sequence
        {"name": "linear_256x576x576", "kind": "linear", "tokens": 256, "n_in": 576, "n_out": 576,
         "backward": False},
        # the smallest whole block a program trains: B1 T256, checkpointed, from host arrays
        {"name": "block_smollm2_t256", "kind": "block", "width": "smollm2-135m", "batch": 1,
         "seq": 256, "checkpoint": True},
        # MLP of a small fine-tuning step: SmolLM2-135M at B4 T512
        dict(_mlp(2048, 576, 1536), name="mlp_smollm2_2048"),
        # MLP of an ordinary one: Qwen3-0.6B at B4 T1024
        dict(_mlp(4096, 1024, 3072), name="mlp_qwen3_0.6b_4096"),
        # MLP of the flagship step: Qwen3-1.7B at B8 T4096
        dict(_mlp(32768, 2048, 6144), name="mlp_qwen3_1.7b_32768"),
        # attention of one ragged document: LLaMA-3.2-1B widths at B1 T1000
        dict(_attn(1, 1000, "llama3.2-1b"), name="attn_llama_t1000"),
        # attention of the flagship step
        dict(_attn(8, 4096, "qwen3-1.7b"), name="attn_qwen3_1.7b_b8_t4096"),
        # LM head + loss of a small step, where about half the tokens are the prompt's
        dict(_head(2048, 576, 49152, 0.5), name="head_smollm2_2048_half"),
        # one chunk of the flagship step's LM head, most of its rows active
        dict(_head(1024, 2048, 151936, 0.95), name="head_qwen3_1.7b_1024"),
        # clip and update of a whole small model
        {"name": "optim_smollm2", "kind": "optim", "width": "smollm2-135m", "layers": 30},
        # prompt of a chat turn, batch 1
        {"name": "prefill_qwen3_0.6b_509", "kind": "prefill", "width": "qwen3-0.6b", "batch": 1,
         "seq": 509},
        # one token of batch-1 generation on the flagship model
        {"name": "decode_qwen3_1.7b_1024", "kind": "decode", "width": "qwen3-1.7b", "batch": 1,
         "seq": 1024},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "mlp", "attn", "head", "optim", "block", "prefill",
                       "decode"])
    if kind == "linear":
        width = rng.choice(sorted(WIDTHS))
        h, i, nh, nk, d = WIDTHS[width][:5]
        n_in, n_out = rng.choice([(h, nh * d), (h, nk * d), (nh * d, h), (h, i), (i, h)])
        return {"kind": kind, "tokens": _log(rng, 9, 16384), "n_in": n_in, "n_out": n_out,
                "backward": rng.random() < 0.5}
    if kind == "mlp":
        h, i = WIDTHS[rng.choice(sorted(WIDTHS))][:2]
        return _mlp(_log(rng, 64, 8192), h, i)
    if kind == "attn":
        seq = _log(rng, 32, 4096)
        return _attn(rng.randint(1, max(1, min(8, 8192 // seq))), seq, rng.choice(sorted(WIDTHS)))
    if kind == "head":
        w = WIDTHS[rng.choice(sorted(WIDTHS))]
        top = 4096 if w[6] < 100000 else 1024
        return _head(_log(rng, 33, top), w[0], w[6], rng.uniform(0.2, 1.0))
    if kind == "optim":
        width = rng.choice(["smollm2-135m", "smollm2-360m", "qwen3-0.6b"])
        return {"kind": kind, "width": width, "layers": rng.randint(1, 12)}
    if kind == "block":
        return {"kind": kind, "width": rng.choice(["smollm2-135m", "smollm2-360m", "qwen3-0.6b"]),
                "batch": rng.randint(1, 4), "seq": _log(rng, 16, 512),
                "checkpoint": rng.random() < 0.7}
    width = rng.choice(["smollm2-135m", "smollm2-360m", "qwen3-0.6b"])
    if kind == "prefill":
        return {"kind": kind, "width": width, "batch": rng.randint(1, 2), "seq": _log(rng, 16, 2048)}
    return {"kind": kind, "width": width, "batch": rng.randint(1, 8), "seq": _log(rng, 16, 1500)}


# ------------------------------------------------------------------ inputs


def _p(t):
    return C.c_void_p(t.data_ptr())


class _Calls:
    """Buffers a program holds and the calls it makes on them, in order."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda").manual_seed(int(seed))
        self.calls, self.keep = [], []

    def normal(self, *shape, std=1.0, mean=0.0):
        t = torch.randn(*shape, device="cuda", dtype=F32, generator=self.gen)
        return t.mul_(std).add_(mean)

    def empty(self, *shape, dtype=F32):
        t = torch.empty(*shape, device="cuda", dtype=dtype)
        self.keep.append(t)
        return t

    def scratch(self, nbytes):
        t = self.empty(max(1, (int(nbytes) + 3) // 4))
        return _p(t), int(nbytes)

    def add(self, name, *args):
        self.calls.append((name, tuple(_p(a) if isinstance(a, torch.Tensor) else a for a in args)))
        self.keep.extend(a for a in args if isinstance(a, torch.Tensor))

    def gemm(self, ta, tb, a, b, c, beta=0.0):
        """c = op(a) op(b) + beta c."""
        m, k = (a.shape[1], a.shape[0]) if ta else a.shape
        n = b.shape[0] if tb else b.shape[1]
        ws, wsb = self.scratch(capi.lib().ember_gemm_f32_workspace_bytes(m, n, k, 1))
        self.add("ember_gemm_f32_ws", int(ta), int(tb), m, n, k, 1.0, a, a.shape[1], 0, b,
                 b.shape[1], 0, beta, c, n, 0, 1, ws if wsb else None, wsb, None)

    def gemm_add(self, a, b, d, c):
        """c = a b^T + d."""
        (m, k), n = a.shape, b.shape[0]
        ws, wsb = self.scratch(capi.lib().ember_gemm_f32_workspace_bytes(m, n, k, 1))
        self.add("ember_gemm_f32_add", 0, 1, m, n, k, 1.0, a, k, b, k, d, n, c, n,
                 ws if wsb else None, wsb, None)

    def rms_bwd(self, dy, x, w, r, dx, dw, eps):
        rows, h = x.shape
        ws, wsb = self.scratch(capi.lib().ember_rmsnorm_bwd_workspace_bytes(rows, h))
        self.add("ember_rmsnorm_bwd", dy, x, w, r, dx, dw, rows, h, eps, ws, wsb, None)

    def run(self):
        for name, args in self.calls:
            capi.call(name, *args)


def _linear_inputs(c, k):
    x = k.normal(c["tokens"], c["n_in"])
    w = k.normal(c["n_out"], c["n_in"], std=0.02)
    dy = k.normal(c["tokens"], c["n_out"], std=1e-3)
    return x, w, dy


def _prepare_linear(c, seed):
    k = _Calls(seed)
    x, w, dy = _linear_inputs(c, k)
    if not c["backward"]:
        y = k.empty(c["tokens"], c["n_out"])
        k.gemm(False, True, x, w, y)
        return k, {"y": y}
    dx, dw = torch.empty_like(x), torch.empty_like(w)
    k.gemm(True, False, dy, x, dw)
    k.gemm(False, False, dy, w, dx)
    return k, {"dx": dx, "dw": dw}


def _mlp_inputs(c, k):
    n, h, i = c["tokens"], c["hidden"], c["inter"]
    return {"x": k.normal(n, h), "norm": k.normal(h, std=0.1, mean=1.0),
            "gate": k.normal(i, h, std=0.02), "up": k.normal(i, h, std=0.02),
            "down": k.normal(h, i, std=0.02), "dy": k.normal(n, h, std=1e-3)}


def _prepare_mlp(c, seed):
    k = _Calls(seed)
    n, h, i, eps = c["tokens"], c["hidden"], c["inter"], 1e-6
    t = _mlp_inputs(c, k)
    xn, r, g, u, a, y = (k.empty(n, h), k.empty(n), k.empty(n, i), k.empty(n, i), k.empty(n, i),
                         k.empty(n, h))
    da, dg, du, dxn, dx = (k.empty(n, i), k.empty(n, i), k.empty(n, i), k.empty(n, h),
                           k.empty(n, h))
    dn, dwg, dwu, dwd = k.empty(h), k.empty(i, h), k.empty(i, h), k.empty(h, i)
    k.add("ember_rmsnorm_fwd", t["x"], t["norm"], xn, r, n, h, eps, None)
    k.gemm(False, True, xn, t["gate"], g)
    k.gemm(False, True, xn, t["up"], u)
    k.add("ember_swiglu_fwd", g, u, a, n * i, None)
    k.gemm_add(a, t["down"], t["x"], y)
    k.gemm(True, False, t["dy"], a, dwd)
    k.gemm(False, False, t["dy"], t["down"], da)
    k.add("ember_swiglu_bwd", g, u, da, dg, du, n * i, None)
    k.gemm(True, False, dg, xn, dwg)
    k.gemm(True, False, du, xn, dwu)
    k.gemm(False, False, dg, t["gate"], dxn)
    k.gemm(False, False, du, t["up"], dxn, beta=1.0)
    k.rms_bwd(dxn, t["x"], t["norm"], r, dx, dn, eps)
    k.add("ember_accumulate", dx, t["dy"], n * h, None)
    return k, {"y": y, "dx": dx, "dnorm": dn, "dgate": dwg, "dup": dwu, "ddown": dwd}


def _attn_inputs(c, k):
    n, h, d = c["batch"] * c["seq"], c["hidden"], c["head_dim"]
    q, kv = c["heads"] * d, c["kv_heads"] * d
    t = {"x": k.normal(n, h), "norm": k.normal(h, std=0.1, mean=1.0),
         "wq": k.normal(q, h, std=0.02), "wk": k.normal(kv, h, std=0.02),
         "wv": k.normal(kv, h, std=0.02), "wo": k.normal(h, q, std=0.02),
         "dy": k.normal(n, h, std=1e-3)}
    if c["qk_norm"]:
        t["nq"], t["nk"] = k.normal(d, std=0.1, mean=1.0), k.normal(d, std=0.1, mean=1.0)
    return t


def _prepare_attn(c, seed):
    k = _Calls(seed)
    lib = capi.lib()
    B, T, h, H, Hk, D, eps = (c["batch"], c["seq"], c["hidden"], c["heads"], c["kv_heads"],
                              c["head_dim"], c["eps"])
    n, scale = B * T, 1.0 / math.sqrt(D)
    t = _attn_inputs(c, k)
    fr = (C.c_float * (D // 2))()
    capi.check(lib.ember_rope_freqs_host(fr, D, c["theta"], 0.0, 1.0, 4.0, 8192), "freqs")
    xn, r = k.empty(n, h), k.empty(n)
    q, kk, v, o = k.empty(n, H * D), k.empty(n, Hk * D), k.empty(n, Hk * D), k.empty(n, H * D)
    qr, kr, lse, y = k.empty(n, H * D), k.empty(n, Hk * D), k.empty(B * H * T), k.empty(n, h)
    rq, rk = k.empty(n * H), k.empty(n * Hk)
    k.add("ember_rmsnorm_fwd", t["x"], t["norm"], xn, r, n, h, eps, None)
    k.gemm(False, True, xn, t["wq"], q)
    k.gemm(False, True, xn, t["wk"], kk)
    k.gemm(False, True, xn, t["wv"], v)
    if c["qk_norm"]:
        k.add("ember_qknorm_rope_fwd", q, t["nq"], qr, rq, n * H, H, T, D, eps, 0, fr, None)
        k.add("ember_qknorm_rope_fwd", kk, t["nk"], kr, rk, n * Hk, Hk, T, D, eps, 0, fr, None)
    else:
        k.add("ember_rope", q, qr, B, T, H, D, 0, fr, 1.0, None)
        k.add("ember_rope", kk, kr, B, T, Hk, D, 0, fr, 1.0, None)
    k.add("ember_attn_fwd", qr, kr, v, o, lse, B, T, H, Hk, D, scale, None)
    k.gemm_add(o, t["wo"], t["x"], y)

    do, dqr, dkr, dv = k.empty(n, H * D), k.empty(n, H * D), k.empty(n, Hk * D), k.empty(n, Hk * D)
    dq, dk, dxn, dx = k.empty(n, H * D), k.empty(n, Hk * D), k.empty(n, h), k.empty(n, h)
    out = {"y": y, "dx": dx, "dnorm": k.empty(h)}
    for name, like in (("dwq", "wq"), ("dwk", "wk"), ("dwv", "wv"), ("dwo", "wo")):
        out[name] = torch.empty_like(t[like])
    k.gemm(True, False, t["dy"], o, out["dwo"])
    k.gemm(False, False, t["dy"], t["wo"], do)
    # dS for 32 KV rows at a time, as the C++ layer does under its own budget
    wsb = lib.ember_attn_bwd_workspace_bytes_min(B, T, H) + min(
        B * Hk, 32) * lib.ember_attn_bwd_ds_row_bytes(T, H, Hk)
    ws, wsb = k.scratch(wsb)
    k.add("ember_attn_bwd", qr, kr, v, o, lse, do, dqr, dkr, dv, B, T, H, Hk, D, scale, ws, wsb,
          None)
    if c["qk_norm"]:
        out["dnq"], out["dnk"] = k.empty(D), k.empty(D)
        for g, x, w, rs, dxx, dw, rows, heads in ((dqr, q, "nq", rq, dq, "dnq", n * H, H),
                                                  (dkr, kk, "nk", rk, dk, "dnk", n * Hk, Hk)):
            ws, wsb = k.scratch(lib.ember_rmsnorm_bwd_workspace_bytes(rows, D))
            k.add("ember_qknorm_rope_bwd", g, x, t[w], rs, dxx, out[dw], rows, heads, T, D, eps, 0,
                  fr, ws, wsb, None)
    else:
        k.add("ember_rope", dqr, dq, B, T, H, D, 0, fr, -1.0, None)
        k.add("ember_rope", dkr, dk, B, T, Hk, D, 0, fr, -1.0, None)
    k.gemm(True, False, dq, xn, out["dwq"])
    k.gemm(True, False, dk, xn, out["dwk"])
    k.gemm(True, False, dv, xn, out["dwv"])
    k.gemm(False, False, dq, t["wq"], dxn)
    k.gemm(False, False, dk, t["wk"], dxn, beta=1.0)
    k.gemm(False, False, dv, t["wv"], dxn, beta=1.0)
    k.rms_bwd(dxn, t["x"], t["norm"], r, dx, out["dnorm"], eps)
    k.add("ember_accumulate", dx, t["dy"], n * h, None)
    k.keep.append(fr)
    return k, out


def _head_inputs(c, k):
    n, h, v = c["tokens"], c["hidden"], c["vocab"]
    t = {"h": k.normal(n, h), "w": k.normal(v, h, std=0.02),
         "tgt": torch.randint(0, v, (n,), device="cuda", generator=k.gen)}
    # the prompts' tokens count for nothing; the rest is trained on
    pick = torch.rand(n, device="cuda", generator=k.gen) < c["active"]
    pick[0] = True
    t["mask"] = pick.to(F32)
    return t


def _prepare_head(c, seed):
    k = _Calls(seed)
    lib = capi.lib()
    n, h, v = c["tokens"], c["hidden"], c["vocab"]
    rows = (n + 15) // 16 * 16
    t = _head_inputs(c, k)
    idx, one = k.empty(n + 1, dtype=torch.int64), torch.ones(1, device="cuda")
    count = C.c_void_p(idx.data_ptr() + 8 * n)
    hc, logits, dhc = k.empty(rows, h), k.empty(rows, v), k.empty(rows, h)
    lse, row_loss, loss, msum = k.empty(n), k.empty(n), k.empty(1), k.empty(1)
    dh, dw = k.empty(n, h), k.empty(v, h)

    def dyn(ta, tb, m, nn, kk, a, b, out, dim):
        wsb = lib.ember_gemm_f32_workspace_bytes(m, nn, kk, 1) if dim == 0 else 0
        ws, wsb = k.scratch(wsb)
        k.add("ember_gemm_f32_dyn", int(ta), int(tb), m, nn, kk, 1.0, a, a.shape[1], b, b.shape[1],
              0.0, out, nn, count, 0, dim, ws if wsb else None, wsb, None)

    k.add("ember_mask_rows", t["mask"], n, idx, count, None)
    k.add("ember_fill", row_loss, n, 0.0, None)
    k.add("ember_fill", dh, n * h, 0.0, None)
    k.add("ember_rows_gather", t["h"], h, h, idx, count, 0, rows, hc, None)
    dyn(False, True, rows, v, h, hc, t["w"], logits, 0)
    k.add("ember_ce_masked_rows_idx", logits, t["tgt"], t["mask"], idx, count, 0, n, v, lse,
          row_loss, None)
    k.add("ember_ce_masked_reduce", row_loss, t["mask"], n, loss, msum, None)
    k.add("ember_ce_masked_bwd_idx", logits, t["tgt"], t["mask"], lse, idx, count, 0, n, v, one,
          msum, logits, None)
    dyn(False, False, n, h, v, logits, t["w"], dhc, 0)
    k.add("ember_rows_scatter", dhc, h, idx, count, 0, n, dh, h, None)
    dyn(True, False, v, h, rows, logits, hc, dw, 1)
    return k, {"loss": loss, "dh": dh, "dw": dw}


def _sizes(c):
    h, i, nh, nk, d, qk, v = WIDTHS[c["width"]][:7]
    layer = [h, nh * d * h, nk * d * h, nk * d * h, h * nh * d] + ([d, d] if qk else [])
    layer += [h, i * h, i * h, h * i]
    return [v * h] + layer * c["layers"] + [h]


def _optim_inputs(c, k):
    total = sum(_sizes(c))
    p, g = k.normal(total, std=0.02), k.normal(total, std=1e-3)
    m, v = k.normal(total, std=1e-4), k.normal(total, std=1e-4).square_()
    return p, g, m, v


OPT = dict(lr=1e-4, beta1=0.9, beta2=0.95, eps=1e-8, wd=0.1, step=10, max_norm=1.0)


def _prepare_optim(c, seed):
    k = _Calls(seed)
    p, g, m, v = _optim_inputs(c, k)
    sizes = _sizes(c)
    at = np.concatenate([[0], np.cumsum(sizes)[:-1]])
    cnt = len(sizes)
    ptrs = (C.c_void_p * cnt)(*[g.data_ptr() + 4 * int(a) for a in at])
    szs = (C.c_int64 * cnt)(*sizes)
    out = k.empty(1)
    ws1, wsb1 = k.scratch(capi.lib().ember_sumsq_workspace_bytes(cnt))
    ws2, wsb2 = k.scratch(capi.lib().ember_scale_multi_workspace_bytes(cnt))
    bc1, bc2 = 1.0 - OPT["beta1"] ** OPT["step"], 1.0 - OPT["beta2"] ** OPT["step"]
    args = []
    for a, s in zip(at, sizes):
        four = [C.c_void_p(t.data_ptr() + 4 * int(a)) for t in (p, g, m, v)]
        wd = OPT["wd"] if s > 10000 else 0.0  # the norm weights are in the group without decay
        args.append((*four, s, OPT["lr"], OPT["beta1"], OPT["beta2"], OPT["eps"], wd, bc1, bc2,
                     None))
    keep = (p, g, m, v, ptrs, szs, out)

    def step():
        capi.call("ember_sumsq_multi", ptrs, szs, cnt, _p(out), ws1, wsb1, None)
        norm = math.sqrt(out.item())  # the host decides whether to scale
        if norm > OPT["max_norm"]:
            capi.call("ember_scale_multi", ptrs, szs, cnt, OPT["max_norm"] / (norm + 1e-6), ws2,
                      wsb2, None)
        for a in args:
            capi.call("ember_adamw", *a)

    k.run, k.keep = step, k.keep + list(keep)
    return k, {"p": p, "m": m, "v": v}


def _trainer(c, seed, layers=None, vocab=None):
    cfg = TR.preset(c["width"])
    # plain RoPE: long-context frequency scaling changes values, not work
    cfg.rope_factor = 0.0
    if layers:
        cfg.num_layers, cfg.vocab_size = layers, vocab
    return TR.Trainer(cfg, seed=int(seed), init_std=0.02, norm_value=1.0)


class _Block:
    def __init__(self, c, seed):
        self.tr = _trainer(c, seed, layers=1, vocab=256)
        rng = np.random.default_rng(int(seed))
        shape = (c["batch"], c["seq"], self.tr.cfg.hidden_size)
        self.x = rng.standard_normal(shape, dtype=np.float32)
        self.dy = rng.standard_normal(shape, dtype=np.float32) * np.float32(1e-3)
        self.ck = c["checkpoint"]

    def run(self):
        self.tr.zero_grad()
        y, dx = self.tr.block_step(0, self.x, self.dy, checkpoint=self.ck)
        return {"y": y, "dx": dx}


class _Generate:
    def __init__(self, c, seed):
        self.tr = _trainer(c, seed)
        rng = np.random.default_rng(int(seed))
        self.ids = rng.integers(0, self.tr.cfg.vocab_size, (c["batch"], c["seq"] + 1))
        self.decode, self.seq = c["kind"] == "decode", c["seq"]
        self.cache = self.tr.kv_cache(c["batch"], c["seq"] + 64)
        if self.decode:
            self.tr.forward(self.ids[:, : self.seq], self.cache, 0, last_only=True)

    def run(self):
        if self.decode:
            out = self.tr.forward(self.ids[:, self.seq:], self.cache, self.seq, last_only=True)
        else:
            out = self.tr.forward(self.ids[:, : self.seq], self.cache, 0, last_only=True)
        return {"logits": out}


def prepare(case, seed):
    kind = case["kind"]
    if kind == "block":
        return _Block(case, seed), None
    if kind in ("prefill", "decode"):
        return _Generate(case, seed), None
    return {"linear": _prepare_linear, "mlp": _prepare_mlp, "attn": _prepare_attn,
            "head": _prepare_head, "optim": _prepare_optim}[kind](case, seed)


def run(state):
    what, out = state
    got = what.run()
    return got if out is None else out


# ------------------------------------------------------------------ work


def _attn_work(B, T, h, H, Hk, D, passes):
    """(bytes, flops) of the attention layer's forward (1), or forward and backward (3)."""
    n, q, kv = B * T, H * D, Hk * D
    weights = 2 * q * h + 2 * kv * h
    flops = 2.0 * n * weights * passes + 4.0 * B * H * D * (T * (T + 1) / 2) * passes
    return weights, flops


def work(case):
    c, kind = case, case["kind"]
    if kind == "linear":
        n, i, o = c["tokens"], c["n_in"], c["n_out"]
        if not c["backward"]:
            return {"bytes": 4.0 * (n * i + i * o + n * o), "flops": 2.0 * n * i * o}
        return {"bytes": 4.0 * (n * o + 2 * n * i + 2 * i * o), "flops": 4.0 * n * i * o}
    if kind == "mlp":
        n, h, i = c["tokens"], c["hidden"], c["inter"]
        return {"bytes": 4.0 * (4 * n * h + 6 * i * h), "flops": 18.0 * n * h * i}
    if kind == "attn":
        B, T, h, H, Hk, D = (c["batch"], c["seq"], c["hidden"], c["heads"], c["kv_heads"],
                             c["head_dim"])
        w, f = _attn_work(B, T, h, H, Hk, D, 3)
        return {"bytes": 4.0 * (4 * B * T * h + 2 * w), "flops": f}
    if kind == "head":
        n, h, v = max(1, round(c["tokens"] * c["active"])), c["hidden"], c["vocab"]
        return {"bytes": 4.0 * (n * h + 2 * v * h + c["tokens"] * h), "flops": 6.0 * n * h * v}
    if kind == "optim":
        n = float(sum(_sizes(c)))
        return {"bytes": 32.0 * n, "flops": 16.0 * n}  # g twice: its norm decides its scale
    h, i, H, Hk, D, _, v, layers = WIDTHS[c["width"]][:8]
    B, T = c["batch"], c["seq"]
    if kind == "block":
        w, f = _attn_work(B, T, h, H, Hk, D, 3)
        return {"bytes": 4.0 * (4 * B * T * h + 2 * (w + 3 * i * h)),
                "flops": f + 18.0 * B * T * h * i}
    w, _ = _attn_work(B, T, h, H, Hk, D, 1)
    per = w + 3 * i * h
    kv = 2.0 * B * T * Hk * D * layers
    if kind == "prefill":
        attn = 4.0 * B * H * D * (T * (T + 1) / 2) * layers
        return {"bytes": 4.0 * (layers * per + v * h + kv + B * v),
                "flops": 2.0 * B * T * per * layers + attn + 2.0 * B * v * h}
    return {"bytes": 4.0 * (layers * per + v * h + kv + B * v),
            "flops": 2.0 * B * (per * layers + v * h) + 4.0 * B * H * D * T * layers}


def tolerance(case):
    # About four times what the path shows against 64-bit sums (32-bit sums of up to 32768
    # products in a layer; whole models carry a layer's rounding through those that follow),
    # and twenty of those for the one furthest of some millions of values.
    rel = {"linear": 8e-6, "mlp": 8e-6, "attn": 1.2e-5, "head": 7e-6, "optim": 3e-7,
           "block": 1e-6, "prefill": 5e-6, "decode": 5e-6}[case["kind"]]
    return {"rel": rel, "max": 20 * rel}


# ------------------------------------------------------------------ 64-bit results


def _rms64(x, w, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w


def _rope64(x, theta):
    """x [B,T,H,D]: pairs (i, i + D/2), the angle one 32-bit product as the models define it."""
    B, T, H, D = x.shape
    i = torch.arange(D // 2, dtype=torch.float64, device=x.device)
    freq = torch.pow(torch.tensor(theta, dtype=torch.float64, device=x.device),
                     -2.0 * i / D).to(F32)
    ang = (torch.arange(T, device=x.device).to(F32)[:, None] * freq[None]).double()
    cos, sin = ang.cos()[None, :, None], ang.sin()[None, :, None]
    a, b = x[..., : D // 2], x[..., D // 2:]
    return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)


def _one_head64(q, k, v):
    s = (q @ k.t()) / math.sqrt(q.shape[1])
    t = torch.arange(q.shape[0], device=q.device)
    s = s.masked_fill(t[None, :] > t[:, None], float("-inf"))
    return torch.softmax(s, -1) @ v


def _attend64(q, k, v):
    """Causal GQA attention, one (batch, head) at a time so that 64-bit scores fit."""
    B, _, H, _ = q.shape
    group = H // k.shape[2]
    rows = []
    for b in range(B):
        heads = [torch.utils.checkpoint.checkpoint(_one_head64, q[b, :, i], k[b, :, i // group],
                                                   v[b, :, i // group], use_reentrant=False)
                 for i in range(H)]
        rows.append(torch.stack(heads, 1))
    return torch.stack(rows)


def _attn_layer64(x, t, B, T, H, Hk, D, theta, eps):
    n = B * T
    xn = _rms64(x, t["norm"], eps)
    q, k, v = ((xn @ t[w].t()).reshape(B, T, -1, D) for w in ("wq", "wk", "wv"))
    if "nq" in t:
        q, k = _rms64(q, t["nq"], eps), _rms64(k, t["nk"], eps)
    o = _attend64(_rope64(q, theta), _rope64(k, theta), v)
    return x + o.reshape(n, H * D) @ t["wo"].t()


def _mlp64(x, t, eps):
    xn = _rms64(x, t["norm"], eps)
    return x + (torch.nn.functional.silu(xn @ t["gate"].t()) * (xn @ t["up"].t())) @ t["down"].t()


def _grads64(t, fn):
    leaf = {name: v.double().requires_grad_(name != "dy") for name, v in t.items()}
    dy = leaf.pop("dy")
    y = fn(leaf)
    y.backward(dy)
    return y.detach(), {name: v.grad for name, v in leaf.items()}


def _layers64(tr, c, x):
    """Hidden states after every block, in 64 bits, and a reader of the weights."""
    eps = WIDTHS[c["width"]][9]
    h, i, H, Hk, D, qk = WIDTHS[c["width"]][:6]
    names = {n: j for j, n in enumerate(tr.names)}

    def param(name, *shape):
        return torch.from_numpy(tr.get_param(names[name])).cuda().double().reshape(shape)

    B, T = x.shape[:2]
    for layer in range(tr.cfg.num_layers):
        at = "model.layers.%d." % layer
        t = {"norm": param(at + "input_layernorm.weight", h),
             "wq": param(at + "self_attn.q_proj.weight", H * D, h),
             "wk": param(at + "self_attn.k_proj.weight", Hk * D, h),
             "wv": param(at + "self_attn.v_proj.weight", Hk * D, h),
             "wo": param(at + "self_attn.o_proj.weight", h, H * D)}
        if qk:
            t["nq"] = param(at + "self_attn.q_norm.weight", D)
            t["nk"] = param(at + "self_attn.k_norm.weight", D)
        y = _attn_layer64(x.reshape(B * T, h), t, B, T, H, Hk, D, tr.cfg.rope_theta, eps)
        m = {"norm": param(at + "post_attention_layernorm.weight", h),
             "gate": param(at + "mlp.gate_proj.weight", i, h),
             "up": param(at + "mlp.up_proj.weight", i, h),
             "down": param(at + "mlp.down_proj.weight", h, i)}
        x = _mlp64(y, m, eps).reshape(B, T, h)
    return x, param


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "linear":
        x, w, dy = (v.double() for v in _linear_inputs(c, _Calls(seed)))
        return {"dx": dy @ w, "dw": dy.t() @ x} if c["backward"] else {"y": x @ w.t()}
    if kind == "mlp":
        y, g = _grads64(_mlp_inputs(c, _Calls(seed)), lambda t: _mlp64(t["x"], t, 1e-6))
        return {"y": y, "dx": g["x"], "dnorm": g["norm"], "dgate": g["gate"], "dup": g["up"],
                "ddown": g["down"]}
    if kind == "attn":
        y, g = _grads64(_attn_inputs(c, _Calls(seed)), lambda t: _attn_layer64(
            t["x"], t, c["batch"], c["seq"], c["heads"], c["kv_heads"], c["head_dim"], c["theta"],
            c["eps"]))
        out = {"y": y, "dx": g["x"], "dnorm": g["norm"]}
        out.update({"d" + n: g[n] for n in ("wq", "wk", "wv", "wo")})
        if c["qk_norm"]:
            out.update(dnq=g["nq"], dnk=g["nk"])
        return out
    if kind == "head":
        t = _head_inputs(c, _Calls(seed))
        h, w = t["h"].double().requires_grad_(), t["w"].double().requires_grad_()
        rows = t["mask"].nonzero()[:, 0]  # all weights are 0 or 1
        loss = torch.nn.functional.cross_entropy(h[rows] @ w.t(), t["tgt"][rows])
        loss.backward()
        return {"loss": loss.detach().reshape(1), "dh": h.grad, "dw": w.grad}
    if kind == "optim":
        p, g, m, v = (x.double() for x in _optim_inputs(c, _Calls(seed)))
        norm = math.sqrt(g.square().sum().item())
        if norm > OPT["max_norm"]:
            g = g * (OPT["max_norm"] / (norm + 1e-6))
        m = OPT["beta1"] * m + (1 - OPT["beta1"]) * g
        v = OPT["beta2"] * v + (1 - OPT["beta2"]) * g.square()
        bc1, bc2 = 1.0 - OPT["beta1"] ** OPT["step"], 1.0 - OPT["beta2"] ** OPT["step"]
        wd = torch.cat([torch.full((s,), OPT["wd"] if s > 10000 else 0.0, device="cuda",
                                   dtype=torch.float64) for s in _sizes(c)])
        p = p - OPT["lr"] * ((m / bc1) / ((v / bc2).sqrt() + OPT["eps"]) + wd * p)
        return {"p": p, "m": m, "v": v}
    if kind == "block":
        s = _Block(c, seed)
        x = torch.from_numpy(s.x).cuda().double().requires_grad_()
        y, _ = _layers64(s.tr, c, x)
        y.backward(torch.from_numpy(s.dy).cuda().double())
        return {"y": y.detach(), "dx": x.grad}
    if c["width"] == "qwen3-1.7b":
        return None  # copying its weights out takes too long
    s = _Generate(c, seed)
    with torch.no_grad():
        ids = torch.from_numpy(s.ids if kind == "decode" else s.ids[:, :-1]).cuda()
        h, v = WIDTHS[c["width"]][0], WIDTHS[c["width"]][6]
        emb = torch.from_numpy(s.tr.get_param(s.tr.names.index("model.embed_tokens.weight")))
        emb = emb.cuda().double().reshape(v, h)
        x, param = _layers64(s.tr, c, emb[ids])
        x = _rms64(x[:, -1:], param("model.norm.weight", h), WIDTHS[c["width"]][9])
        return {"logits": x @ emb.t()}

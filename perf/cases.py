"""Performance cases of the speculative-decoding verify path.

Each case is one call (or one pair of calls) that a program makes through the
library's public entry points with its data already on the GPU:

  linear     cgx_matmul_int4_dev: x [M, K] times a device-resident INT4 weight
  attention  cgx_attention_int4_kv_dev over an INT4 KV cache (chain or tree mask)
  flash      cg_flash_attention_forward on fp32 Q, K, V
  kv         cgx_kv_cache_int4_write of new positions, cg_kv_cache_int4_get of all
  verify     cgx_verify_chain_batch_dev on batches of drafted chains
  model      cgx_model_forward of the decoder stack on a filled context

The sizes are those of the benchmark's stacks: the 7B shape (d 4096, 32 heads
over 8 KV heads of 128, FFN 11008, vocabulary 32000 or 128256), the tiny
decoder (12 layers, d 768, 12 heads of 64, FFN 3072), gamma 4 and contexts of
1024 to 4096; `draw` spreads over the ranges around them.
"""
from __future__ import annotations

import ctypes as C
import math

import torch

import cogito_amd
from cogito_amd.capi import (CgFlashAttnParams, CgTensor, CgTensorQuant, CgxModelConfig,
                             last_error)

# layers, d, heads, KV heads, head_dim, FFN, vocabulary
_STACKS = {
    "7b": (2, 4096, 32, 8, 128, 11008, 32000),
    "7b_1layer": (1, 4096, 32, 8, 128, 11008, 32000),
    "tiny": (12, 768, 12, 12, 64, 3072, 32000),
}
_MASK_NONE, _MASK_CAUSAL, _MASK_WINDOW = 0, 1, 2


def _linear(M, K, N, gs, **name):
    return dict(name, kind="linear", M=M, K=K, N=N, gs=gs)


def _attention(Nq, ctx, H, Hk, D, tree, **name):
    return dict(name, kind="attention", Nq=Nq, ctx=ctx, H=H, Hk=Hk, D=D, tree=tree)


def _flash(B, Nq, Nk, H, Hk, D, mask, window, lse, **name):
    return dict(name, kind="flash", B=B, Nq=Nq, Nk=Nk, H=H, Hk=Hk, D=D, mask=mask,
                window=window, lse=lse)


def _kv(T, pos, H, D, gs, **name):
    return dict(name, kind="kv", T=T, pos=pos, H=H, D=D, gs=gs)


def _verify(B, gamma, V, T, top_k, top_p, ratios, agree, **name):
    return dict(name, kind="verify", B=B, gamma=gamma, V=V, T=T, top_k=top_k, top_p=top_p,
                ratios=ratios, agree=agree)


def _model(stack, M, ctx, n_logits, **name):
    return dict(name, kind="model", stack=stack, M=M, ctx=ctx, n_logits=n_logits)


def listed():
    return [
        # one decoded token through the 7B shape's output projection: the
        # smallest linear call, one launch
        _linear(1, 4096, 4096, 128, name="linear_decode"),
        # the gate|up product of a verified chain (gamma 4 and the bonus row)
        _linear(5, 4096, 22016, 128, name="linear_verify"),
        # the down projection of eight chains verified together
        _linear(40, 11008, 4096, 128, name="linear_batch"),
        # a prompt of an odd length through one half of the FFN
        _linear(509, 4096, 11008, 128, name="linear_prompt"),
        # one layer's verify attention at context 4096
        _attention(5, 4096, 32, 8, 128, False, name="attention_verify"),
        # one layer's attention of a 512-token prompt chunk after 2048 tokens
        _attention(512, 2048, 32, 8, 128, False, name="attention_prompt"),
        # the fp32 flash forward of a prompt of an odd length
        _flash(1, 1021, 1021, 32, 8, 128, _MASK_CAUSAL, 0, True, name="flash_prompt"),
        # one layer's cache fill of a prompt chunk, and the cache read back
        _kv(512, 1536, 8, 128, 128, name="kv_append_get"),
        # one chain verified (the benchmark's acceptance workload): latency
        _verify(1, 4, 32000, 1.0, 0, 1.0, False, 0.0, name="verify_chain"),
        # 64 chains at the large vocabulary: the largest verify
        _verify(64, 4, 128256, 1.0, 0, 1.0, False, 0.0, name="verify_64_chains"),
        # one chain under nucleus sampling (the tiny decoder's loop), with the
        # acceptance ratios
        _verify(1, 4, 32000, 0.8, 0, 0.9, True, 0.0, name="verify_top_p"),
        # a prompt chunk through two layers of the 7B shape and its lm_head
        _model("7b", 256, 2048, 5, name="model_prompt"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "attention", "attention", "flash", "kv",
                       "verify", "verify", "model"])
    if kind == "linear":
        if rng.random() < 0.15:
            # a weight outside the tiled layouts (any K, N and group): the
            # reference-order kernel
            return _linear(_log_int(rng, 1, 12), _log_int(rng, 100, 1200) * 2,
                           _log_int(rng, 100, 2000) * 2, rng.choice([32, 40, 100, 128]))
        gs = rng.choice([128, 128, 128, 64, 32])
        K = 256 * _log_int(rng, 3, 43)
        N = gs * _log_int(rng, 768 // gs, 22016 // gs)
        M = _log_int(rng, 1, 512)
        while M > 1 and M * K * N > 509 * 4096 * 11008:
            M //= 2
        return _linear(M, K, N, gs)
    if kind == "attention":
        H, Hk, D = rng.choice([(32, 8, 128), (32, 8, 128), (12, 12, 64), (32, 32, 128), (8, 1, 64),
                               (28, 4, 128)])
        tree = rng.random() < 0.25
        Nq = _log_int(rng, 2, 64) if tree else _log_int(rng, 1, 512)
        ctx = _log_int(rng, 64, 8192)
        while Nq > 1 and Nq * (ctx + Nq) * H * D > 512 * 2560 * 32 * 128:
            Nq //= 2
        return _attention(Nq, ctx, H, Hk, D, tree)
    if kind == "flash":
        H, Hk, D = rng.choice([(32, 8, 128), (12, 12, 64), (16, 2, 96), (8, 8, 32), (16, 16, 128)])
        B = rng.choice([1, 1, 2, 3])
        Nq = _log_int(rng, 1, 1021)
        mask = rng.choice([_MASK_CAUSAL, _MASK_CAUSAL, _MASK_NONE, _MASK_WINDOW])
        Nk = _log_int(rng, Nq, 2042) if mask == _MASK_NONE else Nq
        while B > 1 and B * Nq * Nk * H * D > 1021 * 1021 * 32 * 128:
            B -= 1
        while Nk > Nq and B * Nq * Nk * H * D > 1021 * 1021 * 32 * 128:
            Nk = max(Nq, Nk // 2)
        return _flash(B, Nq, Nk, H, Hk, D, mask, rng.choice([16, 128, 300]), rng.random() < 0.5)
    if kind == "kv":
        D = rng.choice([128, 128, 64])
        return _kv(_log_int(rng, 1, 1024), rng.choice([0, _log_int(rng, 1, 1024)]),
                   rng.choice([8, 12, 32]), D, rng.choice([D, D, D // 2, 32]))
    if kind == "verify":
        V = rng.choice([32000, 128256, 50257, _log_int(rng, 1000, 128256)])
        top_k, top_p = rng.choice([(0, 1.0), (0, 1.0), (0, 0.9), (0, 0.95), (50, 1.0), (40, 0.9)])
        filtered = top_k > 0 or top_p < 1.0
        gamma = rng.choice([1, 2, 3, 4, 4, 5, 7])
        B = _log_int(rng, 1, 8 if filtered else 64)
        while B > 1 and B * (2 * gamma + 1) * V > 64 * 9 * 128256:
            B //= 2
        return _verify(B, gamma, V, rng.choice([1.0, 0.7, 0.8]), top_k, top_p,
                       rng.random() < 0.4, rng.choice([0.0, 0.8, 0.95]))
    M = _log_int(rng, 1, 256)
    return _model(rng.choice(["7b", "7b_1layer", "tiny"]), M, _log_int(rng, 32, 3072),
                  min(M, rng.choice([1, 5])))


# ---------------------------------------------------------------- helpers

def _lib():
    lib = cogito_amd.load()
    if lib.cgx_init(0):
        raise RuntimeError(last_error(lib))
    return lib


def _check(lib, rc):
    if rc:
        raise RuntimeError(last_error(lib))


def _gen(seed, salt=0):
    return torch.Generator(device="cuda").manual_seed(seed * 7919 + salt)


def _normal(g, *shape, std=1.0):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32) * std


class _Handle:
    """A library object that is freed with its last reference."""

    def __init__(self, ptr, free):
        if not ptr:
            raise RuntimeError(last_error(_lib()))
        self.ptr, self._free = ptr, free

    def __del__(self):
        self._free(self.ptr)


def _fptr(t):
    return C.cast(t.data_ptr(), C.POINTER(C.c_float))


def _tensor(t):
    """A cg_tensor over a torch tensor's memory."""
    c = CgTensor()
    c.data = _fptr(t)
    c.ndim, c.size, c.ref_count = t.dim(), t.numel(), 1
    for i, n in enumerate(t.shape):
        c.shape[i] = n
    return c


def _tiled(K, N, gs):
    return K % 256 == 0 and N % 16 == 0 and gs % 16 == 0 and N % gs == 0


def _linear_inputs(c, seed):
    """Uniform nibbles, fp16-valued scales U(0.005, 0.02), x ~ N(0, 1)."""
    g = _gen(seed)
    n = c["K"] * c["N"]
    nib = torch.randint(0, 256, (n // 2,), generator=g, device="cuda", dtype=torch.uint8)
    ng = -(-n // c["gs"])
    scales = (torch.rand(ng, generator=g, device="cuda") * 0.015 + 0.005).half().float()
    return nib, scales, _normal(g, c["M"], c["K"])


def _attention_inputs(c, seed):
    g = _gen(seed)
    n = c["ctx"] + c["Nq"]
    k, v = _normal(g, n, c["Hk"], c["D"]), _normal(g, n, c["Hk"], c["D"])
    q = _normal(g, c["Nq"], c["H"], c["D"])
    # a draft tree, breadth first: node i hangs below a node of the first half
    # of those before it (-1: below the cached prefix)
    r = torch.Generator().manual_seed(seed)
    parents = [-1 if i == 0 else int(torch.randint(0, (i + 1) // 2, (1,), generator=r))
               for i in range(c["Nq"])]
    return k, v, q, parents


def _kept(z, top_k, top_p):
    """Logits with those outside the top-k list and the nucleus at -inf."""
    if top_k > 0:
        kth = torch.topk(z, min(top_k, z.shape[-1])).values[..., -1:]
        z = torch.where(z >= kth, z, -math.inf)
    if top_p < 1.0:
        p, order = torch.softmax(z.double(), -1).sort(descending=True, stable=True)
        before = p.cumsum(-1) - p
        keep = torch.zeros_like(z, dtype=torch.bool).scatter(-1, order, before < top_p)
        z = torch.where(keep, z, -math.inf)
    return z


def _verify_inputs(c, seed):
    """Logits N(0, 2^2) (`agree`: the draft's correlation with the target's),
    drafted ids drawn from the draft's filtered distribution."""
    g = _gen(seed)
    B, gamma, V = c["B"], c["gamma"], c["V"]
    target = _normal(g, B, gamma + 1, V, std=2.0)
    a = c["agree"]
    draft = a * target[:, :gamma] + math.sqrt(1.0 - a * a) * _normal(g, B, gamma, V, std=2.0)
    draft = draft.contiguous()
    tok = torch.empty(B, gamma, dtype=torch.int32, device="cuda")
    for b in range(B):
        z = _kept(draft[b] / c["T"], c["top_k"], c["top_p"])
        e = torch.empty_like(z).exponential_(generator=g)
        tok[b] = (z - e.log()).argmax(-1)
    u = torch.rand(B, gamma + 1, generator=g, device="cuda")
    return target, draft, tok, u


# ------------------------------------------------------------ the interface

def prepare(case, seed):
    lib, c = _lib(), case
    s = {"lib": lib, "case": c}
    if c["kind"] == "linear":
        nib, scales, x = _linear_inputs(c, seed)
        q = CgTensorQuant()
        shape = (C.c_int * 2)(c["K"], c["N"])
        q.data = C.cast(nib.data_ptr(), C.POINTER(C.c_uint8))
        q.scales = _fptr(scales)
        q.shape = C.cast(shape, C.POINTER(C.c_int))
        q.ndim, q.size, q.quant_type, q.group_size = 2, c["K"] * c["N"], 2, c["gs"]
        q.num_groups, q.symmetric = scales.numel(), True
        torch.cuda.synchronize()
        s["w"] = _Handle(lib.cgx_quant_to_device(C.byref(q)), lib.cg_tensor_quant_free)
        s["x"] = x
        s["y"] = torch.zeros(c["M"], c["N"], device="cuda")
    elif c["kind"] == "attention":
        k, v, q, parents = _attention_inputs(c, seed)
        n = c["ctx"] + c["Nq"]
        torch.cuda.synchronize()
        s["cache"] = _Handle(lib.cg_kv_cache_int4_new(1, n, c["Hk"], c["D"], c["D"]),
                             lib.cg_kv_cache_int4_free)
        _check(lib, lib.cgx_kv_cache_int4_write(s["cache"].ptr, 0, 0, k.data_ptr(), v.data_ptr(), n))
        _check(lib, lib.cgx_kv_cache_int4_set_len(s["cache"].ptr, n))
        _check(lib, lib.cgx_synchronize())
        s["q"], s["o"] = q, torch.zeros_like(q)
        s["parents"] = (C.c_int * c["Nq"])(*parents)
    elif c["kind"] == "flash":
        g = _gen(seed)
        q = _normal(g, c["B"], c["Nq"], c["H"], c["D"])
        k = _normal(g, c["B"], c["Nk"], c["Hk"], c["D"])
        v = _normal(g, c["B"], c["Nk"], c["Hk"], c["D"])
        o = torch.zeros_like(q)
        lse = torch.zeros(c["B"], c["H"], c["Nq"], device="cuda") if c["lse"] else None
        p = CgFlashAttnParams()
        p.Q, p.K, p.V, p.O = q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr()
        p.batch_size, p.seqlen_q, p.seqlen_k = c["B"], c["Nq"], c["Nk"]
        p.n_heads, p.n_heads_k, p.d_head = c["H"], c["Hk"], c["D"]
        p.scale = 1.0 / math.sqrt(c["D"])
        p.mask_type, p.window_size = c["mask"], c["window"]
        p.softmax_lse = lse.data_ptr() if lse is not None else None
        s.update(q=q, k=k, v=v, o=o, lse=lse, params=p)
    elif c["kind"] == "kv":
        g = _gen(seed)
        n = c["pos"] + c["T"]
        old_k, old_v = _normal(g, n, c["H"], c["D"]), _normal(g, n, c["H"], c["D"])
        s["k"], s["v"] = _normal(g, c["T"], c["H"], c["D"]), _normal(g, c["T"], c["H"], c["D"])
        s["ko"], s["vo"] = torch.zeros_like(old_k), torch.zeros_like(old_v)
        s["tko"], s["tvo"] = _tensor(s["ko"]), _tensor(s["vo"])
        torch.cuda.synchronize()
        s["cache"] = _Handle(lib.cg_kv_cache_int4_new(1, n, c["H"], c["D"], c["gs"]),
                             lib.cg_kv_cache_int4_free)
        _check(lib, lib.cgx_kv_cache_int4_write(s["cache"].ptr, 0, 0, old_k.data_ptr(),
                                                old_v.data_ptr(), n))
        _check(lib, lib.cgx_kv_cache_int4_set_len(s["cache"].ptr, n))
        _check(lib, lib.cgx_synchronize())
    elif c["kind"] == "verify":
        s["target"], s["draft"], s["tok"], s["u"] = _verify_inputs(c, seed)
        s["out"] = torch.full((c["B"], c["gamma"] + 1), -1, dtype=torch.int32, device="cuda")
        s["n"] = torch.full((c["B"],), -1, dtype=torch.int32, device="cuda")
        s["ratio"] = torch.zeros(c["B"], c["gamma"], device="cuda") if c["ratios"] else None
    else:
        L, d, H, Hk, hd, ff, V = _STACKS[c["stack"]]
        cfg = CgxModelConfig(n_layers=L, d_model=d, n_heads=H, n_kv_heads=Hk, head_dim=hd,
                             d_ff=ff, vocab=V, group_size=128, kv_group_size=hd,
                             max_seq=c["ctx"] + c["M"], max_tokens=c["M"], rope_theta=10000.0,
                             norm_eps=1e-5, init_std=0.02, max_batch=1)
        s["m"] = _Handle(lib.cgx_model_new(C.byref(cfg), seed, None), lib.cgx_model_free)
        _check(lib, lib.cgx_model_fill_context(s["m"].ptr, c["ctx"], seed + 1))
        _check(lib, lib.cgx_synchronize())
        s["tok"] = torch.randint(0, V, (c["M"],), generator=_gen(seed), device="cuda",
                                 dtype=torch.int32)
        s["logits"] = torch.zeros(c["n_logits"], V, device="cuda")
    torch.cuda.synchronize()
    return s


def run(s):
    lib, c = s["lib"], s["case"]
    if c["kind"] == "linear":
        _check(lib, lib.cgx_matmul_int4_dev(s["x"].data_ptr(), c["M"], s["w"].ptr,
                                            s["y"].data_ptr()))
        return s["y"]
    if c["kind"] == "attention":
        _check(lib, lib.cgx_attention_int4_kv_dev(
            s["q"].data_ptr(), c["Nq"], c["H"], s["cache"].ptr, 0, int(c["tree"]),
            s["parents"] if c["tree"] else None, s["o"].data_ptr()))
        return s["o"]
    if c["kind"] == "flash":
        lib.cg_flash_attention_forward(C.byref(s["params"]))
        return {"o": s["o"], "lse": s["lse"]}
    if c["kind"] == "kv":
        _check(lib, lib.cgx_kv_cache_int4_write(s["cache"].ptr, 0, c["pos"], s["k"].data_ptr(),
                                                s["v"].data_ptr(), c["T"]))
        lib.cg_kv_cache_int4_get(s["cache"].ptr, 0, C.byref(s["tko"]), C.byref(s["tvo"]))
        return {"k": s["ko"], "v": s["vo"]}
    if c["kind"] == "verify":
        _check(lib, lib.cgx_verify_chain_batch_dev(
            s["target"].data_ptr(), s["draft"].data_ptr(), s["tok"].data_ptr(), s["u"].data_ptr(),
            c["B"], c["gamma"], c["V"], c["T"], c["top_k"], c["top_p"], s["out"].data_ptr(),
            s["n"].data_ptr(), s["ratio"].data_ptr() if c["ratios"] else None))
        return {"tokens": s["out"], "n": s["n"], "ratio": s["ratio"]}
    # the chunk after the context; the rollback that a rejected chunk gets
    _check(lib, lib.cgx_model_truncate(s["m"].ptr, c["ctx"]))
    _check(lib, lib.cgx_model_forward(s["m"].ptr, s["tok"].data_ptr(), c["M"], c["n_logits"],
                                      s["logits"].data_ptr()))
    return s["logits"]


def work(case):
    c = case
    if c["kind"] == "linear":
        M, K, N = c["M"], c["K"], c["N"]
        return {"bytes": K * N // 2 + -(-K * N // c["gs"]) * 4 + 4 * M * (K + N),
                "flops": 2 * M * K * N}
    if c["kind"] == "attention":
        n = c["ctx"] + c["Nq"]
        seen = c["Nq"] * c["ctx"] + c["Nq"] * (c["Nq"] + 1) // 2
        return {"bytes": 2 * n * c["Hk"] * (c["D"] // 2 + 4) + 8 * c["Nq"] * c["H"] * c["D"],
                "flops": 4 * seen * c["H"] * c["D"]}
    if c["kind"] == "flash":
        nq, nk = c["Nq"], c["Nk"]
        seen = {_MASK_NONE: nq * nk, _MASK_CAUSAL: nq * (nq + 1) // 2,
                _MASK_WINDOW: sum(min(nk, q + c["window"] + 1) - max(0, q - c["window"])
                                  for q in range(nq))}[c["mask"]]
        rows = c["B"] * nq * c["H"]
        return {"bytes": 8 * rows * c["D"] + 8 * c["B"] * nk * c["Hk"] * c["D"] +
                (4 * rows if c["lse"] else 0),
                "flops": 4 * c["B"] * seen * c["H"] * c["D"]}
    if c["kind"] == "kv":
        row = c["H"] * c["D"]
        packed = row // 2 + row // c["gs"] * 4
        n = c["pos"] + c["T"]
        # new rows in, packed out; every packed row in, values out
        return {"bytes": 2 * (c["T"] * (4 * row + packed) + n * (packed + 4 * row)), "flops": 0}
    if c["kind"] == "verify":
        return {"bytes": 4 * c["B"] * (2 * c["gamma"] + 1) * c["V"], "flops": 0}
    L, d, H, Hk, hd, ff, V = _STACKS[c["stack"]]
    M, n = c["M"], c["ctx"] + c["M"]
    layer = d * (H + 2 * Hk) * hd + H * hd * d + 3 * d * ff
    seen = M * c["ctx"] + M * (M + 1) // 2
    packed = 0.5 + 4 / 128
    return {"bytes": int((L * layer + d * V) * packed + L * 2 * n * Hk * (hd // 2 + 4) +
                         4 * M * d + 4 * c["n_logits"] * V),
            "flops": 2 * M * L * layer + 2 * c["n_logits"] * d * V + 4 * L * seen * H * hd}


def tolerance(case):
    """About four times what other orders of the same sums show.  Measured
    against 64 bits: linear 3e-7 (hi + lo fp16 terms, fp32 sums), flash 3.3e-7
    (fp32 products), attention 7.7e-6 (22-bit probabilities under a result
    that cancels to a few per cent of its terms).  A model's logits pass
    through the INT4 rounding of the new K and V rows, where a changed last
    bit moves a value by a quantisation step: 8e-4 between one chunk of 256
    tokens and the same tokens in chunks of 16."""
    c = case
    if c["kind"] == "linear":
        # shapes outside the tiled layouts run in the reference's order, bit
        # for bit
        return {"rel": 1.2e-6} if _tiled(c["K"], c["N"], c["gs"]) else "exact"
    if c["kind"] == "attention":
        return {"rel": 3e-5}
    if c["kind"] == "flash":
        return {"rel": 1.4e-6}
    if c["kind"] == "model":
        return {"rel": 3.3e-3, "max": 0.04}
    # whole values, the cache's dequantised values and the acceptance ratios
    # are the reference's own
    return "exact"


# ------------------------------------------------------- plain 64-bit results

def _quantized(x, gs):
    """x [..., D] through the cache's INT4 rounding, groups of gs values."""
    t = x.reshape(-1, gs)
    # a tensor divisor: torch multiplies by the reciprocal of a scalar one
    s = t.abs().amax(1, keepdim=True) / torch.full((1, 1), 7.0, device=t.device)
    s = torch.where(s < 1e-8, torch.ones_like(s), s)
    r = (t / s).double()
    q = (r.sign() * (r.abs() + 0.5).floor()).clamp(-8, 7)
    return (q * s.double()).reshape(x.shape)


def _softmax_pv(q, k, v, visible):
    """[Nq, D], [Nk, D], [Nk, D] and a boolean [Nq, Nk] (None: all)."""
    z = q @ k.t().contiguous() / math.sqrt(q.shape[-1])
    if visible is not None:
        z = z.masked_fill(~visible, -math.inf)
    return torch.softmax(z, -1) @ v, torch.logsumexp(z, -1)


def exact(case, seed):
    c = case
    if c["kind"] == "linear":
        nib, scales, x = _linear_inputs(c, seed)
        b = nib.to(torch.int16)
        w = torch.stack([b & 15, b >> 4], 1).reshape(-1)
        w = torch.where(w > 7, w - 16, w).double()
        group = torch.arange(w.numel(), device="cuda") // c["gs"]
        w = (w * scales.double()[group]).reshape(c["K"], c["N"])
        return x.double() @ w
    if c["kind"] == "attention":
        k, v, q, parents = _attention_inputs(c, seed)
        kq, vq = _quantized(k, c["D"]), _quantized(v, c["D"])
        nq, n = c["Nq"], c["ctx"] + c["Nq"]
        vis = torch.ones(nq, n, dtype=torch.bool)
        if c["tree"]:
            vis[:, c["ctx"]:] = False
            for i in range(nq):
                j = i
                while j >= 0:
                    vis[i, c["ctx"] + j] = True
                    j = parents[j]
        else:
            vis[:, c["ctx"]:] = torch.ones(nq, nq, dtype=torch.bool).tril()
        vis = vis.cuda()
        o = torch.empty(nq, c["H"], c["D"], dtype=torch.float64, device="cuda")
        for h in range(c["H"]):
            hk = h * c["Hk"] // c["H"]
            o[:, h] = _softmax_pv(q[:, h].double(), kq[:, hk].contiguous(), vq[:, hk].contiguous(),
                                  vis)[0]
        return o
    if c["kind"] == "flash":
        g = _gen(seed)
        q = _normal(g, c["B"], c["Nq"], c["H"], c["D"]).double()
        k = _normal(g, c["B"], c["Nk"], c["Hk"], c["D"]).double()
        v = _normal(g, c["B"], c["Nk"], c["Hk"], c["D"]).double()
        i = torch.arange(c["Nq"], device="cuda")[:, None]
        j = torch.arange(c["Nk"], device="cuda")[None]
        vis = {_MASK_NONE: None, _MASK_CAUSAL: j <= i,
               _MASK_WINDOW: (j - i).abs() <= c["window"]}[c["mask"]]
        o = torch.empty_like(q)
        lse = torch.empty(c["B"], c["H"], c["Nq"], dtype=torch.float64, device="cuda")
        for b in range(c["B"]):
            for h in range(c["H"]):
                hk = h * c["Hk"] // c["H"]
                o[b, :, h], lse[b, h] = _softmax_pv(q[b, :, h].contiguous(),
                                                    k[b, :, hk].contiguous(),
                                                    v[b, :, hk].contiguous(), vis)
        return {"o": o, "lse": lse if c["lse"] else None}
    if c["kind"] == "kv":
        g = _gen(seed)
        n = c["pos"] + c["T"]
        k, v = _normal(g, n, c["H"], c["D"]), _normal(g, n, c["H"], c["D"])
        k[c["pos"]:], v[c["pos"]:] = _normal(g, c["T"], c["H"], c["D"]), \
            _normal(g, c["T"], c["H"], c["D"])
        return {"k": _quantized(k, c["gs"]), "v": _quantized(v, c["gs"])}
    if c["kind"] == "verify" and c["ratios"]:
        # the draws turn on fp32 running sums: no 64-bit value for the tokens
        target, draft, tok, _ = _verify_inputs(c, seed)
        x = tok.long()[..., None]

        def prob(z):
            z = _kept(z / c["T"], c["top_k"], c["top_p"]).double()
            return torch.softmax(z, -1).gather(-1, x)[..., 0]
        ratio = (prob(target[:, :-1].contiguous()) / prob(draft)).clamp(max=1.0)
        return {"tokens": None, "n": None, "ratio": ratio}
    return None

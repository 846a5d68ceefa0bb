"""The work that users of this package have it do, as cases that can be timed and compared.

A case is one pass through the public entry points:

  linear    `apply_delta` on one projection -- what a single wrapped layer or a `QuantLinear` costs
  layer     the four projections of a decoder layer (fused q/k/v, o, fused gate/up, down) wrapped by
            `create_delta_manager` and run on one batch, `set_delta_mapping` included
  fused     the same seven projections held as separate weights, q/k/v and gate/up in one
            `apply_delta_batch` call each
  vocab     embedding lookup and output projection over full per-delta tables
  merge     a packed delta added to its base weight (export of a merged model)
  compress  a fine-tuned weight's delta compressed by magnitude
  hessian   two calibration batches accumulated by `SparseGPT.add_batch`
  sweep     the Hessian-weighted 2:4 sweep of one projection, scales and packing included

`listed()` holds the sizes of the benchmark's configurations (decode of 1, 32, 64 and 128 tokens
and prefill of 8192) with a chunk of mixed requests, a 4-bit prefill and the offline work beside
them; `draw()` takes other sizes from the same ranges.  Weights, deltas and activations follow the
distributions the benchmark configures: N(0, 0.02), N(0, 1e-3), N(0, 1).
"""
import math

import numpy as np
import torch
import torch.nn as nn

from deltazip_amd import (DeltaConfig, DeltaMapping, SparseGPT, apply_delta, apply_delta_batch, apply_delta_embed,
                          apply_delta_uncompressed, compress_delta, create_delta_manager, merge, ops, tile_base,
                          token_order)
from deltazip_amd.synthetic import gaussian_native_stack

DEV = "cuda:0"


# ---------------------------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------------------------


def listed():
    return [
        # one sequence, one projection: launch and host latency are the whole of it
        dict(name="decode-1-linear", kind="linear", tokens=1, k=4096, n=4096, bits=4, group=-1, slots=1, mix="uniform",
             tiled=True),
        # a decode batch of eight tenants, the headline workload
        dict(name="decode-32-fused", kind="fused", tokens=32, hidden=4096, inter=11008, bits=2, group=-1, slots=8,
             mix="uniform"),
        # a bursty multi-tenant decode batch: few popular deltas, many rare ones
        dict(name="decode-64-zipf", kind="layer", tokens=64, hidden=4096, inter=11008, bits=4, group=128, slots=32,
             mix="zipf"),
        # a full decode batch, nearly every token another tenant's
        dict(name="decode-128-layer", kind="layer", tokens=128, hidden=4096, inter=11008, bits=2, group=-1, slots=64,
             mix="uniform"),
        # one scheduler step that mixes a few short prompts, some of them of the base model; ragged
        dict(name="chunk-333-layer", kind="layer", tokens=333, hidden=5120, inter=13824, bits=2, group=-1, slots=16,
             mix="requests"),
        # a prefill batch of 16 prompts of 512 tokens, each of its own tenant
        dict(name="prefill-8192-layer", kind="layer", tokens=8192, hidden=5120, inter=13824, bits=2, group=-1, slots=16,
             mix="blocks"),
        # prompts of ragged lengths over 4-bit deltas with grouped scales
        dict(name="prefill-1999-layer", kind="layer", tokens=1999, hidden=4096, inter=11008, bits=4, group=128, slots=8,
             mix="requests"),
        # the two ends of the model in a decode step whose deltas bring their own vocabulary tables
        dict(name="decode-32-vocab", kind="vocab", tokens=32, hidden=4096, vocab=32000, slots=8, mix="uniform"),
        # a tenant's model written out as plain weights, or its delta warmed up for a dense path
        dict(name="merge-mlp", kind="merge", k=4096, n=11008, bits=4, group=128),
        # a fine-tuned projection turned into a servable delta without calibration data
        dict(name="compress-mlp", kind="compress", k=4096, n=11008, bits=2, group=-1),
        # calibration: layer inputs of two sequences of 2048 tokens
        dict(name="hessian-4096", kind="hessian", k=4096, tokens=2048),
        # calibration: one attention projection swept
        dict(name="sweep-4096", kind="sweep", k=4096, n=4096, bits=4),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _bits_group(rng):
    return rng.choice([(2, -1), (2, -1), (4, 128), (4, -1), (2, 128), (4, 64)])


def draw(rng):
    kind = rng.choice(["linear"] * 3 + ["layer"] * 4 + ["fused"] * 2 + ["vocab", "merge", "compress", "hessian", "sweep"])
    mix = rng.choice(["uniform", "zipf", "requests"])
    if kind == "linear":
        bits, group = _bits_group(rng)
        return dict(kind=kind, tokens=_log(rng, 1, 4096), k=256 * _log(rng, 2, 54), n=32 * _log(rng, 16, 864), bits=bits,
                    group=group, slots=_log(rng, 1, 32), mix=mix, tiled=rng.random() < 0.7)
    if kind == "fused":
        bits, group = _bits_group(rng)
        return dict(kind=kind, tokens=_log(rng, 1, 128), hidden=256 * _log(rng, 4, 20), inter=256 * _log(rng, 8, 54),
                    bits=bits, group=group, slots=_log(rng, 1, 32), mix=mix)
    if kind == "layer":
        bits, group = _bits_group(rng)
        return dict(kind=kind, tokens=_log(rng, 1, 8192), hidden=256 * _log(rng, 4, 20), inter=256 * _log(rng, 8, 54),
                    bits=bits, group=group, slots=_log(rng, 1, 64), mix=mix)
    if kind == "vocab":
        return dict(kind=kind, tokens=_log(rng, 1, 256), hidden=256 * _log(rng, 4, 16), vocab=64 * _log(rng, 64, 500),
                    slots=_log(rng, 1, 8), mix=mix)
    if kind in ("merge", "compress"):
        bits, group = _bits_group(rng)
        return dict(kind=kind, k=256 * _log(rng, 2, 54), n=32 * _log(rng, 16, 432), bits=bits, group=group)
    if kind == "hessian":
        return dict(kind=kind, k=64 * _log(rng, 8, 64), tokens=_log(rng, 17, 2048))
    return dict(kind="sweep", k=256 * _log(rng, 2, 16), n=32 * _log(rng, 4, 128), bits=rng.choice([2, 4]))


# ---------------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------------


def _ids(case, rs):
    """Slot of every token (-1: the base model), in the order the scheduler delivers them: decode
    batches sorted by delta, prompts one after the other."""
    t, s, mix = case["tokens"], case["slots"], case["mix"]
    if mix == "blocks":
        return np.arange(t) * s // t
    if mix == "requests":
        cuts = np.sort(rs.randint(0, t, size=max(1, min(2 * s, t // 40))))
        owner = rs.randint(-1, s, size=len(cuts) + 1)
        return owner[np.searchsorted(cuts, np.arange(t), side="right")]
    if mix == "zipf":
        p = np.arange(1, s + 1, dtype=np.float64) ** -1.5
        return np.sort(rs.choice(s, size=t, p=p / p.sum()))
    return np.sort(rs.randint(0, s, size=t))


def _present(case):
    """Distinct deltas a batch is expected to meet."""
    t, s, mix = case["tokens"], case["slots"], case["mix"]
    if mix == "blocks":
        return min(s, t)
    if mix == "requests":
        return s * (1 - (1 - 1 / (s + 1)) ** (max(1, min(2 * s, t // 40)) + 1))
    p = np.arange(1, s + 1, dtype=np.float64) ** -1.5 if mix == "zipf" else np.ones(s)
    return float(np.sum(1 - (1 - p / p.sum()) ** t))


def _weight(n, k, gen):
    return (torch.randn((n, k), device=DEV, generator=gen) * 0.02).half()


def _acts(t, k, gen):
    return torch.randn((t, k), device=DEV, generator=gen).half()


class _DecoderLayer(nn.Module):
    """The projections of a decoder layer under the names the manager looks for."""
    packed_modules_mapping = {"qkv_proj": ["q_proj", "k_proj", "v_proj"], "gate_up_proj": ["gate_proj", "up_proj"]}
    supported_delta_modules = ["qkv_proj", "o_proj", "gate_up_proj", "down_proj"]

    def __init__(self, hidden, inter, gen):
        super().__init__()
        for name, k, n in _fused_shapes(hidden, inter):
            lin = nn.Linear(k, n, bias=False, device="meta", dtype=torch.float16)
            lin.weight = nn.Parameter(_weight(n, k, gen), requires_grad=False)
            setattr(self, name, lin)


def _fused_shapes(h, i):
    return [("qkv_proj", h, 3 * h), ("o_proj", h, h), ("gate_up_proj", h, 2 * i), ("down_proj", i, h)]


def _group(case, k):
    return k if case["group"] == -1 or k % case["group"] else case["group"]


def prepare(case, seed):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    rs = np.random.RandomState(seed % (1 << 32))
    kind = case["kind"]
    s = {"kind": kind}
    if kind == "linear":
        k, n = case["k"], case["n"]
        w = _weight(n, k, gen)
        s["q"], s["m"], s["sc"] = gaussian_native_stack(k, n, case["bits"], _group(case, k), case["slots"], DEV, gen)
        s["w"], s["tiles"] = w, tile_base(w) if case["tiled"] else None
        s["x"] = _acts(case["tokens"], k, gen)
        s["idx"] = torch.from_numpy(_ids(case, rs)).to(DEV)
    elif kind == "fused":
        h, i = case["hidden"], case["inter"]
        s["idx"] = torch.from_numpy(_ids(case, rs)).to(DEV)
        s["slots"] = case["slots"]
        s["calls"] = []
        for k, ns in ((h, (h, h, h)), (h, (h,)), (h, (i, i)), (i, (h,))):
            ws = [_weight(n, k, gen) for n in ns]
            stacks = [gaussian_native_stack(k, n, case["bits"], _group(case, k), case["slots"], DEV, gen) for n in ns]
            s["calls"].append((_acts(case["tokens"], k, gen), [v[0] for v in stacks], [v[2] for v in stacks],
                               [v[1] for v in stacks], ws, [tile_base(w) for w in ws]))
    elif kind == "layer":
        h, i, t, slots = case["hidden"], case["inter"], case["tokens"], case["slots"]
        model = _DecoderLayer(h, i, gen)
        mgr = create_delta_manager(model, max_num_seqs=t, max_num_batched_tokens=t, vocab_size=32000,
                                   delta_config=DeltaConfig(max_deltas=slots, max_bitwidth=case["bits"],
                                                            group_size=case["group"]))
        for layer in mgr.modules.values():
            n, k = layer.base_shape
            layer.qweight_stacked, layer.meta_stacked, layer.scales_stacked = gaussian_native_stack(
                k, n, case["bits"], _group(case, k), slots, DEV, gen)
            layer.bitwidth = [case["bits"]] * slots
        mgr.delta_index_to_id = list(range(1, slots + 1))
        ids = tuple(int(v) + 1 for v in _ids(case, rs))
        s["mgr"], s["mapping"] = mgr, DeltaMapping(ids, ids[-1:])
        s["xs"] = [(getattr(model, name), _acts(t, k, gen)) for name, k, _ in _fused_shapes(h, i)]
    elif kind == "vocab":
        t, h, v, slots = case["tokens"], case["hidden"], case["vocab"], case["slots"]
        s["embed"] = torch.empty((slots, v, h), dtype=torch.float16, device=DEV)
        s["head"] = torch.empty((slots, v, h), dtype=torch.float16, device=DEV)
        for table in (s["embed"], s["head"]):
            for d in range(slots):
                table[d] = _weight(v, h, gen)
        s["embed0"], s["head0"] = _weight(v, h, gen), _weight(v, h, gen)
        s["tok"] = torch.randint(0, v, (t,), device=DEV, generator=gen)
        s["idx"] = torch.from_numpy(_ids(case, rs)).to(DEV)
        s["x"] = _acts(t, h, gen)
    elif kind == "merge":
        k, n = case["k"], case["n"]
        q, m, sc = gaussian_native_stack(k, n, case["bits"], _group(case, k), 1, DEV, gen)
        s.update(w=_weight(n, k, gen), q=q[0], m=m[0], sc=sc[0], bits=case["bits"])
    elif kind == "compress":
        k, n = case["k"], case["n"]
        s.update(delta=torch.randn((n, k), device=DEV, generator=gen) * 1e-3, bits=case["bits"], group=_group(case, k))
    elif kind == "hessian":
        k, t = case["k"], case["tokens"]
        s["layer"] = nn.Linear(k, 32, bias=False, dtype=torch.float16, device=DEV)
        s["batches"] = [_acts(t, k, gen).view(1, t, k) for _ in range(2)]
    else:
        k, n = case["k"], case["n"]
        x = torch.randn((k + 512, k), device=DEV, generator=gen)
        x[:, 1:] += 0.5 * x[:, :-1].clone()          # neighbouring inputs of a real layer are correlated
        hess = (x.t() @ x) * (2.0 / x.shape[0])
        hess.diagonal().add_(0.01 * hess.diagonal().mean())
        inv = torch.cholesky_inverse(torch.linalg.cholesky(hess))
        s["hinv"] = torch.linalg.cholesky(inv, upper=True).contiguous()
        s["delta"], s["bits"] = torch.randn((n, k), device=DEV, generator=gen) * 1e-3, case["bits"]
    return s


# ---------------------------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------------------------


def run(s):
    kind = s["kind"]
    if kind == "linear":
        return apply_delta(s["x"], s["q"], s["sc"], s["m"], s["idx"], s["w"], base_tiled=s["tiles"])
    if kind == "fused":
        order = token_order(s["idx"], s["slots"]) if s["idx"].numel() > 32 else None
        out = []
        for x, q, sc, m, w, tiles in s["calls"]:
            out += apply_delta_batch(x, q, sc, m, s["idx"], w, order=order, base_tiled=tiles)
        return out
    if kind == "layer":
        s["mgr"].set_delta_mapping(s["mapping"])
        return [module(x)[0] for module, x in s["xs"]]
    if kind == "vocab":
        return (apply_delta_embed(s["tok"], s["embed"], s["idx"], s["embed0"]),
                apply_delta_uncompressed(s["x"], s["head"], s["idx"], s["head0"]))
    if kind == "merge":
        return merge(s["w"], s["q"], s["m"], s["sc"], s["bits"])
    if kind == "compress":
        return compress_delta(s["delta"], s["bits"], s["group"])
    if kind == "hessian":
        gpt = SparseGPT(s["layer"])
        for batch in s["batches"]:
            gpt.add_batch(batch)
        return gpt.H
    w = s["delta"].clone()                            # the sweep leaves the compressed values in its place
    scale32, scale16 = ops.quant_scales(w, s["bits"])
    losses = ops.obs_sweep(w, s["hinv"], scale32.view(-1), s["bits"], 2, 4)
    codes, meta = ops.pack_2of4(w, scale32, s["bits"])
    return codes, meta, scale16, losses, w


# ---------------------------------------------------------------------------------------------
# what a pass cannot do without, and how exact it is
# ---------------------------------------------------------------------------------------------


def _linear_work(t, k, n, bits, group, present):
    delta = k * n * bits // 16 + k * n // 8 + 2 * n * (k // group)
    # every token meets the base weight; its delta has half as many values
    return np.array([2 * k * n + present * delta + 2 * t * k + 2 * t * n + 8 * t, 3.0 * t * k * n])


def work(case):
    kind = case["kind"]
    if kind == "linear":
        k = case["k"]
        b, f = _linear_work(case["tokens"], k, case["n"], case["bits"], _group(case, k), _present(case))
    elif kind in ("fused", "layer"):
        b, f = sum(_linear_work(case["tokens"], k, n, case["bits"], _group(case, k), _present(case))
                   for _, k, n in _fused_shapes(case["hidden"], case["inter"]))
    elif kind == "vocab":
        t, h, v = case["tokens"], case["hidden"], case["vocab"]
        b, f = 2 * _present(case) * v * h + 2 * t * v + 6 * t * h + 24 * t, 2.0 * t * v * h
    elif kind == "merge":
        k, n = case["k"], case["n"]
        b, f = 4 * k * n + k * n * case["bits"] // 16 + k * n // 8 + 2 * n * (k // _group(case, k)), 1.0 * k * n
    elif kind == "compress":
        k, n = case["k"], case["n"]
        b, f = 4 * k * n + k * n * case["bits"] // 16 + k * n // 8 + 2 * n * (k // _group(case, k)), 2.0 * k * n
    elif kind == "hessian":
        k, t = case["k"], case["tokens"]
        b, f = 2 * 2 * t * k + 4 * k * k, 2 * (1.0 * t * k * (k + 1))      # H is symmetric
    else:
        k, n = case["k"], case["n"]
        b = 4 * n * k * 2 + 4 * k * k // 2 + k * n * case["bits"] // 16 + k * n // 8 + 6 * n
        f = 1.0 * n * k * k
    return {"bytes": float(b), "flops": float(f)}


def tolerance(case):
    if case["kind"] in ("merge", "compress", "sweep"):
        return "exact"                                # every operation's rounding is specified
    if case["kind"] == "hessian":
        # fp32 sums over up to 4096 tokens; against the same sums in 64 bits: rel 9e-7, max 5.7e-6
        return {"rel": 4e-6, "max": 2.5e-5}
    # fp32 sums rounded to fp16 once; against the same sums in 64 bits: rel 2.1e-4, max 4.9e-4 (all sizes)
    return {"rel": 8e-4, "max": 2e-3}

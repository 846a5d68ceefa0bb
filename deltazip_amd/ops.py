"""Operator layer: the reference's delta ops, backed by the HIP kernels in libdz_amd.so.

Mirrors
  serving/vllm/delta/deltazip_marlin.py:10-19   apply_delta(x, qweight_stacked, scales_stacked,
                                                meta_stacked, indices, base_weight) -> y
  serving/vllm/delta/deltazip.py:14-77          add_delta / add_delta_slice (in-place y +=)
of eth-easl/deltazip.  Tensor names and roles are the reference's; the bit layout inside
`qweight`/`meta` is this project's native gfx950 layout (see csrc/dz_layout.h), produced from the
reference's GPTQ-style tensors by `repack_gptq_to_native`.

PyTorch is used for device memory and streams only; all arithmetic happens in the library.
"""
from __future__ import annotations

import ctypes as C
import math
from collections import Counter
from functools import lru_cache
from typing import Dict, NamedTuple, Optional, Sequence, Tuple

import torch

from . import _lib

MAX_TOKENS_FUSED = 128

# ---------------------------------------------------------------------------------------------
# layout helpers
# ---------------------------------------------------------------------------------------------


def native_sizes(K: int, N: int, bits: int, group_size: int = -1) -> Tuple[int, int, int]:
    """(codes_bytes, meta_bytes, scales_bytes) of one delta in the native layout."""
    cb, mb, sb = C.c_size_t(), C.c_size_t(), C.c_size_t()
    _lib.check(_lib.lib().dz_native_sizes(K, N, bits, group_size, C.byref(cb), C.byref(mb), C.byref(sb)),
               "dz_native_sizes")
    return cb.value, mb.value, sb.value


_sizes = lru_cache(maxsize=4096)(native_sizes)      # of the calls' path: by the sizes alone


def _slot_bytes_differ(q, m, sc, sizes) -> bool:
    cb, mb, sb = sizes
    return (_slot_numel(q) * q.element_size() != cb or _slot_numel(m) * m.element_size() != mb
            or _slot_numel(sc) * sc.element_size() != sb)


def stacked_shapes(K: int, N: int, bits: int, group_size: int = -1):
    """Shapes (without the leading slot dimension) of the three stacked tensors, following
    layers_marlin.py:311-333: qweight [K/(pf*4), 2N] int32, meta [N, K/16] int16, scales [G, N]."""
    native_sizes(K, N, bits, group_size)  # validates
    pf = 32 // bits
    g = 1 if group_size in (-1, K) else K // group_size
    return (K // (pf * 4), 2 * N), (N, K // 16), (g, N)


def repack_gptq_to_native(qweight: torch.Tensor, qzeros: torch.Tensor, scales: torch.Tensor,
                          g_idx: Optional[torch.Tensor], bits: int):
    """GPTQ-style tensors of one delta (as QuantLinear.pack writes them,
    deltazip/nn_modules/qlinear_cuda.py:144-244) -> (qweight, meta, scales) CPU tensors in the
    native layout, shaped as `stacked_shapes` says.  Host work, done once per delta; stands where
    the reference calls its checkpoint converter (deltazip/utils/converter.py:13-101)."""
    if bits not in (2, 4):
        raise NotImplementedError("Only 2 and 4 bits are supported.")
    qweight = qweight.detach().cpu().contiguous()
    qzeros = qzeros.detach().cpu().contiguous()
    scales = scales.detach().cpu().contiguous()
    if qweight.dtype != torch.int32 or qzeros.dtype != torch.int32 or scales.dtype != torch.float16:
        raise ValueError("qweight/qzeros must be int32 and scales float16")
    pf = 32 // bits
    K, N = qweight.shape[0] * pf, qweight.shape[1]
    G = scales.shape[0]
    if scales.shape != (G, N) or qzeros.shape != (G, N // pf) or K % G:
        raise ValueError("inconsistent qzeros/scales shapes")
    group_size = -1 if G == 1 else K // G
    gi = None
    if g_idx is not None:
        gi = g_idx.detach().cpu().to(torch.int32).contiguous()
        if gi.numel() != K:
            raise ValueError("g_idx must have K entries")
    (qs, ms, ss) = stacked_shapes(K, N, bits, group_size)
    out_q = torch.empty(qs, dtype=torch.int32)
    out_m = torch.empty(ms, dtype=torch.int16)
    out_s = torch.empty(ss, dtype=torch.float16)
    rc = _lib.lib().dz_repack_2of4(qweight.data_ptr(), qzeros.data_ptr(), scales.data_ptr(),
                                   gi.data_ptr() if gi is not None else None, K, N, bits, group_size,
                                   out_q.data_ptr(), out_m.data_ptr(), out_s.data_ptr())
    _lib.check(rc, "dz_repack_2of4")
    return out_q, out_m, out_s


def unrepack_native_to_gptq(qweight: torch.Tensor, meta: torch.Tensor, scales: torch.Tensor, K: int, N: int,
                            bits: int):
    """One delta in the native layout -> (qweight, qzeros, scales, g_idx) CPU tensors in the
    reference's GPTQ-style format (QuantLinear.pack, deltazip/nn_modules/qlinear_cuda.py:144-244):
    qweight int32 [K*bits/32, N], qzeros int32 [G, N*bits/32], scales fp16 [G, N], g_idx int32 [K].
    The inverse of `repack_gptq_to_native`; host work."""
    if bits not in (2, 4):
        raise NotImplementedError("Only 2 and 4 bits are supported.")
    qweight = qweight.detach().cpu().contiguous()
    meta = meta.detach().cpu().contiguous()
    scales = scales.detach().cpu().contiguous()
    if scales.dtype != torch.float16 or scales.numel() % N:
        raise ValueError("scales must be float16 [G, N]")
    G = scales.numel() // N
    group_size = -1 if G == 1 else K // G
    cb, mb, sb = native_sizes(K, N, bits, group_size)
    if (qweight.numel() * qweight.element_size() != cb or meta.numel() * meta.element_size() != mb
            or scales.numel() * 2 != sb):
        raise ValueError("tensors do not match the native layout for these sizes")
    pf = 32 // bits
    out_q = torch.empty((K // pf, N), dtype=torch.int32)
    out_z = torch.empty((G, N // pf), dtype=torch.int32)
    out_s = torch.empty((G, N), dtype=torch.float16)
    out_g = torch.empty(K, dtype=torch.int32)
    rc = _lib.lib().dz_unrepack_2of4(qweight.data_ptr(), meta.data_ptr(), scales.data_ptr(), K, N, bits, group_size,
                                     out_q.data_ptr(), out_z.data_ptr(), out_s.data_ptr(), out_g.data_ptr())
    _lib.check(rc, "dz_unrepack_2of4")
    return out_q, out_z, out_s, out_g


# The host's half of a call over a small layer is longer than the kernel: what it looks up more than once is looked up
# here.  (The raw handle without the Stream object around it: 0.3 against 3.6 us.)
_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)
_current_device = getattr(torch._C, "_cuda_getDevice", None)


def _stream() -> int:
    if _raw_stream is None or _current_device is None:
        return torch.cuda.current_stream().cuda_stream
    return _raw_stream(_current_device())


def _slot_numel(stacked: torch.Tensor) -> int:
    """Values of one slot of a stacked tensor (IndexError where there is none)."""
    shape = stacked.shape
    return stacked.numel() // shape[0] if shape and shape[0] else stacked[0].numel()


def _need_cuda(*ts):
    for t in ts:
        if t is not None and not t.is_cuda:
            raise ValueError("tensors must live on the GPU (there is no CPU implementation)")


def dequant(qweight: torch.Tensor, meta: torch.Tensor, scales: torch.Tensor, K: int, N: int,
            bits: int) -> torch.Tensor:
    """One native delta -> fp16 [N, K] on the GPU; bit-exact with QuantLinear.unpack
    (deltazip/nn_modules/qlinear_cuda.py:246-329)."""
    _need_cuda(qweight, meta, scales)
    G = scales.numel() // N
    out = torch.empty((N, K), dtype=torch.float16, device=qweight.device)
    rc = _lib.lib().dz_dequant(qweight.data_ptr(), meta.data_ptr(), scales.data_ptr(), K, N, bits,
                               -1 if G == 1 else K // G, out.data_ptr(), _stream())
    _lib.check(rc, "dz_dequant")
    return out


def merge(base_weight: torch.Tensor, qweight, meta, scales, bits: int) -> torch.Tensor:
    """W_base + dequant(delta) as fp16 [N, K] (deltazip/utils/generate.py:9-20 at fp16 storage)."""
    _need_cuda(base_weight, qweight, meta, scales)
    N, K = base_weight.shape
    G = scales.numel() // N
    out = torch.empty_like(base_weight)
    rc = _lib.lib().dz_merge(base_weight.data_ptr(), qweight.data_ptr(), meta.data_ptr(),
                             scales.data_ptr(), K, N, bits, -1 if G == 1 else K // G, out.data_ptr(),
                             _stream())
    _lib.check(rc, "dz_merge")
    return out


def segment(indices: torch.Tensor, num_slots: int, report: bool = False):
    """(perm [T] int32, seg_off [S+2] int32): tokens grouped by delta id, id -1 first.  `report`: an id
    outside [-1, S) sets bit 0 of the status word of this stream's workspace."""
    _need_cuda(indices)
    if indices.dtype != torch.int64:
        raise ValueError("indices must be int64")
    T = indices.numel()
    perm = torch.empty(T, dtype=torch.int32, device=indices.device)
    off = torch.empty(num_slots + 2, dtype=torch.int32, device=indices.device)
    status = _workspace(indices.device, 1, 256, 32).data_ptr() if report else None
    _lib.check(_lib.lib().dz_segment_status(indices.data_ptr(), T, num_slots, perm.data_ptr(), off.data_ptr(), status,
                                            _stream()), "dz_segment")
    return perm, off


SHORT_ROWS = 128               # row blocks of the kernel for few tokens per delta (DZ_SHORT_ROWS)
MAX_SLOTS_SEGMENT = 768        # DZ_MAX_SLOTS_SEGMENT


class RowBlocks:
    """A batch of more than 128 tokens ordered by delta id and cut into row blocks of one delta each
    (what dz_segment and dz_build_tiles write): depends on the indices only, so it can be made once
    per batch and passed to every layer call of the step (`order=`).  `tiles` are blocks of up to
    256 tokens, `short` blocks of up to 128 for the kernel with the smaller tile; either may be None.
    `mixed`: tables of blocks of several deltas (MixedTable), full and small ones, or None.  Up to 128 tokens these
    are all there is, and `order` is the token order for layers that go another way.
    They serve the side of a graph capture they were made on (`captured`), see `_usable_blocks`.
    `mix`: what the maker knew of the batch on the host, or None; `host_picks`: both tables hold all rows."""
    __slots__ = ("perm", "tiles", "max_tiles", "T", "S", "short", "max_short", "captured", "mix", "host_picks", "mixed", "order")

    def __init__(self, perm, tiles, max_tiles, T, S, short=None, max_short=0, mix=None, host_picks=False, mixed=None,
                 order=None):
        self.perm, self.tiles, self.max_tiles, self.T, self.S = perm, tiles, max_tiles, T, S
        self.short, self.max_short, self.mix, self.host_picks = short, max_short, mix, host_picks
        self.mixed, self.order = mixed, order
        self.captured = torch.cuda.is_current_stream_capturing()


class MixedTable(NamedTuple):
    """What dz_build_mixed writes: the table, how many blocks it has room for, and the most deltas of one."""
    table: torch.Tensor
    max_blocks: int
    deltas: int


class DecodeBlocks:
    """The blocks of several deltas of a decode step, made by the first eager call on each stream of a layer that takes
    them: a step that is replayed from a graph reads the token order and never asks, and the tables belong to the stream
    whose calls read them.  `ids`: of the tokens, any, one per delta and one for the base model, `met` of them; `indices`
    may be longer."""
    __slots__ = ("indices", "S", "ids", "met", "deltas", "made")

    def __init__(self, indices, S, ids, met, deltas):
        self.indices, self.S, self.ids, self.met, self.deltas, self.made = indices, S, ids, met, deltas, {}

    def for_layer(self, N: int, K: int, order: torch.Tensor):
        """What a layer of that size passes on as `order`, given the token order."""
        T = len(self.ids)
        if not mixes_at_decode(T, K, N, self.met) or torch.cuda.is_current_stream_capturing():
            return order
        stream = _stream()
        if stream not in self.made:
            self.made[stream] = row_blocks(self.indices[:T], self.S, mix=batch_mix(self.ids), deltas=self.deltas, order=order)
        return self.made[stream]


MIXED_BLOCKS = ((8, 4), (4, 2))   # (tiles of 16 tokens, deltas) of a block: full, small (DZ_MIXED_*)


def mixed_deltas(bits: int, grouped: bool) -> int:
    """Most deltas of a full block: a delta's words stay in registers while its block is multiplied, and at 4 bits
    and with scales that change along K three deltas' fit beside the sums."""
    return 4 if bits == 2 and not grouped else 3


@lru_cache(maxsize=4096)
def _mixed_plan(T: int, K: int, N: int) -> Optional[Tuple[int, int]]:
    """How a batch of more than 128 tokens takes blocks of several deltas: (0 for full blocks, 1 for small
    ones; parts K is cut into), or None where they do not pay.  By the sizes alone, so that above 512 tokens a token's
    result depends on neither the mix nor its place in the batch.  Up to 512 it may: `_in_mixed_blocks` and `_short_chunks`
    may choose another kernel, and where this plan has more than one part the device takes a number of them by the blocks
    that the batch came to (`_parts_of_blocks`), in every call, direct ones and replays among them.  Another kernel or number
    of parts is another order of fp32 sums.

    Fitted to 2240 timed batches of 129 to 1700 tokens and 3780 of 129 to 8192 (1 to 64 slots, sorted ids and
    requests, both bit widths, K from 512 to 13824, N to 27648): the choice takes 6.6 % longer in the mean than
    the best of two to five sizes of blocks and five of parts.  Against the faster of the other kernels (one delta
    per block; chunks of the decode kernel), in the mean: 129 tokens 1.28 times as fast, 333 1.33, 1000 1.29,
    2000 1.22, 8192 1.11.
      small blocks   where the full ones' workgroups would leave most of the 256 CUs idle: a block of half as
                     many tiles walks K in less time (2048 x 2048, 230 tokens: in the mean 1.42 against
                     1.23 times as fast as before; 4096 x 12288 of 333: 1.12 against 1.27); but a batch has more
                     blocks than T / 64, and from 224 workgroups by that count they were a second wave (2560
                     x 10240, 401 tokens of 3 deltas, 4-bit: full 50, small 67 us, one delta per block 60)
      parts          each a walk over its share of K, and one more pass over the sums at 3 TB/s (13824 x 5120,
                     333 tokens of 10 deltas: 1 / 2 / 3 / 4 / 6 parts 222 / 135 / 112 / 146 / 124 us, one delta per
                     block 160; the estimate takes 4, for it counts T / 128 blocks, 3, where there are 4); one where the host takes longer to launch
                     the sums than the walk takes (1536 x 1536, 263 tokens: 26.6 in 3 parts, 21.2 in one)
      K <= 1024      the walk is too short to pay for a workgroup's start unless there are several waves of them
                     (1024 x 8192: 129 tokens 14 / 19 us, 640 tokens 1.24 times as fast)"""
    if T <= MAX_TOKENS_FUSED or 2 * T * K >= 1 << 31:
        return None                                   # (32-bit offsets)
    if K <= 1024 and -(-T // 128) * -(-N // 128) <= 384:
        return None
    small = -(-N // 256) * T / 128 < (112 if K <= 3072 else 25)
    return int(small), _parts(T, K, N, -(-T // (64 if small else 128)), 1.0 if small else 1.7, 25)


def _parts(T: int, K: int, N: int, blocks: int, slab_us: float, host_us: float = 0) -> int:
    """Parts of K for so many blocks: what a wave of workgroups takes to start and to walk its part of K, alone
    and with all CUs busy, and the pass over the partial sums.  `host_us`: one part if it takes no longer."""
    wide, steps, best = -(-N // 256), K // 256, None
    for parts in (1, 2, 3, 4, 6):
        if parts > steps:
            break
        groups = wide * blocks * parts
        waves = -(-groups // 256) if groups <= 1024 else groups / 256
        cost = waves * (8 + -(-steps // parts) * 4 * slab_us * (0.6 + 0.4 * min(1.0, groups / 256)))
        if parts > 1:
            cost += 3 + 8 * T * N * parts / 3e6
        if best is None or cost < best[0]:
            best = (cost, parts)
        if parts == 1 and cost <= host_us:
            break
    return best[1]


@lru_cache(maxsize=4096)
def _parts_of_blocks(T: int, K: int, N: int, S: int, plan: Tuple[int, int], most_deltas: int) -> Tuple[int, int]:
    """What `_mixed_plan`'s number of parts becomes with a better guess at the number of blocks, which is not T / 128: where
    they fill the GPU a little more than once, one more is another wave of workgroups.  (parts, less than 0 where
    the device may take others by the blocks it makes; the most there can be), by `dz_mixed_parts`.
      up to 512 tokens   where a token's result may depend on the mix, the device picks, if there is a launch for the sums in
                         any case (333 tokens of 8 deltas in four blocks, three parts instead of four: 13824 x 5120 129 ->
                         100 us, 5120 x 5120 54 -> 46).  Of 700 drawn projections it takes another number in 250, 13 %
                         less in the mean; 20 of the 700 take 2 % and more longer, the worst 26 %: blocks of few tokens,
                         which end early, and whose second round is not the whole one that the estimate has.  Against the
                         best number for each 1.3 % longer in the mean, the usual one 7.2 %
      above              by the sizes alone: another number of parts if it is the faster one for all numbers of blocks that
                         there can be, from full ones to all slots in use and blocks that end by their deltas; or, of five slots
                         and more in full blocks, twice as many, if those are faster from four fifths of the slots (or a prompt of
                         40 tokens each) on that end half a tile early in the mean.  One in 77 drawn
                         projections; 500 of them timed both ways, a mix each: 6.9 % less in the mean, 39 take 2 % more and
                         the worst 14 % (1999 tokens of 8 deltas, 4-bit, 17 blocks, two parts for one: 4096 x 4096 127 to 146
                         us -> 116 to 126, 11008 x 4096 317 to 372 -> 280 to 314).  With the second range for any
                         number of parts it was one in 29, 8 % less in the mean, but 15 % of them took 2 % more and the worst 37 %"""
    L, (small, parts) = _lib.lib(), plan
    if T <= 4 * MAX_TOKENS_FUSED:
        if parts == 1:
            return 1, 1
        return -parts, L.dz_mixed_most_parts(T, K, N, parts)
    rows, deltas = 16 * MIXED_BLOCKS[small][0], min(S + 1, T // 16)
    early, ended = lambda d: -(-(T + 8 * d) // rows), lambda d: -(-d // most_deltas)
    made = L.dz_mixed_parts_between(T, K, N, -(-T // rows), early(deltas) + ended(deltas) + 1, parts, 0)
    if made == parts <= 3 and not small and S >= 5:
        d = min(4 * deltas // 5, T // 40)
        made = L.dz_mixed_parts_between(T, K, N, max(early(d), ended(d)), early(deltas) + ended(deltas) - 1, parts, 2 * parts)
    return made, made


def mixes_at_decode(T: int, K: int, N: int, deltas: int) -> bool:
    """Whether a batch of 33 to 128 tokens of so many deltas (the base model counts as one) goes in blocks of several
    deltas: the decode kernel makes its products once per 32 tokens and delta, a block once per 16 tokens and never
    twice for a weight it has in registers; with many deltas the blocks are many and short.  By 840 timed calls over
    layers of 20 M weights and more, in the mean and at worst: 33 tokens of up to 8 deltas 1.37 / 0.96 times as
    fast, 48 and 64 tokens of 1 or 2 1.34 / 0.92 (of 7 or 8 1.14 / 0.81: left as they are), 96 tokens of up to 8
    1.41 / 0.97, 128 of up to 8 1.66 / 1.14 and of 13 to 16 1.33 / 0.97 (of more 1.01 / 0.77).  5120 x 27648,
    2-bit, 128 tokens of 4 / 8 / 16 deltas: 194 -> 102, 209 -> 132, 253 -> 230 us; 13824 x 5120: 122 -> 51, 129 -> 67, 151 ->
    104.  Smaller layers take about the time of their calls' host half either way (a layer of 2048/5632, 100 tokens of
    4 deltas: 116 / 125 us)."""
    if not 32 < T <= MAX_TOKENS_FUSED or K * N < 24 << 20:
        return False
    return deltas <= (16 if T > 112 else 8 if T > 64 or T <= 40 else 2)


@lru_cache(maxsize=4096)
def decode_step_mixes(T: int, bits: int, deltas: int, projections: Tuple[Tuple[Tuple[int, int], int], ...]) -> bool:
    """Whether a decode step over `projections`, ((K, N), how many), makes tables for blocks of several deltas: where
    one of them would take such blocks, and the decode kernel keeps the GPU busy for longer than the host needs to
    launch the step.  A layer call takes the host some 30 us, 3 more over blocks (a second launch, the sums' tensor),
    and the blocks are looked up by every projection.  By 190 timed layers of four projections
    that went in blocks: below 160 us of the decode kernel, as `_route_us` has it, 120 us became 130
    (2048/8448, 81 tokens of 4 deltas, 4-bit), at 160 and above 1.22 times as fast in the mean, 0.94 at worst."""
    if not any(mixes_at_decode(T, k, n, deltas) for (k, n), _ in projections):
        return False
    mix = _even_mix(T, deltas)
    return sum(c * _route_us(T, k, n, bits, mix)[0] for (k, n), c in projections) >= 40 * sum(c for _, c in projections)


@lru_cache(maxsize=4096)
def _decode_plan(T: int, K: int, N: int, deltas: int) -> Tuple[int, int]:
    """`_mixed_plan` of such a batch, whose number of blocks is taken to be that of its deltas over four (at 4 bits and with
    grouped scales there are three to a block, and the base model's tokens have blocks of their own).  A token's result
    so depends on how many deltas share the batch, by the order of fp32 sums."""
    return 0, _parts(T, K, N, max(1, -(-deltas // 4)), 1.7)


def _in_mixed_blocks(T: int, K: int, N: int, S: int, mix: Optional["BatchMix"]) -> Optional[Tuple[int, int]]:
    """`_mixed_plan` but for batches whose mix the host knows to suit another kernel: a few tokens of each of many
    deltas over a long and narrow layer go in chunks (11008 x 4096, 129 tokens of 55 deltas: 180 against 261 us),
    and over a short one, where the row blocks are one wave of workgroups, in row blocks (1536 x 3072, 170 tokens
    of 20 deltas: 18 / 27)."""
    plan = _mixed_plan(T, K, N) if 0 < S <= MAX_SLOTS_SEGMENT else None
    if plan is not None and mix is not None:
        if takes_fused_chunks(T, S) and 3 * mix.deltas > T and K >= 2 * N:
            return None
        if K <= 2560 and 20 * mix.blocks >= T and mix.blocks * -(-N // 128) <= 512:
            return None
    return plan


@lru_cache(maxsize=4096)
def _short_chunks(T: int, K: int, N: int, bits: int, S: int) -> bool:
    """Whether a call that would have to make its own table goes in chunks of the decode kernel, of which there are few
    and short ones: it takes the host 28 us to launch two of them, and 37 to launch the table, the product and the sum
    of its parts.  By 300 timed calls of 129 to 512 tokens the two meet at an estimate (`_route_us`) of 36 us: at 28 to
    32 us chunks take 29.7 us and blocks 37.2 (2304 x 1088, 4-bit, 237 tokens of one slot: 31.6 and 45.2 while the
    order and the table were two launches), at 40 to 44 us 40.6 and 37.3.  The line lies a tenth below, the estimate being
    that good."""
    return (takes_fused_chunks(T, S) and _most_blocks_unknown(T, K, N, bits, S) == 0
            and _route_us(T, K, N, bits, _even_mix(T, S))[0] < 33)


class BatchMix(NamedTuple):
    """What the choice between the kernels looks at: deltas in the batch (the base model counts as
    one), row blocks of 128 tokens, tokens of the most popular delta, and the deltas met by each chunk
    of 128 tokens, summed."""
    deltas: int
    blocks: int
    longest: int
    met: int


def batch_mix(ids: Sequence[int]) -> BatchMix:
    """The mix of a batch whose delta ids the host has (any ids: one per delta, one for the base model)."""
    counts = Counter(ids).values()
    return BatchMix(len(counts), sum([-(-c // SHORT_ROWS) for c in counts]), max(counts),
                    sum([len(set(ids[r:r + MAX_TOKENS_FUSED])) for r in range(0, len(ids), MAX_TOKENS_FUSED)]))


def _even_mix(T: int, deltas: int) -> BatchMix:
    """That many deltas (or one per token), as many tokens of each, sorted."""
    d = min(deltas, T)
    return BatchMix(d, d * -(-T // (SHORT_ROWS * d)), T // d, d + -(-T // MAX_TOKENS_FUSED) - 1)


@lru_cache(maxsize=4096)
def _route_us(T: int, K: int, N: int, bits: int, mix: BatchMix) -> Tuple[float, float]:
    """What a batch of a few hundred tokens takes in chunks of the fused kernel, and in row blocks of 128
    tokens.  A row block costs much the same whether it holds 2 tokens or 60,
    because it reads the base weight again, and walks all of K; a chunk of 128 reads the base weight once
    for all its deltas and splits K where there are few features.

    Estimates in us, fitted to 10597 timed calls over tiles (129 to 512 tokens of 1 to 64 deltas, sorted and
    in requests; K from 512 to 13824, N to 27648; 2 bits and 4) and within a fifth of 90 % of them.  What
    they choose is 0.5 % slower in the mean than the faster route; row blocks throughout were 14 % and up
    to 5.4 times, chunks throughout 77 % and 5.7 times.  Chunks / row blocks,
    sorted, 2-bit:
      5120 x 27648, 129 tokens of 4 / 16 / 64 deltas   251 / 307 / 557 against 138 / 376 / 1103 us
                    256                                388 / 433 / 698 against 177 / 386 / 1224
                    512                                769 / 798 / 1064 against 297 / 425 / 1356
      4096 x 4096,  129 tokens of 1 / 4 / 16 deltas    47 / 47 / 54 against 57 / 39 / 44
      13824 x 1024, 129 tokens of 1 / 4 / 16 deltas    48 / 49 / 53 against 173 / 119 / 110
                    512                                119 / 123 / 127 against 178 / 176 / 108
    Row blocks come in waves of 512 workgroups, two per CU: a single wave's time is that of its longest
    block's walk, and of sharing a CU; several are bound by their products.  Chunks: two launches each,
    the products of every 32 tokens, the deltas' words, and the start of each workgroup."""
    k, weight = K / 1024, K * N / 2**20
    groups = mix.blocks * -(-N // 128)
    waves, chunks, turns = -(-groups // 512), -(-T // MAX_TOKENS_FUSED), -(-T // 32)
    if waves == 1:
        start, walk, full, shared = (7.3, 7.7, 5.6, 6.1) if bits == 2 else (6.5, 9.9, 5.0, 6.7)
        rows_us = start + k * (walk + full * (min(mix.longest, SHORT_ROWS) / SHORT_ROWS)**2
                               + shared * max(0, groups - 256) / 256)
    else:
        start, walk, token = (2.8, 8.5, 14.1) if bits == 2 else (2.6, 11.0, 13.1)
        rows_us = waves * (start + k * (walk + token * T / (SHORT_ROWS * mix.blocks)))
    walk, turn, delta, shared = (0.63, 0.287, 0.0416, 0.07) if bits == 2 else (0.69, 0.300, 0.0770, 0.119)
    chunks_us = (chunks * (11.3 + walk * k) + weight * (turn * turns + delta * mix.met - shared * chunks)
                 + 0.153 * N / 1024 * turns)
    return chunks_us, rows_us


def _in_chunks(costs: Tuple[float, float]) -> bool:
    return costs[0] < 0.98 * costs[1]                 # (closer estimates say nothing: row blocks)


def _one_wave_of_long_blocks(T: int, N: int, bits: int) -> bool:
    """Where a single delta's two blocks of 256 tokens beat its four of 128: their tiles of 256 features
    then fill the 256 CUs once, nearly (512 tokens, 2-bit, 5120 x 27648 223 against 257 us, 8192 x
    28672 361 / 395, 4096 x 32768 194 / 221; with fewer tiles, 5120 x 24576, 222 / 204; 448 tokens 235 /
    242; at 4 bits never: 257 / 249)."""
    return bits == 2 and 448 < T <= 512 and 208 < 2 * -(-N // 256) <= 256


def _usable_blocks(order, T: int, S: int) -> Optional[RowBlocks]:
    """`order` if it holds row blocks this call can use, else None: the call then makes its own from the
    indices.  A captured call does so unless the blocks were made under capture too: a replay must
    read the indices as they are then, and the tables of a batch that is over may have been given
    back.  (Blocks made under capture hold nothing before the first replay: no eager call takes them.)"""
    if not isinstance(order, RowBlocks) or order.captured != torch.cuda.is_current_stream_capturing():
        return None
    if order.T == T and order.S == S:
        return order
    if takes_fused_chunks(T, S):
        return None                                   # (at these sizes a stale order was never an error)
    raise ValueError("row blocks were made for another batch size or number of slots")


def _block_table(T: int, num_slots: int, rows: int, device):
    n = (T + rows - 1) // rows + min(num_slots + 1, T)
    return torch.empty((n, 4), dtype=torch.int32, device=device), n


@lru_cache(maxsize=4096)
def _most_mixed_blocks(T: int, S: int, tiles: int, deltas: int) -> int:
    return _lib.lib().dz_mixed_blocks(T, S, tiles, deltas)


def _mixed_table(T: int, S: int, small: int, deltas: int, device, behind: int = 0) -> MixedTable:
    tiles, most = MIXED_BLOCKS[small]
    deltas = min(deltas, most)
    n = _most_mixed_blocks(T, S, tiles, deltas)
    # DZ_MIXED_HEADER words and n times sizeof(dz_mixed_block)
    return MixedTable(torch.empty(4 + n * (2 + 4 * 4 + 128) + behind, dtype=torch.int32, device=device), n, deltas)


def own_mixed_table(indices: torch.Tensor, S: int, small: int, deltas: int) -> MixedTable:
    """The one table a call needs, from the ids, in one launch; the token order is left behind its blocks.  Bad ids are
    reported at the sizes that chunks of the decode kernel can serve, as that kernel does."""
    _need_cuda(indices)
    if indices.dtype != torch.int64:
        raise ValueError("indices must be int64")
    T = indices.numel()
    made = _mixed_table(T, S, small, deltas, indices.device, T)
    table = made.table.data_ptr()
    status = _workspace(indices.device, 1, 256, 32).data_ptr() if takes_fused_chunks(T, S) else None
    _lib.check(_lib.lib().dz_order_mixed(indices.data_ptr(), T, S, MIXED_BLOCKS[small][0], made.deltas,
                                         table + 4 * (made.table.numel() - T), table, made.max_blocks, status, _stream()),
               "dz_order_mixed")
    return made


def row_blocks(indices: torch.Tensor, num_slots: int, long_only: bool = False, mix: Optional[BatchMix] = None,
               device_picks: bool = False, features: Optional[int] = None, deltas: int = 3,
               order: Optional[torch.Tensor] = None, mixed: bool = True) -> RowBlocks:
    """Row blocks of a prefill-sized batch, as the reference converts its mapping once per batch
    (serving/vllm/delta/models.py:421-435).  Small launches, nothing read back to the host.

    Which of the two kernels serves the batch.  Tiles of 256 features x 256 tokens want full
    blocks and some 256 of them; tiles of 128 x 128 read the weights twice as often but fill the GPU
    with a quarter of the tokens and multiply few rows that are not there.
      up to 1024 tokens   short blocks: even with a single delta there are too few long ones to fill
                          the GPU (5120 x 5120, 2-bit, 1024 tokens, 1 / 16 / 64 deltas: 116 / 153 / 276
                          against 192 / 246 / 649 us; 5120 x 27648: 435 / 630 / 1443 against 810 / 1000 /
                          3468), but for `_one_wave_of_long_blocks`
      above, 256 tokens   long blocks: they are at least half full, and at 8192 tokens of 16 deltas
      per slot and more   or fewer the larger tile is the faster one at 2 bits (5120 x 27648: 3113
                          against 3499; 4096 x 12288: 1133 against 1243; 4 bits: equal)
      between             the number of deltas in the batch is known on the device only: it picks
                          (dz_build_tiles_either), and both products are launched, one of them empty --
                          but for layers so narrow that long blocks would fill at most half the GPU,
                          where short ones win and a second launch is felt (512 x 2048, 1500 tokens
                          of 12 slots: 57 against 50 us)
    `long_only`: the table of 256-token blocks alone, whatever the batch.  `mix`: batch_mix() of the
    same ids, if the host has them: calls of a few hundred tokens then choose between these blocks and
    chunks of the fused kernel by it.  `device_picks`: as between, whatever the batch.  `features`: of the
    widest layer they are for, if known.

    Layers with a base weight take the batch in blocks of several deltas where those pay (`_mixed_plan`): their
    tables are made in the same launch.  `deltas`: `mixed_deltas` of the layers (a layer that can hold more in a block reads
    tables made for three all the same, one that can hold fewer makes its own).  `order`: token_order() of the same
    indices, for a batch of up to 128 tokens: the table of full blocks is then all that is made (mixes_at_decode).  `mixed`: False
    leaves the blocks of several deltas out, for a call that has turned them down."""
    indices = indices.reshape(-1)
    if not indices.is_contiguous():
        raise ValueError("indices must be contiguous")
    T = indices.numel()
    if mixed and order is not None and T <= MAX_TOKENS_FUSED and not long_only:   # (a decode step takes full blocks only)
        full = own_mixed_table(indices, num_slots, 0, deltas)
        return RowBlocks(full.table[-T:], None, 0, T, num_slots, mix=mix, mixed=[full, None], order=order)
    # (at the sizes chunks of the fused kernel can serve, bad ids are reported as that kernel does)
    perm, seg_off = segment(indices, num_slots, not long_only and takes_fused_chunks(T, num_slots))
    L, dev, st = _lib.lib(), indices.device, _stream()
    narrow = features is not None and -(-features // 256) * -(-T // 256) <= 128 and T < 256 * (num_slots + 1)
    small = not long_only and not device_picks and (T <= 1024 or narrow)
    tiles, n, short, ns = None, 0, None, 0
    host_picks = small and mix is not None and mix.deltas == 1 and 448 < T <= 512
    if not small or host_picks:
        tiles, n = _block_table(T, num_slots, 256, dev)
    if small or device_picks or (not long_only and T < 256 * (num_slots + 1)):
        short, ns = _block_table(T, num_slots, SHORT_ROWS, dev)
    either = tiles is not None and short is not None and not host_picks
    if mixed and not long_only:
        made = [_mixed_table(T, num_slots, small_ones, deltas, dev) for small_ones in (0, 1)]
        ptr = lambda t: None if t is None else t.data_ptr()
        _lib.check(L.dz_build_tables(seg_off.data_ptr(), perm.data_ptr(), num_slots, T, ptr(tiles), n, ptr(short), ns,
                                     int(either), made[0].deltas, made[0].table.data_ptr(), made[0].max_blocks,
                                     made[1].table.data_ptr(), made[1].max_blocks, st), "dz_build_tables")
        return RowBlocks(perm, tiles, n, T, num_slots, short, ns, mix, host_picks, made, order)
    if either:
        _lib.check(L.dz_build_tiles_either(seg_off.data_ptr(), num_slots, tiles.data_ptr(), n, short.data_ptr(), ns, st),
                   "dz_build_tiles_either")
    else:
        if tiles is not None:
            _lib.check(L.dz_build_tiles(seg_off.data_ptr(), num_slots, tiles.data_ptr(), n, st), "dz_build_tiles")
        if short is not None:
            _lib.check(L.dz_build_tiles_rows(seg_off.data_ptr(), num_slots, SHORT_ROWS, short.data_ptr(), ns, st),
                       "dz_build_tiles_rows")
    return RowBlocks(perm, tiles, n, T, num_slots, short, ns, mix, host_picks)


def apply_delta_embed(x: torch.Tensor, delta_weights: torch.Tensor, indices: torch.Tensor,
                      base_weight: torch.Tensor) -> torch.Tensor:
    """Embedding lookup where every token reads the table of its own delta
    (serving/vllm/delta/deltazip_marlin.py:56-86): out[t] = delta_weights[indices[t]][x[t]], or
    base_weight[x[t]] for indices[t] == -1.  x [T] int64 token ids, delta_weights [S, V, H] fp16,
    base_weight [V, H] fp16; returns [T, H] fp16."""
    _need_cuda(x, delta_weights, indices, base_weight)
    if x.dtype != torch.int64 or indices.dtype != torch.int64:
        raise ValueError("token ids and indices must be int64")
    if delta_weights.dtype != torch.float16 or base_weight.dtype != torch.float16:
        raise ValueError("embedding tables must be float16")
    S, V, H = delta_weights.shape
    if tuple(base_weight.shape) != (V, H) or not delta_weights.is_contiguous() or not base_weight.is_contiguous():
        raise ValueError("base_weight must be [V, H] like each delta table, all contiguous")
    T = x.numel()
    if indices.numel() != T:
        raise ValueError("one index per token is required")
    out = torch.empty((T, H), dtype=torch.float16, device=x.device)
    rc = _lib.lib().dz_embedding_select(x.reshape(-1).contiguous().data_ptr(), indices.contiguous().data_ptr(),
                                        base_weight.data_ptr(), delta_weights.data_ptr(), V * H, S,
                                        out.data_ptr(), T, V, H, H, _stream())
    _lib.check(rc, "dz_embedding_select")
    return out.view(*x.shape, H)


def apply_delta_uncompressed(x: torch.Tensor, delta_weights: torch.Tensor, indices: torch.Tensor,
                             base_embedding: torch.Tensor) -> torch.Tensor:
    """Per-row dense product against the row's own full weight
    (serving/vllm/delta/deltazip_marlin.py:21-53, the lm_head of LogitsProcessorWithDelta):
    out[t] = x[t] @ delta_weights[indices[t]]^T, or x[t] @ base_embedding^T for indices[t] == -1.
    Where the reference loops over torch.unique(indices) on the host, the rows are grouped by id
    and cut into row blocks on the device (dz_segment, dz_build_tiles) and one launch multiplies
    every block by its own table (dz_gemm_f16_select), reading and writing the rows in place
    through the token order: three launches (four where the device picks the block length), nothing
    gathered, scattered or read back to the host, so the call can be captured in a HIP graph."""
    _need_cuda(x, delta_weights, indices, base_embedding)
    if x.dtype != torch.float16 or delta_weights.dtype != torch.float16 or base_embedding.dtype != torch.float16:
        raise ValueError("x and the weights must be float16")
    S, N, K = delta_weights.shape
    T = x.shape[0]
    if x.dim() != 2 or x.shape[1] != K or tuple(base_embedding.shape) != (N, K) or indices.numel() != T:
        raise ValueError("shapes: x [T, K], delta_weights [S, N, K], base_embedding [N, K], indices [T]")
    if not (delta_weights.is_contiguous() and base_embedding.is_contiguous() and x.is_contiguous()):
        raise ValueError("x and the weights must be contiguous")
    # The kernel whose weights go straight into registers is the faster one up to 600 rows, whatever the
    # number of tables (32000 x 4096, 32 / 256 / 600 rows of 8 tables: 421 / 464 / 523 against 368 / 389 /
    # 423 us, of one: 102 / 156 / 286 against 56 / 104 / 244); at 1024 tiles of 256 x 256 are (582 against
    # 691), unless there are too few of them to fill the GPU (4096 x 1024: 46 against 32).
    short = K % 256 == 0 and N % 32 == 0 and (
        T <= 600 or (T <= 1024 and ((N + 255) // 256) * ((T + 255) // 256) <= 64))
    indices = indices.reshape(-1)
    if not indices.is_contiguous():
        raise ValueError("indices must be contiguous")
    L, st = _lib.lib(), _stream()
    perm, seg_off = segment(indices, S)               # (ids without a table take the base table, unreported)
    out = torch.empty((T, N), dtype=torch.float16, device=x.device)
    # A segment of more than 128 rows puts a second, short block over the whole table.  From 225 rows on,
    # where that is likely, and where two, three or four long blocks fill a wave of workgroups by four
    # fifths or more, the device picks them if short ones overflow theirs (256 rows, 32000 x 4096, two
    # tables: long 170, short 203 us; a table and the base table 172 / 204 at 300; one table 168 / 119);
    # the launch that does nothing costs 4 us.
    wide = (N + 255) // 256
    either = short and 224 < T <= 512 and 52 <= wide <= 128 and 256 // wide * wide > 208
    tables = []
    for rows, used in ((256, either or not short), (SHORT_ROWS, short)):
        tables.append(_block_table(T, S, rows, x.device) if used else (None, 0))
    (tiles, n), (few, nf) = tables
    if either:
        _lib.check(L.dz_build_tiles_either_for(seg_off.data_ptr(), S, N, tiles.data_ptr(), n, few.data_ptr(), nf, st),
                   "dz_build_tiles_either_for")
    elif short:
        _lib.check(L.dz_build_tiles_rows(seg_off.data_ptr(), S, SHORT_ROWS, few.data_ptr(), nf, st), "dz_build_tiles_rows")
    else:
        _lib.check(L.dz_build_tiles(seg_off.data_ptr(), S, tiles.data_ptr(), n, st), "dz_build_tiles")
    for table, rows, fn in ((tiles, n, L.dz_gemm_f16_select), (few, nf, L.dz_gemm_f16_select_rows)):
        if table is not None:
            _lib.check(fn(x.data_ptr(), base_embedding.data_ptr(), delta_weights.data_ptr(), N * K, table.data_ptr(), rows,
                          perm.data_ptr(), out.data_ptr(), T, K, N, 0, N, st), "dz_gemm_f16_select")
    return out


_minus_one_ids: Dict[int, torch.Tensor] = {}


def _minus_ones(device) -> torch.Tensor:
    idx = device.index if device.index is not None else torch.cuda.current_device()
    if idx not in _minus_one_ids:
        _minus_one_ids[idx] = torch.full((MAX_TOKENS_FUSED,), -1, dtype=torch.int64, device=device)
    return _minus_one_ids[idx]


def compress_delta(delta: torch.Tensor, bits: int, group_size: int = -1):
    """fp32 delta [N, K] on the GPU -> (qweight, meta, scales) of one slot in the native layout:
    symmetric scales from the un-pruned values, 2:4 magnitude pruning, round-to-nearest codes
    (deltazip/core/quant.py:9-18, 48-130; core/sparsegpt.py:64-66, 123-135 with an identity
    Hessian).  The same bytes as compressing and packing the reference's way and converting with
    `repack_gptq_to_native`."""
    _need_cuda(delta)
    if bits not in (2, 4):
        raise NotImplementedError("Only 2 and 4 bits are supported.")
    if delta.dtype != torch.float32 or delta.dim() != 2 or not delta.is_contiguous():
        raise ValueError("delta must be a contiguous float32 [N, K] tensor")
    N, K = delta.shape
    qs, ms, ss = stacked_shapes(K, N, bits, group_size)
    q = torch.empty(qs, dtype=torch.int32, device=delta.device)
    m = torch.empty(ms, dtype=torch.int16, device=delta.device)
    s = torch.empty(ss, dtype=torch.float16, device=delta.device)
    ws = torch.empty(ss, dtype=torch.float32, device=delta.device)
    rc = _lib.lib().dz_compress_2of4(delta.data_ptr(), K, N, bits, group_size, q.data_ptr(), m.data_ptr(),
                                     s.data_ptr(), ws.data_ptr(), _stream())
    _lib.check(rc, "dz_compress_2of4")
    return q, m, s


def quant_scales(delta: torch.Tensor, bits: int, group_size: int = -1, mse: bool = False, norm: float = 2.4,
                 grid: int = 100, maxshrink: float = 0.8):
    """Symmetric scales of the reference's Quantizer.find_params (deltazip/core/quant.py:48-130,
    perchannel, sym) for an fp32 delta [N, K] on the GPU: (scale32 [G, N] fp32, scale16 [G, N] fp16).
    mse=True runs the reference's search over the clipping range (quant.py:85-101) with its
    `norm`, `grid` and `maxshrink`."""
    _need_cuda(delta)
    if delta.dtype != torch.float32 or delta.dim() != 2 or not delta.is_contiguous():
        raise ValueError("delta must be a contiguous float32 [N, K] tensor")
    N, K = delta.shape
    _, _, ss = stacked_shapes(K, N, bits, group_size)
    s32 = torch.empty(ss, dtype=torch.float32, device=delta.device)
    s16 = torch.empty(ss, dtype=torch.float16, device=delta.device)
    if mse:
        rc = _lib.lib().dz_quant_scales_mse(delta.data_ptr(), K, N, bits, group_size, float(norm), int(grid),
                                            float(maxshrink), s32.data_ptr(), s16.data_ptr(), _stream())
        _lib.check(rc, "dz_quant_scales_mse")
    else:
        rc = _lib.lib().dz_quant_scales(delta.data_ptr(), K, N, bits, group_size, s32.data_ptr(), s16.data_ptr(), _stream())
        _lib.check(rc, "dz_quant_scales")
    return s32, s16


def pack_2of4(w: torch.Tensor, scale32: torch.Tensor, bits: int, group_size: int = -1):
    """(qweight, meta) of one slot in the native layout from fp32 values [N, K] that are 2:4 sparse and
    on the grid of `scale32` [G, N] (what `obs_sweep` leaves behind)."""
    _need_cuda(w, scale32)
    if w.dtype != torch.float32 or w.dim() != 2 or not w.is_contiguous():
        raise ValueError("w must be a contiguous float32 [N, K] tensor")
    N, K = w.shape
    qs, ms, ss = stacked_shapes(K, N, bits, group_size)
    if scale32.dtype != torch.float32 or tuple(scale32.shape) != tuple(ss) or not scale32.is_contiguous():
        raise ValueError("scale32 must be a contiguous float32 [G, N] tensor")
    q = torch.empty(qs, dtype=torch.int32, device=w.device)
    m = torch.empty(ms, dtype=torch.int16, device=w.device)
    rc = _lib.lib().dz_pack_2of4(w.data_ptr(), scale32.data_ptr(), K, N, bits, group_size, q.data_ptr(), m.data_ptr(),
                                 _stream())
    _lib.check(rc, "dz_pack_2of4")
    return q, m


def hessian_add(H: torch.Tensor, x: torch.Tensor, nsamples: int, batch: int) -> int:
    """H <- H * n/(n+b) + (sqrt(2/(n+b)) x)^T (sqrt(2/(n+b)) x) in place for x [T, K] (fp16 or fp32),
    as SparseGPT.add_batch does for a linear layer (deltazip/core/sparsegpt.py:27-40); returns n + b."""
    _need_cuda(H, x)
    K = H.shape[0]
    if H.dtype != torch.float32 or tuple(H.shape) != (K, K) or not H.is_contiguous():
        raise ValueError("H must be a contiguous float32 [K, K] tensor")
    if x.dim() != 2 or x.shape[1] != K or x.dtype not in (torch.float16, torch.float32) or not x.is_contiguous():
        raise ValueError("x must be a contiguous [T, K] float16 or float32 tensor")
    n = nsamples + batch
    rc = _lib.lib().dz_hessian_add(H.data_ptr(), x.data_ptr(), int(x.dtype == torch.float16), x.shape[0], K,
                                   float(nsamples / n), math.sqrt(2.0 / n), _stream())
    _lib.check(rc, "dz_hessian_add")
    return n


def obs_sweep(W: torch.Tensor, hinv_upper: torch.Tensor, scale: Optional[torch.Tensor], bits: int = 4,
              prunen: int = 2, prunem: int = 4) -> torch.Tensor:
    """The column sweep of SparseGPT.fasterprune (deltazip/core/sparsegpt.py:92-146) over W [N, K] fp32
    in place: n:m pruning by w^2 / diag(hinv)^2, rounding to the grid of `scale` [N] (None: no
    rounding), error compensation along the rows of `hinv_upper`.  Returns the per-row losses [N]."""
    _need_cuda(W, hinv_upper, scale)
    N, K = W.shape
    if W.dtype != torch.float32 or not W.is_contiguous():
        raise ValueError("W must be a contiguous float32 [N, K] tensor")
    if hinv_upper.dtype != torch.float32 or tuple(hinv_upper.shape) != (K, K) or not hinv_upper.is_contiguous():
        raise ValueError("hinv_upper must be a contiguous float32 [K, K] tensor")
    if scale is not None and (scale.dtype != torch.float32 or scale.numel() != N or not scale.is_contiguous()):
        raise ValueError("scale must be a contiguous float32 tensor with one entry per row")
    err = torch.empty((2, N, 128), dtype=torch.float32, device=W.device)
    loss = torch.zeros(N, dtype=torch.float32, device=W.device)
    rc = _lib.lib().dz_obs_sweep_ahead(W.data_ptr(), hinv_upper.data_ptr(),
                                       scale.data_ptr() if scale is not None else None, N, K, bits, prunen, prunem,
                                       err.data_ptr(), loss.data_ptr(), _stream())
    _lib.check(rc, "dz_obs_sweep_ahead")
    return loss


def token_order(indices: torch.Tensor, num_slots: int, out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Order in which the fused kernel takes the tokens of a batch of up to 128 tokens (int32 [T]):
    depends on the indices only, so it can be computed once per batch and passed to every layer
    call of the step (`order=`), as the reference converts its mapping once per batch
    (serving/vllm/delta/models.py:421-435)."""
    _need_cuda(indices, out)
    T = indices.numel()
    if indices.dtype != torch.int64 or not indices.is_contiguous():
        raise ValueError("indices must be a contiguous int64 tensor")
    if out is None:
        out = torch.empty(T, dtype=torch.int32, device=indices.device)
    elif out.dtype != torch.int32 or out.numel() < T or not out.is_contiguous():
        raise ValueError("out must be a contiguous int32 tensor with at least T entries")
    _lib.check(_lib.lib().dz_token_order(indices.data_ptr(), T, num_slots, out.data_ptr(), _stream()), "dz_token_order")
    return out[:T]


def map_ids(token_ids: torch.Tensor, prompt_ids: Optional[torch.Tensor], slot_ids: torch.Tensor,
            max_deltas: int, vocab_size: int, extra_vocab_size: int, base_indices: torch.Tensor,
            sampler_indices: Optional[torch.Tensor] = None,
            sampler_indices_padded: Optional[torch.Tensor] = None,
            embeddings_indices: Optional[torch.Tensor] = None,
            n_missing: Optional[torch.Tensor] = None) -> None:
    """Delta ids -> slot indices on the device, written into the given int64 tensors (the index
    tensors of convert_mapping, serving/vllm/delta/models.py:69-145).  token_ids [T], prompt_ids [P]
    or None, slot_ids [S]: int64 on the GPU; the outputs are the manager's persistent buffers
    (at least T resp. P long; embeddings_indices [2, >= T])."""
    _need_cuda(token_ids, prompt_ids, slot_ids, base_indices, sampler_indices, sampler_indices_padded,
               embeddings_indices, n_missing)
    for t in (token_ids, prompt_ids, slot_ids, base_indices, sampler_indices, sampler_indices_padded,
              embeddings_indices):
        if t is not None and t.dtype != torch.int64:
            raise ValueError("id and index tensors must be int64")
    T = token_ids.numel()
    P = 0 if prompt_ids is None else prompt_ids.numel()
    if base_indices.numel() < T or (P and (sampler_indices is None or sampler_indices.numel() < P)):
        raise ValueError("index buffers are shorter than the batch")
    if sampler_indices_padded is not None and sampler_indices_padded.numel() < P:
        raise ValueError("index buffers are shorter than the batch")
    ld = 0
    if embeddings_indices is not None:
        if embeddings_indices.dim() != 2 or embeddings_indices.shape[0] != 2 or embeddings_indices.stride(1) != 1:
            raise ValueError("embeddings_indices must be [2, n] with contiguous rows")
        ld = embeddings_indices.stride(0)
    ptr = lambda t: None if t is None else t.data_ptr()
    rc = _lib.lib().dz_map_ids(token_ids.data_ptr(), T, ptr(prompt_ids), P, slot_ids.data_ptr(),
                               slot_ids.numel(), max_deltas, vocab_size, extra_vocab_size,
                               base_indices.data_ptr(), ptr(sampler_indices), ptr(sampler_indices_padded),
                               ptr(embeddings_indices), ld, ptr(n_missing), _stream())
    _lib.check(rc, "dz_map_ids")


# ---------------------------------------------------------------------------------------------
# workspace: zero-filled once per device, reused by every call on that device
# ---------------------------------------------------------------------------------------------
# one per (device, stream): calls that share a workspace must be ordered on one stream
_workspaces: Dict[Tuple[int, int], torch.Tensor] = {}


WS_HEADER_BYTES = 256          # the status word sits in front of the token order and the partial sums

STATUS_BAD_ID = 1              # a delta id outside [-1, S) was met and treated as -1
STATUS_SUM_MISSING = 2         # a partial sum of a K-slice did not arrive: that call's output is invalid


@lru_cache(maxsize=4096)
def _workspace_bytes(T: int, K: int, N: int) -> int:
    return _lib.lib().dz_workspace_bytes(T, K, N)


def _workspace(device: torch.device, T: int, K: int, N: int) -> torch.Tensor:
    need = _workspace_bytes(T, K, N)
    idx = device.index
    key = (torch.cuda.current_device() if idx is None else idx, _stream())
    ws = _workspaces.get(key)
    if ws is None or ws.numel() < need:
        new = torch.zeros(max(need, 1 << 20), dtype=torch.uint8, device=device)
        if ws is not None:
            # the status word of the buffer that is left behind is carried over (same stream: after
            # the calls that may still set it)
            new[:WS_HEADER_BYTES].copy_(ws[:WS_HEADER_BYTES])
        _workspaces[key] = ws = new
        _status_polls.pop(key, None)
    return ws


def workspace_status(device=None) -> int:
    """Status words of the device's workspaces, OR-ed (bit 0: a delta id outside [-1, S) was seen
    and treated as -1; bit 1: a partial sum did not arrive).  Synchronises; meant for debugging
    and tests -- the serving path uses `poll_status`."""
    idx = torch.cuda.current_device() if device is None else torch.device(device).index
    status = 0
    for (i, _), ws in _workspaces.items():
        if i == idx:
            status |= int(ws[:4].view(torch.int32).item())
    return status


class DeltaKernelError(RuntimeError):
    """A launch of the fused kernel reported that its output is invalid."""


_warned_bad_id = False


def raise_for_status(word: int, where: str = "multi-delta linear") -> None:
    """What a status word means to the caller.  Bit 1 -> DeltaKernelError (a RuntimeError, as every
    failure of the reference's ops is a Python exception); bit 0 -> one warning per process."""
    global _warned_bad_id
    if word & STATUS_SUM_MISSING:
        raise DeltaKernelError(
            f"{where}: a partial sum of a K dimension split over workgroups did not arrive within the kernel's "
            "bounded wait; the outputs of the calls since the last check are invalid (status bit 1). The "
            "workspace has been cleared; repeat the step.")
    if word & STATUS_BAD_ID and not _warned_bad_id:
        _warned_bad_id = True
        import warnings
        warnings.warn(f"{where}: a delta id outside [-1, S) was met and served as -1 (base weight only; status bit 0)",
                      RuntimeWarning, stacklevel=3)


# (device, stream) -> (pinned int32[1], event of the copy that fills it)
_status_polls: Dict[Tuple[int, int], Tuple[torch.Tensor, "torch.cuda.Event"]] = {}


def _clear_workspace(ws: torch.Tensor, word: int) -> None:
    """After a reported failure: empty the partial-sum slots (late slices may have left values in
    them that later calls would take for ready) and drop the reported bits."""
    if word & STATUS_SUM_MISSING:
        ws[WS_HEADER_BYTES:].zero_()
    ws[:4].zero_()


def poll_status(device=None, wait: bool = False) -> None:
    """The serving path's look at the status words, without a synchronisation of its own: every call
    evaluates the copy the previous call started (if it has completed, or after waiting for it when
    `wait` is set) and starts the next one, a 4-byte device-to-host copy into pinned memory on the
    workspace's stream.  Raises DeltaKernelError / warns as `raise_for_status` says; a reported
    failure also clears the workspace.  With `wait` the current state is read as well (this
    synchronises with the workspace's stream)."""
    if not _workspaces:
        return                                        # no fused call has run yet (or no GPU at all)
    idx = None if device is None else torch.device(device).index
    if idx is None:
        idx = torch.cuda.current_device()
    found = 0
    for key, ws in list(_workspaces.items()):
        if key[0] != idx:
            continue
        stream = torch.cuda.ExternalStream(key[1], device=ws.device) if key[1] else torch.cuda.default_stream(ws.device)
        pending = _status_polls.pop(key, None)
        host = pending[0] if pending is not None else torch.zeros(1, dtype=torch.int32, pin_memory=True)
        word = 0
        if pending is not None:
            if wait:
                pending[1].synchronize()
            if pending[1].query():
                word = int(host[0])
            else:
                _status_polls[key] = pending          # not in yet: looked at by the next call
                continue
        with torch.cuda.stream(stream):
            if wait:
                # the state as of now, too
                host.copy_(ws[:4].view(torch.int32), non_blocking=True)
                stream.synchronize()
                word |= int(host[0])
            if word:
                _clear_workspace(ws, word)            # before the next copy is started
            if not wait:
                ev = torch.cuda.Event()
                host.copy_(ws[:4].view(torch.int32), non_blocking=True)
                ev.record()
                _status_polls[key] = (host, ev)
        found |= word
    if found:
        raise_for_status(found)


# ---------------------------------------------------------------------------------------------
# the ops
# ---------------------------------------------------------------------------------------------


def _infer(qweight_stacked, scales_stacked, N: int):
    """(K, bits, group_size, S) from the stacked tensors' shapes."""
    S = qweight_stacked.shape[0]
    words = qweight_stacked[0].numel()
    G = scales_stacked[0].numel() // N
    return S, words, G


def tile_base(weight: torch.Tensor) -> torch.Tensor:
    """The base weight [N, K] in the tiled form the fused kernel streams fastest (`dz_tile_base`):
    a tensor of the same shape and dtype whose bytes are the tiles.  A layer converts its base
    weight once and hands it to `multi_delta_linear` / `apply_delta_batch` (`base_tiled=`); calls of
    every size read the tiles when they are given."""
    _need_cuda(weight)
    if weight.dtype != torch.float16 or weight.dim() != 2 or not weight.is_contiguous():
        raise ValueError("weight must be a contiguous float16 [N, K] tensor")
    N, K = weight.shape
    out = torch.empty_like(weight)
    _lib.check(_lib.lib().dz_tile_base(weight.data_ptr(), K, N, out.data_ptr(), _stream()), "dz_tile_base")
    return out


def untile_base(tiled: torch.Tensor) -> torch.Tensor:
    """Inverse of `tile_base`: the row-major [N, K] weight from its tiles (plain tensor ops; not on
    any hot path).  Tile (np, kb) holds fragments (s, j, h); position 16*g + i of a fragment holds
    W[32*np + 16*s + i][256*kb + 64*j + 16*g + 8*h + e], e = 0..7."""
    if tiled.dtype != torch.float16 or tiled.dim() != 2 or not tiled.is_contiguous():
        raise ValueError("tiled must be a contiguous float16 [N, K] tensor")
    N, K = tiled.shape
    if N % 32 or K % 256:
        raise ValueError("N must be a multiple of 32 and K of 256")
    t = tiled.view(N // 32, K // 256, 2, 4, 2, 4, 16, 8)          # np kb s j h g i e
    return t.permute(0, 2, 6, 1, 3, 5, 4, 7).reshape(N, K).contiguous()   # np s i | kb j g h e


def _check_tiled(base_tiled, base_weight, N: int, K: int, device) -> None:
    if base_tiled.shape != (N, K) or base_tiled.dtype != torch.float16 \
            or not base_tiled.is_contiguous() or base_tiled.device != device \
            or (base_weight is not None and base_weight.numel() and base_tiled.shape != base_weight.shape):
        raise ValueError("base_tiled must be tile_base(base_weight): float16 [N, K], contiguous, on x's device")


def takes_fused_chunks(T: int, S: int) -> bool:
    """Whether a batch above the fused kernel's 128 tokens may go through it in chunks of 128: sizes at
    which that can be faster than row blocks (`_route_us`; always where there are more than 768
    slots, which `segment` cannot order)."""
    return T <= 3 * MAX_TOKENS_FUSED or (T <= 4 * MAX_TOKENS_FUSED and S >= 16)


@lru_cache(maxsize=4096)
def _most_blocks_unknown(T: int, K: int, N: int, bits: int, S: int) -> Optional[int]:
    """`_most_row_blocks` where only the device knows the mix.  Over wide layers all slots in use favour
    the chunks, a few prompts of some 64 tokens the row blocks (5120 x 27648, 2-bit, 129 tokens of 64 slots: 557
    against 1103 us and 251 against 135; 256 tokens of 32: 534 / 728 and 392 / 196).  Where that differs, and
    by more than the 8 to 15 us that launching both costs, the device takes the row blocks up to the
    number with which they are the faster route; it does not look at their lengths, so they count as
    full.  Otherwise the route that loses less between the two."""
    def costs(deltas, longest=None):
        mix = _even_mix(T, deltas)
        return _route_us(T, K, N, bits, mix if longest is None else mix._replace(longest=longest, blocks=deltas))
    many, few = costs(S), costs(min(S, 1 + T // 64), SHORT_ROWS)
    if few[0] < few[1] or many[1] - many[0] < 30:
        return 0 if many[0] * few[0] < many[1] * few[1] else None
    lo, hi = -(-T // SHORT_ROWS), min(S, T)
    while lo < hi:
        mid = (lo + hi + 1) // 2
        chunks, rows = costs(mid, SHORT_ROWS)
        lo, hi = (mid, hi) if rows <= chunks else (lo, mid - 1)
    return lo


def _most_row_blocks(T: int, K: int, N: int, bits: int, S: int, blocks: Optional[RowBlocks]) -> Optional[int]:
    """The faster route: None stands for row blocks, 0 for chunks, a number for the row blocks if there
    are no more of them, by the device's count.  A caller that has the ids on the host says so with
    order=row_blocks(..., mix=batch_mix(ids)); its row blocks without a mix are taken as they are."""
    if not takes_fused_chunks(T, S):
        return None
    if S > MAX_SLOTS_SEGMENT:
        return 0
    if blocks is not None:
        return 0 if blocks.mix is not None and _in_chunks(_route_us(T, K, N, bits, blocks.mix)) else None
    return _most_blocks_unknown(T, K, N, bits, S)


def multi_delta_linear(x: torch.Tensor, base_weight: Optional[torch.Tensor], qweight_stacked,
                       scales_stacked, meta_stacked, indices: torch.Tensor, *, bits: int,
                       out: Optional[torch.Tensor] = None, accumulate: bool = False,
                       order: Optional[torch.Tensor] = None,
                       base_tiled: Optional[torch.Tensor] = None) -> torch.Tensor:
    """y = x @ W_base^T + x @ dequant(delta[indices])^T.  `out` may be a column slice of a wider
    tensor (last-dim stride 1); with accumulate=True the result is added to it.  `order`: what the
    caller already has for this batch -- the result of `token_order(indices, S)` (up to 128
    tokens) or of `row_blocks(indices, S)` (more).
    `base_tiled`: `tile_base(base_weight)`, read instead of the row-major weight (the results are
    the same bit for bit); base_weight may then be None -- a layer that keeps only the tiled copy.
    The order of the fp32 sums goes by the sizes, and at 129 to 512 tokens also by the ids of the batch: the other tokens'
    deltas set the number of blocks, and that the parts K is cut into, also when a graph is replayed over other ids."""
    _need_cuda(x, base_weight, qweight_stacked, scales_stacked, meta_stacked, indices)
    if x.dtype != torch.float16:
        raise ValueError("x must be float16")
    if indices.dtype != torch.int64:
        raise ValueError("indices must be int64")
    if bits not in (2, 4):
        raise NotImplementedError("Only 2 and 4 bits are supported.")
    x2 = x if x.dim() == 2 else x.reshape(-1, x.shape[-1])
    if not x2.is_contiguous():
        x2 = x2.contiguous()
    T, K = x2.shape
    if indices.dim() != 1:
        indices = indices.reshape(-1)
    if indices.shape[0] != T or not indices.is_contiguous():
        raise ValueError("indices must be a contiguous vector with one entry per token")
    S = qweight_stacked.shape[0]
    N = scales_stacked.shape[-1]
    device = x.device
    if base_tiled is not None:
        _check_tiled(base_tiled, base_weight, N, K, device)
        if base_weight is not None and base_weight.numel() == 0:
            base_weight = None
    if base_weight is not None:
        if base_weight.dtype != torch.float16 or base_weight.shape != (N, K) or not base_weight.is_contiguous():
            raise ValueError("base_weight must be a contiguous float16 [N, K] tensor")
    G = _slot_numel(scales_stacked) // N
    group_size = -1 if G == 1 else K // G
    cb, mb, _ = _sizes(K, N, bits, group_size)
    if (_slot_numel(qweight_stacked) * qweight_stacked.element_size() != cb
            or _slot_numel(meta_stacked) * meta_stacked.element_size() != mb
            or not qweight_stacked.is_contiguous() or not meta_stacked.is_contiguous()
            or not scales_stacked.is_contiguous() or scales_stacked.dtype != torch.float16):
        raise ValueError("stacked delta tensors do not match the native layout for these sizes")
    if out is None:
        if accumulate:
            raise ValueError("accumulate needs an output tensor")
        out = torch.empty((T, N), dtype=torch.float16, device=device)
        ldy = N
    else:
        if out.dtype != torch.float16 or out.dim() != 2 or out.shape != (T, N) or out.stride(1) != 1:
            raise ValueError("out must be float16 [T, N] with unit column stride")
        ldy = out.stride(0)
    if T > MAX_TOKENS_FUSED:
        blocks = _usable_blocks(order, T, S)
        plan = None
        if ((base_weight is not None or base_tiled is not None)
                and (not _short_chunks(T, K, N, bits, S) if blocks is None else blocks.mixed is not None)):
            plan = _in_mixed_blocks(T, K, N, S, blocks.mix if blocks is not None else None)
        if plan is not None:
            return prefill.multi_delta_linear_mixed(x2, base_weight, qweight_stacked, scales_stacked, meta_stacked, indices,
                                                    bits=bits, out=out, accumulate=accumulate, blocks=blocks,
                                                    plan=(plan[0], *_parts_of_blocks(
                                                        T, K, N, S, plan, 2 if plan[0] else mixed_deltas(bits, G > 1))),
                                                    base_tiled=base_tiled)
        most = _most_row_blocks(T, K, N, bits, S, blocks)
        if most is not None:
            ws = _workspace(device, MAX_TOKENS_FUSED, K, N)
            w, tiled = (base_tiled, 1) if base_tiled is not None else (base_weight, 0)
            delta = (qweight_stacked.data_ptr(), meta_stacked.data_ptr(), scales_stacked.data_ptr())
            shape = (T, K, N, 1 if accumulate else 0, ldy)
            wptr, over, L, st = w.data_ptr() if w is not None else None, None, _lib.lib(), _stream()
            if most:                                  # the row blocks if there are few, else the chunks
                perm, seg_off = segment(indices, S, True)
                table = torch.empty(4 * most + 1, dtype=torch.int32, device=device)
                over = table[4 * most:].data_ptr()
                _lib.check(L.dz_build_tiles_rows_upto(seg_off.data_ptr(), S, SHORT_ROWS, most, table.data_ptr(), most,
                                                      over, st), "dz_build_tiles_rows_upto")
                _lib.check(L.dz_multi_delta_gemm_rows(x2.data_ptr(), wptr, tiled, *delta, S, bits, group_size,
                                                      table.data_ptr(), most, perm.data_ptr(), out.data_ptr(), *shape, st),
                           "dz_multi_delta_gemm_rows")
            _lib.check(L.dz_multi_delta_linear_chunks(x2.data_ptr(), wptr, tiled, *delta, indices.data_ptr(),
                                                      out.data_ptr(), T, K, N, S, bits, group_size, *shape[3:], over,
                                                      ws.data_ptr(), ws.numel(), st), "dz_multi_delta_linear_chunks")
            return out
        return prefill.multi_delta_linear_prefill(x2, base_weight, qweight_stacked, scales_stacked, meta_stacked,
                                                  indices, bits=bits, out=out, accumulate=accumulate, blocks=blocks,
                                                  base_tiled=base_tiled)
    blocks, met = None, T
    if isinstance(order, RowBlocks):
        if (order.order is not None and order.T == T and order.S == S and order.mix is not None
                and order.captured == torch.cuda.is_current_stream_capturing()):
            blocks, met = order, order.mix.deltas
    elif order is None and T > 64 and S <= 4 and K * N >= 40 << 20:
        # A call that has to make its own table takes 8 us for it: large layers over few slots only (5120 x 13824, 100
        # tokens of 4 slots 104 -> 70 us; 4096 x 12288, 4-bit, 128 tokens of 8 106 / 111).
        met = S
    if (met < T and (base_weight is not None or base_tiled is not None) and 0 < S <= MAX_SLOTS_SEGMENT
            and mixes_at_decode(T, K, N, met)):
        parts = _decode_plan(T, K, N, met)[1]
        return prefill.multi_delta_linear_mixed(x2, base_weight, qweight_stacked, scales_stacked, meta_stacked, indices,
                                                bits=bits, out=out, accumulate=accumulate,
                                                plan=(0, parts, parts), blocks=blocks, base_tiled=base_tiled)
    ws = _workspace(device, T, K, N)
    w, tiled = (base_tiled, 1) if base_tiled is not None else (base_weight, 0)
    rc = _lib.lib().dz_multi_delta_linear_ordered(
        x2.data_ptr(), w.data_ptr() if w is not None else None, tiled, qweight_stacked.data_ptr(), meta_stacked.data_ptr(),
        scales_stacked.data_ptr(), indices.data_ptr(), out.data_ptr(), T, K, N, S, bits, group_size, 1 if accumulate else 0,
        ldy, _order_ptr(order, T, device), ws.data_ptr(), ws.numel(), _stream())
    _lib.check(rc, "dz_multi_delta_linear")
    return out


def _bits_from_shapes(qweight_stacked: torch.Tensor, K: int, N: int) -> int:
    words = _slot_numel(qweight_stacked)
    bits = words * 64 // (K * N)  # words = K*N*bits/64
    if bits not in (2, 4) or words * 64 != K * N * bits:
        raise ValueError("cannot infer the bit width from qweight_stacked")
    return bits


def apply_delta(x: torch.Tensor, qweight_stacked: torch.Tensor, scales_stacked: torch.Tensor,
                meta_stacked: torch.Tensor, indices: torch.Tensor, base_weight: torch.Tensor,
                order: Optional[torch.Tensor] = None, base_tiled: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Drop-in for serving/vllm/delta/deltazip_marlin.py:10-19.  Returns a new [T, N] tensor;
    indices == -1 selects the base weight only.  (`order`: optional, see `token_order`; `base_tiled`:
    optional, see `tile_base`.)"""
    N, K = base_tiled.shape if base_tiled is not None else base_weight.shape
    bits = _bits_from_shapes(qweight_stacked, K, N)
    y = multi_delta_linear(x, base_weight, qweight_stacked, scales_stacked, meta_stacked, indices, bits=bits,
                           order=order, base_tiled=base_tiled)
    return y if x.dim() == 2 else y.view(*x.shape[:-1], N)


def _order_ptr(order: Optional[torch.Tensor], T: int, device) -> Optional[int]:
    if isinstance(order, RowBlocks):
        if order.order is None or order.T != T:
            raise ValueError("row blocks are for batches above %d tokens; pass token_order() here" % MAX_TOKENS_FUSED)
        # (a captured call makes its own from the indices, as it makes its own row blocks)
        order = order.order if order.captured == torch.cuda.is_current_stream_capturing() else None
    if order is None or T <= 32:
        return None
    if (not order.is_cuda or order.device != device or order.dtype != torch.int32 or order.numel() < T
            or not order.is_contiguous()):
        raise ValueError("order must be a contiguous int32 GPU tensor with one entry per token")
    return order.data_ptr()


def apply_delta_batch(x, qweight_stacked: Sequence[torch.Tensor], scales_stacked: Sequence[torch.Tensor],
                      meta_stacked: Sequence[torch.Tensor], indices: torch.Tensor,
                      base_weight: Sequence[torch.Tensor], order: Optional[torch.Tensor] = None,
                      base_tiled: Optional[Sequence[torch.Tensor]] = None):
    """`apply_delta` for up to 4 projections that share the tokens -- q/k/v or gate/up held as
    separate weights, which the reference fuses into one layer
    (serving/vllm/delta/layers_marlin.py:281-487) -- in one launch.  `x` is one [T, K] tensor for
    all or a sequence with one per projection; `order` is what `token_order(indices, S)` returned
    for this batch, if the caller has it; returns the list of [T, N_j] outputs."""
    n = len(base_weight)
    xs = [x] * n if isinstance(x, torch.Tensor) else list(x)
    if not (len(xs) == len(qweight_stacked) == len(scales_stacked) == len(meta_stacked) == n) or not 1 <= n <= 4:
        raise ValueError("one x / qweight / scales / meta / base weight per projection, at most 4 projections")
    K = base_weight[0].shape[1]
    if any(v.shape[-1:] != (w.shape[1],) for v, w in zip(xs, base_weight)):
        raise ValueError("x must be [.., K], as wide as the base weight")
    T = xs[0].shape[0] if xs[0].dim() == 2 else xs[0].reshape(-1, K).shape[0]
    bits = _bits_from_shapes(qweight_stacked[0], K, base_weight[0].shape[0])
    G = _slot_numel(scales_stacked[0]) // base_weight[0].shape[0]
    S = qweight_stacked[0].shape[0]
    if T > MAX_TOKENS_FUSED:
        blocks = order if isinstance(order, RowBlocks) else None
        # row blocks made once serve the projections that would make the same ones
        shared = [q.shape[0] == S and (blocks is not None or (
                      _in_mixed_blocks(T, K, w.shape[0], S, None) is not None and not _short_chunks(T, K, w.shape[0], bits, S))
                      or _most_row_blocks(T, K, w.shape[0], bits, S, None) is None)
                  for q, w in zip(qweight_stacked, base_weight)]
        if blocks is None and sum(shared) > 1 and S <= MAX_SLOTS_SEGMENT and indices.is_cuda \
                and indices.dtype == torch.int64 and indices.numel() == T and indices.is_contiguous():
            blocks = row_blocks(indices, S, features=max(w.shape[0] for w in base_weight), deltas=mixed_deltas(bits, G > 1))
        if blocks is not None and (blocks.T != T or blocks.S != S):
            blocks = None
        return [apply_delta(xs[j], qweight_stacked[j], scales_stacked[j], meta_stacked[j], indices, base_weight[j],
                            order=blocks if shared[j] else None,
                            base_tiled=None if base_tiled is None else base_tiled[j])
                for j in range(n)]
    _need_cuda(indices, *xs, *qweight_stacked, *scales_stacked, *meta_stacked, *base_weight)
    if indices.dtype != torch.int64 or indices.numel() != T or not indices.is_contiguous():
        raise ValueError("indices must be a contiguous int64 tensor with one entry per token")
    group_size = -1 if G == 1 else K // G
    x2s, outs, Ns = [], [], []
    for j in range(n):
        N = base_weight[j].shape[0]
        x2 = xs[j] if xs[j].dim() == 2 else xs[j].reshape(-1, K)
        if (x2.dtype != torch.float16 or base_weight[j].dtype != torch.float16 or base_weight[j].shape[1] != K
                or x2.shape[0] != T or not x2.is_contiguous() or not base_weight[j].is_contiguous()):
            raise ValueError("x and base weights must be contiguous float16 with the same K and T")
        q, m, sc = qweight_stacked[j], meta_stacked[j], scales_stacked[j]
        if (q.shape[0] != S or _slot_bytes_differ(q, m, sc, _sizes(K, N, bits, group_size)) or sc.dtype != torch.float16
                or not (q.is_contiguous() and m.is_contiguous() and sc.is_contiguous())):
            raise ValueError("stacked delta tensors do not match the native layout for these sizes")
        x2s.append(x2); Ns.append(N)
        outs.append(torch.empty((T, N), dtype=torch.float16, device=x2.device))
    vp = C.c_void_p * n
    ptrs = lambda ts: vp(*[t.data_ptr() for t in ts])
    ws = _workspace(x2s[0].device, T, K, sum(Ns))
    entry, bases = _lib.lib().dz_multi_delta_linear_batch, base_weight
    if base_tiled is not None:
        if len(base_tiled) != n:
            raise ValueError("one tiled base weight per projection")
        for j in range(n):
            _check_tiled(base_tiled[j], base_weight[j], Ns[j], K, x2s[j].device)
        entry, bases = _lib.lib().dz_multi_delta_linear_batch_tiled, base_tiled
    rc = entry(
        n, ptrs(x2s), ptrs(bases), ptrs(qweight_stacked), ptrs(meta_stacked), ptrs(scales_stacked),
        indices.data_ptr(), ptrs(outs), (C.c_int * n)(*Ns), (C.c_int * n)(*Ns), T, K, S, bits, group_size, 0,
        _order_ptr(order, T, indices.device), ws.data_ptr(), ws.numel(), _stream())
    _lib.check(rc, "dz_multi_delta_linear_batch")
    return [y if v.dim() == 2 else y.view(*v.shape[:-1], y.shape[1]) for y, v in zip(outs, xs)]


def add_delta(y: torch.Tensor, x: torch.Tensor, qweight: torch.Tensor, qzeros, scales: torch.Tensor,
              g_idx, indices: torch.Tensor, meta: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Drop-in for serving/vllm/delta/deltazip.py:14-37: y[i] += x[i] @ dequant(W[indices[i]])^T,
    in place.  `qzeros` and `g_idx` are accepted for signature compatibility and unused: the native
    layout is symmetric with g_idx = k // group_size (checked when the delta was repacked)."""
    if meta is None:
        raise ValueError("meta (2:4 positions) is required")
    K = x.shape[-1]
    N = scales.shape[-1]
    bits = _bits_from_shapes(qweight, K, N)
    y2 = y.view(-1, y.shape[-1])
    multi_delta_linear(x, None, qweight, scales, meta, indices, bits=bits, out=y2, accumulate=True)
    return y


def add_delta_slice(y: torch.Tensor, x: torch.Tensor, qweight, qzeros, scales, g_idx, indices,
                    scale: float, y_offset: int, y_slice_size: int, *, buffer=None,
                    meta: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Drop-in for serving/vllm/delta/deltazip.py:40-77: as add_delta, into the column slice
    y[:, y_offset : y_offset + y_slice_size].  `scale` is ignored, as it is by the reference."""
    if meta is None:
        raise ValueError("meta (2:4 positions) is required")
    K = x.shape[-1]
    N = scales.shape[-1]
    if N != y_slice_size:
        raise ValueError("y_slice_size must equal the delta's output features")
    bits = _bits_from_shapes(qweight, K, N)
    y2 = y.view(-1, y.shape[-1])[:, y_offset:y_offset + y_slice_size]
    multi_delta_linear(x, None, qweight, scales, meta, indices, bits=bits, out=y2, accumulate=True)
    return y


def apply_delta_into(x: torch.Tensor, qweight_stacked: torch.Tensor, qzeros_stacked, scales_stacked: torch.Tensor,
                     g_idx_stacked, indices: torch.Tensor, output: torch.Tensor, *,
                     meta_stacked: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Drop-in for the in-place, seven-argument apply_delta of serving/vllm/delta/deltazip.py:78-100:
    output[i] += x[i] @ dequant(W[indices[i]])^T for all leading dimensions flattened, returned with
    output's shape.  `meta_stacked` carries the 2:4 positions of the native layout (the reference's
    add_delta takes them as `meta`, deltazip.py:22); `qzeros_stacked` / `g_idx_stacked` are unused, as
    in `add_delta`."""
    x2 = x.view(-1, x.shape[-1])
    out2 = output.view(-1, output.shape[-1])
    add_delta(out2, x2, qweight_stacked, qzeros_stacked, scales_stacked, g_idx_stacked, indices.view(-1),
              meta=meta_stacked)
    return out2.view_as(output)


def apply_delta_packed_nslice(x: torch.Tensor, qweight_stacked: Sequence[torch.Tensor], qzeros_stacked,
                              scales_stacked: Sequence[torch.Tensor], g_idx_stacked, indices: torch.Tensor,
                              output: torch.Tensor, output_slices: Sequence[int], *,
                              meta_stacked: Optional[Sequence[torch.Tensor]] = None,
                              order: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Drop-in for serving/vllm/delta/deltazip.py:103-153: a layer made of several sublayers packed
    side by side (q/k/v, gate/up).  For slice j with n_j = output_slices[j] output features,
    output[:, off_j : off_j + n_j] += x @ dequant(W_j[indices])^T, off_j the sum of the slices before
    it; index -1 adds nothing.  Up to 128 tokens and 4 slices go in one launch (every slice a call
    of dz_multi_delta_linear_batch that adds into its columns of `output`); larger batches take one
    add_delta_slice per slice like the reference.  `meta_stacked[j]`: 2:4 positions of slice j."""
    n = len(output_slices)
    if meta_stacked is None:
        raise ValueError("meta_stacked (2:4 positions of every slice) is required")
    if not (len(qweight_stacked) >= n and len(scales_stacked) >= n and len(meta_stacked) >= n):
        raise ValueError("one qweight / scales / meta per output slice is required")
    K = x.shape[-1]
    x2 = x.view(-1, K)
    ind = indices.view(-1)
    out2 = output.view(-1, output.shape[-1])
    T = x2.shape[0]
    if sum(output_slices) > out2.shape[1]:
        raise ValueError("output_slices exceed the width of output")
    Ns = [int(v) for v in output_slices]
    offs = [sum(Ns[:j]) for j in range(n)]
    fits = (1 <= n <= 4 and T <= MAX_TOKENS_FUSED and out2.dtype == torch.float16 and out2.stride(1) == 1
            and out2.stride(0) % 4 == 0 and all(o % 4 == 0 for o in offs))
    if not fits:
        for j in range(n):
            add_delta_slice(out2, x2, qweight_stacked[j], None, scales_stacked[j], None, ind, 1.0, offs[j], Ns[j],
                            meta=meta_stacked[j])
        return out2.view_as(output)
    _need_cuda(x2, ind, out2, *qweight_stacked[:n], *scales_stacked[:n], *meta_stacked[:n])
    if x2.dtype != torch.float16 or not x2.is_contiguous():
        raise ValueError("x must be contiguous float16")
    if ind.dtype != torch.int64 or ind.numel() != T or not ind.is_contiguous():
        raise ValueError("indices must be a contiguous int64 tensor with one entry per token")
    if out2.shape[0] != T:
        raise ValueError("output must have one row per token")
    bits = _bits_from_shapes(qweight_stacked[0], K, Ns[0])
    S = qweight_stacked[0].shape[0]
    G = _slot_numel(scales_stacked[0]) // Ns[0]
    group_size = -1 if G == 1 else K // G
    for j in range(n):
        q, m, sc = qweight_stacked[j], meta_stacked[j], scales_stacked[j]
        if (q.shape[0] != S or _slot_bytes_differ(q, m, sc, _sizes(K, Ns[j], bits, group_size)) or sc.dtype != torch.float16
                or not (q.is_contiguous() and m.is_contiguous() and sc.is_contiguous())):
            raise ValueError("stacked delta tensors do not match the native layout for these sizes")
    vp = C.c_void_p * n
    esz = out2.element_size()
    ws = _workspace(x2.device, T, K, sum(Ns))
    rc = _lib.lib().dz_multi_delta_linear_batch(
        n, vp(*[x2.data_ptr()] * n), vp(*[None] * n), vp(*[qweight_stacked[j].data_ptr() for j in range(n)]),
        vp(*[meta_stacked[j].data_ptr() for j in range(n)]), vp(*[scales_stacked[j].data_ptr() for j in range(n)]),
        ind.data_ptr(), vp(*[out2.data_ptr() + offs[j] * esz for j in range(n)]), (C.c_int * n)(*Ns),
        (C.c_int * n)(*[out2.stride(0)] * n), T, K, S, bits, group_size, 1, _order_ptr(order, T, ind.device),
        ws.data_ptr(), ws.numel(), _stream())
    _lib.check(rc, "dz_multi_delta_linear_batch")
    return out2.view_as(output)


def set_ksplit(nsplit: int) -> None:
    """Benchmark hook: force the number of K chunks of the fused kernel (0 = automatic)."""
    _lib.lib().dz_set_ksplit(int(nsplit))


from . import prefill  # noqa: E402  (which reads this module when it is called)

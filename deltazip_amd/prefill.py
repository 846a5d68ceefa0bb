"""Prefill-sized calls (T > 128) on the matrix cores.

The reference's exllama backend switches, above 50 rows, to "reconstruct the weight, then a dense
half-precision GEMM" (serving/csrc/quantization/deltazip/exllama/cuda/q_gemm.cu:118-137).  Here
the delta is never reconstructed in memory: dz_multi_delta_gemm multiplies the base weight on the
dense matrix-core instructions and each token block's delta, straight from its packed form, on
the 2:4-sparse ones, into the same fp32 accumulators (base and delta are not summed in fp16
first, which would cost about 5e-5 of the output range in absolute error).
"""
from __future__ import annotations

from typing import Optional

import torch

from . import _lib, ops


def gemm_f16(x: torch.Tensor, w: torch.Tensor, out: Optional[torch.Tensor] = None,
             accumulate: bool = False, w2: Optional[torch.Tensor] = None) -> torch.Tensor:
    """out[T, N] (+)= x[T, K] @ w[N, K]^T (+ x @ w2^T) on the matrix cores."""
    T, K = x.shape
    N = w.shape[0]
    if out is None:
        out = torch.empty((T, N), dtype=torch.float16, device=x.device)
    st = ops._stream()
    if w2 is None:
        rc = _lib.lib().dz_gemm_f16(x.data_ptr(), w.data_ptr(), out.data_ptr(), T, K, N,
                                    1 if accumulate else 0, out.stride(0), st)
    else:
        rc = _lib.lib().dz_gemm_f16_pair(x.data_ptr(), w.data_ptr(), w2.data_ptr(), out.data_ptr(), T, K, N,
                                         1 if accumulate else 0, out.stride(0), st)
    _lib.check(rc, "dz_gemm_f16")
    return out


def multi_delta_linear_prefill(x2, base_weight, qweight_stacked, scales_stacked, meta_stacked, indices,
                               *, bits: int, out: torch.Tensor, accumulate: bool, blocks=None,
                               base_tiled=None) -> torch.Tensor:
    """T > 128: tokens are ordered by delta id on the device (dz_segment), the order is cut into
    row blocks of one delta each (ops.row_blocks) and dz_multi_delta_gemm or dz_multi_delta_gemm_rows multiplies
    every block by the base weight and by its delta in packed form.  Nothing is read back to the
    host, gathered, scattered or dequantised to memory.  `blocks`: ops.row_blocks(indices, S) when
    the caller made it once for the batch (else made here, per call).  `base_tiled`: the base weight
    in tiles (ops.tile_base), read instead of base_weight when given."""
    T, K = x2.shape
    N = scales_stacked.shape[-1]
    S = qweight_stacked.shape[0]
    G = ops._slot_numel(scales_stacked) // N
    group_size = -1 if G == 1 else K // G
    # the kernel addresses an operand with 31-bit byte offsets: very long batches go in pieces
    max_rows = ((1 << 31) - 1) // (2 * K)
    if T > max_rows:
        step = max(256, max_rows // 256 * 256)
        for r in range(0, T, step):
            multi_delta_linear_prefill(x2[r:r + step], base_weight, qweight_stacked, scales_stacked, meta_stacked,
                                       indices[r:r + step].contiguous(), bits=bits, out=out[r:r + step],
                                       accumulate=accumulate, base_tiled=base_tiled)
        return out
    lib = _lib.lib()
    stream = ops._stream()
    one_wave = ops._one_wave_of_long_blocks(T, N, bits)
    if blocks is None:
        blocks = ops.row_blocks(indices, S, device_picks=S == 1 and one_wave, features=N, mixed=False)
    take_long, take_short = blocks.tiles is not None, blocks.short is not None
    if blocks.host_picks:
        take_long, take_short = one_wave, not one_wave
    if not (take_long or take_short):
        raise ValueError("these row blocks hold no blocks of one delta")
    row_major = base_weight.data_ptr() if base_weight is not None else None
    if take_long:
        fn, wptr = lib.dz_multi_delta_gemm, row_major
        if base_tiled is not None:
            fn, wptr = lib.dz_multi_delta_gemm_tiled, base_tiled.data_ptr()
        rc = fn(x2.data_ptr(), wptr, qweight_stacked.data_ptr(), meta_stacked.data_ptr(), scales_stacked.data_ptr(),
                S, bits, group_size, blocks.tiles.data_ptr(), blocks.max_tiles, blocks.perm.data_ptr(),
                out.data_ptr(), T, K, N, 1 if accumulate else 0, out.stride(0), stream)
        _lib.check(rc, "dz_multi_delta_gemm")
    if take_short:
        rc = lib.dz_multi_delta_gemm_rows(
            x2.data_ptr(), base_tiled.data_ptr() if base_tiled is not None else row_major,
            1 if base_tiled is not None else 0, qweight_stacked.data_ptr(), meta_stacked.data_ptr(),
            scales_stacked.data_ptr(), S, bits, group_size, blocks.short.data_ptr(), blocks.max_short,
            blocks.perm.data_ptr(), out.data_ptr(), T, K, N, 1 if accumulate else 0, out.stride(0), stream)
        _lib.check(rc, "dz_multi_delta_gemm_rows")
    return out


def multi_delta_linear_mixed(x2, base_weight, qweight_stacked, scales_stacked, meta_stacked, indices, *, bits: int,
                             out: torch.Tensor, accumulate: bool, plan, blocks=None, base_tiled=None) -> torch.Tensor:
    """The layer over blocks that hold the tokens of several deltas (dz_multi_delta_gemm_mixed), with a base weight.
    `plan`: (0 for full blocks, 1 for small ones; parts of K, or less than 0 where the device may take others; the most there can be).  `blocks`: as for multi_delta_linear_prefill; without them, or where they
    were made for more deltas than this layer's block can hold, the call makes the table it needs."""
    small, parts, most = plan
    T, K = x2.shape
    N, S = scales_stacked.shape[-1], qweight_stacked.shape[0]
    G = ops._slot_numel(scales_stacked) // N
    L, stream = _lib.lib(), ops._stream()
    deltas = ops.mixed_deltas(bits, G > 1)
    table = blocks.mixed[small] if blocks is not None else None
    if table is None or table.deltas > deltas:
        table = ops.own_mixed_table(indices, S, small, deltas)
    sums = torch.empty(most * T * N, dtype=torch.float32, device=x2.device) if most > 1 else None
    w = base_tiled if base_tiled is not None else base_weight
    rc = L.dz_multi_delta_gemm_mixed(
        x2.data_ptr(), w.data_ptr(), 1 if base_tiled is not None else 0, qweight_stacked.data_ptr(),
        meta_stacked.data_ptr(), scales_stacked.data_ptr(), S, bits, -1 if G == 1 else K // G, table.table.data_ptr(),
        table.max_blocks, table.deltas, out.data_ptr(), T, K, N, 1 if accumulate else 0, out.stride(0), parts,
        sums.data_ptr() if sums is not None else None, stream)
    _lib.check(rc, "dz_multi_delta_gemm_mixed")
    return out

"""GPU parity tests: every entry point is called through the C ABI (via the ctypes wrapper) and
compared with the CPU oracle on the same seeded inputs.  Dequantised deltas must match bit for
bit; layer outputs within TOL = 1e-2 max relative error (fp16 outputs vs the fp32 reference)."""
import glob
import os

import numpy as np
import pytest
import torch

from oracle import dz_oracle as o
from deltazip_amd import ops
from _util import TOL, make_problem, run_layer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits", [2, 4])
@pytest.mark.parametrize("gs", [-1, 64, 128, 256])
def test_dequant_bit_exact(dev, bits, gs):
    p = make_problem(96, 768, bits, gs, 2, 1, "single", 100 + bits + max(gs, 0), dev)
    for d in range(2):
        got = ops.dequant(p["q"][d], p["m"][d], p["s"][d], 768, 96, bits).cpu().numpy()
        assert np.array_equal(got.view(np.uint16), np.ascontiguousarray(p["dts"][d].T).view(np.uint16))


@pytest.mark.parametrize("bits", [2, 4])
def test_dequant_extreme_scales(dev, bits):
    """Subnormal, tiny and huge fp16 scales: one rounding of the exact product, no flush to zero."""
    k, n = 256, 32
    zp = 2 ** (bits - 1)
    rng = np.random.default_rng(5)
    codes = np.full((k, n), zp, dtype=np.uint8)
    pos = rng.integers(0, 4, size=(k // 4, n))
    for g in range(k // 4):                       # one non-zero code per group of 4
        codes[4 * g + pos[g], np.arange(n)] = rng.integers(0, 2 ** bits, size=n)
    scales = np.array([6e-8, 1.2e-7, 3e-6, 6.1e-5, 1e-3, 0.5, 1000.0, 8000.0] * 4, dtype=np.float16).reshape(1, n)
    qw, qz, sc, gi = o.pack_codes_gptq(codes, np.full((1, n), zp), scales, bits)
    ref = o.dequant_gptq(qw, qz, sc, gi, bits)
    q, m, s = ops.repack_gptq_to_native(torch.from_numpy(qw), torch.from_numpy(qz), torch.from_numpy(sc),
                                        torch.from_numpy(gi), bits)
    got = ops.dequant(q.to(dev), m.to(dev), s.to(dev), k, n, bits).cpu().numpy()
    assert np.array_equal(got.view(np.uint16), np.ascontiguousarray(ref.T).view(np.uint16))
    assert np.any((ref != 0) & (np.abs(ref.astype(np.float32)) < 6.1e-5))   # subnormals were exercised


def test_merge_is_fp32_add_rounded_once(dev):
    p = make_problem(64, 512, 4, -1, 1, 1, "single", 31, dev)
    got = ops.merge(p["wb"], p["q"][0], p["m"][0], p["s"][0], 4).cpu().numpy()
    ref = (p["wb_np"].astype(np.float32) + p["dts"][0].T.astype(np.float32)).astype(np.float16)
    assert np.array_equal(got.view(np.uint16), ref.view(np.uint16))


@pytest.mark.parametrize("t,s", [(1, 1), (9, 8), (128, 5), (1000, 3), (4099, 17)])
def test_segment(dev, t, s):
    rng = np.random.default_rng(t)
    ids = rng.integers(-1, s, size=t).astype(np.int64)
    ids[::7] = s + 3                               # out-of-range ids count as -1
    perm, off = ops.segment(torch.from_numpy(ids).to(dev), s)
    key = np.where((ids < 0) | (ids >= s), -1, ids)
    assert np.array_equal(perm.cpu().numpy(), np.argsort(key, kind="stable"))
    counts = [(key == v).sum() for v in range(-1, s)]
    assert off.cpu().numpy().tolist() == [0] + np.cumsum(counts).tolist()


CASES = [
    # n, k, bits, gs, deltas, tokens, ids
    (64, 512, 2, -1, 3, 5, "uniform"),
    (64, 512, 4, -1, 3, 16, "uniform"),
    (96, 768, 2, -1, 2, 1, "single"),
    (96, 768, 4, 64, 2, 17, "uniform"),
    (128, 1024, 2, 128, 4, 32, "uniform"),
    (128, 1024, 4, 128, 4, 32, "zipf"),
    (160, 1280, 2, -1, 8, 31, "uniform"),
    (256, 1024, 2, -1, 6, 48, "uniform"),
    (256, 1024, 4, -1, 6, 64, "zipf"),
    (256, 2048, 2, 256, 5, 100, "uniform"),
    (256, 1024, 4, 128, 12, 128, "zipf"),
    (32, 256, 2, -1, 1, 33, "single"),
]


@pytest.mark.parametrize("n,k,bits,gs,nd,t,kind", CASES)
def test_layer_parity(dev, n, k, bits, gs, nd, t, kind):
    p = make_problem(n, k, bits, gs, nd, t, kind, 1000 + n + k + t, dev)
    if t > 2:
        p["ids_np"][1] = -1
        p["ids"] = torch.from_numpy(p["ids_np"]).to(dev)
    y = run_layer(p).cpu().numpy()
    ref = o.forward_ref(p["x_np"], p["wb_np"], p["dts"], p["ids_np"])
    assert o.rel_err(y, ref) <= TOL
    assert ops.workspace_status() == 0


def test_edge_cases(dev):
    p = make_problem(64, 512, 4, -1, 2, 12, "uniform", 77, dev)
    base = o.forward_ref(p["x_np"], p["wb_np"], p["dts"], np.full(12, -1))
    # every token base-only == plain linear layer
    p["ids"] = torch.full((12,), -1, dtype=torch.int64, device=dev)
    assert o.rel_err(run_layer(p).cpu().numpy(), base) <= TOL
    # no slots at all (S = 0 is not allowed by the stacked tensors; one reset slot stands in)
    # a reset slot (zero scales) contributes exactly nothing
    p["s"].zero_()
    p["ids"] = torch.zeros(12, dtype=torch.int64, device=dev)
    y0 = run_layer(p)
    p["ids"] = torch.full((12,), -1, dtype=torch.int64, device=dev)
    assert torch.equal(y0, run_layer(p))


def test_out_of_range_ids_are_flagged_and_treated_as_base(dev):
    p = make_problem(64, 512, 2, -1, 2, 8, "uniform", 78, dev)
    ids = p["ids_np"].copy(); ids[3] = 2; ids[5] = -7
    p["ids"] = torch.from_numpy(ids).to(dev)
    y = run_layer(p).cpu().numpy()
    assert ops.workspace_status() & 1
    ids_eff = np.where((ids < 0) | (ids >= 2), -1, ids)
    assert o.rel_err(y, o.forward_ref(p["x_np"], p["wb_np"], p["dts"], ids_eff)) <= TOL
    ops._workspaces.clear()                        # fresh (zeroed) status word for later tests


GOLDEN = sorted(glob.glob(os.path.join(os.path.dirname(__file__), "golden", "*.npz")))


@pytest.mark.parametrize("path", GOLDEN, ids=[os.path.basename(p)[:-4] for p in GOLDEN])
def test_golden_fixtures(dev, path):
    g = np.load(path)
    bits = int(g["bits"])
    nd = sum(1 for k in g.files if k.endswith("_qweight"))
    qs, ms, ss = [], [], []
    for d in range(nd):
        q, m, s = ops.repack_gptq_to_native(*(torch.from_numpy(g[f"d{d}_{k}"]) for k in
                                              ("qweight", "qzeros", "scales", "g_idx")), bits)
        K, N = g[f"d{d}_dequant_t"].shape
        got = ops.dequant(q.to(dev), m.to(dev), s.to(dev), K, N, bits).cpu().numpy()
        assert np.array_equal(got.view(np.uint16), np.ascontiguousarray(g[f"d{d}_dequant_t"].T).view(np.uint16))
        qs.append(q); ms.append(m); ss.append(s)
    q, m, s = (torch.stack(v).to(dev) for v in (qs, ms, ss))
    x = torch.from_numpy(g["x"]).to(dev); ids = torch.from_numpy(g["ids"]).to(dev)
    y = ops.apply_delta(x, q, s, m, ids, torch.from_numpy(g["w_base"]).to(dev)).cpu().numpy()
    assert o.rel_err(y, g["y_ref"]) <= TOL
    yd = torch.zeros_like(torch.from_numpy(g["y_delta_only"])).half().to(dev)
    ops.add_delta(yd, x, q, None, s, None, ids, meta=m)
    assert o.rel_err(yd.cpu().numpy(), g["y_delta_only"]) <= TOL


def test_add_delta_slices_qkv_and_gate_up(dev):
    """In-place y[:, off:off+n] += x @ delta^T per output slice (deltazip.py:40-153)."""
    k, t = 512, 20
    slices = (128, 64, 64)                         # q, k, v
    probs = [make_problem(n, k, 4, -1, 3, t, "uniform", 300 + i, dev) for i, n in enumerate(slices)]
    ids_np = probs[0]["ids_np"]; ids = probs[0]["ids"]; x = probs[0]["x"]; x_np = probs[0]["x_np"]
    y0 = (torch.randn(t, sum(slices), device=dev) * 0.05).half()
    y = y0.clone()
    off = 0
    for p, n in zip(probs, slices):
        ops.add_delta_slice(y, x, p["q"], None, p["s"], None, ids, 1.0, off, n, meta=p["m"])
        off += n
    torch.cuda.synchronize()
    off = 0
    for p, n in zip(probs, slices):
        ref = y0[:, off:off + n].float().cpu().numpy() + o.forward_ref(x_np, None, p["dts"], ids_np)
        assert o.rel_err(y[:, off:off + n].cpu().numpy(), ref) <= TOL
        off += n
    # whole-width form
    p = probs[0]
    yy = torch.zeros(t, 128, dtype=torch.float16, device=dev)
    assert ops.add_delta(yy, x, p["q"], None, p["s"], None, ids, meta=p["m"]) is yy
    assert o.rel_err(yy.cpu().numpy(), o.forward_ref(x_np, None, p["dts"], ids_np)) <= TOL


@pytest.mark.parametrize("t,bits,gs", [(20, 4, -1), (100, 2, -1), (7, 4, 128), (300, 2, -1)])
def test_apply_delta_packed_nslice_and_in_place_apply_delta(dev, t, bits, gs):
    """The packed-sublayer op and the in-place apply_delta of the reference's non-fused module
    (deltazip.py:78-153), through its own names: every slice of `output` gains x @ delta_j^T of the
    token's delta, a base-only token (-1) gains nothing, columns outside the slices stay as they were."""
    from deltazip_amd import deltazip as dzmod
    k = 512
    slices = (128, 64, 96)
    nd = 4
    mixed = np.random.default_rng(t).integers(-1, nd, t).astype(np.int64)
    mixed[:2] = (-1, nd - 1)
    probs = [make_problem(n, k, bits, gs, nd, t, mixed, 700 + i, dev) for i, n in enumerate(slices)]
    ids_np = probs[0]["ids_np"]; ids = probs[0]["ids"]; x = probs[0]["x"]; x_np = probs[0]["x_np"]
    width = sum(slices) + 32                       # 32 columns that belong to no slice
    lead = (2, t // 2) if t % 2 == 0 else (t,)     # leading dimensions are flattened by the ops
    y0 = (torch.randn(*lead, width, device=dev) * 0.05).half()
    y = y0.clone()
    xin = x.view(*y.shape[:-1], k)
    got = dzmod.apply_delta_packed_nslice(xin, [p["q"] for p in probs], [None] * 3, [p["s"] for p in probs],
                                          [None] * 3, ids.view(*y.shape[:-1]), y, slices,
                                          meta_stacked=[p["m"] for p in probs])
    torch.cuda.synchronize()
    assert got.shape == y.shape and got.data_ptr() == y.data_ptr()
    y2, y02 = y.view(-1, width), y0.view(-1, width)
    off = 0
    for p, n in zip(probs, slices):
        ref = y02[:, off:off + n].float().cpu().numpy() + o.forward_ref(x_np, None, p["dts"], ids_np)
        assert o.rel_err(y2[:, off:off + n].cpu().numpy(), ref) <= TOL
        base_rows = torch.from_numpy(ids_np < 0).to(dev)
        assert torch.equal(y2[base_rows, off:off + n], y02[base_rows, off:off + n])
        off += n
    assert torch.equal(y2[:, off:], y02[:, off:])
    # the same slices one by one give the same bits (one launch or three)
    y3 = y0.clone().view(-1, width)
    off = 0
    for p, n in zip(probs, slices):
        ops.add_delta_slice(y3, x, p["q"], None, p["s"], None, ids, 1.0, off, n, meta=p["m"])
        off += n
    assert torch.equal(y3, y2)
    # in-place apply_delta over the first slice's delta
    p = probs[0]
    z0 = (torch.randn(*y.shape[:-1], slices[0], device=dev) * 0.05).half()
    z = z0.clone()
    out = dzmod.apply_delta(xin, p["q"], None, p["s"], None, ids.view(*y.shape[:-1]), z, meta_stacked=p["m"])
    torch.cuda.synchronize()
    assert out.shape == z.shape and out.data_ptr() == z.data_ptr()
    ref = z0.view(-1, slices[0]).float().cpu().numpy() + o.forward_ref(x_np, None, p["dts"], ids_np)
    assert o.rel_err(z.view(-1, slices[0]).cpu().numpy(), ref) <= TOL


def test_deterministic_and_order_independent(dev):
    p = make_problem(128, 1024, 2, -1, 5, 32, "uniform", 55, dev)
    y1 = run_layer(p); y2 = run_layer(p)
    assert torch.equal(y1, y2)                     # run-to-run bit identical (no float atomics)
    perm = torch.randperm(32, device=dev)
    q = dict(p); q["x"] = p["x"][perm].contiguous(); q["ids"] = p["ids"][perm].contiguous()
    assert torch.equal(run_layer(q), y1[perm])     # a token's result does not depend on its position
    srt = torch.argsort(p["ids"], stable=True)
    q["x"] = p["x"][srt].contiguous(); q["ids"] = p["ids"][srt].contiguous()
    assert torch.equal(run_layer(q), y1[srt])


@pytest.mark.parametrize("t", [32, 100])
def test_k_split_variants_agree(dev, t):
    p = make_problem(64, 2048, 4, 128, 3, t, "uniform", 66, dev)
    ref = o.forward_ref(p["x_np"], p["wb_np"], p["dts"], p["ids_np"])
    try:
        for ns in (1, 2, 3, 8):
            ops.set_ksplit(ns)
            assert o.rel_err(run_layer(p).cpu().numpy(), ref) <= TOL
            assert torch.equal(run_layer(p), run_layer(p))
    finally:
        ops.set_ksplit(0)


def test_indices_are_read_at_call_time(dev):
    """The manager rewrites the index buffer between steps (models.py:421-430); the layer must see it."""
    p = make_problem(64, 512, 4, -1, 3, 8, "uniform", 88, dev)
    buf = torch.zeros(16, dtype=torch.int64, device=dev)
    view = buf[:8]
    for ids in ([0, 1, 2, -1, 0, 1, 2, -1], [2, 2, 2, 2, -1, -1, 0, 0]):
        buf[:8].copy_(torch.tensor(ids))
        y = ops.apply_delta(p["x"], p["q"], p["s"], p["m"], view, p["wb"]).cpu().numpy()
        assert o.rel_err(y, o.forward_ref(p["x_np"], p["wb_np"], p["dts"], np.array(ids))) <= TOL


def test_gemm_f16(dev):
    from deltazip_amd.prefill import gemm_f16
    torch.manual_seed(0)
    x = torch.randn(300, 512, device=dev).half(); w = (torch.randn(256, 512, device=dev) * 0.05).half()
    y = gemm_f16(x, w)
    ref = x.float() @ w.float().t()
    assert o.rel_err(y.float().cpu().numpy(), ref.cpu().numpy()) <= 2e-3
    y2 = y.clone(); gemm_f16(x, w, y2, accumulate=True)
    assert o.rel_err(y2.float().cpu().numpy(), 2 * ref.cpu().numpy()) <= 3e-3


@pytest.mark.parametrize("kind", ["blocks", "uniform"])
def test_prefill_sized_call(dev, kind):
    """T > 128: per-segment merge + matrix-core GEMM; sorted (one delta per request) and unsorted."""
    p = make_problem(256, 1024, 2, -1, 4, 400, kind, 99, dev)
    y = run_layer(p).cpu().numpy()
    ref = o.forward_ref(p["x_np"], p["wb_np"], p["dts"], p["ids_np"])
    assert o.rel_err(y, ref) <= TOL


@pytest.mark.parametrize("bits,with_x", [(2, 0), (2, 1), (4, 1)])
def test_read_only_yardstick_runs_on_the_fused_launch_geometry(dev, bits, with_x):
    """dz_probe_read: the launch bench.py times beside the fused kernel reads the tiled base weight and
    the packed words of the first D slots with the fused kernel's grid and writes nothing (its sink
    stays as it was)."""
    import ctypes as C
    from deltazip_amd import _lib
    p1 = make_problem(256, 1024, bits, -1, 4, 32, "uniform", 3, dev)
    p2 = make_problem(96, 1024, bits, -1, 4, 32, "uniform", 4, dev)
    tiles = [ops.tile_base(p["wb"]) for p in (p1, p2)]
    sink = torch.full((64,), 7, dtype=torch.int32, device=dev)
    arr = lambda ts: (C.c_void_p * 2)(*[t.data_ptr() for t in ts])
    rc = _lib.lib().dz_probe_read(2, arr([p1["x"], p2["x"]]), arr(tiles), arr([p1["q"], p2["q"]]),
                                  arr([p1["m"], p2["m"]]), (C.c_int * 2)(256, 96), 32, 1024, bits, 4, with_x,
                                  sink.data_ptr(), torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert rc == 0 and bool((sink == 7).all())


def test_row_blocks_made_once_per_batch(dev):
    """ops.row_blocks(indices, S) made once and passed as `order` to several calls gives, bit for
    bit, what each call gives when it orders the batch itself; blocks of another batch are refused."""
    p = make_problem(256, 1024, 2, -1, 4, 700, "uniform", 5, dev)
    blocks = ops.row_blocks(p["ids"], 4)
    assert blocks.T == 700 and blocks.S == 4 and blocks.perm.dtype == torch.int32
    y0 = run_layer(p)
    for _ in range(2):
        y1 = ops.multi_delta_linear(p["x"], p["wb"], p["q"], p["s"], p["m"], p["ids"], bits=2, order=blocks)
        torch.cuda.synchronize()
        assert torch.equal(y0, y1)
    with pytest.raises(ValueError):
        ops.multi_delta_linear(p["x"][:600], p["wb"], p["q"], p["s"], p["m"], p["ids"][:600].contiguous(), bits=2,
                               order=blocks)
    with pytest.raises(ValueError):
        ops.multi_delta_linear(p["x"][:64], p["wb"], p["q"], p["s"], p["m"], p["ids"][:64].contiguous(), bits=2,
                               order=blocks)


@pytest.mark.parametrize("t", [1, 100, 128])
def test_prefill_call_of_decode_size(dev, t):
    """The product over blocks of one delta called directly with up to 128 rows, the size of the last piece of a very
    long batch: every row is written, or added to."""
    from deltazip_amd.prefill import multi_delta_linear_prefill
    p = make_problem(96, 512, 2, -1, 3, t, "uniform", t, dev)
    ref = o.forward_ref(p["x_np"], p["wb_np"], p["dts"], p["ids_np"])
    base = o.make_x(t, 96, 5)
    for accumulate in (False, True):
        y = torch.from_numpy(base).to(dev) if accumulate else torch.full((t, 96), float("nan"), dtype=torch.float16, device=dev)
        multi_delta_linear_prefill(p["x"], p["wb"], p["q"], p["s"], p["m"], p["ids"], bits=2, out=y, accumulate=accumulate)
        torch.cuda.synchronize()
        assert o.rel_err(y.cpu().numpy(), ref + (base.astype(np.float32) if accumulate else 0)) <= TOL


@pytest.mark.parametrize("n,k,bits,gs,nd", [(32, 256, 2, -1, 3), (96, 512, 4, -1, 2), (160, 768, 2, 64, 4),
                                            (288, 1024, 4, 128, 3), (128, 512, 2, -1, 1)])
def test_short_row_blocks(dev, n, k, bits, gs, nd):
    """dz_multi_delta_gemm_rows over blocks at the edges of its token tiles (1, 15, 16, 17 .. 127, 128 tokens
    and one of 200, taken in two parts), unsorted rows, row-major and tiled base weight, in place and
    without a base weight, against the kernel for long blocks and the oracle.  2-bit deltas: the same
    products in the same order, so equal bits; 4-bit: the long kernel adds all base products first."""
    from deltazip_amd import _lib
    L = _lib.lib()
    sizes = [1, 15, 16, 17, 32, 33, 48, 49, 64, 65, 96, 97, 127, 128, 200]
    t = sum(sizes)
    p = make_problem(n, k, bits, gs, nd, t, "uniform", 900 + n, dev)
    perm = np.random.default_rng(n).permutation(t).astype(np.int32)
    rows, ids, r = [], np.empty(t, dtype=np.int64), 0
    for i, c in enumerate(sizes):
        slot = i % (nd + 1) - 1
        rows.append([r, r + c, slot, 0])
        ids[perm[r:r + c]] = slot
        r += c
    rows += [[0, 0, -1, 0]] * 2                       # unused entries
    tiles = torch.tensor(rows, dtype=torch.int32, device=dev)
    pd, st = torch.from_numpy(perm).to(dev), torch.cuda.current_stream().cuda_stream
    wt = ops.tile_base(p["wb"])

    def call(short, w, tiled, y, acc):
        args = (p["q"].data_ptr(), p["m"].data_ptr(), p["s"].data_ptr(), nd, bits, gs, tiles.data_ptr(), len(rows),
                pd.data_ptr(), y.data_ptr(), t, k, n, acc, y.stride(0), st)
        wp = None if w is None else w.data_ptr()
        assert (L.dz_multi_delta_gemm_rows(p["x"].data_ptr(), wp, tiled, *args) if short
                else L.dz_multi_delta_gemm(p["x"].data_ptr(), wp, *args)) == 0
        torch.cuda.synchronize()
        return y
    new = lambda: torch.zeros(t, n + 8, device=dev, dtype=torch.float16)[:, :n]
    for w, tiled in ((p["wb"], 0), (wt, 1), (None, 0)):
        for acc in (0, 1):
            y, y0 = new(), new()
            if acc:
                y += 0.5
                y0 += 0.5
            call(True, w, tiled, y, acc)
            # (the long kernel takes at most 256 rows a block: all of these)
            call(False, None if w is None else p["wb"], 0, y0, acc)
            if bits == 2:
                assert torch.equal(y, y0)
            ref = o.forward_ref(p["x_np"], None if w is None else p["wb_np"], p["dts"], ids) + 0.5 * acc
            assert o.rel_err(y.float().cpu().numpy(), ref) <= TOL
            assert o.rel_err(y0.float().cpu().numpy(), ref) <= TOL


def test_bad_ids_of_mid_size_batches_are_reported(dev):
    """An id outside [-1, S) is served as -1 and sets bit 0 of the status word, as at decode sizes."""
    p = make_problem(64, 256, 2, -1, 3, 200, "uniform", 5, dev)
    run_layer(p)
    ops.poll_status(wait=True)
    assert ops.workspace_status() == 0
    good = run_layer(dict(p, ids=torch.where(p["ids"] == 1, torch.full_like(p["ids"], -1), p["ids"])))
    assert ops.workspace_status() == 0
    bad = run_layer(dict(p, ids=torch.where(p["ids"] == 1, torch.full_like(p["ids"], 7), p["ids"])))
    assert torch.equal(good, bad) and ops.workspace_status() == ops.STATUS_BAD_ID
    warned, ops._warned_bad_id = ops._warned_bad_id, True
    ops.poll_status(wait=True)                        # clears it
    ops._warned_bad_id = warned
    assert ops.workspace_status() == 0


@pytest.mark.parametrize("n,lens,long", [(32000, [0, 126, 130], True), (32000, [0, 120, 128], False), (32000, [0, 256, 0], False),
                                         (32000, [13, 243, 0], True), (16384, [64, 0, 192], False), (16384, [60, 130, 300], True),
                                         (24576, [0, 126, 130], False), (32000, [100, 100, 100], False)])
def test_projection_picks_blocks_by_waves(dev, n, lens, long):
    """Long blocks where they fill one wave of workgroups and short ones overflow theirs; the rows' results
    are those of each row's own table (fp32 sums rounded once to fp16, as for the short blocks)."""
    from deltazip_amd import _lib
    k, t, L = 256, sum(lens), _lib.lib()
    seg = torch.from_numpy(np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)).to(dev)
    tabs = [torch.full((8, 4), 77, dtype=torch.int32, device=dev) for _ in range(2)]
    assert L.dz_build_tiles_either_for(seg.data_ptr(), 2, n, tabs[0].data_ptr(), 8, tabs[1].data_ptr(), 8,
                                       torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    step, at = (256 if long else 128), np.concatenate([[0], np.cumsum(lens)])
    want = [[a, min(a + step, int(at[s + 1])), s - 1, 0] for s in range(3) for a in range(int(at[s]), int(at[s + 1]), step)]
    want += [[0, 0, -1, 0]] * (8 - len(want))
    assert tabs[not long].cpu().tolist() == want and tabs[long].cpu().tolist() == [[0, 0, -1, 0]] * 8
    g = torch.Generator().manual_seed(n)
    x = torch.randn(t, k, generator=g).half()
    tables = (torch.randn(3, n, k, generator=g) * 0.02).half()
    ids = torch.from_numpy(np.random.default_rng(t).permutation(np.repeat(np.arange(3) - 1, lens)))
    xd, td = x.to(dev), tables.to(dev)
    got = ops.apply_delta_uncompressed(xd, td[1:].contiguous(), ids.to(dev), td[0].contiguous()).cpu().double()
    for i in range(0, t, 7):
        ref = x[i].double() @ tables[int(ids[i]) + 1].double().t()
        assert ((got[i] - ref).abs() <= 2.0**-10 * ref.abs() + 1e-4).all()
    assert L.dz_build_tiles_either_for(seg.data_ptr(), 2, 0, tabs[0].data_ptr(), 8, tabs[1].data_ptr(), 8, None) == -2
    assert L.dz_build_tiles_either_for(seg.data_ptr(), 2, n, tabs[0].data_ptr(), 8, None, 8, None) == -1


def test_output_projection_does_not_report_ids(dev):
    """apply_delta_uncompressed serves an id without a table from the base table and leaves the fused
    kernel's status word alone, at every size."""
    stack, base = torch.randn(2, 64, 256, device=dev).half(), torch.randn(64, 256, device=dev).half()
    ops.poll_status(wait=True)
    for t in (40, 200, 700):
        x = torch.randn(t, 256, device=dev).half()
        ids = torch.arange(t, device=dev) % 4 - 1          # 2 has no table
        y = ops.apply_delta_uncompressed(x, stack, ids, base)
        assert torch.equal(y, ops.apply_delta_uncompressed(x, stack, torch.where(ids == 2, -1, ids), base))
        torch.cuda.synchronize()
        assert ops.workspace_status() == 0, t


@pytest.mark.parametrize("n,k,s,t", [(32, 256, 3, 1), (96, 512, 8, 33), (160, 768, 2, 128), (4128, 256, 5, 129),
                                     (288, 1024, 1, 300), (64, 512, 20, 1024)])
def test_select_over_short_blocks(dev, n, k, s, t):
    """apply_delta_uncompressed where its row blocks are short: every row against its own table in 64 bits
    (fp32 sums rounded once to fp16: half a unit of 2^-11, and as much again for the sums), and the
    kernel for long blocks on the same rows."""
    from deltazip_amd import _lib
    g = torch.Generator().manual_seed(n + t)
    x = torch.randn(t, k, generator=g).half()
    stack, base = (torch.randn(s, n, k, generator=g) * 0.02).half(), (torch.randn(n, k, generator=g) * 0.02).half()
    ids = torch.randint(-1, s, (t,), generator=g)
    tables = torch.cat([base[None], stack]).double()
    want = torch.stack([x[i].double() @ tables[int(ids[i]) + 1].t() for i in range(t)])
    xd, sd, bd, idd = x.to(dev), stack.to(dev), base.to(dev), ids.to(dev)
    got = ops.apply_delta_uncompressed(xd, sd, idd, bd)
    blocks = ops.row_blocks(idd, s, long_only=True)
    other = torch.empty_like(got)
    assert _lib.lib().dz_gemm_f16_select(xd.data_ptr(), bd.data_ptr(), sd.data_ptr(), n * k, blocks.tiles.data_ptr(),
                                         blocks.max_tiles, blocks.perm.data_ptr(), other.data_ptr(), t, k, n, 0, n,
                                         torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    for y in (got, other):
        assert ((y.cpu().double() - want).abs() <= 2.0**-10 * want.abs() + 1e-4).all()


@pytest.mark.parametrize("lens,short", [([0, 300, 20, 5], True), ([0, 512, 250, 0], False), ([10, 0, 0, 0], True),
                                        ([192, 192, 192, 192], False), ([191, 192, 192, 192], True)])
def test_build_tiles_either(dev, lens, short):
    """All rows go into the table whose blocks suit them -- long blocks from three quarters full on --
    and the other table is empty."""
    from deltazip_amd import _lib
    L = _lib.lib()
    off = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    seg = torch.from_numpy(off).to(dev)
    tabs = [torch.full((16, 4), 77, dtype=torch.int32, device=dev) for _ in range(2)]
    assert L.dz_build_tiles_either(seg.data_ptr(), len(lens) - 1, tabs[0].data_ptr(), 16, tabs[1].data_ptr(), 16,
                                   torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    step = 128 if short else 256
    want = [[a, min(a + step, int(off[s + 1])), s - 1, 0] for s in range(len(lens))
            for a in range(int(off[s]), int(off[s + 1]), step)]
    want += [[0, 0, -1, 0]] * (16 - len(want))
    assert tabs[short].cpu().tolist() == want and tabs[not short].cpu().tolist() == [[0, 0, -1, 0]] * 16
    assert L.dz_build_tiles_either(seg.data_ptr(), len(lens) - 1, tabs[0].data_ptr(), 16, None, 16, None) == -1


@pytest.mark.parametrize("t,nd", [(129, 3), (256, 40), (300, 4), (512, 17)])
def test_mid_size_batches_over_few_slots_and_many(dev, t, nd):
    """Between 129 tokens and a few hundred: the call's own choice, row blocks, and -- the same deltas
    scattered over more slots than the token sort can take -- chunks of 128 tokens through the fused
    kernel, also into a column slice.  All match the oracle."""
    from deltazip_amd.prefill import multi_delta_linear_prefill
    assert ops.takes_fused_chunks(t, nd) and not ops.takes_fused_chunks(513, 64) and not ops.takes_fused_chunks(400, 4)
    p = make_problem(96, 512, 2, -1, nd, t, "uniform", 77 + t, dev)
    ref = o.forward_ref(p["x_np"], p["wb_np"], p["dts"], p["ids_np"])
    y = run_layer(p)
    assert o.rel_err(y.cpu().numpy(), ref) <= TOL
    y2 = torch.empty_like(y)
    multi_delta_linear_prefill(p["x"], p["wb"], p["q"], p["s"], p["m"], p["ids"], bits=2, out=y2, accumulate=False)
    torch.cuda.synchronize()
    assert o.rel_err(y2.cpu().numpy(), ref) <= TOL
    # 1000 slots, in arbitrary order
    S, rng = 1000, np.random.default_rng(t)
    where, mixed = rng.choice(S, nd, replace=False), rng.permutation(t)
    stacks = {}
    for key in ("q", "m", "s"):
        stacks[key] = torch.zeros((S,) + tuple(p[key].shape[1:]), dtype=p[key].dtype, device=dev)
        stacks[key][torch.from_numpy(where).to(dev)] = p[key]
    slots = np.where(p["ids_np"] >= 0, where[np.maximum(p["ids_np"], 0)], -1)
    assert ops._most_row_blocks(t, 512, 96, 2, S, None) == 0
    wide = torch.zeros(t, 96 + 64, device=dev, dtype=torch.float16)
    ops.multi_delta_linear(p["x"][torch.from_numpy(mixed).to(dev)], p["wb"], stacks["q"], stacks["s"], stacks["m"],
                           torch.from_numpy(slots[mixed]).to(dev), bits=2, out=wide[:, 32:128])
    torch.cuda.synchronize()
    assert not wide[:, :32].any() and not wide[:, 128:].any()
    assert o.rel_err(wide[:, 32:128].cpu().numpy(), ref[mixed]) <= TOL
    # in place, delta only, into a column slice
    wide = torch.zeros(t, 96 + 64, device=dev, dtype=torch.float16)
    ops.add_delta_slice(wide, p["x"], p["q"], None, p["s"], None, p["ids"], 1.0, 32, 96, meta=p["m"])
    torch.cuda.synchronize()
    dref = ref - p["x_np"].astype(np.float32) @ p["wb_np"].astype(np.float32).T
    assert float(wide[:, :32].abs().max()) == 0 and float(wide[:, 128:].abs().max()) == 0
    assert np.abs(wide[:, 32:128].float().cpu().numpy() - dref).max() <= 2e-2 * np.abs(dref).max()


@pytest.mark.parametrize("n,k,bits,gs,nd,t", [(64, 512, 2, -1, 3, 1), (96, 768, 4, 128, 5, 16), (256, 4096, 2, -1, 8, 32),
                                              (160, 1024, 2, 64, 7, 33), (128, 2048, 4, -1, 12, 100), (512, 4096, 2, -1, 9, 128),
                                              (256, 1024, 2, -1, 6, 200)])   # 200 tokens: row blocks
def test_tiled_base_weight_gives_the_same_bits(dev, n, k, bits, gs, nd, t):
    """The base weight converted to tiles (dz_tile_base) feeds the fused kernel the same operands in the
    same order: outputs equal the row-major call bit for bit, single and batched, and match the oracle.
    The conversion itself is a pure rearrangement (every value kept, at the position dz_layout.h gives)."""
    p = make_problem(n, k, bits, gs, nd, t, "uniform", 3000 + n + t, dev)
    tiled = ops.tile_base(p["wb"])
    w, tl = p["wb_np"], tiled.cpu().numpy().reshape(-1)
    for (np_, kb, s_, j, h, lane) in [(0, 0, 0, 0, 0, 0), (n // 32 - 1, k // 256 - 1, 1, 3, 1, 63), (0, k // 256 - 1, 1, 2, 0, 37)]:
        off = ((np_ * (k // 256) + kb) * 16384 + ((s_ * 4 + j) * 2 + h) * 1024 + lane * 16) // 2
        i, g = lane % 16, lane // 16
        row, col = 32 * np_ + 16 * s_ + i, 256 * kb + 64 * j + 16 * g + 8 * h
        assert np.array_equal(tl[off:off + 8], w[row, col:col + 8])
    assert np.array_equal(np.sort(tl.view(np.uint16)), np.sort(w.reshape(-1).view(np.uint16)))
    y0 = run_layer(p)
    y1 = ops.apply_delta(p["x"], p["q"], p["s"], p["m"], p["ids"], p["wb"], base_tiled=tiled)
    torch.cuda.synchronize()
    assert torch.equal(y0, y1)
    assert o.rel_err(y1.cpu().numpy(), o.forward_ref(p["x_np"], p["wb_np"], p["dts"], p["ids_np"])) <= TOL
    b0 = ops.apply_delta_batch(p["x"], [p["q"]] * 2, [p["s"]] * 2, [p["m"]] * 2, p["ids"], [p["wb"]] * 2)
    b1 = ops.apply_delta_batch(p["x"], [p["q"]] * 2, [p["s"]] * 2, [p["m"]] * 2, p["ids"], [p["wb"]] * 2,
                               base_tiled=[tiled] * 2)
    torch.cuda.synchronize()
    assert torch.equal(b0[0], b1[0]) and torch.equal(b0[1], b1[1])
    with pytest.raises(ValueError):
        ops.apply_delta(p["x"], p["q"], p["s"], p["m"], p["ids"], p["wb"], base_tiled=tiled[:, : k // 2])
    from deltazip_amd import _lib
    assert _lib.lib().dz_tile_base(p["wb"].data_ptr(), k, n, p["wb"].data_ptr(), None) != 0      # not in place
    assert _lib.lib().dz_tile_base(p["wb"].data_ptr(), k - 64, n, tiled.data_ptr(), None) != 0    # whole k-blocks only


def test_tiled_base_weight_wide_launch(dev):
    """12288 output rows (q, k and v of a 4096-wide model fused), split in K: the K split depends on
    the shapes only, so both forms of the base weight give the same bits here, too."""
    p = make_problem(12288, 2048, 2, -1, 4, 24, "uniform", 77, dev)
    ref = o.forward_ref(p["x_np"], p["wb_np"], p["dts"], p["ids_np"])
    y0 = run_layer(p)
    y1 = ops.apply_delta(p["x"], p["q"], p["s"], p["m"], p["ids"], p["wb"], base_tiled=ops.tile_base(p["wb"]))
    torch.cuda.synchronize()
    assert o.rel_err(y0.cpu().numpy(), ref) <= TOL
    assert torch.equal(y0, y1)


def test_fused_layer_calls_replay_from_a_graph(dev):
    """What a serving loop does with a decode step: the layer calls -- a single projection over the
    tiled base weight, two projections in one launch at 64 tokens (token order computed inside the
    call), a split-K launch -- are captured once into a HIP graph and replayed after the ids were
    rewritten in place, with eager work and synchronisations between the replays.  Every replay
    equals the eager call bit for bit: nothing in the path reads back to the host, allocates or
    depends on state a replay would find changed (the split-K workspace is left empty by every launch)."""
    a = make_problem(256, 4096, 2, -1, 6, 24, "uniform", 501, dev)      # split in K
    b = make_problem(160, 1024, 4, 128, 9, 64, "uniform", 502, dev)     # two chunks of tokens, grouped scales
    tiled = ops.tile_base(a["wb"])

    def step():
        y0 = ops.apply_delta(a["x"], a["q"], a["s"], a["m"], a["ids"], a["wb"], base_tiled=tiled)
        y1 = ops.apply_delta_batch(b["x"], [b["q"]] * 2, [b["s"]] * 2, [b["m"]] * 2, b["ids"], [b["wb"]] * 2)
        return y0, y1[0], y1[1]

    step()                                                               # one-time set-up outside the capture
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(side):
        with torch.cuda.graph(graph, stream=side):
            outs = step()
    torch.cuda.current_stream().wait_stream(side)
    rng = np.random.default_rng(5)
    for rep in range(4):
        ia, ib = rng.integers(-1, 6, size=24), rng.integers(-1, 9, size=64)
        if rep == 2:
            ia[:], ib[:] = -1, 3                                         # base only / one delta for every token
        a["ids"].copy_(torch.from_numpy(ia).to(dev))
        b["ids"].copy_(torch.from_numpy(ib).to(dev))
        eager = step()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        for got, want in zip(outs, eager):
            assert torch.equal(got, want), rep
        assert o.rel_err(outs[0].cpu().numpy(), o.forward_ref(a["x_np"], a["wb_np"], a["dts"], ia)) <= TOL
        assert o.rel_err(outs[2].cpu().numpy(), o.forward_ref(b["x_np"], b["wb_np"], b["dts"], ib)) <= TOL


def test_gemm_grouped(dev):
    """Grouped GEMM through the C ABI: ragged row blocks, a block without second weight, rows that no
    block covers (left untouched), an N that is not a multiple of the 256-wide tile, and the
    second-product-only form (w = NULL)."""
    from deltazip_amd import _lib
    L = _lib.lib()
    torch.manual_seed(1)
    T, K, N, G = 700, 512, 352, 3
    x = torch.randn(T, K, device=dev).half()
    w = (torch.randn(N, K, device=dev) * 0.05).half()
    w2 = (torch.randn(G, N, K, device=dev) * 0.05).half()
    blocks = [(0, 100, -1), (100, 356, 2), (356, 390, 2), (390, 391, 0), (400, 656, 1), (656, 700, 1)]
    tiles = torch.tensor([(lo, hi, g, 0) for lo, hi, g in blocks], dtype=torch.int32, device=dev)
    st = torch.cuda.current_stream().cuda_stream
    for with_base in (True, False):
        y = torch.full((T, N), 7.0, dtype=torch.float16, device=dev)
        rc = L.dz_gemm_f16_grouped(x.data_ptr(), w.data_ptr() if with_base else None, w2.data_ptr(), N * K,
                                   tiles.data_ptr(), len(blocks), y.data_ptr(), T, K, N, 0, N, st)
        assert rc == 0
        torch.cuda.synchronize()
        ref = torch.full((T, N), 7.0, dtype=torch.float32, device=dev)
        for lo, hi, g in blocks:
            r = x[lo:hi].float() @ w.float().t() if with_base else None
            if g >= 0:
                d = x[lo:hi].float() @ w2[g].float().t()
                r = d if r is None else r + d
            if r is not None:
                ref[lo:hi] = r
        assert o.rel_err(y.float().cpu().numpy(), ref.cpu().numpy()) <= 2e-3
        assert torch.equal(y[391:400], torch.full((9, N), 7.0, dtype=torch.float16, device=dev))
    # argument checks happen before the launch
    assert L.dz_gemm_f16_grouped(x.data_ptr(), w.data_ptr(), w2.data_ptr(), N * K, None, 1, y.data_ptr(),
                                 T, K, N, 0, N, st) != 0
    assert L.dz_gemm_f16_grouped(x.data_ptr(), w.data_ptr(), w2.data_ptr(), N * K, tiles.data_ptr(), 1,
                                 y.data_ptr(), T, K + 8, N, 0, N, st) != 0


def test_segment_limits(dev):
    ids = torch.zeros(10, dtype=torch.int64, device=dev)
    perm = torch.empty(10, dtype=torch.int32, device=dev)
    from deltazip_amd import _lib
    off = torch.empty(2000, dtype=torch.int32, device=dev)
    st = torch.cuda.current_stream().cuda_stream
    assert _lib.lib().dz_segment(ids.data_ptr(), 10, 768, perm.data_ptr(), off.data_ptr(), st) == 0
    assert _lib.lib().dz_segment(ids.data_ptr(), 10, 769, perm.data_ptr(), off.data_ptr(), st) != 0
    torch.cuda.synchronize()


@pytest.mark.parametrize("t", [33, 64, 97, 128])
def test_unsorted_batches_above_32_tokens(dev, t):
    """33..128 tokens in arbitrary order with many deltas: the device-side ordering must bring every
    token back to its own output row."""
    p = make_problem(96, 768, 4, 128, 20, t, "uniform", 4242 + t, dev)
    p["ids_np"][::7] = -1
    p["ids"] = torch.from_numpy(p["ids_np"]).to(dev)
    y = run_layer(p).cpu().numpy()
    ref = o.forward_ref(p["x_np"], p["wb_np"], p["dts"], p["ids_np"])
    assert o.rel_err(y, ref) <= TOL
    assert ops.workspace_status() == 0


@pytest.mark.parametrize("t,kind", [(64, "zipf"), (128, "zipf"), (100, "single"), (77, "uniform")])
def test_dealt_chunks_skewed_mixes_and_many_slots(dev, t, kind):
    """33..128 tokens: the tokens are dealt to the 32-token chunks by delta (popular deltas split,
    rare ones spread); whatever the mix, every token must get its own delta's result in its own
    row -- also with far more slots than the sort used for long batches can take, most of them
    empty."""
    nd = 24
    p = make_problem(64, 512, 2, -1, nd, t, kind, 5150 + t, dev)
    S = 1000                                         # slots; deltas sit in scattered ones
    where = np.random.default_rng(t).choice(S, nd, replace=False)
    q = torch.zeros((S,) + tuple(p["q"].shape[1:]), dtype=p["q"].dtype, device=dev)
    m = torch.zeros((S,) + tuple(p["m"].shape[1:]), dtype=p["m"].dtype, device=dev)
    s = torch.zeros((S,) + tuple(p["s"].shape[1:]), dtype=p["s"].dtype, device=dev)
    idx = torch.from_numpy(where).to(dev)
    q[idx], m[idx], s[idx] = p["q"], p["m"], p["s"]
    ids_np = p["ids_np"].copy()
    slots_np = np.where(ids_np >= 0, where[np.maximum(ids_np, 0)], -1)
    slots_np[5] = -1
    ids_np[5] = -1
    perm = np.random.default_rng(t + 1).permutation(t)          # arbitrary arrival order
    y = ops.apply_delta(p["x"][torch.from_numpy(perm).to(dev)], q, s, m, torch.from_numpy(slots_np[perm]).to(dev),
                        p["wb"])
    torch.cuda.synchronize()
    ref = o.forward_ref(p["x_np"][perm], p["wb_np"], p["dts"], ids_np[perm])
    assert o.rel_err(y.cpu().numpy(), ref) <= TOL
    assert ops.workspace_status() == 0


PREFILL_CASES = [
    # n, k, bits, gs, deltas, tokens, ids
    (256, 1024, 2, -1, 4, 400, "uniform"),
    (352, 768, 4, -1, 3, 129, "uniform"),
    (352, 768, 2, 128, 5, 700, "zipf"),
    (512, 512, 4, 64, 2, 300, "blocks"),
    (96, 256, 2, -1, 9, 1000, "uniform"),
    (288, 1280, 4, 256, 6, 515, "uniform"),
]


@pytest.mark.parametrize("n,k,bits,gs,nd,t,kind", PREFILL_CASES)
def test_packed_delta_gemm_parity(dev, n, k, bits, gs, nd, t, kind):
    """T > 128 over row blocks, long ones (dz_multi_delta_gemm) and whatever the call chooses: unsorted
    ids, tokens without a delta, N that is not a multiple of the 256-wide tile, grouped scales, then
    the delta-only and accumulate forms."""
    p = make_problem(n, k, bits, gs, nd, t, kind, 4000 + n + k + t, dev)
    p["ids_np"][::7] = -1
    p["ids"] = torch.from_numpy(p["ids_np"]).to(dev)
    for order in (ops.row_blocks(p["ids"], nd, long_only=True), None):
        y = ops.apply_delta(p["x"], p["q"], p["s"], p["m"], p["ids"], p["wb"], order=order)
        torch.cuda.synchronize()
        ref = o.forward_ref(p["x_np"], p["wb_np"], p["dts"], p["ids_np"])
        assert o.rel_err(y.cpu().numpy(), ref) <= TOL
        # delta only, accumulated onto an existing output (the add_delta form)
        y0 = torch.from_numpy(o.make_x(t, n, 5)).to(dev)
        y1 = y0.clone()
        ops.multi_delta_linear(p["x"], None, p["q"], p["s"], p["m"], p["ids"], bits=bits, out=y1, accumulate=True,
                               order=order)
        torch.cuda.synchronize()
        ref_d = o.forward_ref(p["x_np"], None, p["dts"], p["ids_np"]) + y0.float().cpu().numpy()
        assert o.rel_err(y1.cpu().numpy(), ref_d) <= TOL
        # delta only, not accumulated: rows without a delta are zero
        y2 = ops.multi_delta_linear(p["x"], None, p["q"], p["s"], p["m"], p["ids"], bits=bits, order=order)
        torch.cuda.synchronize()
        assert (y2[torch.from_numpy(p["ids_np"] < 0).to(dev)] == 0).all()
        assert o.rel_err(y2.cpu().numpy(), o.forward_ref(p["x_np"], None, p["dts"], p["ids_np"])) <= TOL


def test_build_tiles(dev):
    from deltazip_amd import _lib
    L = _lib.lib()
    off = [0, 10, 10, 600, 601, 1113, 1113]          # S = 4: segments of 10, 0, 590, 1, 512, 0 rows
    seg = torch.tensor(off, dtype=torch.int32, device=dev)
    tiles = torch.full((12, 4), 77, dtype=torch.int32, device=dev)
    assert L.dz_build_tiles(seg.data_ptr(), 5, tiles.data_ptr(), 12, torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    got = tiles.cpu().tolist()
    want = [[0, 10, -1, 0], [10, 266, 1, 0], [266, 522, 1, 0], [522, 600, 1, 0], [600, 601, 2, 0],
            [601, 857, 3, 0], [857, 1113, 3, 0]]
    assert got[:7] == want and all(r == [0, 0, -1, 0] for r in got[7:])
    assert L.dz_build_tiles(None, 5, tiles.data_ptr(), 12, None) == -1
    assert L.dz_build_tiles(seg.data_ptr(), 5000, tiles.data_ptr(), 12, None) == -2


@pytest.mark.parametrize("n,k,bits,gs", [(32, 256, 4, -1), (64, 512, 2, -1), (96, 768, 4, 128), (160, 1024, 2, 64),
                                         (256, 2048, 4, 256)])
def test_compressor_matches_reference_pipeline(dev, n, k, bits, gs):
    """dz_compress_2of4 against the oracle's restatement of the reference's pipeline (scales from the
    un-pruned delta, 2:4 by magnitude, quantise, GPTQ pack) followed by the repacker: same bytes.
    Rows that are all zero, rows without a negative value, magnitude ties and values that quantise to
    the zero-point are all present."""
    rng = np.random.default_rng(n + k + bits)
    d = (rng.standard_normal((n, k)) * 1e-3).astype(np.float32)
    d[3] = 0.0                                        # all-zero row: range (-1, 1)
    d[5] = np.abs(d[5])                               # no negative value: range (0, max)
    d[7, :64] = np.float32(2e-3) * rng.integers(-2, 3, 64)   # many exact ties and exact zeros
    d[9] *= 1e-4                                      # tiny values next to ...
    d[9, 17] = 1.0                                    # ... one large one: most codes are the zero-point
    codes, scales16, zeros, keep = o.compress_delta(d, bits, gs)
    qw, qz, sc, gi = o.pack_codes_gptq(codes, zeros, scales16, bits)
    want_c, want_m, want_s = o.repack_native(qw, qz, sc, gi, bits)
    q, m, s = ops.compress_delta(torch.from_numpy(d).to(dev), bits, gs)
    torch.cuda.synchronize()
    assert q.cpu().numpy().view(np.uint32).tobytes() == want_c.tobytes()
    assert m.cpu().numpy().view(np.uint32).tobytes() == want_m.tobytes()
    assert np.array_equal(s.cpu().numpy().view(np.uint16), want_s.view(np.uint16))
    # and it dequantises (on the GPU) to the reference dequantisation of those GPTQ tensors
    got = ops.dequant(q, m, s, k, n, bits).cpu().numpy()
    assert np.array_equal(got.view(np.uint16), np.ascontiguousarray(o.dequant_gptq(qw, qz, sc, gi, bits).T).view(np.uint16))


@pytest.mark.parametrize("bits,gs,k", [(2, -1, 1280), (4, -1, 5632), (4, 64, 1280), (2, 128, 256), (4, 256, 768),
                                       (2, 192, 768)])
def test_compressor_at_code_boundaries(dev, bits, gs, k):
    """Byte for byte the oracle's result where a product with the scale's reciprocal could round another way
    than the quotient: values at and one unit beside every half code, for scales over the whole range
    of fp32, and rows whose scale is below or above what the reciprocal is used for."""
    n, maxq, rng = 64, 2**bits - 1, np.random.default_rng(bits + k)
    g = k if gs == -1 else gs
    d = np.empty((n, k), np.float32)
    for r in range(n):
        top = np.float32(rng.uniform(0.5, 1) * 10.0 ** rng.uniform(-30, 30))
        if r == 1:
            top = np.float32(1e-39)
        if r == 2:
            top = np.float32(2e37)
        sc = np.float32(np.float32(2) * top / np.float32(maxq))
        v = ((rng.integers(-maxq - 1, maxq + 1, k) / 2.0).astype(np.float32) * sc).astype(np.float32)
        v = np.where(rng.random(k) < 0.5, np.nextafter(v, np.float32(rng.choice([-np.inf, np.inf]))), v)
        v = np.clip(v, -top, top)
        v[::g] = -top
        d[r] = v
    codes, scales16, zeros, _ = o.compress_delta(d, bits, gs)
    qw, qz, sc16, gi = o.pack_codes_gptq(codes, zeros, scales16, bits)
    want_c, want_m, want_s = o.repack_native(qw, qz, sc16, gi, bits)
    q, m, s = ops.compress_delta(torch.from_numpy(d).to(dev), bits, gs)
    torch.cuda.synchronize()
    assert np.array_equal(s.cpu().numpy().view(np.uint16), want_s.view(np.uint16))
    assert q.cpu().numpy().view(np.uint32).tobytes() == want_c.tobytes()
    assert m.cpu().numpy().view(np.uint32).tobytes() == want_m.tobytes()


def test_compressor_argument_checks(dev):
    with pytest.raises(ValueError):
        ops.compress_delta(torch.zeros(32, 256, device=dev, dtype=torch.float16), 4)
    with pytest.raises(NotImplementedError):
        ops.compress_delta(torch.zeros(32, 256, device=dev), 3)
    with pytest.raises(ValueError):
        ops.compress_delta(torch.zeros(32, 200, device=dev), 4)
    with pytest.raises(ValueError):
        ops.compress_delta(torch.zeros(32, 256), 4)


@pytest.mark.parametrize("bits,gs,t,ns,k", [(2, -1, 32, (128, 128, 128), 1024), (4, 128, 7, (64, 256), 1024),
                                            (2, -1, 64, (96, 32, 32, 160), 1024), (4, -1, 128, (64, 64), 1024),
                                            (2, -1, 32, (64, 96), 4096),
                                            # 2-bit deltas with scale groups of 64: the kernel variant under the
                                            # highest register pressure (it once spilled a register that an
                                            # in-flight load was still to fill)
                                            (2, 64, 32, (160, 160), 1024), (2, 64, 102, (96, 96), 768),
                                            (2, 64, 65, (32, 32), 4096), (2, 64, 7, (64, 32), 512)])
def test_batched_calls_equal_separate_calls(dev, bits, gs, t, ns, k):
    """Projections that share the tokens, in one launch: every output is bit for bit what the
    separate call gives when both split K the same way (1024 columns are never split; for 4096
    the split is pinned, since a batch chooses it by the n-pairs of all its calls and the fp32
    partial sums are then added in a different order), and matches the oracle."""
    nd = 5
    if k > 1024:
        ops.set_ksplit(2)
    try:
        _batched_equal_separate(dev, bits, gs, t, ns, k, nd)
    finally:
        ops.set_ksplit(0)
    if k > 1024:     # with the launch's own choice of split: equal within the parity bound
        ps = [make_problem(n, k, bits, gs, nd, t, "uniform", 700 + 10 * j + n, dev) for j, n in enumerate(ns)]
        ys = ops.apply_delta_batch(ps[0]["x"], [p["q"] for p in ps], [p["s"] for p in ps], [p["m"] for p in ps],
                                   ps[0]["ids"], [p["wb"] for p in ps])
        torch.cuda.synchronize()
        for p, y in zip(ps, ys):
            assert o.rel_err(y.cpu().numpy(), o.forward_ref(ps[0]["x_np"], p["wb_np"], p["dts"], ps[0]["ids_np"])) <= TOL


def _batched_equal_separate(dev, bits, gs, t, ns, k, nd):
    ps = [make_problem(n, k, bits, gs, nd, t, "uniform", 700 + 10 * j + n, dev) for j, n in enumerate(ns)]
    ids = ps[0]["ids"]
    ids_np = ps[0]["ids_np"]
    x = ps[0]["x"]
    ys = ops.apply_delta_batch(x, [p["q"] for p in ps], [p["s"] for p in ps], [p["m"] for p in ps], ids,
                               [p["wb"] for p in ps])
    torch.cuda.synchronize()
    for p, y in zip(ps, ys):
        sep = ops.apply_delta(x, p["q"], p["s"], p["m"], ids, p["wb"])
        torch.cuda.synchronize()
        assert torch.equal(y, sep)
        ref = o.forward_ref(ps[0]["x_np"], p["wb_np"], p["dts"], ids_np)
        assert o.rel_err(y.cpu().numpy(), ref) <= TOL
    # one x per projection
    ys2 = ops.apply_delta_batch([p["x"] for p in ps], [p["q"] for p in ps], [p["s"] for p in ps],
                                [p["m"] for p in ps], ids, [p["wb"] for p in ps])
    torch.cuda.synchronize()
    for p, y in zip(ps, ys2):
        assert torch.equal(y, ops.apply_delta(p["x"], p["q"], p["s"], p["m"], ids, p["wb"]))
    with pytest.raises(ValueError):
        ops.apply_delta_batch(x, [ps[0]["q"]] * 5, [ps[0]["s"]] * 5, [ps[0]["m"]] * 5, ids, [ps[0]["wb"]] * 5)


@pytest.mark.parametrize("n,k,bits,gs,nd,t,present", [
    (256, 8192, 2, -1, 9, 129, None), (96, 8192, 4, 128, 3, 300, None), (128, 8192, 2, 64, 17, 256, None),   # few features
    (256, 512, 4, 64, 2, 150, 1), (2048, 256, 2, -1, 24, 200, 3), (96, 256, 2, -1, 5, 384, None),            # short walks
    (27648, 256, 2, -1, 1, 512, None), (27648, 256, 2, -1, 1, 449, None), (27648, 256, 2, -1, 3, 512, 1),     # wide, one delta
    (27648, 256, 2, -1, 1, 512, 0)])
def test_every_route_of_a_mid_size_batch(dev, n, k, bits, gs, nd, t, present):
    """129 to 512 tokens by whatever route the sizes, the slots and -- where the host knows it -- the mix choose
    (test_route_of_a_mid_size_call names them): the direct call, the call with the manager's row blocks, and several
    projections at once."""
    p = make_problem(n, k, bits, gs, nd, t, "uniform", n + t, dev)
    if present is not None:
        p["ids_np"] = np.where(p["ids_np"] >= present, present - 1, p["ids_np"])
    else:
        p["ids_np"] = p["ids_np"].copy()
    p["ids_np"][7:9] = nd - 1 if present is None else max(present - 1, 0)
    if present == 0:                                  # one slot, a third of the tokens
        p["ids_np"][::3] = 0
    p["ids"] = torch.from_numpy(p["ids_np"]).to(dev)
    ref = o.forward_ref(p["x_np"], p["wb_np"], p["dts"], p["ids_np"])
    tiled = ops.tile_base(p["wb"])
    assert (ops._most_row_blocks(t, k, n, bits, nd, None) == 0) == (k == 8192)
    known = ops.row_blocks(p["ids"], nd, mix=ops.batch_mix((p["ids_np"] + 1).tolist()))
    for order in (None, known, ops.row_blocks(p["ids"], nd)):
        for base in (None, tiled):
            y = ops.apply_delta(p["x"], p["q"], p["s"], p["m"], p["ids"], p["wb"], order=order, base_tiled=base)
            torch.cuda.synchronize()
            assert o.rel_err(y.cpu().numpy(), ref) <= TOL
    for y in ops.apply_delta_batch(p["x"], [p["q"]] * 2, [p["s"]] * 2, [p["m"]] * 2, p["ids"], [p["wb"]] * 2):
        assert o.rel_err(y.cpu().numpy(), ref) <= TOL


class _Recorded:
    """The library, with the names of the products it launches written down."""

    def __init__(self, lib, names):
        self.lib, self.names = lib, names

    def __getattr__(self, name):
        if name.startswith("dz_multi_delta"):
            self.names.add(name.removeprefix("dz_multi_delta_"))
        return getattr(self.lib, name)


@pytest.mark.parametrize("n,k,bits,gs,nd,t,present,base,order,route", [
    # without a base weight: one delta per block, or chunks of the decode kernel
    (256, 8192, 2, -1, 9, 129, None, False, None, {"linear_chunks"}), (96, 8192, 4, 128, 3, 300, None, False, None, {"linear_chunks"}),
    (128, 8192, 2, 64, 17, 256, None, False, "known", {"linear_chunks"}), (96, 256, 2, -1, 5, 384, None, False, None, {"gemm_rows"}),
    (2048, 256, 2, -1, 24, 200, 3, False, "known", {"gemm_rows"}), (27648, 256, 2, -1, 3, 512, 2, False, "known", {"gemm_rows"}),
    (27648, 256, 2, -1, 3, 512, 1, False, "known", {"gemm"}),                            # 256-token blocks, one wave of them
    (27648, 256, 2, -1, 1, 512, None, False, None, {"gemm", "gemm_rows"}),               # the device picks
    # with one: blocks of several deltas ...
    (256, 8192, 2, -1, 9, 129, None, True, None, {"gemm_mixed"}), (96, 8192, 4, 128, 3, 300, None, True, "known", {"gemm_mixed"}),
    (27648, 256, 2, -1, 1, 449, None, True, "known", {"gemm_mixed"}), (128, 2560, 2, 64, 3, 160, None, True, "plain", {"gemm_mixed"}),
    # ... but for a short walk, a few tokens of each of many deltas, short walks in one wave of row blocks, few short chunks
    (96, 256, 2, -1, 5, 384, None, True, None, {"gemm_rows"}), (96, 8192, 2, -1, 44, 129, None, True, "known", {"linear_chunks"}),
    (256, 1280, 2, -1, 20, 170, None, True, "known", {"gemm_rows"}), (704, 1792, 4, 64, 1, 213, None, True, None, {"linear_chunks"})])
def test_route_of_a_mid_size_call(dev, monkeypatch, n, k, bits, gs, nd, t, present, base, order, route):
    """129 to 512 tokens: the products that are launched, by name, and what they give.  `order`: with row blocks whose
    maker knew the mix, or did not, or the ids alone."""
    from deltazip_amd import _lib
    p = make_problem(n, k, bits, gs, nd, t, np.arange(t) % (present or nd), n + t, dev)
    blocks = None
    if order is not None:
        blocks = ops.row_blocks(p["ids"], nd, mix=ops.batch_mix(p["ids_np"].tolist()) if order == "known" else None,
                                deltas=ops.mixed_deltas(bits, gs != -1))
    names, lib = set(), _lib.lib()
    monkeypatch.setattr(_lib, "lib", lambda: _Recorded(lib, names))
    y = ops.multi_delta_linear(p["x"], p["wb"] if base else None, p["q"], p["s"], p["m"], p["ids"], bits=bits, order=blocks)
    torch.cuda.synchronize()
    assert names == route
    assert o.rel_err(y.cpu().numpy(), o.forward_ref(p["x_np"], p["wb_np"] if base else None, p["dts"], p["ids_np"])) <= TOL


@pytest.mark.parametrize("n,k,bits,gs", [(352, 512, 2, -1), (96, 768, 4, 128)])
@pytest.mark.parametrize("t,nd,long", [(1025, 7, False), (1300, 16, False), (1025, 6, True), (1300, 5, True)])
def test_either_table_above_1024_tokens(dev, n, k, bits, gs, t, nd, long):
    """The device puts all rows into long or into short blocks and both products are launched, one over an
    empty table (`long`: ids that fill long blocks); a call that knows how narrow its layer is launches
    the short blocks alone.  Tiles, rows and no base weight, plain and added into a column slice."""
    p = make_problem(n, k, bits, gs, nd, t, "uniform", 17 * t + nd, dev)
    if long:                                              # two deltas of 256 * m tokens, the rest with another
        p["ids_np"] = np.where(np.arange(t) < 256, 1, np.where(np.arange(t) < 768, 4, 0))
    p["ids_np"] = np.random.default_rng(t).permutation(p["ids_np"])
    p["ids"] = torch.from_numpy(p["ids_np"]).to(dev)
    either = ops.row_blocks(p["ids"], nd)
    torch.cuda.synchronize()
    used = [bool((tab[:, 1] > tab[:, 0]).any()) for tab in (either.tiles, either.short)]
    assert used == [long, not long]
    narrow = ops.row_blocks(p["ids"], nd, features=n)
    assert narrow.tiles is None and narrow.short is not None
    assert ops.row_blocks(p["ids"], nd, features=1 << 16).tiles is not None
    base = o.make_x(t, n, 5)
    for w, tiled in ((p["wb"], None), (None, ops.tile_base(p["wb"])), (None, None)):
        ref = o.forward_ref(p["x_np"], None if w is None and tiled is None else p["wb_np"], p["dts"], p["ids_np"])
        for order in (either, narrow, None):
            for accumulate in (False, True):
                wide = torch.zeros(t, n + 32, dtype=torch.float16, device=dev)
                y = wide[:, 16:16 + n]
                y.copy_(torch.from_numpy(base) if accumulate else torch.full((t, n), float("nan")))
                ops.multi_delta_linear(p["x"], w, p["q"], p["s"], p["m"], p["ids"], bits=bits, out=y,
                                       accumulate=accumulate, order=order, base_tiled=tiled)
                torch.cuda.synchronize()
                want = ref + (base.astype(np.float32) if accumulate else 0)
                assert o.rel_err(y.float().cpu().numpy(), want) <= TOL
                assert not wide[:, :16].any() and not wide[:, 16 + n:].any()


@pytest.mark.parametrize("n,k,bits,gs,t", [(96, 512, 2, -1, 200), (160, 1024, 4, 128, 129), (32, 256, 2, 64, 384)])
@pytest.mark.parametrize("spare", [0, 3, -1])
def test_device_chooses_between_row_blocks_and_chunks(dev, monkeypatch, n, k, bits, gs, t, spare):
    """One launch of each is made and one of them does nothing, by the number of row blocks: exactly as many
    as the limit, fewer, and one more (`spare`: the limit over the number); every token is written once."""
    p = make_problem(n, k, bits, gs, 6, t, "uniform", 40 + n + t, dev)
    p["ids_np"][::9] = -1
    p["ids"] = torch.from_numpy(p["ids_np"]).to(dev)
    limit = ops.batch_mix((p["ids_np"] + 1).tolist()).blocks + spare
    called = []
    monkeypatch.setattr(ops, "_most_row_blocks", lambda *a: called.append(a) or limit)
    base = o.make_x(t, n, 5)
    for w, tiled in ((p["wb"], None), (p["wb"], ops.tile_base(p["wb"])), (None, None)):
        ref = o.forward_ref(p["x_np"], None if w is None else p["wb_np"], p["dts"], p["ids_np"])
        for accumulate in (False, True):
            wide = torch.zeros(t, n + 32, dtype=torch.float16, device=dev)
            y = wide[:, 16:16 + n]
            y.copy_(torch.from_numpy(base) if accumulate else torch.full((t, n), float("nan")))
            ops.multi_delta_linear(p["x"], w, p["q"], p["s"], p["m"], p["ids"], bits=bits, out=y, accumulate=accumulate,
                                   base_tiled=tiled)
            torch.cuda.synchronize()
            want = ref + (base.astype(np.float32) if accumulate else 0)
            assert o.rel_err(y.float().cpu().numpy(), want) <= TOL
            assert not wide[:, :16].any() and not wide[:, 16 + n:].any()
    assert len(called) == 6


@pytest.mark.parametrize("t", [200, 700])
def test_batched_calls_over_stacks_of_different_slot_counts(dev, t):
    """Above the fused kernel's sizes every projection is served by its own number of slots: an id that is
    in the first stack and beyond the second counts as -1 there, as in the separate call."""
    ps = [make_problem(96, 512, 2, -1, nd, t, "uniform", 60 + nd, dev) for nd in (5, 3)]
    x, ids = ps[0]["x"], ps[0]["ids"]
    args = [[p[key] for p in ps] for key in ("q", "s", "m")]
    for order in (None, ops.row_blocks(ids, 5), ops.row_blocks(ids, 3)):
        ys = ops.apply_delta_batch(x, *args, ids, [p["wb"] for p in ps], order=order)
        torch.cuda.synchronize()
        for p, y, nd in zip(ps, ys, (5, 3)):
            assert torch.equal(y, ops.apply_delta(x, p["q"], p["s"], p["m"], ids, p["wb"]))
            seen = np.where(ps[0]["ids_np"] < nd, ps[0]["ids_np"], -1)
            assert o.rel_err(y.cpu().numpy(), o.forward_ref(ps[0]["x_np"], p["wb_np"], p["dts"], seen)) <= TOL
    warned, ops._warned_bad_id = ops._warned_bad_id, True
    ops.poll_status(wait=True)                            # clears what ids beyond three slots have set
    ops._warned_bad_id = warned


@pytest.mark.parametrize("t,kind", [(33, "uniform"), (64, "zipf"), (128, "uniform"), (20, "uniform")])
def test_token_order_is_a_permutation_and_reusable(dev, t, kind):
    """dz_token_order: a permutation of the tokens in which every delta's tokens are contiguous; passing
    it to the layer call gives bit for bit what the call computes with its own grouping."""
    p = make_problem(64, 512, 4, -1, 12, t, kind, 808 + t, dev)
    order = ops.token_order(p["ids"], 12)
    torch.cuda.synchronize()
    od = order.cpu().numpy()
    assert sorted(od.tolist()) == list(range(t))
    dealt = p["ids_np"][od]
    if t > 32:
        for c in range(0, t, 32):                      # inside a chunk every delta forms one run
            ch = dealt[c:c + 32]
            runs = 1 + int((ch[1:] != ch[:-1]).sum())
            assert runs == len(set(ch.tolist()))
    y0 = ops.apply_delta(p["x"], p["q"], p["s"], p["m"], p["ids"], p["wb"])
    y1 = ops.apply_delta(p["x"], p["q"], p["s"], p["m"], p["ids"], p["wb"], order=order)
    torch.cuda.synchronize()
    assert torch.equal(y0, y1)
    assert o.rel_err(y1.cpu().numpy(), o.forward_ref(p["x_np"], p["wb_np"], p["dts"], p["ids_np"])) <= TOL



def test_batched_calls_after_a_wide_single_call(dev):
    """The arrival counters of a batch must not sit where an earlier, wider call kept partial sums:
    a launch with three K chunks over 1024 rows (384 KiB of partial sums), then a batch whose
    second call follows 128 rows; every result must still match the oracle."""
    wide = make_problem(1024, 3072, 2, -1, 2, 31, "uniform", 41, dev)
    try:
        ops.set_ksplit(3)
        ref = o.forward_ref(wide["x_np"], wide["wb_np"], wide["dts"], wide["ids_np"])
        assert o.rel_err(run_layer(wide).cpu().numpy(), ref) <= TOL
        ops.set_ksplit(4)
        k, nd, t = 2048, 5, 32
        ns = (128, 96, 32, 160)
        ps = [make_problem(n, k, 2, -1, nd, t, "uniform", 900 + 10 * j + n, dev) for j, n in enumerate(ns)]
        ids, x = ps[0]["ids"], ps[0]["x"]
        ys = ops.apply_delta_batch(x, [p["q"] for p in ps], [p["s"] for p in ps], [p["m"] for p in ps], ids,
                                   [p["wb"] for p in ps])
        torch.cuda.synchronize()
        for p, y in zip(ps, ys):
            ref = o.forward_ref(ps[0]["x_np"], p["wb_np"], p["dts"], ps[0]["ids_np"])
            assert o.rel_err(y.cpu().numpy(), ref) <= TOL
    finally:
        ops.set_ksplit(0)


def _mixed_call(p, w, tiled, table, bits, gs, y, acc, parts, deltas):
    from deltazip_amd import _lib
    t, n, k = y.shape[0], y.shape[1], p["x"].shape[1]
    sums = torch.full((parts * t * n,), float("nan"), dtype=torch.float32, device=y.device) if parts > 1 else None
    rc = _lib.lib().dz_multi_delta_gemm_mixed(
        p["x"].data_ptr(), w.data_ptr(), tiled, p["q"].data_ptr(), p["m"].data_ptr(), p["s"].data_ptr(), p["q"].shape[0], bits,
        gs, table.table.data_ptr(), table.max_blocks, deltas, y.data_ptr(), t, k, n, acc, y.stride(0), parts,
        None if sums is None else sums.data_ptr(), torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    torch.cuda.synchronize()
    return y


@pytest.mark.parametrize("n,k,bits,gs,nd,t,tiles,most", [
    (32, 256, 2, -1, 4, 129, 8, 4), (288, 512, 2, -1, 9, 300, 8, 4), (544, 768, 2, 64, 5, 517, 8, 3),
    (256, 1280, 4, 128, 7, 130, 8, 3), (96, 1536, 4, 192, 40, 257, 8, 3), (320, 512, 4, -1, 3, 400, 8, 3),
    (160, 768, 2, 192, 17, 140, 4, 2), (512, 1024, 4, 64, 20, 333, 4, 2), (64, 512, 2, -1, 1, 1000, 8, 4),
    (96, 512, 2, -1, 60, 150, 2, 1)])
def test_blocks_of_several_deltas(dev, n, k, bits, gs, nd, t, tiles, most):
    """dz_build_mixed and dz_multi_delta_gemm_mixed: every token in one row of one block, tiles of one delta,
    blocks within their limits; unsorted ids with base-only tokens, N that is no multiple of 256, whole and split K,
    rows and tiles, plain and added into a column slice.  Unsplit sums are those of the kernel with one delta
    per block, in the same order: equal bits.  Split: fp32 partial sums added once more, within one
    fp16 rounding of the unsplit result and a few fp32 ones."""
    from deltazip_amd import _lib
    L, st = _lib.lib(), torch.cuda.current_stream().cuda_stream
    p = make_problem(n, k, bits, gs, nd, t, "uniform", 77 + n + t, dev)
    p["ids_np"] = p["ids_np"].copy()
    p["ids_np"][::11] = -1
    ids = torch.from_numpy(p["ids_np"]).to(dev)
    perm, off = ops.segment(ids, nd)
    room = L.dz_mixed_blocks(t, nd, tiles, most)
    table = ops.MixedTable(torch.full((4 + room * 146,), 77, dtype=torch.int32, device=dev), room, most)
    assert L.dz_build_mixed(off.data_ptr(), perm.data_ptr(), nd, t, tiles, most, table.table.data_ptr(), room, st) == 0
    torch.cuda.synchronize()
    tab = table.table.cpu().numpy()
    blocks, seen = tab[4:].reshape(room, 146)[:tab[0]], []
    assert 0 < tab[0] <= room
    for b in blocks:
        bt, bd, slot, tend, rows = b[0], b[1], b[2:6], b[14:18], b[18:]
        assert 1 <= bt <= tiles and 0 <= bd <= most
        for tile in range(bt):
            e = int(np.searchsorted(tend[:max(bd, 1)], tile, side="right")) if bd else 0
            held = rows[16 * tile:16 * tile + 16]
            seen += [r for r in held if r >= 0]
            want = slot[e] if bd else -1
            assert all(p["ids_np"][r if r >= 0 else ~r] == want for r in held) and held[0] >= 0
        assert all(r < 0 for r in rows[16 * bt:])
    assert sorted(seen) == list(range(t))

    short = ops._block_table(t, nd, 128, dev)
    assert L.dz_build_tiles_rows(off.data_ptr(), nd, 128, short[0].data_ptr(), short[1], st) == 0
    one = torch.empty(t, n, dtype=torch.float16, device=dev)
    assert L.dz_multi_delta_gemm_rows(p["x"].data_ptr(), p["wb"].data_ptr(), 0, p["q"].data_ptr(), p["m"].data_ptr(),
                                      p["s"].data_ptr(), nd, bits, gs, short[0].data_ptr(), short[1], perm.data_ptr(),
                                      one.data_ptr(), t, k, n, 0, n, st) == 0
    ref = o.forward_ref(p["x_np"], p["wb_np"], p["dts"], p["ids_np"])
    base = torch.from_numpy(o.make_x(t, n, 5)).to(dev)
    for w, tiled in ((p["wb"], 0), (ops.tile_base(p["wb"]), 1)):
        for parts in sorted({1, min(2, k // 256), min(3, k // 256), k // 256}):
            wide = torch.zeros(t, n + 32, dtype=torch.float16, device=dev)
            y = _mixed_call(p, w, tiled, table, bits, gs, torch.full((t, n), float("nan"), dtype=torch.float16, device=dev), 0,
                            parts, most)
            assert o.rel_err(y.cpu().numpy(), ref) <= TOL
            if parts == 1:
                assert torch.equal(y, one)
            else:
                # |sum of parts - sum| <= (parts + K / 8) fp32 roundings of a value below 64, then half a unit each
                assert ((y.float() - one.float()).abs() <= 2.0**-10 * one.float().abs() + 2e-3).all()
            y = wide[:, 16:16 + n]
            y.copy_(base)
            _mixed_call(p, w, tiled, table, bits, gs, y, 1, parts, most)
            assert o.rel_err(y.float().cpu().numpy(), ref + base.float().cpu().numpy()) <= TOL
            assert not wide[:, :16].any() and not wide[:, 16 + n:].any()
    if most == 4:                                         # three deltas at most elsewhere
        assert L.dz_multi_delta_gemm_mixed(p["x"].data_ptr(), p["wb"].data_ptr(), 0, p["q"].data_ptr(), p["m"].data_ptr(),
                                           p["s"].data_ptr(), nd, 4, -1, table.table.data_ptr(), room, 4, one.data_ptr(), t, k,
                                           n, 0, n, 1, None, st) == -2


@pytest.mark.parametrize("t,nd", [(1, 1), (129, 0), (200, 5), (1024, 17), (1025, 3), (5000, 768)])
@pytest.mark.parametrize("small", [0, 1])
def test_order_and_table_in_one_launch(dev, t, nd, small):
    """dz_order_mixed writes the order and the blocks that dz_segment and dz_build_mixed write, and reports bad ids."""
    from deltazip_amd import _lib
    L, st = _lib.lib(), torch.cuda.current_stream().cuda_stream
    ids_np = np.random.default_rng(t + nd).integers(-1, nd, t)
    tiles, most = ops.MIXED_BLOCKS[small]
    room = L.dz_mixed_blocks(t, nd, tiles, most)
    for bad in (False, True):
        if bad:
            ids_np[t // 2] = nd + 3
        ids = torch.from_numpy(ids_np).to(dev)
        perm, off = ops.segment(ids, nd)
        want, got = (torch.zeros(4 + room * 146, dtype=torch.int32, device=dev) for _ in range(2))
        order, status = torch.zeros(t, dtype=torch.int32, device=dev), torch.zeros(1, dtype=torch.int32, device=dev)
        assert L.dz_build_mixed(off.data_ptr(), perm.data_ptr(), nd, t, tiles, most, want.data_ptr(), room, st) == 0
        assert L.dz_order_mixed(ids.data_ptr(), t, nd, tiles, most, order.data_ptr(), got.data_ptr(), room, status.data_ptr(),
                                st) == 0
        torch.cuda.synchronize()
        assert torch.equal(order, perm) and int(status) == int(bad) and torch.equal(got, want)
    assert L.dz_order_mixed(ids.data_ptr(), t, 769, tiles, most, order.data_ptr(), got.data_ptr(), room, None, st) != 0
    assert L.dz_order_mixed(ids.data_ptr(), t, nd, tiles, most, order.data_ptr(), got.data_ptr(), room - 1, None, st) != 0


def test_blocks_of_several_deltas_keep_tokens_apart(dev):
    """A block's tokens share tiles of activations and nothing else: an infinite scale reaches its own delta's
    tokens only, an infinite or NaN activation its own token only."""
    p = make_problem(256, 1280, 2, -1, 6, 300, "uniform", 9, dev)
    plan = ops._mixed_plan(300, 1280, 256)
    assert plan is not None
    clean = run_layer(p)
    s = p["s"].clone()
    s[2] = float("inf")
    x = p["x"].clone()
    x[17, 5], x[44, 1000] = float("inf"), float("nan")
    y = run_layer(dict(p, s=s, x=x))
    touched = torch.from_numpy(p["ids_np"] == 2).to(dev)
    touched[[17, 44]] = True
    assert torch.equal(y[~touched], clean[~touched])
    assert not torch.isfinite(y[17]).all() and torch.isnan(y[44]).all()


@pytest.mark.parametrize("t,n,k,parts", [(200, 1280, 2560, 2), (700, 12288, 1280, 1)])
def test_blocks_of_several_deltas_under_capture(dev, t, n, k, parts):
    """A captured call over blocks of several deltas reads the ids of the replay, and gives the eager call's bits,
    with tensors of other sizes made and dropped in between."""
    p = make_problem(n, k, 2, -1, 5, t, "uniform", 3, dev)
    assert ops._mixed_plan(t, k, n)[1] >= parts
    ids = p["ids"].clone()
    tiled = ops.tile_base(p["wb"])
    call = lambda: ops.apply_delta(p["x"], p["q"], p["s"], p["m"], ids, p["wb"], base_tiled=tiled)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(side):
        call()
        torch.cuda.synchronize()
        with torch.cuda.graph(graph, stream=side):
            y = call()
    torch.cuda.current_stream().wait_stream(side)
    rng = np.random.default_rng(t)
    for rep in range(4):
        ids.copy_(torch.from_numpy(rng.integers(-1, 5, t) if rep else np.zeros(t, dtype=np.int64)))
        want = call()
        blocks = ops.row_blocks(ids, 5, deltas=ops.mixed_deltas(2, False))
        known = ops.apply_delta(p["x"], p["q"], p["s"], p["m"], ids, p["wb"], order=blocks, base_tiled=tiled)
        junk = torch.full((1 + rep, t), 1 << 20, dtype=torch.int32, device=dev)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want) and torch.equal(known, want), rep
        del junk


@pytest.mark.parametrize("bits,gs,t,met", [(2, -1, 33, 3), (2, -1, 128, 16), (4, 128, 96, 8), (4, -1, 70, 1)])
def test_decode_batches_of_few_deltas(dev, bits, gs, t, met):
    """33 to 128 tokens of few deltas over a layer of 25 M weights: with the blocks its maker hands on the call
    goes in blocks of several deltas, without them through the decode kernel; the two differ by the order of fp32
    sums (as between parts of K) and one rounding.  Bad ids are reported either way; blocks of another batch
    are refused."""
    from deltazip_amd.synthetic import gaussian_native_stack
    n, k, S = 10240, 2560, 20
    gen = torch.Generator(device=dev).manual_seed(t)
    q, m, s = gaussian_native_stack(k, n, bits, k if gs == -1 else gs, 4, dev, gen)
    q, m, s = (v.repeat((5,) + (1,) * (v.dim() - 1)).contiguous() for v in (q, m, s))
    w, x = (torch.randn(n, k, device=dev, generator=gen) * 0.02).half(), torch.randn(t, k, device=dev, generator=gen).half()
    tiled, ids_np = ops.tile_base(w), np.random.default_rng(t).integers(0, met, t)
    ids_np[:met] = np.arange(met)
    ids_np[t // 2] = -1 if met < 8 else 0
    ids = torch.from_numpy(ids_np).to(dev)
    mix = ops.batch_mix(ids_np.tolist())
    assert ops.mixes_at_decode(t, k, n, mix.deltas)
    order = ops.token_order(ids, S)
    blocks = ops.row_blocks(ids, S, mix=mix, deltas=ops.mixed_deltas(bits, gs != -1), order=order)
    call = lambda o_, i=ids: ops.apply_delta(x, q, s, m, i, w, order=o_, base_tiled=tiled)
    y, y0 = call(blocks), call(order)
    torch.cuda.synchronize()
    assert ((y.float() - y0.float()).abs() <= 2.0**-10 * y0.float().abs() + 2e-3).all()
    assert not torch.equal(y, y0)                          # (it did go the other way)
    assert torch.equal(call(ops.row_blocks(ids, S, order=order)), y0)   # (their maker did not count the deltas)
    with pytest.raises(ValueError):
        ops.apply_delta(x[:32 + 1], q, s, m, ids[:33].contiguous() if t != 33 else torch.cat([ids, ids])[:40], w, order=blocks)
    ops.poll_status(wait=True)
    bad = torch.where(ids == 0, torch.full_like(ids, S + 3), ids)
    base = torch.where(ids == 0, torch.full_like(ids, -1), ids)
    made = [ops.row_blocks(i, S, mix=mix, deltas=3, order=ops.token_order(i, S)) for i in (bad, base)]
    yb, yg = call(made[0], bad), call(made[1], base)
    torch.cuda.synchronize()
    assert torch.equal(yb, yg) and ops.workspace_status() == ops.STATUS_BAD_ID
    warned, ops._warned_bad_id = ops._warned_bad_id, True
    ops.poll_status(wait=True)
    ops._warned_bad_id = warned


def test_decode_blocks_of_each_stream(dev):
    """The tables a decode step's layers make for themselves: one set per stream, equal bits from each and from tables
    handed over, and the token order for a layer that takes no blocks and for a captured call."""
    from deltazip_amd.synthetic import gaussian_native_stack
    n, k, S, t = 10240, 2560, 4, 100
    gen = torch.Generator(device=dev).manual_seed(t)
    q, m, s = gaussian_native_stack(k, n, 4, k, S, dev, gen)
    w, x = (torch.randn(n, k, device=dev, generator=gen) * 0.02).half(), torch.randn(t, k, device=dev, generator=gen).half()
    ids_np = np.random.default_rng(t).integers(-1, S, t)
    ids = torch.from_numpy(ids_np).to(dev)
    order = ops.token_order(ids, S)
    made = ops.DecodeBlocks(ids, S, ids_np.tolist(), len(set(ids_np.tolist())), 3)
    want = ops.apply_delta(x, q, s, m, ids, w, order=ops.row_blocks(ids, S, mix=ops.batch_mix(ids_np.tolist()), order=order))
    assert made.for_layer(1024, 1024, order) is order
    streams = [torch.cuda.current_stream(), torch.cuda.Stream()]
    streams[1].wait_stream(streams[0])
    for turn in range(2):
        for stream in streams:
            with torch.cuda.stream(stream):
                blocks = made.for_layer(n, k, order)
                y = ops.apply_delta(x, q, s, m, ids, w, order=blocks)
            torch.cuda.synchronize()
            assert torch.equal(y, want) and blocks.mixed[1] is None
    assert len(made.made) == 2
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(streams[1]), torch.cuda.graph(graph, stream=streams[1]):
        assert made.for_layer(n, k, order) is order
        y.add_(0)
    torch.cuda.synchronize()


@pytest.mark.parametrize("n,k", [(32, 512), (288, 2048), (64, 2304), (96, 4096), (32, 4352), (288, 8192), (32, 8448), (64, 16384),
                                 (32, 16640)])
@pytest.mark.parametrize("bits", [2, 4])
def test_compressor_of_whole_rows(dev, n, k, bits):
    """One scale per row, at the edges of the k-blocks a wavefront holds and beyond the longest row held whole: the
    bytes of the separate passes (dz_quant_scales, dz_pack_2of4), for ordinary rows and for rows of zeros, of one
    sign, with a single value, with infinities and NaNs."""
    gen = torch.Generator(device=dev).manual_seed(n + k)
    d = torch.randn(n, k, device=dev, generator=gen) * 1e-3
    d[0] = 0
    d[1] = d[1].abs()
    d[2, :] = -0.0
    d[3] = 0
    d[3, k - 1] = -7.0
    d[17, 5], d[18, 256], d[19] = float("inf"), float("nan"), float("nan")
    d[20] = d[20].sign() * 1e-40
    q, m, s = ops.compress_delta(d, bits)
    s32, s16 = ops.quant_scales(d, bits)
    q0, m0 = ops.pack_2of4(d, s32, bits)
    torch.cuda.synchronize()
    assert torch.equal(s.view(torch.int16), s16.view(torch.int16)) and torch.equal(q, q0) and torch.equal(m, m0)


@pytest.mark.parametrize("t", [1, 32, 33, 128])
def test_one_call_with_a_token_order(dev, t):
    """dz_multi_delta_linear_ordered over rows, tiles and no base weight, with the order and without: the bits of the entry
    for several calls."""
    from deltazip_amd import _lib
    n, k, nd = 96, 1280, 5
    p = make_problem(n, k, 2, -1, nd, t, "uniform", 7 * t, dev)
    L, st, tiles = _lib.lib(), torch.cuda.current_stream().cuda_stream, ops.tile_base(p["wb"])
    order = ops.token_order(p["ids"], nd) if t > 32 else None
    ws = torch.zeros(L.dz_workspace_bytes(t, k, n), dtype=torch.uint8, device=dev)
    ref = o.forward_ref(p["x_np"], p["wb_np"], p["dts"], p["ids_np"])
    for w, tiled in ((p["wb"], 0), (tiles, 1), (None, 0)):
        for perm in ([None, order] if order is not None else [None]):
            y = torch.full((t, n), float("nan"), dtype=torch.float16, device=dev)
            assert L.dz_multi_delta_linear_ordered(
                p["x"].data_ptr(), None if w is None else w.data_ptr(), tiled, p["q"].data_ptr(), p["m"].data_ptr(),
                p["s"].data_ptr(), p["ids"].data_ptr(), y.data_ptr(), t, k, n, nd, 2, -1, 0, n,
                None if perm is None else perm.data_ptr(), ws.data_ptr(), ws.numel(), st) == 0
            torch.cuda.synchronize()
            if w is not None:
                assert o.rel_err(y.cpu().numpy(), ref) <= TOL
            want = torch.zeros_like(y)
            ops.multi_delta_linear(p["x"], w if not tiled else None, p["q"], p["s"], p["m"], p["ids"], bits=2, out=want,
                                   accumulate=w is None, order=perm, base_tiled=w if tiled else None)
            assert torch.equal(y, want)
    assert L.dz_multi_delta_linear_ordered(None, None, 0, p["q"].data_ptr(), p["m"].data_ptr(), p["s"].data_ptr(),
                                           p["ids"].data_ptr(), y.data_ptr(), t, k, n, nd, 2, -1, 0, n, None, ws.data_ptr(),
                                           ws.numel(), st) != 0


@pytest.mark.parametrize("n,k,bits,gs,t,usual", [(5120, 2560, 2, -1, 333, 4), (2048, 3072, 4, 128, 512, 3), (1280, 1536, 2, 64, 129, 6),
                                                 (96, 512, 2, -1, 2300, 2)])
def test_parts_of_k_by_the_blocks_a_batch_has(dev, n, k, bits, gs, t, usual):
    """ksplit < 0: the parts that dz_mixed_parts gives for the blocks in the table, bit for bit, from the fewest blocks to more
    than 16, a whole walk among them (nothing to sum, and the sums stay as they are); without room for sums it is refused."""
    from deltazip_amd import _lib
    L, seen = _lib.lib(), set()
    p = make_problem(n, k, bits, gs, 40, t, "uniform", n + t, dev)
    fewest = -(-t // 128)
    room = max(L.dz_mixed_parts(t, k, n, b, usual) for b in range(min(fewest, 16), 17))
    for deltas in (1, 3, 7, 12, 20, 40):
        ids = p["ids"] % deltas
        table = ops.own_mixed_table(ids, 40, 0, 3)
        used = int(table.table[0])
        parts = L.dz_mixed_parts(t, k, n, min(max(used, fewest), 16), usual)
        seen.add(parts)
        args = (p["x"].data_ptr(), p["wb"].data_ptr(), 0, p["q"].data_ptr(), p["m"].data_ptr(), p["s"].data_ptr(), 40, bits, gs,
                table.table.data_ptr(), table.max_blocks, table.deltas)
        st, got = torch.cuda.current_stream().cuda_stream, []
        for ksplit in (parts, -usual):
            y = torch.full((t, n), float("nan"), dtype=torch.float16, device=dev)
            sums = torch.full((room * t * n,), 7.0, dtype=torch.float32, device=dev)
            assert L.dz_multi_delta_gemm_mixed(*args, y.data_ptr(), t, k, n, 0, n, ksplit, sums.data_ptr(), st) == 0
            torch.cuda.synchronize()
            got.append(y)
            if parts == 1:
                assert bool((sums == 7.0).all())
        assert torch.equal(*got) and not torch.isnan(got[0]).any(), (deltas, used, parts)
    assert len(seen) > 1 or t > 512
    assert L.dz_multi_delta_gemm_mixed(*args, y.data_ptr(), t, k, n, 0, n, -usual, None, st) != 0
    assert L.dz_multi_delta_gemm_mixed(*args, y.data_ptr(), t, k, n, 0, n, 0, sums.data_ptr(), st) != 0
    assert L.dz_multi_delta_gemm_mixed(*args, y.data_ptr(), t, k, n, 0, n, -(k // 256) - 1, sums.data_ptr(), st) != 0

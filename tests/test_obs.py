"""Hessian-aware compression on the GPU (dz_hessian_add, dz_obs_sweep, dz_quant_scales,
dz_pack_2of4 through the C ABI) against the oracle's restatement of
deltazip/core/sparsegpt.py:25-146: bit for bit, since both sum in the same order."""
import numpy as np
import pytest
import torch

from oracle import dz_oracle as o
from deltazip_amd import ops
from deltazip_amd.sparsegpt import Quantizer, SparseGPT

pytestmark = pytest.mark.gpu


def _inputs(n, k, tokens, seed):
    rng = np.random.default_rng(seed)
    W = (rng.standard_normal((n, k)) * 0.01).astype(np.float32)
    X = rng.standard_normal((tokens, k)).astype(np.float32)
    X = (X + 0.5 * np.roll(X, 1, axis=1)).astype(np.float16)       # layer inputs are fp16
    return W, X


def test_hessian_add_bit_exact(dev):
    k = 256
    _, xa = _inputs(4, k, 3 * 40, 1)
    _, xb = _inputs(4, k, 77, 2)
    H = torch.zeros(k, k, dtype=torch.float32, device=dev)
    n = ops.hessian_add(H, torch.from_numpy(xa).to(dev), 0, 3)            # 3 samples of 40 tokens
    n = ops.hessian_add(H, torch.from_numpy(xb).float().to(dev), n, 1)    # one more, passed as fp32
    torch.cuda.synchronize()
    Href, nref = o.hessian_add_batch_ref(np.zeros((k, k), np.float32), 0, xa.reshape(3, 40, k))
    Href, nref = o.hessian_add_batch_ref(Href, nref, xb)
    assert n == nref == 4
    assert np.array_equal(H.cpu().numpy(), Href)


@pytest.mark.parametrize("n,k,bits,quant,prune", [(32, 256, 4, True, (2, 4)), (64, 384, 2, True, (2, 4)),
                                                  (32, 256, 4, False, (2, 4)), (40, 256, 4, True, (0, 0)),
                                                  (32, 256, 4, True, (4, 8)), (33, 128, 2, True, (1, 2)),
                                                  (256, 1024, 4, True, (2, 4))])
def test_obs_sweep_bit_exact(dev, n, k, bits, quant, prune):
    W, X = _inputs(n, k, 1024, 10 + n + k + bits)
    H, _ = o.hessian_add_batch_ref(np.zeros((k, k), np.float32), 0, X[:256] if k > 512 else X)
    if k > 512:
        H = H + np.eye(k, dtype=np.float32)                 # fewer samples than columns: keep it well conditioned
    hinv, W0 = o.hinv_upper_ref(H, W)
    scale, _ = o.find_params_sym(W, bits)
    sc = scale[:, 0].copy() if quant else None
    pn, pm = prune
    want, want_loss = o.obs_sweep_ref(W0, hinv, sc, bits, pn, pm)
    Wd = torch.from_numpy(W0.copy()).to(dev)
    loss = ops.obs_sweep(Wd, torch.from_numpy(hinv).to(dev), torch.from_numpy(sc).to(dev) if quant else None,
                         bits, pn, pm)
    torch.cuda.synchronize()
    assert np.array_equal(Wd.cpu().numpy(), want)
    assert np.array_equal(loss.cpu().numpy(), want_loss)
    # with errors of one block in the workspace instead of two: block after block
    from deltazip_amd import _lib
    Wd, hd = torch.from_numpy(W0.copy()).to(dev), torch.from_numpy(hinv).to(dev)
    scd = torch.from_numpy(sc).to(dev) if quant else None
    err, loss = torch.empty(n, 128, device=dev), torch.zeros(n, device=dev)
    assert _lib.lib().dz_obs_sweep(Wd.data_ptr(), hd.data_ptr(), scd.data_ptr() if quant else None, n, k, bits, pn, pm,
                                   err.data_ptr(), loss.data_ptr(), torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    assert np.array_equal(Wd.cpu().numpy(), want)
    assert np.array_equal(loss.cpu().numpy(), want_loss)


@pytest.mark.parametrize("k,tokens,half", [(64, 1, True), (128, 31, True), (192, 33, False), (320, 64, True), (320, 95, False)])
def test_hessian_tiles_bit_exact(dev, k, tokens, half):
    """Edges of the 64-column tiles and 32-token stages; the old value need not be symmetric, since
    either side of the diagonal scales its own."""
    rng = np.random.default_rng(k + tokens)
    x = rng.standard_normal((tokens, k)).astype(np.float16 if half else np.float32)
    H0 = rng.standard_normal((k, k)).astype(np.float32)
    buf = torch.zeros(tokens * k + 1, dtype=torch.float16 if half else torch.float32, device=dev)
    buf[1:] = torch.from_numpy(x).to(dev).view(-1)
    for xd in (torch.from_numpy(x).to(dev), buf[1:].view(tokens, k)):          # aligned, and to its elements only
        H = torch.from_numpy(H0.copy()).to(dev)
        assert ops.hessian_add(H, xd, 2, 1) == 3
        want, _ = o.hessian_add_batch_ref(H0.copy(), 2, x.reshape(1, tokens, k))
        assert np.array_equal(H.cpu().numpy(), want)


@pytest.mark.parametrize("k,tokens,half", [(64, 66, True), (576, 129, False), (1856, 17, True), (1920, 40, True), (2048, 37, False),
                                           (2112, 5, True)])
def test_hessian_rounds_of_tiles_bit_exact(dev, k, tokens, half):
    """Quarter tiles alone (64 to 1856 columns), whole ones alone (1920), whole ones and a few quartered ones (2048,
    2112), at the edges of their 32- and 64-token stages."""
    rng = np.random.default_rng(k + tokens)
    x = rng.standard_normal((tokens, k)).astype(np.float16 if half else np.float32)
    H0 = rng.standard_normal((k, k)).astype(np.float32)
    H = torch.from_numpy(H0.copy()).to(dev)
    assert ops.hessian_add(H, torch.from_numpy(x).to(dev), 2, 1) == 3
    want, _ = o.hessian_add_batch_ref(H0.copy(), 2, x.reshape(1, tokens, k))
    assert np.array_equal(H.cpu().numpy(), want)


def test_hessian_factor_zero_is_still_a_product(dev):
    """scale_x = 0: 0 times an infinite or NaN input is NaN, in the input's rows and columns; only the
    places beyond the last token are filled with zeros."""
    from deltazip_amd import _lib
    k, tokens = 128, 33
    x = torch.ones(tokens, k, dtype=torch.float16, device=dev)
    x[32, 3], x[5, 100] = float("inf"), float("nan")
    H = torch.ones(k, k, device=dev)
    assert _lib.lib().dz_hessian_add(H.data_ptr(), x.data_ptr(), 1, tokens, k, 0.5, 0.0,
                                     torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    want = torch.full((k, k), 0.5)
    for c in (3, 100):
        want[c], want[:, c] = float("nan"), float("nan")
    assert np.array_equal(H.cpu().numpy(), want.numpy(), equal_nan=True)


@pytest.mark.parametrize("n,k,quant,prune", [(1, 128, True, (2, 4)), (17, 256, True, (2, 4)), (17, 256, False, (2, 4)),
                                             (50, 384, True, (1, 8)), (50, 384, False, (3, 8)), (16, 128, True, (1, 2)),
                                             (65, 256, False, (0, 0))])
def test_obs_sweep_values_outside_the_fast_range(dev, n, k, quant, prune):
    """Zeros, values too small or too large for division by a reciprocal, a zero row, rows whose scale
    is out of range and a diagonal entry out of range: the ordinary divisions take over, and the result
    stays the oracle's bit for bit."""
    bits = 4
    W, X = _inputs(n, k, 1024, 90 + n + k)
    H, _ = o.hessian_add_batch_ref(np.zeros((k, k), np.float32), 0, X)
    hinv, W0 = o.hinv_upper_ref(H, W)
    rng = np.random.default_rng(5)
    W0[rng.random((n, k)) < 0.02] = 0
    W0[:, 9] = 0                                                   # a dead column
    W0[rng.random((n, k)) < 0.01] *= np.float32(1e-30)
    if n > 16:
        W0[3, 40] = np.float32(3e13)
        W0[5] = 0
        W0[7] *= np.float32(2.0 ** -60)                            # and with it the row's scale
    if n == 50:
        hinv[k - 3, k - 3] = np.float32(2.0 ** -25)
    sc = o.find_params_sym(W0, bits)[0][:, 0].copy() if quant else None
    pn, pm = prune
    want, want_loss = o.obs_sweep_ref(W0.copy(), hinv, sc, bits, pn, pm)
    Wd = torch.from_numpy(W0.copy()).to(dev)
    loss = ops.obs_sweep(Wd, torch.from_numpy(hinv).to(dev), torch.from_numpy(sc).to(dev) if quant else None,
                         bits, pn, pm)
    torch.cuda.synchronize()
    assert np.array_equal(Wd.cpu().numpy(), want, equal_nan=True)
    assert np.array_equal(loss.cpu().numpy(), want_loss, equal_nan=True)


@pytest.mark.parametrize("prune", [(1, 2), (2, 4), (3, 8)])
def test_obs_sweep_ties_keep_the_lower_column(dev, prune):
    """Columns of a group that are equally far from zero, in the range of the fast turns: the lower ones are pruned first, as
    in the oracle.  With an inverse factor that is diagonal no error travels and every group has ties."""
    n, k = 33, 256
    rng = np.random.default_rng(11)
    W0 = (rng.choice([-2e-3, -1e-3, 1e-3, 2e-3], size=(n, k))).astype(np.float32)
    hinv = np.diag(rng.choice([0.5, 1.0], size=k // 8).repeat(8)).astype(np.float32)
    sc = o.find_params_sym(W0, 4)[0][:, 0].copy()
    want, want_loss = o.obs_sweep_ref(W0.copy(), hinv, sc, 4, *prune)
    Wd = torch.from_numpy(W0.copy()).to(dev)
    loss = ops.obs_sweep(Wd, torch.from_numpy(hinv).to(dev), torch.from_numpy(sc).to(dev), 4, *prune)
    torch.cuda.synchronize()
    assert np.array_equal(Wd.cpu().numpy(), want)
    assert np.array_equal(loss.cpu().numpy(), want_loss)


@pytest.mark.parametrize("n", [2117, 3072])
def test_obs_sweep_of_many_rows_is_that_of_its_parts(dev, n):
    """Rows are swept on their own: a call that carries errors in tiles of which the last go in halves (more than 512 of 64 x
    128 values) gives the bits of calls over a few of the rows, which need none."""
    k, rows = 2304, 1024
    g = torch.Generator(device=dev).manual_seed(n)
    W0 = torch.randn(n, k, device=dev, generator=g) * 1e-3
    hinv = torch.randn(k, k, device=dev, generator=g).mul_(0.02).triu_(1)
    hinv.diagonal().copy_(torch.rand(k, device=dev, generator=g) * 0.5 + 0.5)
    sc = W0.abs().amax(1) / 7
    W = W0.clone()
    loss = ops.obs_sweep(W, hinv, sc, 4, 2, 4)
    for r in range(0, n, rows):
        part = W0[r:r + rows].clone()
        assert torch.equal(ops.obs_sweep(part, hinv, sc[r:r + rows].clone(), 4, 2, 4), loss[r:r + rows])
        assert torch.equal(part, W[r:r + rows])
    assert torch.isfinite(W).all()


@pytest.mark.parametrize("n,k", [(3072, 2688), (3050, 2688), (1024, 2432), (1460, 2304)])
def test_obs_sweep_keeps_the_first_half_round_of_the_rest_whole(dev, n, k):
    """Up to 912 tiles, 400 beyond 512: 256 of those stay whole and 144 go in halves, launch by launch fewer; 272 and 368 tiles,
    of which 16 and 112 go in halves, and fewer, which stay whole.  The bits are
    those of calls over 512 rows, whose tiles (152 and fewer) all stay whole."""
    g = torch.Generator(device=dev).manual_seed(n + k)
    W0 = torch.randn(n, k, device=dev, generator=g) * 1e-3
    hinv = torch.randn(k, k, device=dev, generator=g).mul_(0.02).triu_(1)
    hinv.diagonal().copy_(torch.rand(k, device=dev, generator=g) * 0.5 + 0.5)
    sc = W0.abs().amax(1) / 7
    W = W0.clone()
    loss = ops.obs_sweep(W, hinv, sc, 4, 2, 4)
    for r in range(0, n, 512):
        part = W0[r:r + 512].clone()
        assert torch.equal(ops.obs_sweep(part, hinv, sc[r:r + 512].clone(), 4, 2, 4), loss[r:r + 512])
        assert torch.equal(part, W[r:r + 512])
    assert torch.isfinite(W).all()


@pytest.mark.parametrize("prune", [(0, 0), (1, 2), (2, 4), (3, 8)])
def test_obs_sweep_without_rounding_carries_nan_and_infinity(dev, prune):
    """A weight that is no finite number spoils its row from its column on, and no other row: in the
    places the oracle's sweep has it, the rest bit for bit."""
    n, k = 20, 384
    W, X = _inputs(n, k, 1024, 321)
    H, _ = o.hessian_add_batch_ref(np.zeros((k, k), np.float32), 0, X)
    hinv, W0 = o.hinv_upper_ref(H, W)
    W0[2, 5], W0[4, 130], W0[17, 383] = np.nan, np.nan, np.nan
    W0[6, 64], W0[9, 257] = np.inf, -np.inf
    W0[11, 200], W0[11, 201] = np.nan, np.inf
    with np.errstate(invalid="ignore"):
        want, want_loss = o.obs_sweep_ref(W0.copy(), hinv, None, 4, *prune)
    Wd = torch.from_numpy(W0.copy()).to(dev)
    loss = ops.obs_sweep(Wd, torch.from_numpy(hinv).to(dev), None, 4, *prune)
    torch.cuda.synchronize()
    assert np.isnan(want[2, 200:]).any() and np.isfinite(want[[0, 1, 3, 19]]).all()
    assert np.array_equal(Wd.cpu().numpy(), want, equal_nan=True)
    assert np.array_equal(loss.cpu().numpy(), want_loss, equal_nan=True)


@pytest.mark.parametrize("n,k,bits,gs", [(64, 512, 4, -1), (96, 1024, 2, -1), (32, 512, 4, 128), (64, 256, 2, 64)])
def test_scales_with_the_search_over_the_clipping_range(dev, n, k, bits, gs):
    """dz_quant_scales_mse against the oracle's restatement of quant.py:85-101.  The candidates'
    errors are sums of |d| ** 2.4 whose last bits depend on the pow routine and the order of the
    sum, so where two candidates are within 1e-5 of each other either may win; everywhere else the
    chosen scale is the oracle's, bit for bit."""
    W, _ = _inputs(n, k, 8, 40 + n + bits)
    W[3, 5] = 25 * np.abs(W).max()                                # a row with an outlier
    W[7] = 0                                                      # an all-zero row
    W[9] = np.abs(W[9])                                           # a row without a negative value
    s32, s16 = ops.quant_scales(torch.from_numpy(W).to(dev), bits, gs, mse=True)
    scale, _, errs = o.find_params_sym(W, bits, gs, mse=True, return_errors=True)      # [N, G], [80, N, G]
    plain, _ = o.find_params_sym(W, bits, gs)
    got = s32.cpu().numpy().T                                                            # [N, G]
    assert got.shape == scale.shape
    differ = got != scale
    assert differ.mean() < 0.05
    for r, g in zip(*np.nonzero(differ)):
        cand = np.array([np.float32(np.float32(1 - i / 100) * plain[r, g]) for i in range(80)])
        i_got = int(np.argmin(np.abs(cand - got[r, g])))
        assert abs(cand[i_got] - got[r, g]) <= 1e-6 * got[r, g]                          # one of the candidates ...
        assert errs[i_got, r, g] <= errs[:, r, g].min() * (1 + 1e-5)                     # ... and as good as the best
    assert (got <= plain).all() and (got < plain).any()           # the search only ever shrinks the range
    assert np.array_equal(s16.cpu().numpy().view(np.uint16), s32.cpu().numpy().astype(np.float16).view(np.uint16))
    # the Quantizer front end with the reference's keywords
    from deltazip_amd.sparsegpt import Quantizer
    qz = Quantizer()
    qz.configure(bits, perchannel=True, sym=True, mse=True, norm=2.4, grid=100, maxshrink=0.8)
    qz.find_params(torch.from_numpy(W).to(dev), weight=True)
    if gs == -1:
        assert torch.equal(qz.scale[:, 0], s32[0]) and float(qz.zero[0, 0]) == 2 ** (bits - 1)


@pytest.mark.parametrize("n,k,bits,gs", [(32, 256, 4, 64), (64, 1280, 2, 128), (96, 256, 2, 256), (32, 1280, 4, 256),
                                         (32, 768, 4, 192), (64, 1024, 2, 64), (32, 3072, 4, 1024), (32, 5120, 2, -1)])
def test_scales_of_grouped_columns(dev, n, k, bits, gs):
    """Plain scales for every group length, K / 256 a multiple of four and not: the oracle's, bit for bit,
    with an all-zero row, one without a negative value and one with an outlier."""
    W, _ = _inputs(n, k, 8, 60 + n + bits)
    W[0] = 0
    W[2] = np.abs(W[2])
    W[4, 3] = 30 * np.abs(W).max()
    s32, s16 = ops.quant_scales(torch.from_numpy(W).to(dev), bits, gs)
    scale, _ = o.find_params_sym(W, bits, gs)
    assert np.array_equal(s32.cpu().numpy().T, scale)
    assert np.array_equal(s16.cpu().numpy().T.view(np.uint16), scale.astype(np.float16).view(np.uint16))


def test_scales_and_pack_match_the_reference_pipeline(dev):
    """Values on the grid with two zeros per group of four -> the same native bytes as compressing
    and packing the reference's way (oracle) and converting with the repacker."""
    n, k, bits = 64, 512, 4
    W, X = _inputs(n, k, 512, 3)
    s32, s16 = ops.quant_scales(torch.from_numpy(W).to(dev), bits)
    scale, zero = o.find_params_sym(W, bits)
    assert np.array_equal(s32.cpu().numpy()[0], scale[:, 0])
    assert np.array_equal(s16.cpu().numpy()[0].view(np.uint16), scale[:, 0].astype(np.float16).view(np.uint16))
    H, _ = o.hessian_add_batch_ref(np.zeros((k, k), np.float32), 0, X)
    hinv, W0 = o.hinv_upper_ref(H, W)
    out, _ = o.obs_sweep_ref(W0, hinv, scale[:, 0], bits)
    q, m = ops.pack_2of4(torch.from_numpy(out).to(dev), s32, bits)
    torch.cuda.synchronize()
    codes = o.quantize_codes(out, scale, zero, 2**bits - 1)                    # [N, K]
    qw, qz, sc16, gi = o.pack_codes_gptq(np.ascontiguousarray(codes.T), zero.T.astype(np.int32),
                                         scale.T.astype(np.float16), bits)
    rq, rm, rs = ops.repack_gptq_to_native(torch.from_numpy(qw), torch.from_numpy(qz), torch.from_numpy(sc16),
                                           torch.from_numpy(gi), bits)
    assert torch.equal(q.cpu(), rq) and torch.equal(m.cpu(), rm)
    # and the packed delta dequantises to the swept values rounded to fp16 the reference's way
    dq = ops.dequant(q, m, s16, k, n, bits).cpu().numpy()
    assert np.array_equal(dq, o.dequant_gptq(qw, qz, sc16, gi, bits).T)


def test_sparsegpt_interface_end_to_end(dev):
    """SparseGPT(layer).add_batch / fasterprune / pack with the reference's call sequence
    (deltazip/modeling/_base.py:399-470): the layer ends up holding base + compressed delta, the
    compensation lowers the layer's output error below plain magnitude pruning + rounding."""
    n, k, bits = 64, 256, 4
    rng = np.random.default_rng(7)
    base = (rng.standard_normal((n, k)) * 0.02).astype(np.float16)
    delta, X = _inputs(n, k, 2048, 8)
    target = (base.astype(np.float32) + delta).astype(np.float16)
    layer = torch.nn.Linear(k, n, bias=False, dtype=torch.float16, device=dev)
    layer.weight.data = torch.from_numpy(target).to(dev)
    gpt = SparseGPT(layer)
    gpt.quantizer = Quantizer()
    gpt.quantizer.configure(bits, perchannel=True, sym=True, mse=False)
    xs = torch.from_numpy(X).to(dev)
    for i in range(0, 2048, 512):
        gpt.add_batch(xs[i:i + 512].reshape(4, 128, k), None)
    assert gpt.nsamples == 16
    scale, zero, g_idx, avg_loss, Wc = gpt.fasterprune(0.5, prunen=2, prunem=4, base_weight=torch.from_numpy(base).to(dev))
    torch.cuda.synchronize()
    assert tuple(scale.shape) == (n, 1) and float(zero[0, 0]) == 8 and int(g_idx.abs().sum()) == 0 and avg_loss > 0
    d32 = target.astype(np.float32) - base.astype(np.float32)
    got = Wc.float().cpu().numpy()
    assert ((got.reshape(n, -1, 4) == 0).sum(axis=2) >= 2).all()
    sc, zr = o.find_params_sym(d32, bits)
    plain = o.quantize(np.where(o.prune_2of4_magnitude(d32), d32, np.float32(0)), sc, zr, 15)
    xf = X.astype(np.float32)
    assert np.linalg.norm((d32 - got) @ xf.T) < 0.95 * np.linalg.norm((d32 - plain) @ xf.T)
    assert torch.equal(layer.weight.data, (Wc + torch.from_numpy(base).to(dev)).half())
    q, m, s16 = gpt.pack()
    dq = ops.dequant(q, m, s16, k, n, bits).float().cpu().numpy()
    assert np.allclose(dq, got, rtol=2e-3, atol=1e-7)
    gpt.free()
    with pytest.raises(NotImplementedError):
        SparseGPT(layer).fasterprune(0.5)                       # unstructured sparsity
    with pytest.raises(NotImplementedError):
        SparseGPT(layer).fasterprune(0.0, actorder=True)

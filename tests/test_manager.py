"""Slot manager: bookkeeping on the CPU (no kernels), the oracle's convert_mapping restatement
against hand-computed answers, and on the GPU the device-side mapping and a checkpoint -> manager
-> layer forward pass checked against the oracle."""
from types import SimpleNamespace

import numpy as np
import pytest
import torch
import torch.nn as nn

from oracle import dz_oracle as o
from deltazip_amd import (DeltaConfig, DeltaMapping, DeltaModel, CompressionConfig, LRUCacheDeltaModelManager,
                          DeltaModelManager, create_delta_manager, convert_model)
from deltazip_amd.layers import (LinearWithDelta, MergedQKVParallelLinearWithDelta, MergedColumnParallelLinearWithDelta,
                                 RowParallelLinearWithDelta, VocabParallelEmbeddingWithDelta,
                                 LogitsProcessorWithDelta)
from deltazip_amd.manager import LRUCache
from deltazip_amd import ops

H, I, V = 256, 512, 64


class Attn(nn.Module):
    def __init__(self, dev):
        super().__init__()
        self.qkv_proj = nn.Linear(H, H + 128, bias=False, dtype=torch.float16, device=dev)
        self.o_proj = nn.Linear(H, H, bias=False, dtype=torch.float16, device=dev)


class Mlp(nn.Module):
    def __init__(self, dev):
        super().__init__()
        self.gate_up_proj = nn.Linear(H, 2 * I, bias=False, dtype=torch.float16, device=dev)
        self.down_proj = nn.Linear(I, H, bias=False, dtype=torch.float16, device=dev)


class Block(nn.Module):
    def __init__(self, dev):
        super().__init__()
        self.self_attn, self.mlp = Attn(dev), Mlp(dev)


class Inner(nn.Module):
    def __init__(self, dev, layers):
        super().__init__()
        self.embed_tokens = nn.Embedding(V, H, dtype=torch.float16, device=dev)
        self.layers = nn.ModuleList([Block(dev) for _ in range(layers)])


class ToyLogitsProcessor(nn.Module):
    """The serving engine's LogitsProcessor reduced to what the delta wrapper uses: `vocab_size`
    and a forward that calls `_get_logits(hidden_states, embedding, embedding_bias)`."""

    def __init__(self, vocab_size):
        super().__init__()
        self.vocab_size = vocab_size
        self.scale = 1.0

    def _get_logits(self, hidden_states, embedding, embedding_bias=None):
        return hidden_states @ embedding.t()

    def forward(self, embedding, hidden_states):
        return self._get_logits(hidden_states, embedding, None) * self.scale


class ToyModel(nn.Module):
    """Module tree and class attributes shaped like the serving model
    (model_executor/models/llama.py:299-340)."""
    packed_modules_mapping = {"qkv_proj": ["q_proj", "k_proj", "v_proj"], "gate_up_proj": ["gate_proj", "up_proj"]}
    supported_delta_modules = ["qkv_proj", "o_proj", "gate_up_proj", "down_proj", "embed_tokens", "lm_head"]

    def __init__(self, dev="cpu", layers=1):
        super().__init__()
        self.model = Inner(dev, layers)
        self.lm_head = nn.Linear(H, V, bias=False, dtype=torch.float16, device=dev)
        self.logits_processor = ToyLogitsProcessor(V)
        with torch.no_grad():
            g = torch.Generator().manual_seed(5)
            for p in self.parameters():
                p.copy_((torch.randn(p.shape, generator=g) * 0.02).to(p.dtype))


SHAPES = {"self_attn.q_proj": (H, H), "self_attn.k_proj": (64, H), "self_attn.v_proj": (64, H),
          "self_attn.o_proj": (H, H), "mlp.gate_proj": (I, H), "mlp.up_proj": (I, H), "mlp.down_proj": (H, I)}


def make_delta_model(delta_id, bits, seed):
    """A DeltaModel built the way a checkpoint is read, plus the reference dequantisation [N, K] of
    every fused module."""
    sd, ref = {}, {}
    for j, (name, (n, k)) in enumerate(SHAPES.items()):
        d = o.make_delta(n, k, 1e-3, bits, -1, seed + j)
        for key in ("qweight", "qzeros", "scales", "g_idx"):
            sd[f"model.layers.0.{name}.{key}"] = torch.from_numpy(d[key].copy())
        ref[name] = o.dequant_gptq(d["qweight"], d["qzeros"], d["scales"], d["g_idx"], bits)   # [K, N]
    fused = {"self_attn.qkv_proj": np.concatenate([ref[f"self_attn.{x}_proj"] for x in "qkv"], axis=1),
             "self_attn.o_proj": ref["self_attn.o_proj"],
             "mlp.gate_up_proj": np.concatenate([ref["mlp.gate_proj"], ref["mlp.up_proj"]], axis=1),
             "mlp.down_proj": ref["mlp.down_proj"]}
    g = torch.Generator().manual_seed(seed + 77)
    sd["model.embed_tokens.weight"] = (torch.randn(V, H, generator=g) * 0.02).half()
    sd["lm_head.weight"] = (torch.randn(V, H, generator=g) * 0.02).half()
    sd["model.norm.weight"] = torch.ones(H, dtype=torch.float16)
    fused["model.embed_tokens"] = sd["model.embed_tokens.weight"].numpy()
    fused["lm_head"] = sd["lm_head.weight"].numpy()
    dm = DeltaModel.from_tensors(sd, delta_id, CompressionConfig(bits=bits, prunen=2, prunem=4, sparsity=0.5),
                                 pin_memory=False)
    return dm, fused


# ---------------------------------------------------------------------------------------------
# CPU
# ---------------------------------------------------------------------------------------------
def test_row_blocks_stay_on_their_side_of_a_capture(monkeypatch):
    """Tables made outside a graph capture are gone when the graph is replayed after the next mapping
    (their row numbers would address whatever took their place), and tables made under capture
    hold nothing before a replay: a call on the other side makes its own from the indices."""
    now = [False]
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: now[0])
    perm = torch.arange(200, dtype=torch.int32)
    made = {}
    for now[0] in (False, True):
        made[now[0]] = ops.RowBlocks(perm, None, 0, 200, 3, perm, 1)
    for now[0] in (False, True):
        assert ops._usable_blocks(made[now[0]], 200, 3) is made[now[0]]
        assert ops._usable_blocks(made[not now[0]], 200, 3) is None
        assert ops._usable_blocks(perm, 200, 3) is None and ops._usable_blocks(None, 200, 3) is None
        assert ops._usable_blocks(made[now[0]], 201, 3) is None
    now[0] = False
    late = ops.RowBlocks(perm, None, 0, 600, 3, perm, 1)
    with pytest.raises(ValueError):
        ops._usable_blocks(late, 601, 3)


@pytest.mark.parametrize("t,k,n,plan", [
    (263, 1536, 1536, (1, 1)), (154, 1280, 1280, (1, 1)), (383, 1280, 1280, (1, 1)),      # the host's half: no second launch
    (401, 2560, 10240, (0, 1)), (329, 1280, 13184, (0, 1)), (479, 2560, 8736, (0, 1)),    # no second wave of small blocks
    (333, 2560, 8736, (1, 1)), (200, 2560, 1280, (1, 6))])
def test_plan_of_small_layers(t, k, n, plan):
    """A walk that is over before the host could launch a sum is not cut; small blocks only where they are one wave."""
    assert ops._mixed_plan(t, k, n) == plan


def test_batch_mix_counts_what_the_routes_meet():
    ids = [0] * 5 + [7] * 130 + [9] * 128 + [7] * 1                            # 264 tokens, three chunks
    assert ops.batch_mix(ids) == ops.BatchMix(3, 1 + 2 + 1, 131, 2 + 2 + 2)
    assert ops.batch_mix(tuple(reversed(ids))) == ops.BatchMix(3, 4, 131, 2 + 2 + 2)
    for t, s, want in ((129, 1, (1, 2, 129, 2)), (512, 16, (16, 16, 32, 19)), (300, 2, (2, 4, 150, 4)),
                       (130, 700, (130, 130, 1, 131))):
        assert ops._even_mix(t, s) == ops.BatchMix(*want)


@pytest.mark.parametrize("k,n,bits,t,deltas,chunks,rows", [
    (5120, 27648, 2, 129, 4, 251, 138), (5120, 27648, 2, 129, 16, 307, 376), (5120, 27648, 2, 129, 64, 557, 1103),
    (5120, 27648, 2, 256, 16, 433, 386), (5120, 27648, 2, 256, 24, 478, 540), (5120, 27648, 2, 384, 48, 798, 1016),
    (5120, 27648, 2, 512, 64, 1064, 1356), (5120, 27648, 2, 512, 1, 741, 238), (5120, 5120, 2, 129, 12, 81, 54),
    (5120, 5120, 2, 160, 32, 108, 140), (5120, 5120, 2, 320, 16, 151, 103), (13824, 5120, 2, 129, 1, 160, 184),
    (13824, 5120, 2, 192, 48, 324, 507), (4096, 4096, 2, 129, 1, 48, 58), (4096, 4096, 2, 129, 64, 86, 150),
    (4096, 4096, 2, 512, 48, 143, 119), (5120, 27648, 4, 192, 32, 596, 891), (5120, 27648, 4, 448, 8, 761, 337),
    (4096, 12288, 4, 129, 24, 185, 242), (4096, 12288, 4, 384, 16, 267, 173),
    # few features: the walk over K is one workgroup's, where a chunk splits it
    (13824, 512, 2, 129, 1, 46, 172), (13824, 1024, 2, 512, 4, 123, 176), (13824, 2048, 2, 256, 4, 95, 151),
    (13824, 2048, 2, 512, 16, 188, 131), (13824, 4096, 2, 384, 8, 240, 144), (8192, 1024, 4, 256, 1, 63, 137),
    (4096, 1024, 2, 256, 16, 50, 34), (1024, 4096, 2, 129, 4, 45, 14), (512, 512, 4, 300, 2, 72, 12)])
def test_the_faster_route_is_taken(k, n, bits, t, deltas, chunks, rows):
    """Measured times (us, sorted batches) of both routes on a few hundred tokens: the rule takes the
    faster one where it knows the mix."""
    ids = np.sort(np.random.RandomState(deltas + t).randint(1, deltas + 1, t)).tolist()
    for mix in (ops.batch_mix(ids), ops._even_mix(t, deltas)):
        a, b = ops._route_us(t, k, n, bits, mix)
        assert (a < b) == (chunks < rows)


@pytest.mark.parametrize("k,n,t,slots,most", [(5120, 27648, 129, 64, "device"), (5120, 27648, 256, 32, "device"),
                                              (4096, 12288, 129, 64, "device"),
                                              (5120, 27648, 129, 8, None), (13824, 1024, 256, 8, 0), (4096, 3072, 256, 2, 0),
                                              (512, 512, 300, 2, None), (512, 512, 512, 1000, 0), (1024, 13824, 129, 32, None),
                                              (13824, 512, 400, 4, None), (5120, 27648, 513, 64, None)])
def test_route_of_a_batch_whose_mix_the_host_does_not_know(k, n, t, slots, most):
    """Narrow layers go in chunks whatever the mix, small ones in row blocks; for wide ones over many
    slots the device chooses, and the limit it is given lies where the two estimates meet."""
    got = ops._most_row_blocks(t, k, n, 2, slots, None)
    assert got == most if most != "device" else 2 <= got < slots
    if got:
        for d, rows in ((got, True), (got + 1, False)):
            a, b = ops._route_us(t, k, n, 2, ops._even_mix(t, d)._replace(blocks=d, longest=128))
            assert (b <= a) == rows


@pytest.mark.parametrize("n,bits,t,short,long", [
    (27648, 2, 512, 257, 223), (28672, 2, 512, 395, 361), (32768, 2, 512, 221, 194), (24576, 2, 512, 204, 222),
    (22016, 2, 512, 157, 169), (27648, 2, 640, 320, 585), (15360, 2, 1024, 237, 391), (27648, 4, 512, 249, 257)])
def test_one_delta_takes_long_blocks_where_they_fill_one_wave(n, bits, t, short, long):
    """Measured times (us) of one delta's tokens in blocks of 128 and of 256."""
    assert ops._one_wave_of_long_blocks(t, n, bits) == (long < short)


def test_oracle_convert_mapping_known_answers():
    # slots: [id 7, free, id 3]; manager passes max_deltas = slots + 1 = 4
    base, samp, padded, emb = o.convert_mapping_ref((3, 3, 0, 7, 0), (3, 0, 7), [7, None, 3], 4, 100, 10)
    assert base.tolist() == [2, 2, -1, 0, -1]
    assert samp.tolist() == [2, -1, 0]
    assert padded.tolist() == [0 + 2 * 3, 1 + 3 * 3, 2 + 0 * 3]
    assert emb.tolist() == [[20, 20, 0, 0, 0], [220, 220, 0, 0, 0]]
    with pytest.raises(ValueError):
        o.convert_mapping_ref((5,), (), [7, None, 3], 4, 100, 0)


def test_oracle_table_selection_known_answers():
    base = np.arange(12, dtype=np.float16).reshape(4, 3)                 # row r = [3r, 3r+1, 3r+2]
    stack = np.stack([base + 100, base + 200]).astype(np.float16)
    got = o.embed_select_ref([3, 0, 2], stack, [-1, 1, 0], base)
    assert got.tolist() == [[9, 10, 11], [200, 201, 202], [106, 107, 108]]
    x = np.array([[1, 0, 0], [0, 1, 0], [1, 1, 1]], dtype=np.float16)
    y = o.linear_select_ref(x, stack, [0, -1, 1], base)
    assert y[0].tolist() == [100, 103, 106, 109]         # column 0 of table 0
    assert y[1].tolist() == [1, 4, 7, 10]                # column 1 of the base table
    assert y[2].tolist() == [603, 612, 621, 630]         # row sums of table 1


def test_lru_cache_order_and_callbacks():
    removed = []

    class C(LRUCache):
        def _on_remove(self, key, value):
            removed.append(key)

    c = C(2)
    c.put(1, "a"); c.put(2, "b"); c.get(1); c.put(3, "c")          # 2 is the oldest now
    assert removed == [2] and list(c.keys()) == [1, 3] and len(c) == 2
    c.touch(1); c.remove_oldest()
    assert removed == [2, 3] and 1 in c
    assert c.pop(1) == "a" and removed == [2, 3, 1] and c.pop(9, "x") == "x"


def test_manager_wraps_modules_and_tracks_slots(dzlib):
    model = ToyModel()
    cfg = DeltaConfig(max_deltas=2, max_bitwidth=4, max_cpu_deltas=3)
    mgr = create_delta_manager(model, 8, 64, V, cfg)
    assert isinstance(model.model.layers[0].self_attn.qkv_proj, MergedQKVParallelLinearWithDelta)
    assert isinstance(model.model.layers[0].mlp.gate_up_proj, MergedColumnParallelLinearWithDelta)
    assert isinstance(model.model.layers[0].mlp.down_proj, RowParallelLinearWithDelta)
    assert isinstance(model.model.embed_tokens, VocabParallelEmbeddingWithDelta)
    assert isinstance(model.logits_processor, LogitsProcessorWithDelta) and isinstance(model.lm_head, nn.Linear)
    assert mgr.modules["lm_head"] is model.logits_processor and model.logits_processor.scale == 1.0
    assert sorted(mgr.modules) == ["lm_head", "model.embed_tokens", "model.layers.0.mlp.down_proj",
                                   "model.layers.0.mlp.gate_up_proj", "model.layers.0.self_attn.o_proj",
                                   "model.layers.0.self_attn.qkv_proj"]
    assert mgr.packed_modules["model.layers.0.self_attn.qkv_proj"] == [
        "model.layers.0.self_attn.q_proj", "model.layers.0.self_attn.k_proj", "model.layers.0.self_attn.v_proj"]
    qkv = model.model.layers[0].self_attn.qkv_proj
    assert qkv.indices is mgr.base_indices and qkv.indices_len is mgr.indices_len
    assert model.delta_manager is mgr and mgr.capacity == 3 and mgr.delta_slots == 2

    dms = [make_delta_model(i, 4, 10 * i)[0] for i in (1, 2, 3)]
    assert [mgr.add_delta(d) for d in dms] == [True, True, True] and not mgr.add_delta(dms[0])
    with pytest.raises(RuntimeError, match="No free Delta slots"):
        mgr.add_delta(make_delta_model(4, 4, 40)[0])
    assert len(mgr) == 3 and set(mgr.list_deltas()) == {1, 2, 3} and mgr.get_delta(2) is dms[1]
    assert mgr.activate_delta(2) and not mgr.activate_delta(2) and mgr.activate_delta(1)
    assert mgr.delta_index_to_id == [2, 1]
    with pytest.raises(ValueError, match="No free delta slots"):
        mgr.activate_delta(3)
    # slot 0 of the fused qkv layer holds delta 2's tensors
    want = dms[1].get_delta("model.layers.0.self_attn.qkv_proj")
    assert torch.equal(qkv.qweight_stacked[0].reshape(-1), want.qweight.reshape(-1))
    assert torch.equal(qkv.scales_stacked[0].reshape(-1), want.scales.reshape(-1))
    assert torch.equal(model.model.embed_tokens.delta_weights[0], dms[1].get_delta("model.embed_tokens").weight)
    assert torch.equal(model.logits_processor.weight_stacked[1], dms[0].get_delta("lm_head").weight)
    assert mgr.deactivate_delta(2) and not mgr.deactivate_delta(2)
    assert mgr.delta_index_to_id == [None, 1]
    assert mgr.activate_delta(3) and mgr.delta_index_to_id == [3, 1]
    assert mgr.remove_delta(1) and mgr.delta_index_to_id == [3, None] and not mgr.remove_delta(1)
    mgr.remove_all_deltas()
    assert len(mgr) == 0 and mgr.delta_index_to_id == [None, None]
    # there is no CPU implementation of the mapping kernel
    with pytest.raises(ValueError, match="GPU"):
        mgr.set_delta_mapping(DeltaMapping((0, 0), (0,)))


def test_lru_manager_evicts_least_recently_used(dzlib):
    model = ToyModel()
    mgr = create_delta_manager(model, 8, 64, V, DeltaConfig(max_deltas=2, max_bitwidth=4, max_cpu_deltas=3),
                               delta_manager_cls=LRUCacheDeltaModelManager)
    for i in (1, 2, 3):
        assert mgr.add_delta(make_delta_model(i, 4, 10 * i)[0])
    assert not mgr.add_delta(mgr.get_delta(1))
    mgr.activate_delta(1); mgr.activate_delta(2)
    assert mgr.delta_index_to_id == [1, 2]
    mgr.activate_delta(1)                       # touch: 2 is now the least recently used
    mgr.activate_delta(3)
    assert mgr.delta_index_to_id == [1, 3]
    # host cache is full: the registered delta that was looked up longest ago (1: the second
    # activate_delta(1) returned before reading it) goes, and leaves its GPU slot as well
    mgr.add_delta(make_delta_model(4, 4, 40)[0])
    assert len(mgr) == 3 and set(mgr.list_deltas()) == {2, 3, 4} and mgr.delta_index_to_id == [None, 3]
    assert mgr.remove_oldest_delta() and len(mgr) == 2


def test_model_without_delta_support_is_refused():
    with pytest.raises(ValueError, match="not supported"):
        create_delta_manager(nn.Linear(4, 4), 1, 8, 10, DeltaConfig())


# ---------------------------------------------------------------------------------------------
# GPU
# ---------------------------------------------------------------------------------------------
@pytest.mark.gpu
@pytest.mark.parametrize("T,P,S", [(1, 1, 1), (5, 3, 3), (37, 37, 8), (300, 7, 64), (4096, 129, 700)])
def test_map_ids_matches_reference_loop(dev, T, P, S):
    from deltazip_amd import ops
    rng = np.random.default_rng(T + S)
    table = [None] * S
    resident = rng.choice(np.arange(1, 10 * S + 2), size=max(1, (2 * S) // 3), replace=False).tolist()
    for s_, d in zip(rng.permutation(S)[: len(resident)], resident):
        table[int(s_)] = int(d)
    pool = np.array(resident + [0, 0, -1])
    tok = rng.choice(pool, size=T).astype(np.int64)
    prm = rng.choice(pool, size=P).astype(np.int64)
    vocab, extra = 32000, 3
    tok_nonneg, prm_nonneg = np.maximum(tok, 0), np.maximum(prm, 0)
    want = o.convert_mapping_ref(tok_nonneg.tolist(), prm_nonneg.tolist(), table, S + 1, vocab, extra)
    n = T + 11
    base = torch.full((n,), -7, dtype=torch.long, device=dev)
    samp, padded = torch.full_like(base, -7), torch.full_like(base, -7)
    emb = torch.full((2, n), -7, dtype=torch.long, device=dev)
    missing = torch.zeros(1, dtype=torch.int32, device=dev)
    slots = torch.tensor([d if d is not None else 0 for d in table], dtype=torch.long, device=dev)
    ops.map_ids(torch.from_numpy(tok).to(dev), torch.from_numpy(prm).to(dev), slots, S + 1, vocab, extra,
                base, samp, padded, emb, missing)
    torch.cuda.synchronize()
    assert np.array_equal(base[:T].cpu().numpy(), want[0]) and np.array_equal(samp[:P].cpu().numpy(), want[1])
    assert np.array_equal(padded[:P].cpu().numpy(), want[2]) and np.array_equal(emb[:, :T].cpu().numpy(), want[3])
    # nothing written past the batch, nothing reported missing
    assert (base[T:] == -7).all() and (samp[P:] == -7).all() and (emb[:, T:] == -7).all()
    assert int(missing.item()) == 0
    # an id that is in no slot: -1 and counted
    tok2 = torch.tensor([10 * S + 5], dtype=torch.long, device=dev)
    ops.map_ids(tok2, None, slots, S + 1, vocab, extra, base, n_missing=missing)
    torch.cuda.synchronize()
    assert int(base[0].item()) == -1 and int(missing.item()) == 1


@pytest.mark.gpu
@pytest.mark.parametrize("T,S,V_,H_", [(1, 1, 64, 256), (37, 5, 1000, 264), (300, 9, 512, 4096)])
def test_embedding_select_is_exact(dev, T, S, V_, H_):
    from deltazip_amd import ops
    rng = np.random.default_rng(T)
    base = rng.standard_normal((V_, H_)).astype(np.float16)
    stack = rng.standard_normal((S, V_, H_)).astype(np.float16)
    tok = rng.integers(0, V_, size=T)
    ids = rng.integers(-1, S, size=T)
    got = ops.apply_delta_embed(torch.from_numpy(tok).to(dev), torch.from_numpy(stack).to(dev),
                                torch.from_numpy(ids).to(dev), torch.from_numpy(base).to(dev))
    torch.cuda.synchronize()
    want = o.embed_select_ref(tok, stack, ids, base)
    assert got.dtype == torch.float16 and np.array_equal(got.cpu().numpy().view(np.uint16), want.view(np.uint16))
    # a token id outside the vocabulary gives zeros, ids outside [0, S) read the base table
    got = ops.apply_delta_embed(torch.tensor([V_, 1], device=dev), torch.from_numpy(stack).to(dev),
                                torch.tensor([0, S + 3], device=dev), torch.from_numpy(base).to(dev))
    assert (got[0] == 0).all() and np.array_equal(got[1].cpu().numpy(), base[1])


@pytest.mark.gpu
@pytest.mark.parametrize("T,S,N,K", [(1, 1, 64, 256), (32, 8, 1000, 512), (128, 3, 32000, 256), (300, 4, 512, 320)])
def test_uncompressed_projection_matches_loop(dev, T, S, N, K):
    from deltazip_amd import ops
    rng = np.random.default_rng(T + N)
    base = (rng.standard_normal((N, K)) * 0.05).astype(np.float16)
    stack = (rng.standard_normal((S, N, K)) * 0.05).astype(np.float16)
    x = rng.standard_normal((T, K)).astype(np.float16)
    ids = rng.integers(-1, S, size=T)
    if T > 2:
        ids[0], ids[1] = -1, S - 1
    got = ops.apply_delta_uncompressed(torch.from_numpy(x).to(dev), torch.from_numpy(stack).to(dev),
                                       torch.from_numpy(ids).to(dev), torch.from_numpy(base).to(dev))
    torch.cuda.synchronize()
    want = o.linear_select_ref(x, stack, ids, base)
    assert tuple(got.shape) == (T, N) and o.rel_err(got.float().cpu().numpy(), want) <= 1e-2
    # all rows on the base weight: the plain product
    got = ops.apply_delta_uncompressed(torch.from_numpy(x).to(dev), torch.from_numpy(stack).to(dev),
                                       torch.full((T,), -1, dtype=torch.long, device=dev),
                                       torch.from_numpy(base).to(dev))
    ref = x.astype(np.float32) @ base.astype(np.float32).T
    assert o.rel_err(got.float().cpu().numpy(), ref) <= 1e-2


@pytest.mark.gpu
def test_uncompressed_projection_never_reads_back_to_the_host(dev):
    """The per-delta output projection is captured into a HIP graph -- which any read-back of the
    group sizes to the host would refuse -- and every replay, with eager work and synchronisations
    in between and the ids rewritten in place, gives what the eager call gives."""
    from deltazip_amd import ops
    T, S, N, K = 48, 5, 1000, 512
    rng = np.random.default_rng(99)
    base_np = (rng.standard_normal((N, K)) * 0.05).astype(np.float16)
    stack_np = (rng.standard_normal((S, N, K)) * 0.05).astype(np.float16)
    x_np = rng.standard_normal((T, K)).astype(np.float16)
    base, stack, x = (torch.from_numpy(a).to(dev) for a in (base_np, stack_np, x_np))
    ids = torch.from_numpy(rng.integers(-1, S, size=T)).to(dev)
    ops.apply_delta_uncompressed(x, stack, ids, base)          # first call outside the capture (one-time set-up)
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(side):
        with torch.cuda.graph(graph, stream=side):
            out = ops.apply_delta_uncompressed(x, stack, ids, base)
    torch.cuda.current_stream().wait_stream(side)
    for rep in range(3):
        new_ids = rng.integers(-1, S, size=T)
        if rep == 1:
            new_ids[:] = -1                                     # a batch without any delta
        ids.copy_(torch.from_numpy(new_ids).to(dev))
        eager = ops.apply_delta_uncompressed(x, stack, ids, base)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager), rep
        assert o.rel_err(out.float().cpu().numpy(), o.linear_select_ref(x_np, stack_np, new_ids, base_np)) <= 1e-2


@pytest.mark.gpu
def test_checkpoint_to_manager_to_forward(dev):
    bits = 4
    model = ToyModel(dev)
    base = {n: m.weight.detach().cpu().numpy().copy() for n, m in model.named_modules()
            if isinstance(m, nn.Linear)}
    base_emb = model.model.embed_tokens.weight.detach().cpu().numpy().copy()
    mgr = create_delta_manager(model, 8, 64, V, DeltaConfig(max_deltas=3, max_bitwidth=bits, max_cpu_deltas=4),
                               delta_manager_cls=LRUCacheDeltaModelManager)
    fused = {}
    for did in (11, 12, 13, 14):
        dm, fused[did] = make_delta_model(did, bits, 100 * did)
        mgr.add_delta(dm)
    for did in (12, 11, 13):
        mgr.activate_delta(did)
    assert mgr.delta_index_to_id == [12, 11, 13]
    ids = (11, 11, 0, 13, 12, 12, 0, 13, 11)
    x = torch.from_numpy(o.make_x(len(ids), H, 3)).to(dev)

    def check(ids):
        mgr.set_delta_mapping(DeltaMapping(ids, ids[:2]))
        torch.cuda.synchronize()
        slots = [mgr.delta_index_to_id.index(i) if i > 0 else -1 for i in ids]
        assert mgr.base_indices[: len(ids)].tolist() == slots and list(mgr.indices_len) == [len(ids), 2, 2, len(ids)]
        for name in ("self_attn.qkv_proj", "self_attn.o_proj", "mlp.gate_up_proj"):
            layer = model.get_submodule("model.layers.0." + name)
            y, bias = layer(x)
            torch.cuda.synchronize()
            table = {i: fused[i][name] for i in fused}
            uniq = sorted({i for i in ids if i > 0})
            ref = o.forward_ref(x.cpu().numpy(), base["model.layers.0." + name], [table[i] for i in uniq],
                                np.array([uniq.index(i) if i > 0 else -1 for i in ids]))
            assert bias is None and o.rel_err(y.float().cpu().numpy(), ref) <= 1e-2, name
        # embedding and output projection: the delta's own tables
        slots_np = np.array(slots)
        tok = np.arange(len(ids)) % V
        by_slot = lambda name: np.stack([fused[d][name] if d is not None else np.zeros((V, H), np.float16)
                                         for d in mgr.delta_index_to_id])
        e = model.model.embed_tokens(torch.from_numpy(tok).to(dev))
        assert np.array_equal(e.cpu().numpy(), o.embed_select_ref(tok, by_slot("model.embed_tokens"), slots_np,
                                                                  base_emb))
        logits = model.logits_processor(model.lm_head.weight, x[:2])
        want = o.linear_select_ref(x[:2].cpu().numpy(), by_slot("lm_head"), slots_np[:2], base["lm_head"])
        assert o.rel_err(logits.float().cpu().numpy(), want) <= 1e-2

    check(ids)
    # delta 14 takes the least recently used slot (12's: 11 and 13 were activated after it)
    mgr.activate_delta(14)
    assert mgr.delta_index_to_id == [14, 11, 13]
    check((14, 11, 0, 13, 14, 14, 0, 13, 11))
    with pytest.raises(ValueError, match="not in list"):
        mgr.set_delta_mapping(DeltaMapping((12, 0), (12,)))
    # an unchanged mapping is not converted again
    m = DeltaMapping((11, 0), (11,))
    mgr.set_delta_mapping(m)
    before = mgr._staged
    mgr.set_delta_mapping(DeltaMapping((11, 0), (11,)))
    assert mgr._last_mapping == m and mgr._staged is before


@pytest.mark.gpu
def test_manager_makes_row_blocks_once_for_a_large_batch(dev):
    """A batch above the fused kernel's sizes: the manager orders the tokens by delta and cuts the row
    blocks once, with the mapping, and every layer call of the step uses them; a smaller batch
    afterwards drops them again."""
    bits = 4
    model = ToyModel(dev)
    base = {n: m.weight.detach().cpu().numpy().copy() for n, m in model.named_modules() if isinstance(m, nn.Linear)}
    mgr = create_delta_manager(model, 8, 1024, V, DeltaConfig(max_deltas=3, max_bitwidth=bits, max_cpu_deltas=4),
                               delta_manager_cls=LRUCacheDeltaModelManager)
    fused = {}
    for did in (11, 12):
        dm, fused[did] = make_delta_model(did, bits, 100 * did)
        mgr.add_delta(dm)
        mgr.activate_delta(did)
    rng = np.random.default_rng(5)
    ids = tuple(int(i) for i in rng.choice([0, 11, 12], size=600))
    assert not ops.takes_fused_chunks(len(ids), mgr.delta_slots)
    mgr.set_delta_mapping(DeltaMapping(ids, ids[:2]))
    blocks = mgr.row_blocks[0]
    assert isinstance(blocks, ops.RowBlocks) and blocks.T == 600
    x = torch.from_numpy(o.make_x(len(ids), H, 3)).to(dev)
    for name in ("self_attn.qkv_proj", "mlp.gate_up_proj"):
        layer = model.get_submodule("model.layers.0." + name)
        assert layer.row_blocks is mgr.row_blocks
        y, _ = layer(x)
        torch.cuda.synchronize()
        ref = o.forward_ref(x.cpu().numpy(), base["model.layers.0." + name], [fused[11][name], fused[12][name]],
                            np.array([{0: -1, 11: 0, 12: 1}[i] for i in ids]))
        assert o.rel_err(y.float().cpu().numpy(), ref) <= 1e-2, name
    assert mgr.row_blocks[0] is blocks          # made once, not per layer call
    mgr.set_delta_mapping(DeltaMapping(ids[:9], ids[:2]))
    assert mgr.row_blocks[0] is None


@pytest.mark.gpu
@pytest.mark.parametrize("T", [200, 400, 1100])
def test_wrapped_layers_replay_from_a_graph_with_the_mapping_of_the_day(dev, T):
    """Layers captured above the fused kernel's sizes and replayed after further set_delta_mapping calls,
    with tensors of other sizes made and dropped in between: every replay reads the ids as they are
    then, and equals the eager call of the same mapping bit for bit."""
    model = ToyModel(dev)
    mgr = create_delta_manager(model, 8, 2048, V, DeltaConfig(max_deltas=6, max_bitwidth=4, max_cpu_deltas=6))
    for did in (11, 12, 13):
        mgr.add_delta(make_delta_model(did, 4, 100 * did)[0])
        mgr.activate_delta(did)
    layers = [model.get_submodule("model.layers.0." + n) for n in ("self_attn.qkv_proj", "self_attn.o_proj")]
    x = torch.from_numpy(o.make_x(T, H, 3)).to(dev)
    step = lambda: [layer(x)[0] for layer in layers]
    rng = np.random.default_rng(T)

    def mapping(t):
        ids = tuple(int(i) for i in np.sort(rng.choice([0, 11, 12, 13], size=t, p=rng.dirichlet(np.ones(4)))))
        mgr.set_delta_mapping(DeltaMapping(ids, ids[:2]))
    mapping(T)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(side):
        step()                                       # this stream's workspace is made outside the capture
        torch.cuda.synchronize()
        with torch.cuda.graph(graph, stream=side):
            outs = step()
    torch.cuda.current_stream().wait_stream(side)
    for rep in range(4):
        mapping(9 + 200 * rep)                       # batches of other sizes in between, their tables dropped
        junk = [torch.full((n, 4), 1 << 20, dtype=torch.int32, device=dev) for n in (5, 9, 17, T)]
        mapping(T)
        want = step()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        for a, b in zip(outs, want):
            assert torch.equal(a, b), rep
        del junk


@pytest.mark.gpu
def test_manager_with_one_copy_of_the_base_weights(dev):
    """DeltaConfig.keep_row_major_base=False through the manager: every wrapped projection frees its
    row-major weight, and a decode-sized and a prefill-sized batch give, bit for bit, what a manager
    that keeps both copies gives on the same weights and deltas."""
    bits = 4
    torch.manual_seed(7)
    models = [ToyModel(dev), ToyModel(dev)]
    models[1].load_state_dict(models[0].state_dict())
    cfgs = [DeltaConfig(max_deltas=2, max_bitwidth=bits), DeltaConfig(max_deltas=2, max_bitwidth=bits,
                                                                       keep_row_major_base=False)]
    mgrs = [create_delta_manager(m, 8, 1024, V, c) for m, c in zip(models, cfgs)]
    for mgr in mgrs:
        for did in (11, 12):
            mgr.add_delta(make_delta_model(did, bits, 100 * did)[0])
            mgr.activate_delta(did)
    qkv = [m.get_submodule("model.layers.0.self_attn.qkv_proj") for m in models]
    assert qkv[0].base_layer.weight.numel() > 0 and qkv[1].base_layer.weight.numel() == 0
    assert qkv[1].base_shape == tuple(qkv[0].base_layer.weight.shape)
    rng = np.random.default_rng(11)
    for T in (9, 700):
        ids = tuple(int(i) for i in rng.choice([0, 11, 12], size=T))
        x = torch.from_numpy(o.make_x(T, H, 5)).to(dev)
        outs = []
        for mgr, model in zip(mgrs, models):
            mgr.set_delta_mapping(DeltaMapping(ids, ids[:2]))
            outs.append([model.get_submodule("model.layers.0." + name)(x)[0]
                         for name in ("self_attn.qkv_proj", "self_attn.o_proj", "mlp.gate_up_proj")])
        torch.cuda.synchronize()
        for a, b in zip(*outs):
            assert torch.equal(a, b), T


@pytest.mark.parametrize("t,k,n,plan", [
    (128, 4096, 4096, None), (129, 1024, 8192, None), (2000, 1024, 8192, (0, 1)),        # a short walk
    (129, 5120, 27648, (0, 1)), (8192, 5120, 27648, (0, 1)), (333, 4096, 12288, (0, 1)),  # enough workgroups
    (230, 2048, 2048, (1, 4)), (333, 13824, 5120, (0, 4)), (333, 5120, 5120, (0, 4)),     # few: K in parts
    (300000, 4096, 4096, None)])                                                          # 32-bit offsets
def test_plan_of_blocks_of_several_deltas(t, k, n, plan):
    """By the sizes alone; where the host knows the mix, a few tokens of each of many deltas go elsewhere."""
    assert ops._mixed_plan(t, k, n) == plan
    assert ops._in_mixed_blocks(t, k, n, 769, None) is None
    many = ops._even_mix(t, t)
    assert ops._in_mixed_blocks(t, k, n, 64, None) == plan
    if plan is not None and (k >= 2 * n and t <= 512):
        assert ops._in_mixed_blocks(t, k, n, 64, many) is None


class _Calls:
    """The library with its launches written down instead of made."""

    def __init__(self, lib):
        self.lib, self.names = lib, []

    def __getattr__(self, name):
        if not name.startswith(("dz_build", "dz_order", "dz_multi_delta")):
            return getattr(self.lib, name)
        return lambda *a: self.names.append(name) or 0


@pytest.fixture
def launches(monkeypatch):
    from deltazip_amd import _lib
    calls = _Calls(_lib.lib())
    monkeypatch.setattr(_lib, "lib", lambda: calls)
    monkeypatch.setattr(ops, "_stream", lambda: 0)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda *a: SimpleNamespace(cuda_stream=0))
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    monkeypatch.setattr(ops, "_need_cuda", lambda *a: None)
    monkeypatch.setattr(ops, "_workspace", lambda *a: torch.empty(4))
    monkeypatch.setattr(ops, "segment", lambda ids, s, report=False: (torch.empty(ids.numel(), dtype=torch.int32),
                                                                      torch.empty(s + 2, dtype=torch.int32)))
    return calls.names


@pytest.mark.parametrize("t,order,tables", [(1, False, "short"), (100, False, "short"), (128, False, "short"), (100, True, ""),
                                            (129, False, "short"), (1024, False, "short"), (1025, False, "both"), (9000, False, "long")])
def test_row_blocks_hold_blocks_of_one_delta(launches, t, order, tables):
    """Every batch has them, also one that is as short as a decode step: the last piece of a very long one.  Only blocks
    that come with a token order have none, and the product over blocks of one delta refuses those."""
    from deltazip_amd.prefill import multi_delta_linear_prefill
    ids, s = torch.zeros(t, dtype=torch.int64), 8
    blocks = ops.row_blocks(ids, s, order=torch.zeros(t, dtype=torch.int32) if order else None)
    assert ((blocks.tiles is not None) + 2 * (blocks.short is not None)) == ("", "long", "short", "both").index(tables)
    args = (torch.empty(t, 256, dtype=torch.float16), None, torch.empty(s, 4), torch.empty(s, 1, 32), torch.empty(s, 4), ids)
    out = torch.empty(t, 32, dtype=torch.float16)
    if not tables:
        with pytest.raises(ValueError):
            multi_delta_linear_prefill(*args, bits=2, out=out, accumulate=False, blocks=blocks)
    else:
        assert blocks.mixed is not None and launches == ["dz_build_tables"]
        launches.clear()
        multi_delta_linear_prefill(*args, bits=2, out=out, accumulate=False)   # (makes the table it reads and no other)
        assert [n for n in launches if "build" in n] == ["dz_build_tiles" if tables == "long" else "dz_build_tiles_rows"]
        ops.row_blocks(ids, s, mixed=False)
        assert launches[-1] == {"short": "dz_build_tiles_rows", "long": "dz_build_tiles", "both": "dz_build_tiles_either"}[tables]
        launches.clear()
        multi_delta_linear_prefill(*args, bits=2, out=out, accumulate=False, blocks=blocks)
        assert [n for n in launches if "gemm" in n] == ["dz_multi_delta_gemm"] * (tables != "short") + \
            ["dz_multi_delta_gemm_rows"] * (tables != "long")


@pytest.mark.parametrize("k,t", [(13824, 77673), (13824, 77696), (11008, 97542), (5120, 209792)])
def test_last_piece_of_a_very_long_batch(launches, k, t):
    """A call beyond the kernels' 31-bit offsets goes in pieces, each of them multiplied, also a last one of 1 to 128 rows."""
    from deltazip_amd.prefill import multi_delta_linear_prefill
    assert ops._mixed_plan(t, k, 32) is None
    x = torch.empty(1, k, dtype=torch.float16).expand(t, k)
    multi_delta_linear_prefill(x, None, torch.empty(2, 4), torch.empty(2, 1, 32), torch.empty(2, 4),
                               torch.zeros(1, dtype=torch.int64).expand(t), bits=2, out=torch.empty(t, 32, dtype=torch.float16),
                               accumulate=False)
    tables = [i for i, n in enumerate(launches) if n.startswith("dz_build")]
    assert len(tables) >= 2 and all("gemm" in launches[i + 1] for i in tables[:-1]) and "gemm" in launches[-1]


def _mapped(monkeypatch, layers):
    """A manager on the CPU whose kernels are left out, and which counts projections of these sizes."""
    for name in ("map_ids", "token_order", "poll_status"):
        monkeypatch.setattr(ops, name, lambda *a, **kw: None)
    mgr = create_delta_manager(ToyModel(), 128, 256, V, DeltaConfig(max_deltas=8, max_bitwidth=4, group_size=-1))
    assert dict(mgr._projections) == {(H, H + 128): 1, (H, H): 1, (H, 2 * I): 1, (I, H): 1}
    mgr.delta_index_to_id = list(range(1, 9))
    mgr._projections = tuple(((k, n), 32) for h, i in layers for k, n in ((h, 3 * h), (h, h), (h, 2 * i), (i, h)))
    return mgr


@pytest.mark.parametrize("t,deltas,layers,makes", [
    (81, 4, [(2048, 8448)], False), (52, 2, [(2048, 6144)], False), (51, 2, [(4096, 3584)], False),   # over before the host
    (36, 1, [(1536, 10752)], False), (128, 4, [(256, 512)], False), (128, 8, [(4096, 5000)], True),
    (128, 4, [(4096, 11008)], True), (33, 8, [(5120, 13824)], True), (64, 7, [(5120, 13824)], False)])
def test_decode_step_makes_blocks_where_the_whole_step_gains(monkeypatch, t, deltas, layers, makes):
    """One projection that would take blocks of several deltas is not enough: a step the decode kernel is through with
    before the host has launched it makes none."""
    mgr = _mapped(monkeypatch, layers)
    ids = tuple(1 + i * deltas // t for i in range(t))
    mgr.set_delta_mapping(DeltaMapping(ids, ids[:1]))
    assert (mgr.row_blocks[0] is not None) == makes


def test_decode_blocks_are_made_by_the_layers_that_take_them(monkeypatch, launches):
    """set_delta_mapping itself launches nothing for them (a step that is replayed from a graph reads the token order
    alone); the first eager call of a layer that takes them does, once for every stream, and makes one table."""
    mgr = _mapped(monkeypatch, [(4096, 11008)])
    ids, now, seen = tuple(1 + i // 32 for i in range(128)), SimpleNamespace(stream=7, capturing=False), []
    monkeypatch.setattr(ops, "_stream", lambda: now.stream)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: now.capturing)
    monkeypatch.setattr(ops, "apply_delta", lambda *a, order, base_tiled: seen.append(order))
    mgr.set_delta_mapping(DeltaMapping(ids, ids[:1]))
    assert launches == []
    layer = mgr.model.model.layers[0].mlp.down_proj
    layer.base_tiled = None

    def call(n, k):
        layer.base_shape = (n, k)
        layer.apply_weights(None)
        return seen[-1]
    small = call(4096, 4096)                           # under 24 M weights
    now.capturing = True
    captured = call(4096, 11008)
    now.capturing = False
    assert launches == [] and small.data_ptr() == captured.data_ptr() == mgr.token_order.data_ptr() and small.numel() == 128
    first, again = call(4096, 11008), call(22016, 4096)
    assert first is again and isinstance(first, ops.RowBlocks) and first.mix.deltas == 4
    assert first.order.data_ptr() == mgr.token_order.data_ptr() and first.mixed[0].deltas == 4 - 1 and first.mixed[1] is None
    now.stream = 8
    other = call(4096, 11008)
    assert other is not first and launches == ["dz_order_mixed"] * 2
    now.stream = 7
    assert call(4096, 11008) is first and len(launches) == 2
    mgr.set_delta_mapping(DeltaMapping(ids[:20], ids[:1]))
    assert mgr.row_blocks[0] is None


@pytest.mark.parametrize("t,k,n,bits,slots,route", [
    (155, 2048, 1408, 2, 1, "chunks"), (144, 2560, 736, 4, 21, "chunks"), (210, 2304, 640, 4, 3, "chunks"),   # the host's half
    (200, 2560, 1280, 2, 5, "blocks"), (293, 6656, 1728, 2, 2, "blocks"), (333, 13824, 5120, 2, 16, "blocks"),
    (600, 2560, 1280, 2, 5, "blocks"), (129, 4096, 512, 2, 700, "blocks"), (129, 4096, 512, 2, 769, "chunks")])
def test_route_of_a_call_that_makes_its_own_table(monkeypatch, launches, t, k, n, bits, slots, route):
    """Few short chunks are over before the host has launched the table, the product and its sums; a batch whose tables
    are there goes in blocks of several deltas all the same, and so do projections that share theirs."""
    def called(make):
        launches.clear()
        make()
        return set(launches)
    x, w = torch.empty(t, k, dtype=torch.float16), torch.empty(n, k, dtype=torch.float16)
    ids = torch.zeros(t, dtype=torch.int64)
    qs, ms, ss = ops.stacked_shapes(k, n, bits, -1)
    stack = [torch.empty((slots,) + tuple(v), dtype=d) for v, d in ((qs, torch.int32), (ss, torch.float16), (ms, torch.int16))]
    got = called(lambda: ops.apply_delta(x, *stack, ids, w))
    assert got == ({"dz_multi_delta_linear_chunks"} if route == "chunks" else {"dz_order_mixed", "dz_multi_delta_gemm_mixed"})
    if slots <= 768:
        known = ops.row_blocks(ids, slots, deltas=3)
        assert called(lambda: ops.apply_delta(x, *stack, ids, w, order=known)) == {"dz_multi_delta_gemm_mixed"}


@pytest.mark.parametrize("layers,mixed", [([(256, 512)], False), ([(1024, 1024)], False), ([(256, 512), (4096, 11008)], True)])
def test_mapping_makes_the_tables_its_projections_read(monkeypatch, launches, layers, mixed):
    mgr = _mapped(monkeypatch, layers)
    ids = tuple(1 + i // 32 for i in range(200))
    mgr.set_delta_mapping(DeltaMapping(ids, ids[:1]))
    assert launches == ["dz_build_tables" if mixed else "dz_build_tiles_rows"]
    assert (mgr.row_blocks[0].mixed is not None) == mixed and mgr.row_blocks[0].short is not None


@pytest.mark.parametrize("made_captured,capturing,blocks_go", [(False, False, True), (False, True, False), (True, True, True)])
def test_captured_decode_step_keeps_the_token_order(monkeypatch, made_captured, capturing, blocks_go):
    """A decode batch whose blocks were made outside a capture goes into it with the manager's token order, as a
    batch without blocks does; a prefill batch hands its blocks on either way."""
    seen = []
    monkeypatch.setattr(ops, "apply_delta", lambda *a, order, base_tiled: seen.append(order))
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: capturing)
    blocks, token_order = SimpleNamespace(captured=made_captured), torch.arange(256)
    layer = SimpleNamespace(token_order=token_order, row_blocks=[blocks], base_layer=SimpleNamespace(weight=None),
                            _row_major_dropped=False, base_tiled=None, qweight_stacked=None, scales_stacked=None,
                            meta_stacked=None, indices=token_order)
    for t in (64, 200):
        layer.indices_len = [t]
        LinearWithDelta.apply_weights(layer, None)
    assert (seen[0] is blocks) == blocks_go and (blocks_go or torch.equal(seen[0], token_order[:64]))
    assert seen[1] is blocks


@pytest.mark.parametrize("shape", [(3, 4, 5), (1, 7), (2, 0), (4,), (0, 3), ()])
def test_values_per_slot_without_a_view(shape):
    """The calls' checks count a slot's values by the shape; a stack without slots is refused as indexing it is."""
    t = torch.zeros(shape)
    if shape and shape[0]:
        assert ops._slot_numel(t) == t[0].numel()
    else:
        with pytest.raises(IndexError):
            ops._slot_numel(t)


def test_sizes_are_looked_up_once_and_refused_every_time():
    assert ops._sizes(512, 64, 2, -1) == ops.native_sizes(512, 64, 2, -1) == ops._sizes(512, 64, 2, -1)
    for _ in range(2):
        with pytest.raises(ValueError):
            ops._sizes(500, 64, 2, -1)


def test_parts_by_blocks_keep_the_usual_number_unless_another_is_clearly_faster():
    from deltazip_amd import _lib
    L = _lib.lib()
    for t, k, n in ((333, 13824, 5120), (129, 256, 32), (512, 2560, 1280), (4000, 4096, 4096)):
        for usual in (1, 2, 4, 6):
            if usual > k // 256:
                assert L.dz_mixed_parts(t, k, n, 4, usual) == usual and L.dz_mixed_us(t, k, n, 4, usual) == 0
                continue
            for blocks in (1, 4, 5, 16, 40):
                us = {c: L.dz_mixed_us(t, k, n, blocks, c) for c in {1, 2, 3, 4, 6, usual} if c <= k // 256}
                got, least = L.dz_mixed_parts(t, k, n, blocks, usual), min(us.values())
                assert us[got] == least if least < 0.899 * us[usual] and least < us[usual] - 3.01 else \
                    got == usual or us[got] < us[usual]
    assert ops._parts_of_blocks(333, 5120, 27648, 16, (0, 1), 4) == (1, 1)             # nothing was to be summed
    parts, room = ops._parts_of_blocks(333, 13824, 5120, 16, (0, 4), 4)
    assert parts == -4 and room == max(L.dz_mixed_parts(333, 13824, 5120, b, 4) for b in range(3, 17))
    assert ops._parts_of_blocks(1999, 11008, 4096, 8, (0, 1), 3) == (2, 2)             # by the sizes alone
    assert ops._parts_of_blocks(8192, 13824, 5120, 16, (0, 1), 4) == (1, 1)


@pytest.mark.parametrize("t", [4, 128, 256])
def test_projections_that_share_tokens_refuse_other_widths(launches, t):
    """A batch of projections takes [.., K] as one projection does: tokens of another width are not cut into rows of K,
    whatever the number of rows that would make, and nothing is launched for them."""
    k, n, s = 256, 32, 2
    stacks = [torch.empty(s, k * n * 2 // 64, dtype=torch.int32)] * 2, [torch.empty(s, 1, n, dtype=torch.float16)] * 2, \
        [torch.empty(s, n, k // 16, dtype=torch.int16)] * 2
    w, ids = [torch.empty(n, k, dtype=torch.float16)] * 2, torch.zeros(t, dtype=torch.int64)
    x = torch.empty(t, k, dtype=torch.float16)
    for bad in (x.view(t // 2, 2 * k), x.view(2 * t, k // 2), x.view(2, t // 4, 2 * k), x.view(t * k)):
        for xs in (bad, [x, bad], [bad, x]):
            with pytest.raises(ValueError):
                ops.apply_delta_batch(xs, *stacks, ids, w)
    assert not launches
    for good in (x, x.view(2, t // 2, k), x.view(t, 1, k)):
        assert [y.shape for y in ops.apply_delta_batch(good, *stacks, ids, w)] == [(*good.shape[:-1], n)] * 2
    assert ops.apply_delta_batch(x[0], *stacks, ids[:1], w)[1].shape == (n,)
    narrow = [torch.empty(t, k, dtype=torch.float16), torch.empty(t, 2 * k, dtype=torch.float16)]   # each its own width: a call each
    stacks2 = [stacks[0][0], torch.empty(s, k * n * 4 // 64, dtype=torch.int32)], stacks[1], [stacks[2][0], torch.empty(s, n, k // 8, dtype=torch.int16)]
    both = lambda: ops.apply_delta_batch(narrow, *stacks2, ids, [w[0], torch.empty(n, 2 * k, dtype=torch.float16)])
    if t > 128:
        assert [y.shape for y in both()] == [(t, n)] * 2
    else:
        with pytest.raises(ValueError):
            both()


def test_room_for_sums_is_asked_of_the_function_that_picks_the_parts(monkeypatch):
    """A launch whose parts the device picks writes as many partial sums as that function has it; the caller asks the same
    one, once for a size, and makes no list of blocks of its own."""
    from deltazip_amd import _lib
    L, asked = _lib.lib(), []
    for t in (129, 195, 333, 512, 2300):
        for k, n in ((13824, 10784), (4096, 4096), (5120, 2560), (512, 96)):
            for usual in (1, 2, 4, 6, 15):
                if usual <= k // 256:
                    few = min(-(-t // 128), 16)
                    assert L.dz_mixed_most_parts(t, k, n, usual) == max(L.dz_mixed_parts(t, k, n, b, usual) for b in range(few, 17))

    class Asked:
        def __getattr__(self, name):
            asked.append(name)
            return getattr(L, name)
    monkeypatch.setattr(_lib, "lib", lambda: Asked())
    ops._parts_of_blocks.cache_clear()
    assert [ops._parts_of_blocks(195, 13824, 10784, 2, (0, 2), 4) for _ in range(2)] == [(-2, 6)] * 2
    assert asked == ["dz_mixed_most_parts"]
    ops._parts_of_blocks.cache_clear()


def test_parts_above_512_tokens_cost_few_calls_of_the_library(monkeypatch):
    """Prefill meets a new number of tokens at nearly every step: the estimates behind its parts are made in a call or two, and
    come to what they do one by one."""
    from deltazip_amd import _lib
    L, asked = _lib.lib(), []

    class Asked:
        def __getattr__(self, name):
            asked.append(name)
            return getattr(L, name)
    monkeypatch.setattr(_lib, "lib", lambda: Asked())
    ops._parts_of_blocks.cache_clear()
    for t in (513, 1999, 8192):
        for k, n in ((4096, 4096), (1536, 1536), (11008, 4096)):
            asked.clear()
            assert ops._parts_of_blocks(t, k, n, 8, ops._mixed_plan(t, k, n), 3)[0] >= 1 and len(asked) <= 2
            for few, many in ((1, 1), (-(-t // 128), -(-t // 128)), (-(-t // 128), -(-t // 128) + 5)):
                us = {p: [L.dz_mixed_us(t, k, n, b, p) for b in range(few, many + 1)] for p in (1, 2, 3, 4, 6)}
                for usual, now in us.items():
                    share = {p: sum(v) / sum(now) for p, v in us.items() if all(a < b for a, b in zip(v, now))}
                    for only in (0, 2, 5):
                        may = {usual: 0.9, **{p: v for p, v in share.items() if only in (0, p)}}
                        assert L.dz_mixed_parts_between(t, k, n, few, many, usual, only) == min(may, key=may.get)
    ops._parts_of_blocks.cache_clear()
    assert L.dz_mixed_parts_between(999, 512, 96, 8, 9, 3, 0) == 3 and L.dz_mixed_parts_between(999, 512, 96, 0, 9, 2, 0) == 2


@pytest.mark.parametrize("t,k,n,slots,deltas,usual", [
    (541, 3072, 6656, 6, 2, (1, 1)), (1268, 3072, 3072, 2, 4, (0, 2)), (620, 5888, 4352, 4, 3, (0, 3)),     # full blocks fit one round
    (588, 3840, 3840, 38, 3, (0, 3)), (986, 4096, 4096, 17, 4, (0, 2)), (1876, 11008, 1024, 34, 3, (0, 4))])  # one part leaves CUs idle
def test_parts_above_512_tokens_stay_where_some_mix_would_lose(t, k, n, slots, deltas, usual):
    """Sizes at which a batch whose blocks come out a few more or fewer than the mean took up to 1.3 times as long in the
    other number of parts."""
    assert ops._mixed_plan(t, k, n) == usual and ops._parts_of_blocks(t, k, n, slots, usual, deltas) == (usual[1],) * 2

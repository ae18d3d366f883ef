"""Routed experts with few rows each (16- and 32-row tiles, weights multiplied as whole numbers)
against the oracle, at the edges of a tile; and the 32-row kernels that take the other widths."""
import pytest
import torch

from oracle import moe_oracle as O
from tolerances import assert_close

pytestmark = pytest.mark.gpu

# rows of successive experts: one row, the edges of a 16-row group, of a 32-row tile, several tiles
EDGES = [1, 15, 16, 17, 31, 32, 33, 2, 47, 48, 49, 64, 65, 3]


def _raw(pkg, lw, x, ids):
    """experts() on given routing: its rows [T * 8, H] back in (token, slot) order."""
    gr = pkg.abi.sort_permute(ids, lw.n_experts)
    y = pkg.abi.experts(x, lw.gate_up_q, lw.gate_up_fmt, lw.down_q, lw.down_fmt, gr, 8,
                        pkg._lib.MOE_PATH_MFMA, up_q=lw.up_q)
    torch.cuda.synchronize()
    return y.cpu()[gr["pair_pos"].cpu().long()]


def _ids(T, counts, n_experts, seed):
    """[T, 8] ids in which experts 3, 3 + 7, ... get the given row counts (the last takes the rest)."""
    p = T * 8
    flat = torch.cat([torch.full((n,), (3 + 7 * i) % n_experts, dtype=torch.int32) for i, n in enumerate(counts)])
    assert flat.numel() <= p
    rest = torch.arange(p - flat.numel(), dtype=torch.int32) % 2 + 1
    flat = torch.cat([flat, rest])
    return flat[torch.randperm(p, generator=torch.Generator().manual_seed(seed))].view(T, 8)


def _rel(got, want):
    return float((got.double() - want.double()).norm() / want.double().norm())


# up to 256 tokens 16-row tiles, above 32-row ones; x and the SiLU rows are rounded to f16 (2^-11 / sqrt(12)
# = 1.4e-4 rms each, three of them in a row: 2.4e-4), the weights not at all: 5e-4 is twice that
@pytest.mark.parametrize("fixture,T", [("layer_c0", 64), ("layer_c0", 257), ("layer_q5k", 64),
                                       ("layer_q5k", 257), ("layer_artifact", 100)])
def test_rows_at_tile_edges(pkg, dev, request, fixture, T):
    lw, ow = request.getfixturevalue(fixture)
    x = pkg.synth.make_input(T, seed=T, device=dev)
    ids = _ids(T, EDGES, lw.n_experts, T)
    raw = _raw(pkg, lw, x, ids.to(dev))
    sample = torch.randperm(T, generator=torch.Generator().manual_seed(T))[:48]
    want = O.experts_and_combine(x.cpu()[sample], ids[sample].long(),
                                 torch.ones(len(sample), 8, dtype=torch.bfloat16), ow)["expert_raw"]
    got = raw.view(T, 8, -1)[sample]
    assert_close(got, want, f"{fixture} T={T}")
    assert _rel(got, want) <= 5e-4


def test_one_tile_height_or_the_other_same_bits(pkg, layer_q5k, dev):
    """A row's sums do not depend on the tile it sits in: 256 tokens (16-row tiles) and the same
    tokens among 257 (32-row tiles), Q4_K gate_up and Q5_K down."""
    lw, _ = layer_q5k
    x = pkg.synth.make_input(257, seed=5, device=dev)
    ids = _ids(257, EDGES, lw.n_experts, 6).to(dev)
    a = _raw(pkg, lw, x[:256].contiguous(), ids[:256].contiguous())
    b = _raw(pkg, lw, x, ids)[: 256 * 8]
    assert torch.isfinite(a).all() and torch.equal(a, b)


@pytest.mark.parametrize("fixture", ["layer_c0", "layer_q5k"])
def test_slab_count_does_not_change_the_bits(pkg, dev, request, fixture):
    """16-row tile lists of 80 tiles (the finest slabs) and, with one token more, of 81 (whole ones)."""
    lw, ow = request.getfixturevalue(fixture)
    x = pkg.synth.make_input(17, seed=21, device=dev)
    ids = torch.cat([torch.arange(80, dtype=torch.int32), torch.arange(48, dtype=torch.int32),
                     torch.tensor([80] + list(range(48, 55)), dtype=torch.int32)]).view(17, 8)
    a = _raw(pkg, lw, x[:16].contiguous(), ids[:16].contiguous().to(dev))
    b = _raw(pkg, lw, x, ids.to(dev))
    want = O.experts_and_combine(x[:16].cpu(), ids[:16].long(), torch.ones(16, 8, dtype=torch.bfloat16), ow)["expert_raw"]
    assert torch.equal(a, b[:128])
    assert _rel(a.view(16, 8, -1), want) <= 5e-4


def test_large_and_small_activations(pkg, layer_c0, dev):
    """Rows whose sub-block sums pass 65504 (their SiLU rows saturate, here as on the other tiles), and
    small rows: x 0.05 gives SiLU rows of (0.05 0.9)^2 / 2 = 1e-3, still above f16's subnormals
    (6e-5), so the bound of two roundings holds."""
    lw, ow = layer_c0
    x = pkg.synth.make_input(16, seed=9, device=dev)
    x[:8] *= 8000.0
    x[8:] *= 0.05
    ids = _ids(16, [1, 17, 20], lw.n_experts, 9)
    raw = _raw(pkg, lw, x, ids.to(dev)).view(16, 8, -1)
    want = O.experts_and_combine(x.cpu(), ids.long(), torch.ones(16, 8, dtype=torch.bfloat16), ow)["expert_raw"]
    assert torch.isfinite(raw).all()
    assert _rel(raw[8:], want[8:]) <= 5e-4


def test_other_widths_on_the_32_row_kernels(pkg, dev):
    """hidden 4096: the few-rows kernels of the other widths, against the 160-row ones (whose K order
    they share): the rows of a 256-token call equal those of the same tokens among 257."""
    lw = pkg.synth.make_layer(seed=11, device=dev, n_experts=16, hidden=4096)
    x = pkg.synth.make_input(257, seed=12, device=dev, hidden=4096)
    ids = _ids(257, EDGES[:12], 16, 13).to(dev)
    a = _raw(pkg, lw, x[:256].contiguous(), ids[:256].contiguous())
    b = _raw(pkg, lw, x, ids)[: 256 * 8]
    assert torch.isfinite(a).all() and torch.equal(a, b)


@pytest.mark.parametrize("fixture", ["layer_c0", "layer_artifact"])
@pytest.mark.parametrize("T", [2, 3, 5, 16])
def test_shared_gemv_token_groups_same_bits(pkg, dev, request, fixture, T):
    """Up to 16 tokens the shared expert runs as f32 dots over groups of one, two or four tokens: each
    token's row and gate are those of a call of its own, bit for bit."""
    lw, _ = request.getfixturevalue(fixture)
    args = (lw.shared_gate, lw.shared_up, lw.shared_down, lw.shared_scalar_gate)
    x = pkg.synth.make_input(T, seed=300 + T, device=dev)
    raw, prob = pkg.abi.shared_expert(x, *args)
    one = [pkg.abi.shared_expert(x[t:t + 1].contiguous(), *args) for t in range(T)]
    torch.cuda.synchronize()
    assert torch.equal(raw, torch.cat([r for r, _ in one]))
    assert torch.equal(prob, torch.cat([p for _, p in one]))


# 32-row token tiles up to 256 tokens, 64-row tiles to 896, the 160-row kernels above; x and the SiLU rows
# are rounded to f16, the quants are exact (the bound of the routed rows above)
@pytest.mark.parametrize("T,dtype", [(17, torch.float32), (32, torch.bfloat16), (33, torch.float32),
                                     (257, torch.bfloat16), (321, torch.float32), (896, torch.bfloat16),
                                     (897, torch.float32)])
def test_q8_0_shared_tiles(pkg, layer_artifact, dev, T, dtype):
    lw, ow = layer_artifact
    x = pkg.synth.make_input(T, seed=400 + T, device=dev, dtype=dtype)
    raw, prob = pkg.abi.shared_expert(x, lw.shared_gate, lw.shared_up, lw.shared_down, lw.shared_scalar_gate)
    torch.cuda.synchronize()
    rows = torch.cat([torch.arange(min(T, 40)), torch.tensor([T - 2, T - 1])])
    want = O.shared_expert(x.cpu()[rows], ow)
    assert torch.isfinite(raw).all()
    assert_close(raw.cpu()[rows], want["shared_raw"], f"T={T}")
    if T <= 896:
        assert _rel(raw.cpu()[rows], want["shared_raw"]) <= 5e-4
    assert torch.allclose(prob.cpu()[rows], want["shared_gate_prob"].view(-1), rtol=1e-5, atol=1e-6)


@pytest.mark.parametrize("fixture", ["layer_c0", "layer_artifact"])
@pytest.mark.parametrize("T", [2, 3, 6])
@pytest.mark.parametrize("ties", [False, True])
def test_few_tokens_routed_in_one_launch(pkg, dev, request, fixture, T, ties):
    """2 to 6 tokens: logits, routing and sort of the block in one launch, bit for bit the router call's
    logits, ids and weights (ties: every expert of two groups has the same row), twice on one workspace."""
    import copy
    lw, ow = request.getfixturevalue(fixture)
    if ties:
        lw, ow = copy.copy(lw), copy.copy(ow)
        lw.router = lw.router.clone()
        lw.router[40:60], lw.router[200:230] = lw.router[40].clone(), lw.router[200].clone()
        lw.router_bias = None
    x = pkg.synth.make_input(T, seed=500 + T, device=dev)
    want = pkg.abi.router_topk(x, lw.router, 8, bias=lw.router_bias)
    for _ in range(2):
        got = pkg.abi.block_forward(x, lw, stages=True)
        torch.cuda.synchronize()
        for k in ("router_logits", "topk_ids", "topk_weights"):
            assert torch.equal(got[k].view(want[k].shape), want[k]), k
        if not ties:
            assert_close(got["combined_out"].cpu(), O.moe_block(x.cpu(), ow)["combined_out"], f"T={T}")
    assert pkg.abi.device_error_bits(dev) == 0

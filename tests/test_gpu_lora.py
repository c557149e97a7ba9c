"""Adapters and the backward on the GPU against the oracle (oracle/lora.py,
itself pinned by finite differences in test_lora_oracle.py).

A layer gets adapters on every layer (Model.AddLowRankAdapters), their Down
and Up values are set to the oracle's, and the device's forward, input
gradients and every adapter's gradients must match the oracle under the
device's routing (the device computes router logits in fp32, so flips at
near-ties are allowed as in the other parity tests).  Bars: forward
max|y - r| / max|r| <= 1e-4; gradients the same measure <= 2e-4 (fp32
accumulation over the hidden and vector widths)."""
import numpy as np
import pytest

import gotransformers_amd as gt
from oracle import lora
from tests.moe_fixtures import FLOAT32, FP4, INT8, make_moe
from tests.test_gpu_parity import check_routing, rel_err, say

pytestmark = pytest.mark.gpu

FWD_TOL = 1e-4
GRAD_TOL = 2e-4


@pytest.fixture(scope="module")
def ctx():
    c = gt.Context(0)
    yield c
    c.close()


def keys_of(spec):
    for kind, experts in (("shared", spec.shared), ("routed", spec.routed)):
        for i in range(len(experts)):
            for which in ("gate", "up", "down"):
                yield (kind, i, which)
    yield ("router", 0, None)


def with_adapters(ctx, spec, adapters, rank, alpha):
    m = gt.MixtureOfExperts.from_spec(ctx, spec)
    m.add_adapters(rank, alpha, seed=1)
    for (kind, i, which), ad in adapters.items():
        assert m.adapter_rank(kind, i, which) == ad.down.shape[0]
        m.set_adapter(kind, i, which, ad.down, ad.up)
    return m


CASES = {
    # name: (d, h, E, k, S, precision, clamp, hash, T)
    "small int8 shared": (37, 53, 5, 2, 1, INT8, 0.0, False, 29),
    "small fp4 two shared": (64, 96, 6, 3, 2, FP4, 0.0, False, 17),
    "float32 experts": (40, 24, 4, 2, 0, FLOAT32, 0.0, False, 9),
    "clamped": (48, 40, 4, 2, 1, INT8, 0.3, False, 13),
    "hash routing": (32, 48, 6, 2, 1, FP4, 0.0, True, 11),
    "C2 int8 decode": (1024, 2048, 16, 2, 0, INT8, 0.0, False, 8),
    "C3 fp4 layer": (1024, 512, 64, 6, 1, FP4, 0.0, False, 64),
    # many positions per group: the transposed product on the matrix cores
    # (32-position tiles, the down layer's rows in sixteen chunks) and full
    # tiles of 64 positions in the adapters' kernels
    "many positions per expert": (1024, 128, 4, 1, 1, INT8, 0.0, False, 1024),
    # the matrix-core product over FP4 rows with a partial last panel (d = 200
    # rows of the down layer, its gradient rows 200 floats apart) and half a
    # workgroup of column blocks (h = 40: four blocks)
    "many positions fp4 ragged": (200, 40, 3, 2, 1, FP4, 0.0, False, 256),
    "many positions float32": (48, 40, 2, 1, 0, FLOAT32, 0.0, False, 160),
    # fourteen positions per group on average: eight-position tiles
    "eight-position tiles": (96, 64, 8, 2, 0, INT8, 0.0, False, 56),
}
# adapter rank per case (4 unless listed): 16 fill a block of the projections'
# ranks, five are read one at a time
RANKS = {"many positions per expert": 16, "small fp4 two shared": 5, "clamped": 16}


@pytest.mark.parametrize("name", list(CASES))
def test_adapter_forward_and_backward(ctx, name):
    d, h, E, k, S, prec, clamp, hashed, T = CASES[name]
    rank = RANKS.get(name, 4)
    alpha = 2.0 * rank
    say(f"adapters {name}: d={d} h={h} E={E} k={k} S={S} precision={prec} T={T}")
    spec = make_moe(gt.encode_rows, d=d, h=h, E=E, k=k, S=S, precision=prec, seed=21, std=0.05, router_std=0.05,
                    bias_std=0.02, clamp=clamp, use_hash=hashed)
    rng = np.random.default_rng(22)
    adapters = lora.make_adapters(spec, rank, alpha, rng, up_scale=0.05)
    x = rng.uniform(-1, 1, (T, d))
    ids = rng.integers(0, 10000, T) if hashed else None
    G = rng.uniform(-1, 1, (T, d))
    m = with_adapters(ctx, spec, adapters, rank, alpha)
    try:
        y = m.forward(x, ids)
        r = m.last_routing()
        dx = m.backward(G)
        grads = {key: m.adapter_gradients(*key) for key in keys_of(spec)}
        dx2 = m.backward(G)  # gradients add up over calls
        grads2 = {key: m.adapter_gradients(*key) for key in keys_of(spec)}
        m.zero_adapter_gradients()
        zeroed = m.adapter_gradients("routed", 0, "gate")
    finally:
        m.destroy()
    if not hashed:
        # the oracle's routing, with its own float64 logits including the router adapter
        ref_y, st = lora.forward(spec, adapters, x, ids)
        flips = np.nonzero(np.any(st.chosen != r.chosen, axis=1))[0]
        say(f"[{name}] routing flips: {len(flips)} of {T}")
    ref_y, st = lora.forward(spec, adapters, x, ids, chosen=r.chosen)
    e = rel_err(y, ref_y)
    say(f"[{name}] forward max rel err {e:.2e}")
    assert e <= FWD_TOL
    ref_grads = lora.zero_grads(spec, adapters)
    ref_dx = lora.backward(spec, adapters, st, G, ref_grads)
    e = rel_err(dx, ref_dx)
    say(f"[{name}] input gradient max rel err {e:.2e}")
    assert e <= GRAD_TOL
    assert np.array_equal(dx, dx2)
    worst = 0.0
    for key in keys_of(spec):
        gd, gu = grads[key]
        rd, ru = ref_grads[key]
        if not np.any(rd) and not np.any(ru):  # e.g. the router under hash routing, an unused expert
            assert not np.any(gd) and not np.any(gu), key
            continue
        worst = max(worst, rel_err(gd, rd) if np.any(rd) else 0.0, rel_err(gu, ru) if np.any(ru) else 0.0)
        assert np.allclose(grads2[key][0], 2 * gd, rtol=1e-12, atol=0)
        assert np.allclose(grads2[key][1], 2 * gu, rtol=1e-12, atol=0)
    say(f"[{name}] adapter gradient max rel err {worst:.2e}")
    assert worst <= GRAD_TOL
    assert not np.any(zeroed[0]) and not np.any(zeroed[1])


def test_fresh_adapters_keep_the_output(ctx):
    """Up starts at zero (adapter.go:37-40): the adapter path's forward equals
    the adapter-free layer's to fp32 tolerance, and Down holds values in
    +-1/sqrt(inputs) while Up is zero."""
    say("fresh adapters")
    spec = make_moe(gt.encode_rows, d=64, h=96, E=8, k=2, S=1, precision=INT8, seed=23, std=0.05, bias_std=0.02)
    x = np.random.default_rng(24).uniform(-1, 1, (12, 64))
    m = gt.MixtureOfExperts.from_spec(ctx, spec)
    try:
        plain = m.forward(x, path=gt.PATH_FP32)
        m.add_adapters(8, 16.0, seed=5)
        down, up = m.adapter("routed", 3, "down")
        assert down.shape == (8, 96) and up.shape == (64, 8)
        assert not np.any(up) and np.all(np.abs(down) <= 1 / np.sqrt(96)) and np.any(down)
        assert m.adapter_rank("router", 0) == 8
        adapted = m.forward(x)
        m.remove_adapters()
        again = m.forward(x, path=gt.PATH_FP32)
    finally:
        m.destroy()
    assert rel_err(adapted, plain) <= FWD_TOL
    assert np.array_equal(again, plain)


def test_adapter_errors_mirror_the_reference(ctx):
    say("adapter errors")
    spec = make_moe(gt.encode_rows, d=32, h=32, E=4, k=2, S=0, precision=INT8, seed=25)
    x = np.random.default_rng(26).uniform(-1, 1, (3, 32))
    m = gt.MixtureOfExperts.from_spec(ctx, spec)
    try:
        m.forward(x)
        with pytest.raises(gt.GtmoeError, match="add a low-rank adapter to train around them") as info:
            m.backward(np.zeros((3, 32)))
        assert info.value.code == gt.ERR_UNSUPPORTED
        with pytest.raises(gt.InvalidArgument, match="rank must be at least 1, got 0"):
            m.add_adapters(0, 1.0)
        m.add_adapters(2, 4.0)
        with pytest.raises(gt.InvalidArgument, match="already has adapters"):
            m.add_adapters(2, 4.0)
        with pytest.raises(gt.GtmoeError, match="call Forward before Backward") as info:
            m.backward(np.zeros((3, 32)))
        assert info.value.code == gt.ERR_NOT_READY
        m.forward(x)
        with pytest.raises(gt.InvalidArgument, match="output gradients are 2x32 but the last Forward produced 3x32"):
            m.backward(np.zeros((2, 32)))
        with pytest.raises(gt.InvalidArgument, match="routed expert 4 of 4"):
            m.adapter("routed", 4, "gate")
        import torch
        xd = torch.zeros((3, 32), device="cuda")
        with pytest.raises(gt.GtmoeError, match="runs through gtmoe_forward") as info:
            m.forward_device(3, xd.data_ptr(), xd.data_ptr())
        assert info.value.code == gt.ERR_UNSUPPORTED
    finally:
        m.destroy()


@pytest.mark.parametrize("rank", [3, 16, 17, 20])
@pytest.mark.parametrize("T", [1, 15, 17, 63, 65, 130])
def test_rank_projections_at_the_edges_of_their_tiles(ctx, T, rank):
    """One routed expert (T positions in its group and T in the shared
    expert's): blocks of 16 positions and tiles of 64, partly filled; ranks
    below, at and past 16; output-gradient rows 37 floats apart, hidden widths
    that are not multiples of 16.  The only expert's gate is 1 whatever its
    logit, so the router's gradients are exactly zero; its adapter is tested
    below."""
    d, h = 37, 53
    say(f"rank projections T={T} rank={rank}")
    spec = make_moe(gt.encode_rows, d=d, h=h, E=1, k=1, S=1, precision=INT8, seed=51, std=0.1, router_std=0.1,
                    bias_std=0.02)
    rng = np.random.default_rng(52 + T)
    alpha = 2.0 * rank
    adapters = lora.make_adapters(spec, rank, alpha, rng, up_scale=0.05)
    x = rng.uniform(-1, 1, (T, d))
    G = rng.uniform(-1, 1, (T, d))
    m = with_adapters(ctx, spec, adapters, rank, alpha)
    try:
        y = m.forward(x)
        r = m.last_routing()
        dx = m.backward(G)
        grads = {key: m.adapter_gradients(*key) for key in keys_of(spec)}
    finally:
        m.destroy()
    ref_y, st = lora.forward(spec, adapters, x, None, chosen=r.chosen)
    ref_grads = lora.zero_grads(spec, adapters)
    ref_dx = lora.backward(spec, adapters, st, G, ref_grads)
    assert rel_err(y, ref_y) <= FWD_TOL
    assert rel_err(dx, ref_dx) <= GRAD_TOL
    for key in keys_of(spec):
        for got, want in zip(grads[key], ref_grads[key]):
            if np.any(want):
                assert rel_err(got, want) <= GRAD_TOL, key
            else:
                assert not np.any(got), key


@pytest.mark.parametrize("rank", [3, 16, 17, 20])
@pytest.mark.parametrize("T", [1, 15, 17, 63, 65, 130])
def test_router_adapter_at_the_edges_of_its_tiles(ctx, T, rank):
    """The router's adapter over its own tiles of the T tokens: 21 experts, so
    that its rank is not cut below 20, three of them chosen.  Its projection
    decides the gates (forward outputs) and takes a gradient from them, and its
    input gradients join the layer's."""
    d, h, E, k = 37, 53, 21, 3
    say(f"router adapter T={T} rank={rank}")
    spec = make_moe(gt.encode_rows, d=d, h=h, E=E, k=k, S=1, precision=INT8, seed=53, std=0.1, router_std=0.1,
                    bias_std=0.02)
    rng = np.random.default_rng(54 + T)
    alpha = 2.0 * rank
    adapters = lora.make_adapters(spec, rank, alpha, rng, up_scale=0.3)
    x = rng.uniform(-1, 1, (T, d))
    G = rng.uniform(-1, 1, (T, d))
    m = with_adapters(ctx, spec, adapters, rank, alpha)
    try:
        y = m.forward(x)
        r = m.last_routing()
        dx = m.backward(G)
        down, up = m.adapter_gradients("router", 0)
    finally:
        m.destroy()
    ref_y, st = lora.forward(spec, adapters, x, None, chosen=r.chosen)
    ref_grads = lora.zero_grads(spec, adapters)
    ref_dx = lora.backward(spec, adapters, st, G, ref_grads)
    want_down, want_up = ref_grads[("router", 0, None)]
    assert down.shape == (rank, d) and np.any(want_down) and np.any(want_up)
    assert rel_err(r.gates, st.gates) <= FWD_TOL
    assert rel_err(y, ref_y) <= FWD_TOL
    assert rel_err(dx, ref_dx) <= GRAD_TOL
    assert rel_err(down, want_down) <= GRAD_TOL
    assert rel_err(up, want_up) <= GRAD_TOL
    idle = ~np.isin(np.arange(E), r.chosen)  # no token chose them: their rows of Up's gradients
    assert not np.any(up[idle])


@pytest.mark.parametrize("d", [256, 1000, 1024, 2048, 4096])
def test_rank_projections_round_as_short_sums_do(ctx, d):
    """One token through one expert makes every adapter gradient a rank-one
    matrix: Up's of the gate layer is (its gradient) (A x)^T, Down's of the
    down layer (B^T g) (hidden row)^T.  Their leading singular vectors average
    the products' own rounding away and leave that of the projections A x and
    B^T g over d values.  Sums of 16 products added in 64 bits, rounded once to
    32, stay below 1e-7 (half an ulp of the results alone is 3e-8 on average;
    a model of 16 sequential roundings gives 8e-8); one serial fp32 sum per
    quarter grows with d, 2.9e-7 at 1024 and 5.7e-7 at 4096 values."""
    say(f"rounding of the rank projections, d={d}")
    rank = 64
    spec = make_moe(gt.encode_rows, d=d, h=64, E=1, k=1, S=0, precision=INT8, seed=61, std=0.05, bias_std=0.02)
    rng = np.random.default_rng(62)
    f32 = lambda v: v.astype(np.float32).astype(np.float64)
    adapters = lora.make_adapters(spec, rank, 2.0 * rank, rng, up_scale=0.05)
    for ad in adapters.values():
        ad.down, ad.up = f32(ad.down), f32(ad.up)
    m = with_adapters(ctx, spec, adapters, rank, 2.0 * rank)
    got, want = {"u": [], "t": []}, {"u": [], "t": []}
    try:
        for _ in range(16):
            x, G = f32(rng.standard_normal((1, d))), f32(rng.standard_normal((1, d)))
            m.zero_adapter_gradients()
            m.forward(x)
            m.backward(G)
            up = m.adapter_gradients("routed", 0, "gate")[1]
            down = m.adapter_gradients("routed", 0, "down")[0]
            for key, mat, exact in (("u", up, adapters[("routed", 0, "gate")].down @ x[0]),
                                    ("t", down.T, adapters[("routed", 0, "down")].up.T @ G[0])):
                v = np.linalg.svd(mat, full_matrices=False)[2][0]
                got[key].append(v * (v @ exact))
                want[key].append(exact)
    finally:
        m.destroy()
    for key in got:
        g, w = np.array(got[key]), np.array(want[key])
        e = np.linalg.norm(g - w) / np.linalg.norm(w)
        say(f"[d={d}] {key}: relative error {e:.2e}")
        assert e <= 1e-7, (key, e)


@pytest.mark.parametrize("d,row", [(37, 36), (48, 47), (48, 11)])
def test_an_infinite_row_of_up(ctx, d, row):
    """An infinite value in one row of the down layer's Up makes that rank of
    t = s g Up infinite with the sign of the row's gradient, and with it a row
    of Down's gradients; 37 rows end inside a step of 16 values, whose rest adds
    nothing."""
    say(f"infinite Up value, d={d} row={row}")
    spec = make_moe(gt.encode_rows, d=d, h=32, E=1, k=1, S=0, precision=INT8, seed=63, std=0.1, bias_std=0.02)
    rng = np.random.default_rng(64)
    adapters = lora.make_adapters(spec, 4, 8.0, rng, up_scale=0.05)
    adapters[("routed", 0, "down")].up[row, 2] = np.inf
    x, G = rng.uniform(-1, 1, (1, d)), rng.uniform(-1, 1, (1, d))
    m = with_adapters(ctx, spec, adapters, 4, 8.0)
    try:
        m.forward(x)
        m.backward(G)
        got = m.adapter_gradients("routed", 0, "down")[0]
    finally:
        m.destroy()
    _, st = lora.forward(spec, adapters, x)
    want = lora.zero_grads(spec, adapters)
    with np.errstate(all="ignore"):
        lora.backward(spec, adapters, st, G, want)
    want = want[("routed", 0, "down")][0]
    assert np.all(np.isinf(want[2])) and np.all(np.isfinite(want[[0, 1, 3]]))
    assert np.array_equal(got[2], want[2])
    assert rel_err(got[[0, 1, 3]], want[[0, 1, 3]]) <= GRAD_TOL


@pytest.mark.parametrize("T", [1, 6])
def test_an_infinite_weight_of_an_unchosen_router_row(ctx, T):
    """Router row 3 holds -inf in a column whose inputs are positive, so no
    token chooses expert 3 and the forward is finite.  That column's input
    gradient is a sum over every expert, NaN from the zero logit gradient times
    the weight; the other columns' are not touched by it."""
    say(f"infinite router weight, T={T}")
    d, column = 40, 7
    spec = make_moe(gt.encode_rows, d=d, h=24, E=4, k=2, S=1, precision=INT8, seed=71, std=0.1, router_std=0.1,
                    bias_std=0.02)
    spec.router.weights.values[3, column] = -np.inf
    rng = np.random.default_rng(72)
    adapters = lora.make_adapters(spec, 4, 8.0, rng, up_scale=0.05)
    x, G = rng.uniform(-1, 1, (T, d)), rng.uniform(-1, 1, (T, d))
    x[:, column] = rng.uniform(0.1, 1, T)
    m = with_adapters(ctx, spec, adapters, 4, 8.0)
    try:
        y = m.forward(x)
        r = m.last_routing()
        dx = m.backward(G)
    finally:
        m.destroy()
    assert not np.any(r.chosen == 3)
    with np.errstate(all="ignore"):
        ref_y, st = lora.forward(spec, adapters, x, chosen=r.chosen)
        ref_dx = lora.backward(spec, adapters, st, G, lora.zero_grads(spec, adapters))
    others = np.arange(d) != column
    assert rel_err(y, ref_y) <= FWD_TOL
    assert np.all(np.isnan(dx[:, column]))
    assert rel_err(dx[:, others], ref_dx[:, others]) <= GRAD_TOL

"""Routed experts with few pairs each: chunks of one and two row tiles, on a kernel of their own."""
import numpy as np
import pytest
import torch

import synth
from oracle import mfq_oracle as O

pytestmark = pytest.mark.gpu

# both edges of a tile, chunks of one and two tiles, experts of several chunks; then experts without pairs, which bring the average
# down to the kernel for few pairs
PAIRS = [1, 0, 15, 16, 17, 31, 32, 33, 48, 64, 65, 97] + [0] * 12


@pytest.mark.parametrize("bits,gs,sub", [(4, 24, 6), (3, 24, 5), (2, 16, 5), (5, 28, 7), (4, 32, 6), (4, 16, 6), (4, 48, 6), (2, 32, 5)])
@pytest.mark.parametrize("out,K", [(224, 680), (32, 72)])
def test_chunks_of_one_and_two_tiles(bits, gs, sub, out, K):
    """Against the dequantized weights in 64 bits: fp32 sums of K <= 680 terms, and 2^-11 of a weight for five-bit codes; the gated
    form against the plain call's own sums, half an ulp of fp16."""
    from tyloquant_amd.runtime_moe import NintMoeWeight, build_moe_route_plan
    rng = np.random.default_rng(100 * bits + gs + out)
    E, R = len(PAIRS), 2
    ids = np.repeat(np.arange(E), PAIRS)
    assert len(ids) <= 20 * E
    ids = np.append(ids, [E + 7] * (2 - len(ids) % 2)).astype(np.int32)        # and one or two pairs without an expert
    ids = rng.permutation(ids).reshape(-1, R)
    T = len(ids)
    pool = O.MoePool(np.arange(E, dtype=np.int32), f"NINT{bits}", synth.nint_random(rng, E * out, K, bits, gs, sub))
    w = NintMoeWeight.from_blob(O.pack_nint_moe(O.NintMoeTensor((E, out, K), [pool])))
    dense = w.dequantize().double()
    flat = torch.from_numpy(ids.reshape(-1)).long().cuda()
    for routed, dtype in ((False, torch.bfloat16), (True, torch.float16)):
        x = torch.from_numpy((rng.standard_normal((T, R, K) if routed else (T, K)) * 0.1).astype(np.float32)).to(dtype).cuda()
        rows = (x.reshape(T * R, K) if routed else x.repeat_interleave(R, 0)).double()
        ref = torch.zeros(T * R, out, dtype=torch.float64, device="cuda")
        bound = torch.zeros(T * R, out, dtype=torch.float64, device="cuda")
        for e in range(E):
            at = (flat == e).nonzero().flatten()
            ref[at] = rows[at] @ dense[e].t()
            bound[at] = rows[at].abs() @ dense[e].abs().t()
        route = build_moe_route_plan(torch.from_numpy(ids).cuda(), E)
        got = w(x, route).reshape(T * R, out).double()
        inside = flat < E
        assert float((got - ref)[inside].norm() / ref[inside].norm()) < (1e-5 if bits < 5 else 1e-3)
        assert bool(((got - ref).abs() <= 2e-3 * bound + 1e-30)[inside].all())
        assert bool((got[~inside] == 0).all())
        hidden = w.forward_glu(x, route, out_dtype=torch.float16).reshape(T * R, out // 2).double()
        want = torch.nn.functional.silu(got[:, : out // 2]) * got[:, out // 2:]
        assert float((hidden - want).norm() / want.norm()) < 5e-4
        assert bool((hidden[~inside] == 0).all())


@pytest.mark.parametrize("T,E,R", [(20, 12, 2), (45, 12, 2), (300, 6, 2), (700, 6, 1)])    # few pairs an expert, and many
@pytest.mark.parametrize("bits,gs,sub", [(4, 24, 6), (4, 32, 6), (5, 28, 7)])              # a groupsize of the cohorts', and others
def test_shared_expert_in_the_launches_of_the_routed_ones(T, E, R, bits, gs, sub):
    """Rows of the pairs and of the shared tensor against the dequantized weights in 64 bits, plain from routed rows and gated from
    tokens; an id without an expert, a column of neurons that ends inside a tile."""
    from tyloquant_amd.runtime import load_quant_linear
    from tyloquant_amd.runtime_moe import NintMoeWeight, build_moe_route_plan
    rng = np.random.default_rng(T + E + gs)
    out, K = 160, 296
    w = NintMoeWeight.from_blob(O.pack_nint_moe(synth.moe_random(rng, E, out, K, [(4, 3, 2)[e % 3] for e in range(E)], True)))
    own = load_quant_linear(*O.pack_tensor(synth.nint_random(rng, out, K, bits, gs, sub))).weight
    dense, dense_own = w.dequantize().double(), own.dequantize().double()
    ids = rng.integers(0, E, (T, R)).astype(np.int32)
    ids[3, R - 1] = E + 5
    flat = torch.from_numpy(ids.reshape(-1)).long().cuda()
    route = build_moe_route_plan(torch.from_numpy(ids).cuda(), E)
    assert route.ids_dst is not None
    for routed in (False, True):
        n = T * R
        x = torch.from_numpy((rng.standard_normal((n + T if routed else T, K)) * 0.1).astype(np.float32)).to(torch.bfloat16).cuda()
        rows = x.double() if routed else torch.cat([x.repeat_interleave(R, 0), x]).double()
        ref = torch.zeros(n + T, out, dtype=torch.float64, device="cuda")
        for e in range(E):
            at = (flat == e).nonzero().flatten()
            ref[at] = rows[at] @ dense[e].t()
        ref[n:] = rows[n:] @ dense_own.t()
        got = w.forward_shared(x, route, own, routed=routed).double()
        zero = (flat >= E).nonzero().flatten()
        assert bool((got[zero] == 0).all())
        assert float((got[:n] - ref[:n]).norm() / ref[:n].norm()) < 1e-5
        assert float((got[n:] - ref[n:]).norm() / ref[n:].norm()) < (1e-5 if bits < 5 else 1e-3)
        hidden = w.forward_shared(x, route, own, glu=True, routed=routed).double()
        want = torch.nn.functional.silu(got[:, : out // 2]) * got[:, out // 2:]
        assert float((hidden - want).norm() / want.norm()) < 5e-4
        assert bool((hidden[zero] == 0).all())
    assert w.forward_shared(x[:-1], route, own, routed=True) is None          # not one row per output row


@pytest.mark.parametrize("T,R,K", [(2050, 1, 2048), (2050, 1, 2056), (30, 2, 8192), (30, 2, 8200), (1030, 2, 72)])
@pytest.mark.parametrize("routed", [False, True])
def test_activation_rows_that_registers_hold_and_longer_ones(T, R, K, routed):
    """A wave and four waves a row, rows up to what they hold and one piece more, a row with an infinity and one with a NaN, rows of very
    different magnitudes.  Against the dequantized weights in 64 bits: fp32 sums over K <= 8200 terms, 1e-5 of the sum of the magnitudes."""
    from tyloquant_amd.runtime_moe import NintMoeWeight, build_moe_route_plan
    rng = np.random.default_rng(T + K + routed)
    E, out = 5, 48
    w = NintMoeWeight.from_blob(O.pack_nint_moe(synth.moe_random(rng, E, out, K, [(4, 3, 2)[e % 3] for e in range(E)], True)))
    dense = w.dequantize().double()
    ids = rng.integers(0, E, (T, R)).astype(np.int32)
    ids[3, R - 1] = E + 5
    flat = torch.from_numpy(ids.reshape(-1)).long().cuda()
    n = T * R if routed else T
    x = torch.from_numpy(rng.standard_normal((n, K)).astype(np.float32))
    x[1] *= 1e6
    x[2] *= 1e-6
    x[5, K - 1], x[6, 8] = float("inf"), float("nan")
    x = x.to(torch.bfloat16).cuda()
    route = build_moe_route_plan(torch.from_numpy(ids).cuda(), E)
    got = w(x.reshape(T, R, K) if routed else x, route).reshape(T * R, out).double()
    rows = (x if routed else x.repeat_interleave(R, 0)).double()
    ok = torch.isfinite(rows).all(1) & (flat < E)
    for e in range(E):
        at = (ok & (flat == e)).nonzero().flatten()
        ref, bound = rows[at] @ dense[e].t(), rows[at].abs() @ dense[e].abs().t()
        assert bool(((got[at] - ref).abs() <= 1e-5 * bound + 1e-30).all()), float(((got[at] - ref).abs() / bound).max())
    assert bool((got[flat >= E] == 0).all())
    assert not bool(torch.isfinite(got[~torch.isfinite(rows).all(1) & (flat < E)]).all(1).any())


@pytest.mark.parametrize("T", [61, 300])
@pytest.mark.parametrize("gate,down,foreign,products", [        # products: gate/up calls beside the joint one
    ((4, 24, 6), (4, 24, 6), False, 0), ((4, 24, 6), (6, 24, 7), False, 0), ((5, 28, 7), (8, 48, 7), False, 0),
    ((4, 24, 6), (4, 24, 6), True, 0), ((6, 24, 7), (4, 24, 6), False, 1), ((6, 24, 7), (6, 24, 7), False, 1)])
def test_shared_expert_of_which_one_tensor_cannot_join(T, gate, down, foreign, products, monkeypatch):
    """A feed-forward block whose shared gate/up or down (or the experts' down, with a cohort of another family) keeps its product off the
    joint launch: against the dequantized weights in 64 bits, and no product is made twice.  Bound in the 2-norm: the hidden row is rounded
    to 11 bits, and weights of five bits and more once each where they meet the matrix cores, before and behind it: three roundings of
    at most 2^-11, and 1e-5 for the 32-bit sums."""
    from tyloquant_amd.runtime import load_quant_linear
    from tyloquant_amd.runtime_moe import NintMoeWeight, nint_moe_ffn_forward
    rng = np.random.default_rng(T + gate[1] + down[1])
    E, H, W, R = 12, 288, 96, 2
    bits = [(4, 3, 2, 5)[e % 4] for e in range(E)]
    tg, td = synth.moe_random(rng, E, 2 * W, H, bits, True), synth.moe_random(rng, E, H, W, bits, True)
    if foreign:
        pool = td.pools[0]
        weights = O.quantize_nint8_zero((rng.standard_normal((len(pool.expert_ids) * H, W)) * 0.02).astype(np.float32))
        td.pools[0] = O.MoePool(pool.expert_ids, "NINT8-0", weights)
    gu, dn = (NintMoeWeight.from_blob(O.pack_nint_moe(t)) for t in (tg, td))
    sg, sd = (O.quantize_nint((rng.standard_normal(s) * 0.02).astype(np.float32), *p) for s, p in (((2 * W, H), gate), ((H, W), down)))
    shared = tuple(load_quant_linear(*O.pack_tensor(t)).weight for t in (sg, sd))
    calls, plain = [], NintMoeWeight.forward_glu
    monkeypatch.setattr(NintMoeWeight, "forward_glu", lambda self, *a, **k: (calls.append(1), plain(self, *a, **k))[1])
    x = torch.from_numpy(rng.standard_normal((T, H)).astype(np.float32)).to(torch.bfloat16).cuda()
    logits = torch.from_numpy(rng.standard_normal((T, E)).astype(np.float32)).cuda()
    out, ids, wts = nint_moe_ffn_forward(gu, dn, x, logits, R, normalize=True, shared=shared)
    assert len(calls) == products
    dg, dd, xd = gu.dequantize().double(), dn.dequantize().double(), x.double()
    dsg, dsd = (w.dequantize().double() for w in shared)
    glu = lambda v: torch.nn.functional.silu(v[:, :W]) * v[:, W:]
    ref = glu(xd @ dsg.t()) @ dsd.t()
    for e in range(E):
        t, r = (ids == e).nonzero(as_tuple=True)
        ref[t] += wts[t, r, None].double() * (glu(xd[t] @ dg[e].t()) @ dd[e].t())
    assert float((out.double() - ref).norm() / ref.norm()) < 3 * 2.0 ** -11 + 1e-5

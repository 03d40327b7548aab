"""Q8_0 products on few members per expert against the CPU oracle and the older paths: the streaming kernels
(16-column items, dsx_stream_kernels.hpp) on rows of an odd and an even number of 128-value groups and in each
instance by row length (up to 8, 12, 16 and 32 groups), with second items of an expert, beside the GEMM with the device's choice, in
captures, blocks and the hyper-connection combine; the 32- and 64-column int8 GEMMs with several items of an expert that nearly
every token names; items with one column and with an empty column group, empty slots."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from deepstrix_amd.capi import FMT_MXFP4, FMT_Q8_0
from deepstrix_amd.executor import MoeChain, MoeLayer
from oracle import ref
from tests import helpers as H
from tests.test_gpu_chain import layer_shapes, verify_chain_stepwise
from tests.test_gpu_hc_post import _layer_case

pytestmark = pytest.mark.gpu

ROUTER = dict(router_mode=1, route_scale=2.5, bias_sigma=0.01, clamp=10.0)


def _run(s, T, seed, monkeypatch, named=None):
    """Picks on the first `named` experts (None: all).  Also returns the streaming range."""
    monkeypatch.setattr(MoeLayer, "v3_thresholds_below_experts", None)   # the library's own thresholds
    x, _, _ = H.host_inputs(s, T)
    rng = np.random.default_rng(seed)
    sel = np.stack([rng.permutation(named or s.n_expert)[:2] for _ in range(T)]).astype(np.int32)
    few = rng.random(T) < 0.6                       # most tokens name expert 3: several items
    sel[few, 0] = np.where(sel[few, 1] == 3, sel[few, 0], 3)
    sel[T // 2, 1] = -1                             # an empty slot
    w = rng.uniform(0.05, 0.6, sel.shape).astype(np.float32)
    dw = H.device_weights(s)
    layer, older = MoeLayer(dw, T), MoeLayer(dw, T)
    older.set_tuning(by_expert_chunk=4)             # the by-expert kernels and the int8 GEMM
    dx, ds, dwt = torch.from_numpy(x).cuda(), torch.from_numpy(sel).cuda(), torch.from_numpy(w).cuda()
    out = layer.run(dx, None, selected_in=ds, weights_in=dwt).clone()
    again = layer.run(dx, None, selected_in=ds, weights_in=dwt)
    old = older.run(dx, None, selected_in=ds, weights_in=dwt)
    torch.cuda.synchronize()
    assert torch.equal(out, again)
    hw = H.host_weights(s, experts=range(named or s.n_expert))
    want = ref.moe_forward(hw, x, sel, w)
    # the dots are exact: other orders of the f32 sums, and a mid value at a rounding boundary that takes the
    # neighbouring int8 step (fitted to a column of a down matrix)
    H.assert_parity_up_to_rounding_steps(out.cpu().numpy(), want, hw, sel, f"{s.hidden} x {s.inter} T={T}")
    return out, old, layer.streaming()


# (hidden, inter): gate/up rows of hidden / 128 groups, down rows of inter / 128
@pytest.mark.parametrize("hidden,inter", [(128, 256), (384, 1152), (1024, 640), (1152, 128), (2048, 1408), (2304, 2176), (4096, 512), (512, 4096)])
@pytest.mark.parametrize("T", [2, 5, 15, 16, 60, 111])
def test_all_q8_0_layer_matches_the_oracle(monkeypatch, hidden, inter, T):
    """2 and 5 tokens (1.25 picks per expert): the streaming kernels, which serve matrices over 2 M elements at 15 as
    well; behind them, to 111, the narrow GEMM, which has the bits of the wide one."""
    s = H.Shape(hidden, inter, 8, 2, FMT_Q8_0, FMT_Q8_0, shared=hidden != 1024, seed=800, **ROUTER)
    out, old, streaming = _run(s, T, T, monkeypatch)
    assert streaming == (2, 15 if hidden * inter > 2 << 20 else 5)
    assert torch.equal(out, old) == (T > streaming[1])


@pytest.mark.parametrize("hidden,inter", [(256, 1280), (384, 1536), (640, 1664), (512, 1792), (1280, 2048), (4096, 384)])
@pytest.mark.parametrize("T", [17, 23])
def test_all_q8_0_streaming_with_several_items_of_an_expert(monkeypatch, hidden, inter, T):
    """Under 1.5 picks per expert on 32 experts, but most tokens name one and all of them the shared one: their second
    items begin at member 16 and have one to seven columns.  Down rows of 10 and 12 groups (four waves, padded rows), 13, 14 and 16 (eight
    waves, of which some are a group short)."""
    s = H.Shape(hidden, inter, 32, 2, FMT_Q8_0, FMT_Q8_0, shared=inter != 1664, seed=810, **ROUTER)
    out, old, streaming = _run(s, T, T, monkeypatch, named=6)
    assert streaming == (2, 63 if hidden * inter > 2 << 20 else 23)
    assert H.max_rel(out.cpu().numpy(), old.cpu().numpy()) < 1e-3


def _choice_case(T):
    """64 experts of 2048 x 2048, top-4: streaming to 63 tokens, from 24 on beside the narrow GEMM."""
    s = H.Shape(2048, 2048, 64, 4, FMT_Q8_0, FMT_Q8_0, seed=870, **ROUTER)
    dw = H.device_weights(s)
    layer, gemm = MoeLayer(dw, T), MoeLayer(dw, T)
    gemm.set_tuning(gemm_min_tokens=1)   # the int8 GEMM alone
    assert layer.streaming() == (2, 63) and gemm.streaming() == (0, 0)
    rng = np.random.default_rng(T)
    sets = {}
    for kind, named in (("few", 5), ("spread", 64)):
        sel = np.stack([rng.choice(named, 4, replace=False) for _ in range(T)]).astype(np.int32)
        sets[kind] = (sel, rng.uniform(0.05, 0.6, sel.shape).astype(np.float32))
    return s, dw, layer, gemm, torch.from_numpy(H.host_inputs(s, T)[0]).cuda(), sets


@pytest.mark.parametrize("T", [24, 33, 63])
def test_all_q8_0_picks_on_a_few_experts_take_the_gemm(T):
    """From 1.5 picks per expert on the device chooses: picks on a few experts go to the int8 GEMM, whose bits a layer
    that only has it reproduces, spread ones to the streaming kernels (another order of the sums)."""
    s, dw, layer, gemm, x, sets = _choice_case(T)
    for kind in ("few", "spread", "few"):   # one workspace: the counts of one call say nothing to the next
        sel, w = sets[kind]
        run = lambda l: l.run(x, None, selected_in=torch.from_numpy(sel).cuda(), weights_in=torch.from_numpy(w).cuda()).cpu().numpy()
        out, want = run(layer), run(gemm)
        assert np.array_equal(out, want) == (kind == "few"), kind
        assert H.max_rel(out, want) < 1e-3
        n = T if kind == "few" else 3   # (spread: the experts of three tokens are enough on the host)
        hw = H.host_weights_from_device(s, dw, experts=np.unique(sel[-n:]))
        H.assert_parity_up_to_rounding_steps(out[-n:], ref.moe_forward(hw, x.cpu().numpy()[-n:], sel[-n:], w[-n:]), hw, sel[-n:], kind)


def test_a_captured_all_q8_0_pass_chooses_at_every_replay():
    s, dw, layer, gemm, x, sets = _choice_case(40)
    sets = [tuple(torch.from_numpy(a).cuda() for a in sets[kind]) for kind in ("few", "spread")]
    eager = [layer.run(x, None, selected_in=sel, weights_in=w).clone() for sel, w in sets]
    sel, w = (t.clone() for t in sets[0])
    out = torch.empty_like(x)
    side, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        layer.run(x, None, out=out, selected_in=sel, weights_in=w)
        side.synchronize()
        with torch.cuda.graph(graph, stream=side):
            layer.run(x, None, out=out, selected_in=sel, weights_in=w)
    torch.cuda.synchronize()
    for rep in range(4):
        sel.copy_(sets[rep % 2][0])
        w.copy_(sets[rep % 2][1])
        out.fill_(float(rep))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager[rep % 2]), rep


@pytest.mark.parametrize("hidden,inter,shared", [(512, 256, "none"), (1280, 768, "same"), (1280, 768, "q8_0"),
                                                 (2048, 2048, "none"), (7168, 512, "same")])
@pytest.mark.parametrize("T", [10, 15, 16, 23, 24, 111])
def test_q8_0_down_behind_mxfp4_gate_up_matches_the_oracle(monkeypatch, hidden, inter, shared, T):
    fmts = dict(sh_gate_fmt=FMT_Q8_0, sh_down_fmt=FMT_Q8_0) if shared == "q8_0" else {}
    s = H.Shape(hidden, inter, 8, 2, down_fmt=FMT_Q8_0, shared=shared != "none", seed=820 + T, **fmts, **ROUTER)
    _run(s, T, T, monkeypatch)


@pytest.mark.parametrize("hidden,inter,shared", [(4096, 1280, "none"), (3072, 1536, "same"), (4096, 1792, "q8_0"), (2048, 2048, "same")])
@pytest.mark.parametrize("T", [2, 5, 7])
def test_q8_0_down_streams_behind_mxfp4_gate_up(monkeypatch, hidden, inter, shared, T):
    """Below two picks per expert down takes the streaming kernel as well: rows of 10 and 12 groups (four waves), 14 and 16."""
    fmts = dict(sh_gate_fmt=FMT_Q8_0, sh_down_fmt=FMT_Q8_0) if shared == "q8_0" else {}
    s = H.Shape(hidden, inter, 8, 2, down_fmt=FMT_Q8_0, shared=shared != "none", seed=830 + T, **fmts, **ROUTER)
    monkeypatch.setattr(MoeLayer, "v3_thresholds_below_experts", None)
    layer = MoeLayer(H.device_weights(s), 8)
    assert layer.streaming()[0] == 2 and layer.tuning()["gemm_q8_min_tokens"] == 8
    _run(s, T, T, monkeypatch)


@pytest.mark.parametrize("T", [3, 15])
def test_a_stack_of_all_q8_0_streaming_blocks(monkeypatch, T):
    """h += layer(RMSNorm(h)) in a chain: each block against the oracle, replays of a capture against eager steps."""
    monkeypatch.setattr(MoeLayer, "v3_thresholds_below_experts", None)
    shapes = layer_shapes(H.Shape(2304, 1024, 8, 2, FMT_Q8_0, FMT_Q8_0, seed=880, **ROUTER), 2)
    chain = MoeChain([H.device_weights(s, block=True) for s in shapes], T)
    for layer in chain.layers:
        assert layer.streaming() == (2, 15)
    rng = np.random.default_rng(T)
    chain.capture(T)
    for step in range(3):
        h = rng.normal(0, 1, (T, 2304)).astype(np.float32)
        eager = chain.step(torch.from_numpy(h).cuda()).clone()
        torch.cuda.synchronize()
        replayed = chain.replay(torch.from_numpy(h).cuda()).clone()
        torch.cuda.synchronize()
        assert torch.equal(eager, replayed), step
    final = verify_chain_stepwise(chain, shapes, h, 3 * 2e-3, min_checked=(9 * 2 * T) // 10)   # (the bar of the other chains)
    assert np.array_equal(final, eager.cpu().numpy())


@pytest.mark.parametrize("T", [2, 15])
def test_hyper_connection_combine_behind_all_q8_0_streaming(monkeypatch, T):
    monkeypatch.setattr(MoeLayer, "v3_thresholds_below_experts", None)
    s = H.Shape(2304, 1024, 8, 2, FMT_Q8_0, FMT_Q8_0, seed=885, **ROUTER)
    layer = MoeLayer(H.device_weights(s), T)
    assert layer.streaming() == (2, 15)
    _layer_case(s, layer, T)


@pytest.mark.parametrize("down_fmt", ["all", "down"])
@pytest.mark.parametrize("T", [112, 129, 167, 168])
def test_middle_tile_of_the_down_gemm_matches_the_oracle(monkeypatch, down_fmt, T):
    """28 to 42 picks per expert on a layer whose down product makes a round of workgroups (fewer
    take the narrow tile): down by 64-column items, several of the expert that most tokens name, with one to four column
    groups; the wide tile's bits."""
    s = H.Shape(6144, 256, 8, 2, FMT_Q8_0 if down_fmt == "all" else FMT_MXFP4, FMT_Q8_0, seed=840 + T, **ROUTER)
    out, old, _ = _run(s, T, T, monkeypatch)
    if down_fmt == "all":
        assert torch.equal(out, old)


@pytest.mark.parametrize("hidden,inter", [(128, 1152), (640, 128), (1152, 640), (2048, 1408)])
@pytest.mark.parametrize("T", [168, 201, 239])
def test_middle_tile_of_both_products_matches_the_oracle(monkeypatch, hidden, inter, T):
    """42 to 60 picks per expert: gate/up by 64-column items as well, on rows of 1 to 16 chunks, whose scales come by segments of
    eight with a last one of 1 to 8; the wide tile's bits."""
    s = H.Shape(hidden, inter, 8, 2, FMT_Q8_0, FMT_Q8_0, shared=T != 201, seed=846, **ROUTER)
    out, old, _ = _run(s, T, T, monkeypatch)
    assert torch.equal(out, old)


def test_middle_tile_on_many_workgroups(monkeypatch):
    """48 picks per expert and enough row tiles for many rounds: the middle tile again, the wide one's bits."""
    monkeypatch.setattr(MoeLayer, "v3_thresholds_below_experts", None)
    s = H.Shape(4096, 128, 128, 8, FMT_Q8_0, FMT_Q8_0, shared=True, seed=845, **ROUTER)
    x, logits, _ = H.host_inputs(s, 768)
    dw = H.device_weights(s)
    layer, older = MoeLayer(dw, 768), MoeLayer(dw, 768)
    older.set_tuning(by_expert_chunk=4)
    dx, dl = torch.from_numpy(x).cuda(), torch.from_numpy(logits).cuda()
    out = layer.run(dx, dl).clone()
    assert torch.equal(out, older.run(dx, dl)) and torch.isfinite(out).all()


@pytest.mark.parametrize("named,wide", [(8, True), (16, True), (64, False)])
@pytest.mark.parametrize("hidden", [640, 1152])
def test_gate_up_items_of_128_on_few_hot_experts(monkeypatch, hidden, named, wide):
    """31 picks per expert: the middle tile's launch, which takes the list of 128-column items where 250 tokens name eight or sixteen of
    64 experts (16 row tiles: two rounds of 64-column items, one of 128-column ones); groups of every remainder; the wide tile's bits."""
    monkeypatch.setattr(MoeLayer, "v3_thresholds_below_experts", None)
    T, s = 250, H.Shape(hidden, 1024, 64, 8, FMT_Q8_0, FMT_Q8_0, seed=848, **ROUTER)
    rng = np.random.default_rng(named)
    sel = np.stack([rng.permutation(named)[:8] for _ in range(T)]).astype(np.int32)
    sel[T // 2, 1] = -1
    n = np.append(np.bincount(sel[sel >= 0], minlength=64), T)
    middle, big = (int((-(-n // c)).sum()) for c in (64, 128))
    slots = 2 * torch.cuda.get_device_properties(0).multi_processor_count
    assert (5 * middle >= 7 * big and 5 * -(-big * 16 // slots) <= 3 * -(-middle * 16 // slots)) == wide
    w = rng.uniform(0.05, 0.6, sel.shape).astype(np.float32)
    x, dw = H.host_inputs(s, T)[0], H.device_weights(s)
    layer, older = MoeLayer(dw, T), MoeLayer(dw, T)
    older.set_tuning(by_expert_chunk=4)             # the wide tile alone
    args = dict(selected_in=torch.from_numpy(sel).cuda(), weights_in=torch.from_numpy(w).cuda())
    dx = torch.from_numpy(x).cuda()
    out = layer.run(dx, None, **args).clone()
    old = older.run(dx, None, **args)
    torch.cuda.synchronize()
    assert layer.status() == 0 and torch.equal(out, old)
    hw = H.host_weights(s)
    H.assert_parity_up_to_rounding_steps(out.cpu().numpy(), ref.moe_forward(hw, x, sel, w), hw, sel, f"{hidden} {named}")


def test_rows_longer_than_the_registers_take_the_older_paths(monkeypatch):
    """Gate/up rows of 33 groups: the older paths' bits."""
    s = H.Shape(4224, 256, 8, 2, FMT_Q8_0, FMT_Q8_0, shared=False, seed=850, **ROUTER)
    out, old, _ = _run(s, 15, 5, monkeypatch)
    assert torch.equal(out, old)


@pytest.mark.parametrize("hidden", [128, 384, 1152])
@pytest.mark.parametrize("T", [1, 3, 33])
def test_front_launch_of_q8_0_layers(hidden, T):
    """Router, activation rows and status word in one launch: rows that are no multiple of the wave's 256 elements;
    given logits and the same picks pinned make the same bits."""
    s = H.Shape(hidden, 256, 16, 3, FMT_Q8_0, FMT_Q8_0, shared=False, seed=860, **ROUTER)
    x, logits, bias = H.host_inputs(s, T)
    layer = MoeLayer(H.device_weights(s), T)
    dx = torch.from_numpy(x).cuda()
    out, sel, w = (t.clone() for t in layer.run(dx, torch.from_numpy(logits).cuda(), want_routing=True))
    pinned = layer.run(dx, None, selected_in=sel, weights_in=w)
    torch.cuda.synchronize()
    assert torch.equal(out, pinned)
    rsel, _ = H.oracle_route(s, logits, bias)
    _, scores = ref.router_scores(logits, bias, s.router_mode, s.n_group, s.topk_group)
    sel, w = sel.cpu().numpy(), w.cpu().numpy()
    assert H.routing_mismatch_explained(sel, rsel, scores, s.n_used) == []
    want = ref.moe_forward(H.host_weights(s), x, sel, w)
    H.assert_parity_up_to_rounding_steps(out.cpu().numpy(), want, H.host_weights(s), sel, f"{hidden} T={T}")

"""The streaming kernels for groups of few members (whole row tiles through LDS, columns in registers)
against the CPU oracle: rows of an odd and an even number of super-blocks, each instance by row length
(gate/up: up to 8, 16 and 28 super-blocks, down: up to 4, 8, 16 and 28), groups around the 16- and
32-column items, empty slots, an expert that nearly every token names (several items), no shared expert."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from deepstrix_amd.capi import FMT_Q8_0
from deepstrix_amd.executor import MoeChain, MoeLayer
from oracle import ref
from tests import helpers as H
from tests.test_gpu_chain import layer_shapes, verify_chain_stepwise

pytestmark = pytest.mark.gpu

ROUTER = dict(router_mode=1, route_scale=2.5, bias_sigma=0.01, clamp=10.0)
# (hidden, inter): gate/up rows of hidden / 256 super-blocks, down rows of inter / 256
SHAPES = [(512, 256), (1280, 768), (2048, 1280), (3328, 2304), (4096, 2048), (4352, 1024), (7168, 512), (512, 4352),
          (512, 7168)]


@pytest.mark.parametrize("hidden,inter", SHAPES)
@pytest.mark.parametrize("which", ["first", "23", "33", "last"])
def test_stream_matches_the_oracle(monkeypatch, hidden, inter, which):
    """The first and the last token count that stream, and 23 and 33: 23 (under 6 picks per expert) takes
    16-column items, of which the expert that nearly every token names has two; from 24 on 32-column ones."""
    monkeypatch.setattr(MoeLayer, "v3_thresholds_below_experts", None)   # the library's own thresholds
    s = H.Shape(hidden, inter, 8, 2, shared=hidden != 1280, seed=500, **ROUTER)
    dw = H.device_weights(s)
    first, last = MoeLayer(dw, 1).streaming()
    T = {"first": first, "last": last}.get(which) or int(which)
    assert 9 <= first <= 23 and 33 <= last and first <= T <= last
    x, _, _ = H.host_inputs(s, T)
    rng = np.random.default_rng(T)
    sel = np.stack([rng.permutation(8)[:2] for _ in range(T)]).astype(np.int32)
    sel[:, 0] = np.where(sel[:, 1] == 3, sel[:, 0], 3)     # nearly every token names expert 3
    sel[T // 2, 1] = -1                                    # an empty slot
    w = rng.uniform(0.05, 0.6, sel.shape).astype(np.float32)
    layer = MoeLayer(dw, T)
    dx, ds, dwt = torch.from_numpy(x).cuda(), torch.from_numpy(sel).cuda(), torch.from_numpy(w).cuda()
    out = layer.run(dx, None, selected_in=ds, weights_in=dwt).clone()
    again = layer.run(dx, None, selected_in=ds, weights_in=dwt)
    layer.set_tuning(gemm_min_tokens=1, gemm_narrow_members=1)   # the wide GEMM tile on the same inputs
    gemm = layer.run(dx, None, selected_in=ds, weights_in=dwt).cpu().numpy()
    torch.cuda.synchronize()
    assert torch.equal(out, again)
    out = out.cpu().numpy()
    if inter % 512 == 0 and hidden % 512 == 0:
        # other orders of the same f32 sums; a mid value may round to the neighbouring int8 step
        # (1/127 of its block's largest value)
        assert H.max_rel(out, gemm) < 1e-3 and not np.array_equal(out, gemm)
    H.assert_close(out, ref.moe_forward(H.host_weights(s), x, sel, w), 2e-3, f"{hidden} x {inter} T={T}")


def _items(sel, E, members, shared):
    n = np.bincount(sel[sel >= 0], minlength=E)
    return int((-(-n // members)).sum()) + (-(-len(sel) // members) if shared else 0)


@pytest.mark.parametrize("hidden,inter", SHAPES)
@pytest.mark.parametrize("kind", ["spread", "few"])
@pytest.mark.parametrize("T", [26, 34])
def test_either_width_of_item_gives_the_same_bits(monkeypatch, hidden, inter, kind, T):
    """6 to 9 picks per expert: spread picks make hardly more items of 16 members than of 32, picks on three experts twice as many;
    the first 20 tokens alone (under 6 picks per expert) take items of 16."""
    monkeypatch.setattr(MoeLayer, "v3_thresholds_below_experts", None)
    s = H.Shape(hidden, inter, 8, 2, shared=T == 34, seed=520, **ROUTER)
    layer = MoeLayer(H.device_weights(s), T)
    x, _, _ = H.host_inputs(s, T)
    rng = np.random.default_rng(T)
    sel = np.stack([(2 * t + np.arange(2)) % 8 if kind == "spread" else rng.permutation(3)[:2] for t in range(T)]).astype(np.int32)
    sel[T // 2, 1] = -1
    assert (5 * _items(sel, 8, 16, s.shared) <= 6 * _items(sel, 8, 32, s.shared)) == (kind == "spread")
    w = rng.uniform(0.05, 0.6, sel.shape).astype(np.float32)
    dx, ds, dwt = torch.from_numpy(x).cuda(), torch.from_numpy(sel).cuda(), torch.from_numpy(w).cuda()
    out = layer.run(dx, None, selected_in=ds, weights_in=dwt).clone()
    first = layer.run(dx[:20].contiguous(), None, selected_in=ds[:20].contiguous(), weights_in=dwt[:20].contiguous())
    torch.cuda.synchronize()
    assert torch.equal(out[:20], first)
    H.assert_close(out.cpu().numpy(), ref.moe_forward(H.host_weights(s), x, sel, w), 2e-3, f"{hidden} x {inter} T={T} {kind}")


@pytest.mark.parametrize("kind", ["spread", "few", "same"])
def test_either_width_or_the_gemm(kind):
    """8 picks per expert where the GEMM is offered as well (three lists of items): same picks take it."""
    s = H.Shape(5120, 1536, 160, 6, seed=530, **ROUTER)
    dw = H.device_weights(s)
    layer, gemm = MoeLayer(dw, 220), MoeLayer(dw, 220)
    gemm.set_tuning(gemm_min_tokens=1)
    x = torch.from_numpy(H.host_inputs(s, 220)[0]).cuda()
    sel, w = _picks(s, 220, kind, 530)
    if kind == "few":
        sel = (np.argsort(np.random.default_rng(531).random((220, 60)), axis=1)[:, :6]).astype(np.int32)
    assert (5 * _items(sel, 160, 16, True) <= 6 * _items(sel, 160, 32, True)) == (kind == "spread")
    ds, dwt = torch.from_numpy(sel).cuda(), torch.from_numpy(w).cuda()
    out = layer.run(x, None, selected_in=ds, weights_in=dwt).clone()
    want = gemm.run(x, None, selected_in=ds, weights_in=dwt).clone()
    first = layer.run(x[:90].contiguous(), None, selected_in=ds[:90].contiguous(), weights_in=dwt[:90].contiguous())   # (below gemm_min_tokens)
    torch.cuda.synchronize()
    assert torch.equal(out, want) == (kind == "same") and torch.equal(out[:90], first) == (kind != "same")


@pytest.mark.parametrize("hidden,inter", [(512, 256), (1280, 768), (2048, 1280), (4352, 1024), (7168, 512)])
@pytest.mark.parametrize("T", [2, 10, 15, 16, 47, 64])
@pytest.mark.parametrize("shared", ["none", "same", "q8_0"])
def test_stream_gate_up_beside_a_q8_0_down_matches_the_oracle(monkeypatch, hidden, inter, T, shared):
    """Gate/up from the streaming kernel, down from the by-expert kernel and the int8 GEMM (16 tokens: two
    picks per expert); the shared expert as the extra group or beside it; one expert named by half of the
    tokens and more (47: two 16-column items)."""
    monkeypatch.setattr(MoeLayer, "v3_thresholds_below_experts", None)
    fmts = dict(sh_gate_fmt=FMT_Q8_0, sh_down_fmt=FMT_Q8_0) if shared == "q8_0" else {}
    s = H.Shape(hidden, inter, 16, 2, down_fmt=FMT_Q8_0, shared=shared != "none", seed=700 + T, **fmts, **ROUTER)
    x, _, _ = H.host_inputs(s, T)
    rng = np.random.default_rng(T)
    sel = np.stack([rng.permutation(16)[:2] for _ in range(T)]).astype(np.int32)
    sel[: T // 2, 0] = np.where(sel[: T // 2, 1] == 3, sel[: T // 2, 0], 3)
    sel[T // 2, 1] = -1
    w = rng.uniform(0.05, 0.6, sel.shape).astype(np.float32)
    layer = MoeLayer(H.device_weights(s), T)
    first, last = layer.streaming()   # (2 tokens: where the matrices are large)
    assert first == (2 if hidden * inter > 4 << 20 else 10) and T <= last
    dx, ds, dwt = torch.from_numpy(x).cuda(), torch.from_numpy(sel).cuda(), torch.from_numpy(w).cuda()
    out = layer.run(dx, None, selected_in=ds, weights_in=dwt).clone()
    again = layer.run(dx, None, selected_in=ds, weights_in=dwt)
    torch.cuda.synchronize()
    assert torch.equal(out, again)
    H.assert_close(out.cpu().numpy(), ref.moe_forward(H.host_weights(s), x, sel, w), 2e-3, f"{hidden} x {inter} T={T} {shared}")


def _picks(s, T, kind, seed):
    rng = np.random.default_rng(seed)
    sel = np.stack([rng.choice(s.n_expert, s.n_used, replace=False) for _ in range(T)]).astype(np.int32)
    if kind == "same":
        sel[:] = sel[0]
    return sel, rng.uniform(0.05, 0.6, sel.shape).astype(np.float32)


@pytest.mark.parametrize("shared", ["same", "q8_0", "none"])
def test_picks_on_a_few_experts_take_the_gemm(shared):
    """An all-MXFP4 layer, from gemm_min_tokens on: the device sends picks that all fall on a few experts to
    the GEMM, whose bits a layer that only has the GEMM reproduces, and spread ones to the streaming kernels
    (another order of the sums: other bits, the same values).  300 tokens: 80 or 90 items of 32 members against
    24 or 27 of 128; 100 tokens: 32 or 36, of which the GEMM would leave most of the chip idle."""
    fmts = dict(sh_gate_fmt=FMT_Q8_0, sh_down_fmt=FMT_Q8_0) if shared == "q8_0" else {}
    s = H.Shape(4096, 1024, 128, 8, shared=shared != "none", seed=901, **fmts, **ROUTER)
    dw = H.device_weights(s)
    layer, gemm = MoeLayer(dw, 300), MoeLayer(dw, 300)
    gemm.set_tuning(gemm_min_tokens=1)
    for T in (100, 300):
        x = torch.from_numpy(H.host_inputs(s, T)[0]).cuda()
        for kind in ("same", "spread", "same"):   # one workspace: the counts of one call say nothing to the next
            sel, w = (torch.from_numpy(a).cuda() for a in _picks(s, T, kind, T))
            out = layer.run(x, None, selected_in=sel, weights_in=w)
            want = gemm.run(x, None, selected_in=sel, weights_in=w)
            torch.cuda.synchronize()
            assert torch.equal(out, want) == (T == 300 and kind == "same"), (T, kind)
            assert H.max_rel(out.cpu().numpy(), want.cpu().numpy()) < 1e-3, (T, kind)


@pytest.mark.parametrize("T,experts,streams", [(224, 48, False), (264, 64, True)])
def test_the_device_chooses_by_the_rounds_of_the_gemm(T, experts, streams):
    """Random picks on some of the experts: where the GEMM's items fit one round of the chip (64 at this width),
    more than 56 streaming items go to it; where they make a second round, up to 126 stay."""
    s = H.Shape(4096, 1024, 128, 8, seed=904, **ROUTER)
    dw = H.device_weights(s)
    layer, gemm = MoeLayer(dw, T), MoeLayer(dw, T)
    gemm.set_tuning(gemm_min_tokens=1)
    rng = np.random.default_rng(T)
    sel = np.stack([rng.choice(experts, s.n_used, replace=False) for _ in range(T)]).astype(np.int32)
    count = np.bincount(sel.reshape(-1), minlength=experts)
    items = {c: int((-(-count // c)).sum()) + -(-T // c) for c in (32, 128)}
    assert 1.5 * items[128] < items[32] and 56 < items[32] <= 126 and (items[128] > 64) == streams
    x = torch.from_numpy(H.host_inputs(s, T)[0]).cuda()
    sel, w = torch.from_numpy(sel).cuda(), torch.full((T, s.n_used), 0.3, device="cuda")
    out = layer.run(x, None, selected_in=sel, weights_in=w)
    want = gemm.run(x, None, selected_in=sel, weights_in=w)
    torch.cuda.synchronize()
    assert torch.equal(out, want) == (not streams)
    assert H.max_rel(out.cpu().numpy(), want.cpu().numpy()) < 1e-3


def test_a_captured_pass_chooses_at_every_replay():
    s, T = H.Shape(4096, 1024, 128, 8, seed=902, **ROUTER), 300
    layer = MoeLayer(H.device_weights(s), T)
    x = torch.from_numpy(H.host_inputs(s, T)[0]).cuda()
    sets = [tuple(torch.from_numpy(a).cuda() for a in _picks(s, T, kind, 3)) for kind in ("same", "spread")]
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


def test_the_paths_that_a_caller_asks_for_run(monkeypatch):
    """A by-expert chunk and a decode form that the caller sets decide the path: the same bits as where
    thresholds that leave no other path are set."""
    monkeypatch.setattr(MoeLayer, "v3_thresholds_below_experts", None)
    s = H.Shape(4096, 1280, 32, 2, seed=903, **ROUTER)
    dw = H.device_weights(s)

    def run(T, set_up):
        layer = MoeLayer(dw, T)
        set_up(layer)
        sel, w = (torch.from_numpy(a).cuda() for a in _picks(s, T, "spread", T))
        return layer.run(torch.from_numpy(H.host_inputs(s, T)[0]).cuda(), None, selected_in=sel, weights_in=w)

    by_expert = run(40, lambda l: l.set_tuning(gemm_min_tokens=1 << 30, decode_max_tokens=1))
    assert torch.equal(run(40, lambda l: l.set_tuning(by_expert_chunk=4)), by_expert)
    assert not torch.equal(run(40, lambda l: None), by_expert)
    s = H.Shape(4096, 1280, 64, 2, seed=903, **ROUTER)
    dw = H.device_weights(s)
    one_launch = run(14, lambda l: l.set_tuning(decode_max_tokens=14, gemm_min_tokens=1 << 30))
    for form in (2, 3, 4):
        forced = run(14, lambda l: (l.set_tuning(decode_max_tokens=14, gemm_min_tokens=1 << 30), l.set_decode(form)))
        assert torch.equal(run(14, lambda l: l.set_decode(form)), forced), form
    assert not torch.equal(run(14, lambda l: None), one_launch)


@pytest.mark.parametrize("fmt", ["mxfp4", "q8_0 shared", "q8_0 down"])
@pytest.mark.parametrize("T", [15, 40])
def test_a_stack_of_streaming_blocks(monkeypatch, fmt, T):
    """h += layer(RMSNorm(h)), the residual added behind the streaming kernels and the shared expert inside or
    beside them, in a chain: each block against the oracle, replays of a capture against eager steps."""
    monkeypatch.setattr(MoeLayer, "v3_thresholds_below_experts", None)
    kw = {"mxfp4": {}, "q8_0 shared": dict(sh_gate_fmt=FMT_Q8_0, sh_down_fmt=FMT_Q8_0), "q8_0 down": dict(down_fmt=FMT_Q8_0)}[fmt]
    shapes = layer_shapes(H.Shape(2048, 512, 8, 2, seed=905, **kw, **ROUTER), 2)
    chain = MoeChain([H.device_weights(s, block=True) for s in shapes], T)
    for layer in chain.layers:
        assert layer.streaming()[0] <= T <= layer.streaming()[1]
    rng = np.random.default_rng(T)
    chain.capture(T)
    for step in range(3):
        h = rng.normal(0, 1, (T, 2048)).astype(np.float32)
        eager = chain.step(torch.from_numpy(h).cuda()).clone()
        torch.cuda.synchronize()
        replayed = chain.replay(torch.from_numpy(h).cuda()).clone()
        torch.cuda.synchronize()
        assert torch.equal(eager, replayed), step
    final = verify_chain_stepwise(chain, shapes, h, 3 * 2e-3, min_checked=(9 * 2 * T) // 10)   # (the bar of the other chains)
    assert np.array_equal(final, eager.cpu().numpy())


@pytest.mark.parametrize("hidden,inter,E,k,T", [(4096, 2048, 16, 8, 4), (4096, 2048, 16, 8, 8), (7168, 2048, 64, 8, 4), (2048, 1536, 32, 6, 9),
                                                (1536, 1536, 64, 6, 19), (2048, 1536, 32, 6, 7), (4096, 2048, 16, 8, 3), (4096, 2048, 64, 8, 3)])
@pytest.mark.parametrize("shared", ["none", "same", "q8_0"])
def test_few_tokens_stream_in_the_decode_launch_s_place(monkeypatch, hidden, inter, E, k, T, shared):
    """Half a pick per expert and more: from 28, 48 or 112 picks on by size of a matrix (the last three shapes are short of it; a Q8_0
    shared expert: from 7 tokens); a decode limit set by the caller brings the one-launch form back, the same sums in another order, whose bits the
    token counts short of both ranges have (three tokens on 64 experts)."""
    monkeypatch.setattr(MoeLayer, "v3_thresholds_below_experts", None)
    fmts = dict(sh_gate_fmt=FMT_Q8_0, sh_down_fmt=FMT_Q8_0) if shared == "q8_0" else {}
    s = H.Shape(hidden, inter, E, k, shared=shared != "none", seed=950 + T, **fmts, **ROUTER)
    dw = H.device_weights(s)
    layer, launch = MoeLayer(dw, T), MoeLayer(dw, T)
    launch.set_tuning(decode_max_tokens=16)
    streams = T * k >= (28 if hidden * inter >= 8 << 20 else 48 if hidden * inter >= 3 << 20 else 112) and (shared != "q8_0" or T >= 7)
    assert (T >= layer.streaming()[0]) == streams
    x, _, _ = H.host_inputs(s, T)
    rng = np.random.default_rng(T)
    sel = np.stack([rng.permutation(E)[:k] for _ in range(T)]).astype(np.int32)
    sel[T // 2, 1] = -1
    w = rng.uniform(0.05, 0.6, sel.shape).astype(np.float32)
    dx, ds, dwt = torch.from_numpy(x).cuda(), torch.from_numpy(sel).cuda(), torch.from_numpy(w).cuda()
    out = layer.run(dx, None, selected_in=ds, weights_in=dwt).clone()
    again = layer.run(dx, None, selected_in=ds, weights_in=dwt)
    if T <= 16:
        other = launch.run(dx, None, selected_in=ds, weights_in=dwt)
        assert layer.status() == 0 and launch.status() == 0
        assert torch.equal(out, other) == (not streams and T <= layer.tuning()["decode_max_tokens"])
        assert H.max_rel(out.cpu().numpy(), other.cpu().numpy()) < 1e-3
    torch.cuda.synchronize()
    assert torch.equal(out, again)
    H.assert_close(out.cpu().numpy(), ref.moe_forward(H.host_weights(s, experts=np.unique(sel[sel >= 0])), x, sel, w), 2e-3, f"{hidden} x {inter} T={T} {shared}")


def test_a_stack_of_few_token_streaming_blocks(monkeypatch):
    """The residual is added by the slot-order sum, in place."""
    monkeypatch.setattr(MoeLayer, "v3_thresholds_below_experts", None)
    shapes = layer_shapes(H.Shape(4096, 2048, 16, 8, seed=960, **ROUTER), 2)
    chain = MoeChain([H.device_weights(s, block=True) for s in shapes], 5)
    rng = np.random.default_rng(5)
    chain.capture(5)
    for step in range(3):
        h = rng.normal(0, 1, (5, 4096)).astype(np.float32)
        eager = chain.step(torch.from_numpy(h).cuda()).clone()
        torch.cuda.synchronize()
        replayed = chain.replay(torch.from_numpy(h).cuda()).clone()
        torch.cuda.synchronize()
        assert torch.equal(eager, replayed), step
    final = verify_chain_stepwise(chain, shapes, h, 3 * 2e-3, min_checked=(9 * 2 * 5) // 10)
    assert np.array_equal(final, eager.cpu().numpy())

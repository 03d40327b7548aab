"""The reference's own layer mix -- MXFP4 routed experts beside a Q8_0 shared expert whose
intermediate size differs from the routed one (docs/v41/ARCH_SPEC.md:239,
crates/v4flash-kernels/src/het/dispatch.rs:196-214) -- against the CPU oracle at every token
count that takes a different path: one launch / per-stage decode, by-expert, streaming, grouped GEMM
with the shared expert on the int8 GEMM.  Up to three tokens the Q8_0 shared expert is computed by items
of the one-launch decode path, from four on by the dense kernels on a side stream."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from deepstrix_amd.capi import FMT_Q8_0
from deepstrix_amd.executor import MoeLayer
from oracle import ref
from tests import helpers as H

pytestmark = pytest.mark.gpu

CONTRACT = 2e-3
# Regression bar beside the contract.  The integer dots are exact; what differs from the oracle
# is the order of f32 sums, and through it now and then the rounding of a mid value to int8
# (one step of 1/127 of its block's maximum).  With the Q8_0 shared expert's 32-wide blocks that
# reads up to 1.7e-4 of max|ref| on 64 tokens; three times that is the bar.
REGRESSION = 5e-4

SMALL = H.Shape(1024, 512, 16, 4, sh_gate_fmt=FMT_Q8_0, sh_down_fmt=FMT_Q8_0, sh_inter=384,
                router_mode=1, n_group=4, topk_group=2, route_scale=2.5, bias_sigma=0.01,
                clamp=10.0, seed=1201)
V3 = H.Shape(7168, 2048, 256, 8, sh_gate_fmt=FMT_Q8_0, sh_down_fmt=FMT_Q8_0, sh_inter=1024,
             router_mode=1, n_group=8, topk_group=4, route_scale=2.5, bias_sigma=0.01,
             seed=0xD5EE0F30)


def _check(s, layer, hw, T, modes=(1,)):
    x, logits, bias = H.host_inputs(s, T)
    dx, dl = torch.from_numpy(x).cuda(), torch.from_numpy(logits).cuda()
    rsel, _ = H.oracle_route(s, logits, bias)
    _, scores = ref.router_scores(logits, bias, s.router_mode, s.n_group, s.topk_group)
    for mode in modes:
        layer.set_decode(fused=mode)
        out, sel, w = layer.run(dx, dl, want_routing=True)
        assert layer.status() == 0
        sel, w, out = sel.cpu().numpy(), w.cpu().numpy(), out.cpu().numpy()
        assert H.routing_mismatch_explained(sel, rsel, scores, s.n_used) == []
        want = ref.moe_forward(hw, x, sel, w)     # the oracle on the GPU's routing, unconditionally
        H.assert_close(out, want, CONTRACT, f"T={T} mode={mode}")
        assert H.compare_stats(out, want)["max_over_max"] < REGRESSION, (T, mode)


@pytest.mark.parametrize("T", [1, 2, 3, 5, 6, 7, 9, 14, 16, 64, 130, 300])
def test_small_layer_with_q8_0_shared_expert_of_another_width(T):
    dw = H.device_weights(SMALL)
    layer = MoeLayer(dw, T)
    _check(SMALL, layer, H.host_weights(SMALL), T, modes=(1, 2) if T <= 14 else (1,))


def test_small_layer_pre_norm_block_with_q8_0_shared_expert():
    """h += layer(RMSNorm(h)) with the residual folded into the one-launch decode path (up to six
    tokens: the shared expert inside the launch; more: on the side stream, its rows and the
    residual added behind the join while the launch writes to a row buffer of the workspace)."""
    s = SMALL
    dw = H.device_weights(s, block=True)
    layer = MoeLayer(dw, 8)
    norm_w, router_w = H.host_block_params(s)
    hw = H.host_weights(s)
    rng = np.random.default_rng(3)
    for T in (1, 3, 5, 8):
        h0 = rng.standard_normal((T, s.hidden)).astype(np.float32)
        xn = ref.rms_norm(h0, norm_w, 1e-6)
        logits = ref.router_logits(router_w, xn)
        sel, w = H.oracle_route(s, logits, H.host_inputs(s, 1)[2])
        want = h0 + ref.moe_forward(hw, xn, sel, w)
        h = torch.from_numpy(h0.copy()).cuda()
        layer.block(h)
        assert layer.status() == 0
        H.assert_close(h.cpu().numpy(), want, CONTRACT, f"block T={T}")


@pytest.fixture(scope="module")
def v3_layers():
    """The layer as it is, the same with the streaming kernels off, its bytes on the host."""
    dw = H.device_weights(V3)
    layer, older = MoeLayer(dw, 512), MoeLayer(dw, 512)
    older.set_tuning(by_expert_chunk=4)
    assert layer.streaming() == (7, 575) and older.streaming() == (0, 0)
    return layer, older, H.host_weights_from_device(V3, dw)


@pytest.mark.parametrize("T,streams", [(1, True), (2, True), (4, True), (64, True), (512, True), (64, False), (512, False)])
def test_v3_shape_with_q8_0_shared_expert(T, streams, v3_layers):
    layer, older, hw = v3_layers
    _check(V3, layer if streams else older, hw, T, modes=(1, 2) if T <= 14 else (1,))


@pytest.mark.parametrize("T,streams", [(2, True), (4, True), (12, True), (24, True), (130, True), (12, False), (24, False), (130, False)])
def test_side_stream_shared_expert_under_graph_capture(T, streams, v3_layers):
    """From seven tokens on (decode, by-expert, streaming and GEMM paths alike) the Q8_0 shared expert is
    computed on a stream of its own, forked from and joined to the caller's: a capture of the
    caller's stream must record both branches, and every replay must give what the eager call
    gives -- bitwise, with the program's own work and synchronizations between the replays.
    (Two and four tokens: the shared expert inside the decode launch, no second stream.)"""
    s = V3
    layer = v3_layers[0 if streams else 1]
    layer.set_decode(fused=1)
    x, logits, _ = H.host_inputs(s, T)
    dx, dl = torch.from_numpy(x).cuda(), torch.from_numpy(logits).cuda()
    out = torch.empty((T, s.hidden), dtype=torch.float32, device="cuda")
    layer.run(dx, dl, out=out)
    assert layer.status() == 0
    eager = out.clone()
    side = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        layer.run(dx, dl, out=out)          # warm-up on the capturing stream
        side.synchronize()
        with torch.cuda.graph(graph, stream=side):
            layer.run(dx, dl, out=out)
    torch.cuda.synchronize()
    for rep in range(3):
        out.fill_(float(rep))               # eager work between the replays
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager), rep
        assert layer.status() == 0
    # and the eager path still agrees afterwards
    layer.run(dx, dl, out=out)
    torch.cuda.synchronize()
    assert torch.equal(out, eager)


@pytest.mark.parametrize("T", [1, 2, 5])
def test_q8_0_shared_expert_wider_than_the_routed_ones(T):
    """A shared expert wider than the routed experts cannot sit in the one-launch path's mid rows
    (they are `inter` long): it stays with the dense kernels at every token count."""
    s = H.Shape(1024, 256, 16, 4, sh_gate_fmt=FMT_Q8_0, sh_down_fmt=FMT_Q8_0, sh_inter=384,
                router_mode=1, n_group=4, topk_group=2, route_scale=2.5, bias_sigma=0.01,
                clamp=10.0, seed=1207)
    layer = MoeLayer(H.device_weights(s), T)
    _check(s, layer, H.host_weights(s), T, modes=(1, 2))

"""Q8_0 products on few members per expert against the CPU oracle and the older paths: the streaming kernels
(16-column items, dsx_stream_kernels.hpp) on rows of an odd and an even number of 128-value groups and in each
instance by row length (up to 8, 12, 16 and 32 groups), and the 32- and 64-column int8 GEMMs; items with one column and with
an empty column group, empty slots, an expert that nearly every token names (several items)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from deepstrix_amd.capi import FMT_MXFP4, FMT_Q8_0
from deepstrix_amd.executor import MoeLayer
from oracle import ref
from tests import helpers as H

pytestmark = pytest.mark.gpu

ROUTER = dict(router_mode=1, route_scale=2.5, bias_sigma=0.01, clamp=10.0)


def _run(s, T, seed, monkeypatch):
    monkeypatch.setattr(MoeLayer, "v3_thresholds_below_experts", None)   # the library's own thresholds
    x, _, _ = H.host_inputs(s, T)
    rng = np.random.default_rng(seed)
    sel = np.stack([rng.permutation(s.n_expert)[:2] for _ in range(T)]).astype(np.int32)
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
    want = ref.moe_forward(H.host_weights(s), x, sel, w)
    # the dots are exact: other orders of the f32 sums, and a mid value at a rounding boundary that takes the
    # neighbouring int8 step (fitted to a column of a down matrix)
    H.assert_parity_up_to_rounding_steps(out.cpu().numpy(), want, H.host_weights(s), sel, f"{s.hidden} x {s.inter} T={T}")
    return out, old


# (hidden, inter): gate/up rows of hidden / 128 groups, down rows of inter / 128
@pytest.mark.parametrize("hidden,inter", [(128, 256), (384, 1152), (1024, 640), (1152, 128), (2048, 1408), (2304, 2176), (4096, 512), (512, 4096)])
@pytest.mark.parametrize("T", [2, 15, 16, 60, 111])
def test_all_q8_0_layer_matches_the_oracle(monkeypatch, hidden, inter, T):
    """2 and 15 tokens: the streaming kernels; from 16 (4 picks per expert) to 111: the narrow GEMM, which has the
    bits of the wide one."""
    s = H.Shape(hidden, inter, 8, 2, FMT_Q8_0, FMT_Q8_0, shared=hidden != 1024, seed=800, **ROUTER)
    out, old = _run(s, T, T, monkeypatch)
    assert torch.equal(out, old) == (T >= 16)


@pytest.mark.parametrize("hidden,inter,shared", [(512, 256, "none"), (1280, 768, "same"), (1280, 768, "q8_0"),
                                                 (2048, 2048, "none"), (7168, 512, "same")])
@pytest.mark.parametrize("T", [10, 15, 16, 23, 24, 111])
def test_q8_0_down_behind_mxfp4_gate_up_matches_the_oracle(monkeypatch, hidden, inter, shared, T):
    fmts = dict(sh_gate_fmt=FMT_Q8_0, sh_down_fmt=FMT_Q8_0) if shared == "q8_0" else {}
    s = H.Shape(hidden, inter, 8, 2, down_fmt=FMT_Q8_0, shared=shared != "none", seed=820 + T, **fmts, **ROUTER)
    _run(s, T, T, monkeypatch)


@pytest.mark.parametrize("down_fmt", ["all", "down"])
@pytest.mark.parametrize("T", [112, 129, 167, 168])
def test_middle_tile_of_the_down_gemm_matches_the_oracle(monkeypatch, down_fmt, T):
    """28 to 42 picks per expert: down by 64-column items, several of the expert that most tokens name, with one to
    four column groups; the wide tile's bits."""
    s = H.Shape(512, 512, 8, 2, FMT_Q8_0 if down_fmt == "all" else FMT_MXFP4, FMT_Q8_0, seed=840 + T, **ROUTER)
    out, old = _run(s, T, T, monkeypatch)
    if down_fmt == "all":
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


def test_rows_longer_than_the_registers_take_the_older_paths(monkeypatch):
    """Gate/up rows of 33 groups: the older paths' bits."""
    s = H.Shape(4224, 256, 8, 2, FMT_Q8_0, FMT_Q8_0, shared=False, seed=850, **ROUTER)
    out, old = _run(s, 15, 5, monkeypatch)
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

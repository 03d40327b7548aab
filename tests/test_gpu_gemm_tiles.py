"""The grouped GEMMs of a planar layer with both tiles: small groups on the narrow one (non-temporal loads where a
group is one tile), the others on the wide one, as the picks have it.  The wide tile alone, on the engine's rows, gives
the same bits."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from deepstrix_amd import capi
from deepstrix_amd.executor import MoeLayer
from tests import helpers as H

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def layers():
    s = H.CFG2   # 7168 x 2048, 256 experts, top-8: both tiles from 384 to 1023 tokens
    rows, planar = MoeLayer(H.device_weights(s), 1024), MoeLayer(H.device_weights(s, planar=True), 1024)
    rows.set_tuning(gemm_min_tokens=1, decode_max_tokens=1, gemm_narrow_members=1)
    return s, rows, planar


def _picks(kind, T):
    rng = np.random.default_rng(T)
    if kind == "same":
        sel = np.tile(rng.permutation(256)[:8].astype(np.int32), (T, 1))
    elif kind == "sixteen":
        sel = np.tile(np.arange(248, 256, dtype=np.int32), (T, 1))
        for e in range(min(192, 7 * T // 17)):   # expert e: 15 + e % 3 members, in slot e % 7 of tokens that follow each other
            t0 = (e // 7) * 17
            sel[t0:t0 + 15 + e % 3, e % 7] = e
        sel[T // 2, 7] = -1
    else:
        p = np.ones(256) if kind == "spread" else 1.0 / (1.0 + np.arange(256)) ** 0.8
        g = -np.log(-np.log(rng.uniform(1e-9, 1.0, (T, 256))))   # Gumbel: eight of 256 without replacement
        sel = np.argsort(-(np.log(p) + g), axis=1)[:, :8].astype(np.int32)
    return np.ascontiguousarray(sel), rng.uniform(0.05, 0.6, sel.shape).astype(np.float32)


@pytest.mark.parametrize("T,picks,lists", [(383, "spread", "narrow"), (384, "spread", "both"), (600, "spread", "both"), (600, "skewed", "both"),
                                           (600, "sixteen", "both"), (600, "same", "wide"), (1023, "same", "wide"), (1024, "spread", "wide")])
def test_which_groups_the_two_lists_have(layers, T, picks, lists):
    """The items of either list as the group tables leave them in the workspace."""
    s, _, planar = layers
    sel, w = _picks(picks, T)
    n = np.append(np.bincount(sel[sel >= 0], minlength=256), T)   # (the shared expert: the last group)
    small = n <= 16
    items = lambda c, chunk: int((-(-c // chunk)).sum())
    want = {"narrow": (0, items(n, 16)), "wide": (items(n, 128), 0), "both": (items(n[~small], 128), items(n[small], 16))}[lists]
    planar.workspace.zero_()
    planar.run(torch.from_numpy(H.host_inputs(s, T)[0]).cuda(), None, selected_in=torch.from_numpy(sel).cuda(), weights_in=torch.from_numpy(w).cuda())
    torch.cuda.synchronize()
    up = lambda b: -(-b // 256) * 256
    rows = up(T * s.hidden * 4)   # the regions behind the first list's count: shared scratch, two of rows around the logits
    end = int(capi.lib().dsx_moe_layer_workspace_bytes(planar._h, T))
    ffn_out = end - rows
    first = ffn_out - up(T * 256 * 4) - rows - up(int(capi.lib().dsx_dense_ffn_scratch_bytes(T, s.hidden, s.inter))) - 256
    word = lambda at: int(planar.workspace[at:at + 4].cpu().numpy().view(np.int32)[0])
    second = word(ffn_out + 4 * (1 + 9 * T))
    # (outside the range the one list has the tile that the picks per expert call for)
    got = (word(first), second) if 384 <= T < 1024 else (0, word(first)) if T < 384 else (word(first), 0)
    assert got == want


@pytest.mark.parametrize("T", [32, 383, 384, 600, 1023, 1024])
@pytest.mark.parametrize("picks", ["spread", "skewed", "same", "sixteen"])
def test_both_tiles_give_the_wide_tiles_bits(layers, T, picks):
    """skewed: a tenth of the experts have most of the picks (both lists); same: all tokens name eight experts (the
    wide list alone); sixteen: groups of 15, 16 and 17 members, an empty slot, the rest on a few experts.  From 32 tokens
    on the other layer's threshold of one pick per expert makes its tile the wide one."""
    s, rows, planar = layers
    x = H.host_inputs(s, T)[0]
    sel, w = _picks(picks, T)
    dx, ds, dw = torch.from_numpy(x).cuda(), torch.from_numpy(sel).cuda(), torch.from_numpy(w).cuda()
    want = rows.run(dx, None, selected_in=ds, weights_in=dw)
    got = planar.run(dx, None, selected_in=ds, weights_in=dw).clone()
    again = planar.run(dx, None, selected_in=ds, weights_in=dw)
    torch.cuda.synchronize()
    assert planar.status() == 0 and torch.equal(got, want) and torch.equal(got, again)

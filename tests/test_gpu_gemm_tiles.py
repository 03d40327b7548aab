"""The grouped GEMMs of a planar layer with both tiles: small groups on the narrow one (non-temporal loads where a
group is one tile), the others on the wide one, as the picks have it.  The wide tile alone, on the engine's rows, gives
the same bits."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from deepstrix_amd.executor import MoeLayer
from tests import helpers as H

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def layers():
    s = H.CFG2   # 7168 x 2048, 256 experts, top-8: both tiles from 384 to 1023 tokens
    rows, planar = MoeLayer(H.device_weights(s), 1024), MoeLayer(H.device_weights(s, planar=True), 1024)
    rows.set_tuning(gemm_min_tokens=1, decode_max_tokens=1, gemm_narrow_members=1)
    return s, rows, planar


@pytest.mark.parametrize("T", [12, 383, 384, 600, 1023, 1024])
@pytest.mark.parametrize("picks", ["spread", "skewed", "same", "sixteen"])
def test_both_tiles_give_the_wide_tiles_bits(layers, T, picks):
    """skewed: a tenth of the experts have most of the picks (both lists); same: all tokens name eight experts (the
    wide list alone); sixteen: groups of 15, 16 and 17 members, an empty slot, the rest on a few experts."""
    s, rows, planar = layers
    x = H.host_inputs(s, T)[0]
    rng = np.random.default_rng(T)
    if picks == "same":
        sel = np.tile(rng.permutation(256)[:8].astype(np.int32), (T, 1))
    elif picks == "sixteen":
        sel = np.tile(np.arange(248, 256, dtype=np.int32), (T, 1))
        for e in range(min(192, 7 * T // 17)):   # expert e: 15 + e % 3 members, in slot e % 7 of tokens that follow each other
            t0 = (e // 7) * 17
            sel[t0:t0 + 15 + e % 3, e % 7] = e
        sel[T // 2, 7] = -1
    else:
        p = np.ones(256) if picks == "spread" else 1.0 / (1.0 + np.arange(256)) ** 0.8
        g = -np.log(-np.log(rng.uniform(1e-9, 1.0, (T, 256))))   # Gumbel: eight of 256 without replacement
        sel = np.argsort(-(np.log(p) + g), axis=1)[:, :8].astype(np.int32)
    w = rng.uniform(0.05, 0.6, sel.shape).astype(np.float32)
    dx, ds, dw = torch.from_numpy(x).cuda(), torch.from_numpy(np.ascontiguousarray(sel)).cuda(), torch.from_numpy(w).cuda()
    want = rows.run(dx, None, selected_in=ds, weights_in=dw)
    got = planar.run(dx, None, selected_in=ds, weights_in=dw).clone()
    again = planar.run(dx, None, selected_in=ds, weights_in=dw)
    torch.cuda.synchronize()
    assert planar.status() == 0 and torch.equal(got, want) and torch.equal(got, again)

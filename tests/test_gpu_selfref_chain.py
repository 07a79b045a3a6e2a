"""The chain-resident forward of the self-referential memory (chunks of up to 64 tokens) at the edges of its 16-token
tiles: chunks one token short of, at and behind a tile's end, last chunks of one token, every head size, both value
modes, against the float32 oracle; gradients against the float64 oracle (1e-4, fp32 sums over a chain)."""
import numpy as np
import pytest

from tests.gpu_util import assert_close
from tests.test_gpu_selfref import gpu_run, inputs, oracle_run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("s,C", [(33, 15), (33, 16), (35, 17), (66, 33), (97, 48), (112, 63), (17, 64), (18, 2)])
@pytest.mark.parametrize("d", [16, 32, 64])
@pytest.mark.parametrize("sg", [True, False])
def test_tile_edges(s, C, d, sg):
    mems, x, dy = inputs(2, s, d, seed=s * 100 + C + d)
    print(f"selfref chain s={s} d={d} C={C} sg={sg}", flush=True)
    got = gpu_run(mems, x, dy, C, sg)
    want = oracle_run(mems, x, dy, C, sg, np.float32)
    for n in ("y", "mems", "k", "v", "q", "alpha", "theta", "frozen"):
        assert_close(n, got[n].reshape(want[n].shape), want[n])
    ref = oracle_run(mems, x, dy, C, sg, np.float64)
    for n in ("d_emb", "d_mems"):
        assert_close(n, got[n].reshape(ref[n].shape), ref[n])


@pytest.mark.parametrize("C", [1, 17, 33, 49])
@pytest.mark.parametrize("d", [32, 64])
def test_tiles_of_one_token(C, d):
    """Chunks whose last tile is one token: its exchange and the next tile's first stand a single barrier apart, so the
    waves of a chain must not share the exchanged row between them.  Many chains, equal ones among them: the same bits."""
    B, s = 96, 3 * C + 1
    mems, x, dy = inputs(2, s, d, seed=7 * C + d)
    mems, x, dy = (np.concatenate([a] * (B // 2)) for a in (mems, x, dy))
    got = gpu_run(mems, x, dy, C, True)
    for n in ("y", "mems", "k", "v", "alpha", "theta"):
        a = got[n].reshape(B // 2, -1)
        assert (a == a[:1]).all(), n
    want = oracle_run(mems[:2], x[:2], dy[:2], C, True, np.float32)
    for n in ("y", "k", "v", "alpha", "theta"):
        assert_close(n, got[n].reshape(B, -1)[:2].reshape(want[n].shape), want[n])

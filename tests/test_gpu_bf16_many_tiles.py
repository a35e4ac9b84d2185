"""bf16 experts on either side of the number of M tiles a launch's grid takes
(65,536): up to there the matrix-core GEMMs, beyond it the vector kernels, whose
grids do not grow with the tokens. Every expert gets every token (top-64 of 64), so
few tokens make many tiles; sampled tokens against the oracle's exact block, within
TOL_BF16: a token's 64 rows of about equal weight are each rounded to bf16, 2^-9 of
the row, and partly cancel in the sum."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from oracle import oracle as O  # noqa: E402
from tests.common import rel_err  # noqa: E402
from tests.test_gpu_branches import TOL_BF16, Blk, x_np  # noqa: E402

pytestmark = pytest.mark.gpu


def test_tiles_around_the_grid_limit():
    from helexa_amd import synth
    b = Blk(256, 64, 64, 256, 0, True, synth.FMT_BF16, O.BF16, 31)
    tiles = lambda T: T + 64 + (T + 63) // 64 + 1   # rows / 64, one more an expert, the shared expert's
    for T in (64400, 64700):
        assert (tiles(T) <= 65536) == (T == 64400)
        x = b.x(T, seed=T)
        y = b.block.forward(x)
        assert bool(torch.isfinite(y).all())
        sel = np.array([0, 1, 63, 64, 4096, T // 2, T - 65, T - 1])
        got = y[torch.from_numpy(sel).cuda()].float().cpu().numpy()
        assert rel_err(got, b.ref_tokens(x_np(x), sel)) <= TOL_BF16, T
        del x, y

"""The generic kernels at small token counts: router logits and routing
bit-exact at every pair and group boundary of the router's grids (1 to 9 tokens,
and 56 to 65, where it starts to map token groups to XCDs), and the down kernel
that takes its rows from the decode plan, for row counts around the 16 a
workgroup has in flight, with rows of h held beside the weights and not, one
output row and several a wave, against the oracle."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.test_gpu_branches import TOL_BF16, TOL_F32, TOL_F32_GGUF, Blk, x_np

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,fmt,act", [(264, "FMT_F32", O.F32), (2048, "FMT_BF16", O.BF16), (2304, "FMT_F32", O.F32)])
def test_router_groups(H, fmt, act):
    from helexa_amd import synth
    b = Blk(H, 40, 4, 32, 32, True, getattr(synth, fmt), act, 1100 + H)
    for T in (1, 2, 3, 4, 7, 8, 9, 56, 57, 64, 65):
        x = b.x(T, seed=T)
        got = b.block.router_logits(x).cpu().numpy()
        assert np.array_equal(got.view(np.uint32), b.oracle.logits(x_np(x)).view(np.uint32)), T


# (H, E, k, I, Is): rows of h T (k + 1); 8, 16, 32, 64 lanes a row and several chunks a lane
@pytest.mark.parametrize("H,E,k,I,Is,fmt,act,tol", [
    (64, 8, 3, 64, 64, "FMT_F32", O.F32, TOL_F32), (256, 16, 4, 128, 0, "FMT_F32", O.F32, TOL_F32),
    (256, 16, 15, 768, 768, "FMT_F32", O.F32, TOL_F32), (512, 24, 7, 512, 512, "FMT_BF16", O.BF16, TOL_BF16),
    (512, 9, 2, 256, 512, "FMT_Q8_0", O.F32, TOL_F32_GGUF), (264, 9, 2, 40, 24, "FMT_BF16", O.BF16, TOL_BF16)])
def test_down_rows_from_plan(H, E, k, I, Is, fmt, act, tol):
    from helexa_amd import synth
    b = Blk(H, E, k, I, Is, True, getattr(synth, fmt), act, 1200 + I)
    for T in (1, 2, 4, 5, 8):
        b.check(b.x(T, seed=T), tol, tag=f"generic decode H{H} I{I} T={T}")

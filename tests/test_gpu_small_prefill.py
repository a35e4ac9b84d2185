"""Prompts of 9 to 33 tokens, either side of the count up to which every tile has
at most 32 rows and kernels that hold only those run, with calls of every row
count up to all tokens (2 of 4 experts a token), against the reference's
arithmetic."""
import pytest

from oracle import oracle as O
from tests.test_gpu_branches import TOL_BF16, Blk

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt", ["FMT_Q4_K_M", "FMT_Q8_0", "FMT_BF16"])
@pytest.mark.parametrize("T", [9, 16, 17, 32, 33])
def test_small_prefill(fmt, T):
    from helexa_amd import synth
    b = Blk(512, 4, 2, 512, 512, True, getattr(synth, fmt), O.BF16, 801)
    b.check(b.x(T, seed=T), TOL_BF16, tag=f"{fmt} T={T}")

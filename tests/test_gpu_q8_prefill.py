"""Q8_0 experts in prefill: tiles of 1 to 64 rows and their remainders, calls on
either side of the 64 rows where the reference changes arm, every width the
kernels' chunks allow from the smallest, with and without a shared expert, one
stream and the side stream, against the reference's arithmetic (candle mode),
max-normwise within TOL_BF16: the bf16 rounding of the weighted rows and of the
output, 2^-9 of each, over the f16 rounding of the operands (2^-11) and the rare
code of h one step off."""
import pytest

from oracle import oracle as O
from tests.test_gpu_branches import TOL_BF16, Blk

pytestmark = pytest.mark.gpu


# (H, E, k, I, shared, renormalised, T): rows of an expert's call follow from T k / E
@pytest.mark.parametrize("H,E,k,I,shared,norm", [(256, 4, 2, 256, 256, True), (2048, 64, 8, 512, 512, True),
                                                 (1536, 8, 4, 768, 0, True), (768, 16, 4, 1024, 1024, False)])
@pytest.mark.parametrize("T", [9, 33, 64, 65, 160])
def test_q8_prefill_tiles(H, E, k, I, shared, norm, T):
    from helexa_amd import synth
    b = Blk(H, E, k, I, shared, norm, synth.FMT_Q8_0, O.BF16, 700 + H + E)
    b.check(b.x(T, seed=T), TOL_BF16, tag=f"q8 prefill H{H} I{I} T={T}")


def test_q8_prefill_side_stream():
    from helexa_amd import synth
    b = Blk(512, 16, 4, 256, 256, True, synth.FMT_Q8_0, O.BF16, 701)
    b.check(b.x(2049, seed=2), TOL_BF16, tag="q8 prefill T=2049")


def test_q8_prefill_wide():
    """K beyond the columns whose scales are in LDS at a time (2048): a remainder
    window in gate/up, a whole second one in down"""
    from helexa_amd import synth
    b = Blk(2304, 4, 2, 4096, 0, True, synth.FMT_Q8_0, O.BF16, 702)
    b.check(b.x(40, seed=3), TOL_BF16, tag="q8 prefill H2304 I4096")


@pytest.mark.parametrize("down", ["Q4_K", "Q6_K"])
@pytest.mark.parametrize("T", [33, 160])
def test_q8_gate_up_other_down(down, T):
    """Q8_0 gate and up over k-quant down weights: h is quantised by its own
    kernel there (blocks of 256), on both sides of the 64 rows"""
    from helexa_amd import moe, synth
    fmt = dict(synth.FMT_Q8_0, down=getattr(moe, down), sdown=getattr(moe, down))
    b = Blk(512, 8, 4, 512, 512, True, fmt, O.BF16, 703)
    b.check(b.x(T, seed=4), TOL_BF16, tag=f"q8 gate/up, {down} down T={T}")

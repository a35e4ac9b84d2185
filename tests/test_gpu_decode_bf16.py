"""One token on bf16 experts at the shapes of the overlapped decode kernels:
expert counts at both ends of the range, with and without a shared expert, the
routing bit-exact, the output against the oracle's exact block (one bf16
rounding of f32 sums: TOL_BF16 holds with room) and, through the decoder step,
the residual; the shapes beside them take the generic kernels."""
import pytest

from oracle import oracle as O
from tests.common import rel_err
from tests.test_gpu_branches import TOL_BF16, Blk, x_np

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("E,k,Is", [(257, 10, 512), (512, 10, 512), (300, 10, 0), (256, 10, 512), (300, 9, 512)])
def test_one_token_bf16(E, k, Is):
    import torch
    from helexa_amd import synth
    b = Blk(2048, E, k, 512, Is, True, synth.FMT_BF16, O.BF16, 1000 + E)
    for seed in (1, 2):
        x = b.x(1, seed=seed)
        b.check(x, TOL_BF16, tag=f"bf16 decode E={E} k={k} Is={Is}")
        w = torch.linspace(-0.5, 0.5, 2048, device="cuda")
        n = torch.from_numpy(O.rmsnorm(x_np(x), w.cpu().numpy(), 1e-6, O.BF16)).to(torch.bfloat16)
        ref = x.float().cpu().numpy() + b.ref(x_np(n))
        got = b.block.decoder_mlp_(x.clone(), w, 1e-6).float().cpu().numpy()
        assert rel_err(got, ref) <= TOL_BF16

"""hx_moe_decoder_mlp on prompts: the RMSNorm at the widths where its register
count changes (and beyond, where it loops), the residual added by the combine,
bf16 and f32, a hidden size of more than one combine block, against the oracle:
x + block(rmsnorm(x)), within the tolerance of the block's output."""
import pytest

from oracle import oracle as O
from tests.common import rel_err
from tests.test_gpu_branches import TOL_BF16, TOL_F32, Blk, x_np

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,fmt,act", [(264, "FMT_F32", O.F32), (1024, "FMT_F32", O.F32), (768, "FMT_Q8_0", O.BF16),
                                       (1280, "FMT_BF16", O.BF16), (2304, "FMT_Q4_K_M", O.BF16),
                                       (4352, "FMT_Q8_0", O.BF16)])
@pytest.mark.parametrize("T", [9, 70])
def test_decoder_prefill(H, fmt, act, T):
    import torch
    from helexa_amd import synth
    b = Blk(H, 8, 2, 256, 256, True, getattr(synth, fmt), act, 900 + H)
    x = b.x(T, seed=T)
    w = torch.linspace(-0.5, 0.5, H, device="cuda")
    n = torch.from_numpy(O.rmsnorm(x_np(x), w.cpu().numpy(), 1e-6, act))
    n = n.to(torch.bfloat16) if act == O.BF16 else n
    ref = x.float().cpu().numpy() + b.ref(x_np(n))
    got = b.block.decoder_mlp_(x.clone(), w, 1e-6).float().cpu().numpy()
    assert rel_err(got, ref) <= (TOL_BF16 if act == O.BF16 else TOL_F32)


@pytest.mark.parametrize("act,offset", [(O.BF16, 1), (O.BF16, 4), (O.F32, 1)])
def test_residual_stream_at_any_element(act, offset):
    """a stream that does not start on 16 bytes: same bits as one that does"""
    import torch
    from helexa_amd import synth
    H, T = 768, 21
    b = Blk(H, 8, 2, 256, 256, True, synth.FMT_Q8_0 if act == O.BF16 else synth.FMT_F32, act, 41)
    x = b.x(T, seed=3)
    w = torch.linspace(-0.5, 0.5, H, device="cuda")
    buf = torch.empty(T * H + 8, dtype=x.dtype, device="cuda")
    off = buf[offset:offset + T * H].view(T, H).copy_(x)
    assert off.data_ptr() % 16 != 0
    assert torch.equal(b.block.decoder_mlp_(off, w, 1e-6), b.block.decoder_mlp_(x.clone(), w, 1e-6))

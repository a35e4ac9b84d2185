"""bf16 experts in prefill (the MFMA grouped GEMMs): tiles of 1 to 64 rows and
their remainders, every width the kernels' chunks allow from the smallest, with
and without a shared expert, both routings, against the oracle's exact block.

Tolerance: products are exact and summed in f32 (terms of order 2^-24), so the
distance is the bf16 rounding of the weighted expert rows and of the output,
each at most 2^-9 of the value: max-normwise |y - ref| <= 2^-9 (sum over the
rows of a token of |row| + |y|). The rows of a token partly cancel in y; the sum
of their magnitudes is below 4 max|y| over these inputs, so 5 * 2^-9 < 1e-2
(TOL_BF16)."""
import pytest

from oracle import oracle as O
from tests.test_gpu_branches import TOL_BF16, Blk, x_np

pytestmark = pytest.mark.gpu


# (H, E, k, I, shared, renormalised): rows of an expert's call follow from T k / E
@pytest.mark.parametrize("H,E,k,I,shared,norm", [(256, 4, 2, 256, 256, True), (2048, 64, 8, 512, 512, True),
                                                 (1536, 8, 4, 768, 0, True), (768, 16, 4, 1024, 1024, False)])
@pytest.mark.parametrize("T", [9, 31, 33, 130])
def test_bf16_prefill_tiles(H, E, k, I, shared, norm, T):
    from helexa_amd import synth
    b = Blk(H, E, k, I, shared, norm, synth.FMT_BF16, O.BF16, 500 + H + E)
    b.check(b.x(T, seed=T), TOL_BF16, tag=f"bf16 prefill H{H} I{I} T={T}")


# five to eight tokens (a slot's rows in one half-filled tile, f32 rows, one
# rounding) and four, which stay on the decode GEMVs: slots of up to eight rows,
# groups of eight slots partly filled, more rows a token than the combine holds
# at a time
@pytest.mark.parametrize("H,E,k,I,shared,norm", [(256, 8, 6, 256, 256, True), (2048, 64, 8, 512, 512, True),
                                                 (1536, 9, 6, 768, 0, True), (768, 16, 14, 1024, 1024, False)])
@pytest.mark.parametrize("T", [4, 5, 7, 8])
def test_bf16_few_tokens(H, E, k, I, shared, norm, T):
    import torch
    from helexa_amd import synth
    b = Blk(H, E, k, I, shared, norm, synth.FMT_BF16, O.BF16, 700 + H + E)
    x = b.x(T, seed=T)
    b.check(x, TOL_BF16, tag=f"bf16 few H{H} I{I} T={T}")
    assert b.block.workspace_size(T) <= b.block.workspace_size(T + 1)
    # the residual in the combine, and by itself for a stream off 16 bytes
    w = torch.linspace(-0.5, 0.5, H, device="cuda")
    n = torch.from_numpy(O.rmsnorm(x_np(x), w.cpu().numpy(), 1e-6, O.BF16)).to(torch.bfloat16)
    ref = x.float() + b.block.forward(n.cuda().view_as(x)).float()
    off = torch.empty(T * H + 8, dtype=x.dtype, device="cuda")[1:1 + T * H].view(T, H).copy_(x)
    assert torch.equal(b.block.decoder_mlp_(x.clone(), w, 1e-6), b.block.decoder_mlp_(off, w, 1e-6))
    assert torch.equal(off, ref.bfloat16())


# h goes into the down products as three bf16 parts, of which some are exactly
# zero: an infinite weight must still give the infinity that h itself gives.
# Every output column of expert 0 meets one infinity, at another row of h
@pytest.mark.parametrize("sign", [1.0, -1.0])
@pytest.mark.parametrize("T", [7, 9, 130])
def test_bf16_infinite_down_weights(T, sign):
    import numpy as np
    import torch
    import helexa_amd as hx
    from helexa_amd import synth
    H, E, k, I = 1024, 8, 6, 256
    cfg = hx.TextConfig(hidden_size=H, num_experts=E, num_experts_per_tok=k, moe_intermediate_size=I,
                        shared_expert_intermediate_size=0, norm_topk_prob=True)
    w = synth.make_weights(cfg, synth.FMT_BF16, 21)
    n = torch.arange(H, device="cuda")
    w["down"][1][0, n, n % I] = sign * float("inf")
    b = hx.Qwen3_5MoeBlock.load(cfg, w, act_dtype=hx.BF16)
    x = synth.make_x(cfg, T, 4)
    got = b.forward(x).float().cpu().numpy()
    ref = O.OracleMoe(H, E, k, I, 0, True, O.BF16, synth.to_numpy(w)).forward(x_np(x))
    assert np.isinf(ref).any() and not np.isnan(ref).any()
    fin = np.isfinite(ref)
    assert np.array_equal(got[~fin], ref[~fin])
    assert fin.any() and np.abs(got[fin] - ref[fin]).max() <= TOL_BF16 * np.abs(ref[fin]).max()


@pytest.mark.parametrize("offset", [1, 2, 4])
def test_bf16_few_tokens_output_at_any_element(offset):
    """an output that does not start on 8 bytes: same bits as one that does, and
    nothing beside it written"""
    import torch
    from helexa_amd import synth
    H, T = 768, 7
    b = Blk(H, 16, 6, 256, 256, True, synth.FMT_BF16, O.BF16, 22)
    x = b.x(T, seed=5)
    buf = torch.full((T * H + 16,), 7.0, dtype=x.dtype, device="cuda")
    out = buf[8 + offset:8 + offset + T * H].view(T, H)
    assert torch.equal(b.block.forward(x, out=out), b.block.forward(x))
    assert (buf[:8 + offset] == 7).all() and (buf[8 + offset + T * H:] == 7).all()

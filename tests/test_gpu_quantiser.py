"""The device quantiser at its workgroup edges, byte for byte against the oracle:
row counts around the 128 Q8_0 blocks, 32 Q4_K and 16 Q6_K superblocks a
workgroup takes, sources and destinations off 16-byte alignment, blocks of one
sign (minima of -0), all-zero sub-blocks beside others, and values that sit on
rounding boundaries."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt,per_wg", [(O.Q8_0, 128), (O.Q4_K, 32), (O.Q6_K, 16), (O.BF16, 2048)])
@pytest.mark.parametrize("blocks", [-1, 0, 1])
def test_quantiser_edges(dt, per_wg, blocks):
    import torch
    from helexa_amd import moe as hx
    cols = {O.Q8_0: 32, O.BF16: 1}.get(dt, 256)
    rows = 2 * per_wg + blocks
    g = torch.Generator(device="cuda").manual_seed(41 + blocks)
    base = torch.randn(rows * cols + 4, generator=g, device="cuda") * 0.02
    x = base[:rows * cols].view(rows, cols)
    x[1::5] = x[1::5].abs()
    x[2::5] = -x[2::5].abs()
    x[3::5] = torch.round(x[3::5] * 800) / 2               # halves: rounding boundaries
    x[4::10, : max(1, cols // 2)] = 0.0
    x[9::10] *= 1e-6
    ref = O.quantize(dt, x.cpu().numpy()).reshape(-1)
    assert np.array_equal(hx.quantize(dt, x).cpu().numpy().reshape(-1), ref)
    # a source on a 4-byte boundary, a destination on a 2-byte one; nothing written past its end
    y = base[1:1 + rows * cols].view(rows, cols)
    y.copy_(x.clone())
    out = torch.zeros(ref.size + 34, dtype=torch.uint8, device="cuda")
    hx.check(hx.lib().hx_quantize(dt, y.data_ptr(), rows, cols, out.data_ptr() + 2,
                                  torch.cuda.current_stream().cuda_stream), "hx_quantize")
    got = out.cpu().numpy()
    assert np.array_equal(got[2:2 + ref.size], ref)
    assert not got[2 + ref.size:].any()


@pytest.mark.parametrize("dt", [O.Q8_0, O.Q4_K, O.Q6_K, O.BF16, O.F16])
def test_quantiser_special_values(dt):
    """blocks with infinities, NaN, -0, denormals, values whose squares and sums
    overflow or underflow, and blocks of nothing else"""
    import torch
    from helexa_amd import moe as hx
    inf, nan = np.float32("inf"), np.float32("nan")
    rng = np.random.default_rng(77)
    special = [inf, -inf, nan, -0.0, 1e-45, -1e-40, 3e38, -3e38, 1e20, 1e-20, 2.0 ** -126, 65504.0, 70000.0]
    x = rng.standard_normal((6 * len(special) + 4, 512)).astype(np.float32) * np.float32(0.02)
    for i, v in enumerate(special):
        x[6 * i, 5] = v                      # one in a block
        x[6 * i + 1, 16:48] = v              # a run over sub-blocks
        x[6 * i + 2, 256:] = v               # whole blocks
        x[6 * i + 3, ::7] = v
        x[6 * i + 4] *= v                    # a row scaled by it
        x[6 * i + 5] = np.where(rng.random(512) < 0.5, v, -np.float32(v))
    x[-4], x[-3], x[-2], x[-1] = 0.0, -0.0, nan, inf
    x[-1, ::2] = -inf
    ref = O.quantize(dt, x)
    got = hx.quantize(dt, torch.from_numpy(x).cuda()).cpu().numpy()
    bad = np.unique(np.nonzero(got.reshape(ref.shape) != ref)[0])
    assert bad.size == 0, bad

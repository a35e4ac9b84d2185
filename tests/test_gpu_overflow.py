"""A token of values that overflow, of infinities or of NaN: it is routed to experts
that exist (its probabilities are NaN; where the expert count does not fill the
wave's 64 lanes, the padding's are too, and of a sign that ordered above), and the
other tokens of the call are bit for bit what they are beside an ordinary one. On
every routing path: one token, up to 8, longer calls with the router on the matrix
cores and not; every expert call at most 64 rows either way, so that no arm changes."""
import pytest

torch = pytest.importorskip("torch")

from oracle import oracle as O  # noqa: E402
from tests.test_gpu_branches import Blk  # noqa: E402

pytestmark = pytest.mark.gpu


# 16, 40 and 300 experts: 48, 24 and 212 ids of padding
@pytest.mark.parametrize("H,E,k,I,fmt,act,norm", [(512, 16, 6, 256, "FMT_BF16", O.BF16, True),
                                                  (512, 16, 6, 256, "FMT_Q8_0", O.BF16, True),
                                                  (512, 40, 6, 512, "FMT_Q4_K_M", O.BF16, False),
                                                  (256, 40, 4, 128, "FMT_F32", O.F32, True),
                                                  (2048, 300, 10, 512, "FMT_BF16", O.BF16, True),
                                                  (2048, 300, 10, 512, "FMT_Q8_0", O.BF16, True)])
def test_tokens_isolated_from_an_overflowing_token(H, E, k, I, fmt, act, norm):
    from helexa_amd import synth
    b = Blk(H, E, k, I, I, norm, getattr(synth, fmt), act, 1400 + E)
    for T in (1, 6, 9, 60):
        x = b.x(T, seed=T)
        y0 = b.block.forward(x)
        for bad in (1e38, float("inf"), "nan", "-nan"):
            print(f"[overflow] H={H} E={E} {fmt} T={T} {bad}", flush=True)
            xb = x.clone()
            if isinstance(bad, float):
                xb[T // 2] = bad
            else:   # the bits of a quiet NaN of either sign
                bits = xb.view(torch.int16 if act == O.BF16 else torch.int32)
                bits[T // 2] = (0x7fc0 if bad == "nan" else -0x40) << (0 if act == O.BF16 else 16)
            r = b.block.route(xb)
            ix = r["topk_idx"].cpu().numpy()
            assert ix.min() >= 0 and ix.max() < E
            assert all(len(set(row)) == k for row in ix.tolist())
            y1 = b.block.forward(xb)
            keep = torch.arange(T, device="cuda") != T // 2
            assert torch.isfinite(y1[keep]).all()
            assert torch.equal(y1[keep], y0[keep])
            assert bad == 1e38 or not torch.isfinite(y1[T // 2]).all()

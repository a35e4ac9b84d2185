"""Q8_0 experts in prefill, bit for bit. A code between -32 and 31 under one f16
scale a 256-element run is the same weight in Q8_0 and in Q6_K, so beyond 64 rows
an expert call, where both formats take f16 activations, the two blocks run the
same products: the Q8_0 kernels (weights into registers) have to sum and round
them as the kernels that dequantise into LDS do, f16 h included (rounded once).
Widths of one chunk pair, of several, and with more columns than the scales held
in LDS at a time (2048); 16-row sub-tiles in every number and a remainder."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from oracle import oracle as O  # noqa: E402

pytestmark = pytest.mark.gpu


def both_formats(rng, rows, cols):
    """the same weights as (Q8_0 rows, Q6_K rows)"""
    q = rng.integers(-32, 32, (rows, cols // 256, 256)).astype(np.int8)
    d = (rng.uniform(0.4, 1.6, (rows, cols // 256, 1)) * 1e-3).astype(np.float16)
    b = np.repeat(d[:, :, None, :], 8, axis=2).view(np.uint8)
    q8 = np.concatenate([b, q.reshape(rows, cols // 256, 8, 32).view(np.uint8)], axis=3)
    u = (q + 32).astype(np.uint8).reshape(rows, cols // 256, 2, 4, 32)   # halves, quarters
    ql = np.concatenate([(u[:, :, :, 0] & 15) | ((u[:, :, :, 2] & 15) << 4),
                         (u[:, :, :, 1] & 15) | ((u[:, :, :, 3] & 15) << 4)], axis=3)
    qh = (u[:, :, :, 0] >> 4) | ((u[:, :, :, 1] >> 4) << 2) | ((u[:, :, :, 2] >> 4) << 4) | ((u[:, :, :, 3] >> 4) << 6)
    sc = np.ones((rows, cols // 256, 16), np.uint8)
    q6 = np.concatenate([ql.reshape(rows, -1, 128), qh.reshape(rows, -1, 64), sc, d.view(np.uint8)], axis=2)
    q8, q6 = q8.reshape(rows, -1), q6.reshape(rows, -1)
    assert np.array_equal(O.dequantize(O.Q8_0, q8, cols), O.dequantize(O.Q6_K, q6, cols))
    return q8, q6


@pytest.mark.parametrize("H,I,shared", [(256, 256, True), (512, 768, False), (2304, 256, True), (256, 2304, False)])
def test_q8_prefill_bits(H, I, shared):
    import helexa_amd as hx
    from helexa_amd import synth
    E = 2                                   # top-2 of 2: every call has all tokens
    rng = np.random.default_rng(H + I)
    cfg = hx.TextConfig(hidden_size=H, num_experts=E, num_experts_per_tok=E, moe_intermediate_size=I,
                        shared_expert_intermediate_size=I if shared else 0, norm_topk_prob=True)
    base = synth.make_weights(cfg, synth.FMT_BF16, 5)
    shapes = {k: s for k, s in synth.shapes(cfg).items() if k not in ("router", "seg")}
    w = {k: both_formats(rng, int(np.prod(s[:-1])), s[-1]) for k, s in shapes.items()}

    def block(gate_up, down):
        out = {k: base[k] for k in base if k not in shapes}
        for k in shapes:
            f = down if k in ("down", "sdown") else gate_up
            out[k] = (f, torch.from_numpy(w[k][0 if f == hx.Q8_0 else 1]).cuda())
        return hx.Qwen3_5MoeBlock.load(cfg, out, act_dtype=hx.BF16)

    lds = block(hx.Q6_K, hx.Q6_K)
    regs = [(f, block(*f)) for f in ((hx.Q8_0, hx.Q6_K), (hx.Q6_K, hx.Q8_0), (hx.Q8_0, hx.Q8_0))]
    for T in (65, 80, 97, 128, 300):
        x = synth.make_x(cfg, T, T)
        ref = lds.forward(x)
        assert torch.isfinite(ref).all() and ref.float().abs().max() > 0
        for f, b in regs:
            print(f"[q8 bits] H={H} I={I} T={T} formats {f}", flush=True)
            assert torch.equal(b.forward(x), ref), f

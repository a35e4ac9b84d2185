"""Workspaces over token counts: a buffer sized for T tokens serves every smaller
call. Up to 8 tokens the layout changes with the kernels a call takes (records on
GGUF experts, f32 weighted rows on bf16 experts from 5 tokens and 30 assignments
on), and the shapes here put those changes where the need of fewer tokens is the
larger: wide intermediates and few assignments a token, the step from 8 to 9."""
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu


def make(H, E, k, I, fmt):
    import helexa_amd as hx
    from helexa_amd import synth
    cfg = hx.TextConfig(hidden_size=H, num_experts=E, num_experts_per_tok=k, moe_intermediate_size=I,
                        shared_expert_intermediate_size=I, norm_topk_prob=True)
    return hx.Qwen3_5MoeBlock.load(cfg, synth.make_weights(cfg, getattr(synth, fmt), 9), act_dtype=hx.BF16)


SHAPES = [(256, 64, 4, 1280, "FMT_BF16"), (512, 64, 4, 2304, "FMT_BF16"), (2048, 64, 10, 512, "FMT_BF16"),
          (512, 16, 10, 2048, "FMT_Q8_0"), (256, 16, 4, 512, "FMT_Q4_K_M")]


@pytest.mark.parametrize("H,E,k,I,fmt", SHAPES)
def test_a_buffer_serves_smaller_calls(H, E, k, I, fmt):
    from helexa_amd import synth
    b = make(H, E, k, I, fmt)
    sizes = [b.workspace_size(T) for T in range(25)]
    assert sizes == sorted(sizes), sizes
    for T in (1, 4, 5, 7, 8):
        x = synth.make_x(b.cfg, T, T)
        ws = torch.empty(b.workspace_size(T + 1), dtype=torch.uint8, device="cuda")
        assert torch.equal(b.forward(x, workspace=ws), b.forward(x))


@pytest.mark.parametrize("H,E,k,I,fmt", SHAPES)
def test_own_workspace_serves_smaller_calls(H, E, k, I, fmt):
    """the handle's own workspace, grown by a call of 9 tokens, holds every smaller
    one: they can be captured (growing it is not possible there), and the replays
    equal the eager results"""
    from helexa_amd import synth
    b = make(H, E, k, I, fmt)
    xs = [synth.make_x(b.cfg, T, T) for T in (8, 7, 5)]
    big = synth.make_x(b.cfg, 9, 9)
    b.forward(big)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    outs, g = [torch.zeros_like(x) for x in xs], torch.cuda.CUDAGraph()
    with torch.cuda.stream(s):
        with torch.cuda.graph(g, stream=s):
            for x, o in zip(xs, outs):
                b.forward(x, stream=s, out=o)
    torch.cuda.current_stream().wait_stream(s)
    refs = [b.forward(x) for x in xs]
    for _ in range(3):
        for o in outs:
            o.fill_(float("nan"))
        b.forward(big)
        g.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(o, r) for o, r in zip(outs, refs))

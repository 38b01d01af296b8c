"""The patch convolution as others see it who follow its operations (no GPU needed)."""
import pytest
import torch


def _conv(dtype):
    from lingbot_map_amd.aggregator import PatchConv
    torch.manual_seed(0)
    conv = PatchConv(14, 64).to(dtype)
    return conv, torch.randn(2, 3, 28, 42).to(dtype)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("grad", [False, True])
def test_patch_conv_can_be_traced(dtype, grad):
    conv, images = _conv(dtype)
    with torch.set_grad_enabled(grad):
        want = conv(images)
        traced = torch.fx.symbolic_trace(conv)
        assert torch.equal(traced(images), want)
        assert [n.target for n in traced.graph.nodes if n.op == "call_module"] == ["proj"]
        assert torch.equal(torch.jit.trace(conv, images)(images), want)


def test_patch_conv_compiles_as_one_graph(monkeypatch):
    """Nothing in it that a compiled graph has to be broken for, the question for the kernel's way included (whose answer on
    the CPU is made the one of the GPU)."""
    from lingbot_map_amd import aggregator
    conv, images = _conv(torch.bfloat16)
    monkeypatch.setattr(aggregator, "_plain", lambda *tensors: True)
    with torch.no_grad():
        compiled = torch.compile(conv, backend="eager", fullgraph=True)
        assert torch.equal(compiled(images), conv.proj(images).flatten(2).transpose(1, 2))

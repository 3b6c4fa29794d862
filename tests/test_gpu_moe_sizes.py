"""The MoE layer's scratch and task lists over token counts: a call gives the
same bits whatever max_tokens its context was made with."""
import pytest

from conftest import load_pkg

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_dev(gpu):
    import torch
    return torch, gpu


@pytest.mark.parametrize("n", [2, 17, 64, 65, 300])
def test_call_smaller_than_context(torch_dev, n):
    """calls below the context's max_tokens: the one of up to 64 tokens has
    more task entries than one of 300"""
    torch, dev = torch_dev
    pkg = load_pkg()
    x = torch.randn((n, 512), generator=torch.Generator().manual_seed(n)).to(dev).bfloat16()
    outs = []
    for most in (n, max(n, 300), 4096):
        with pkg.MoeContext(512, 512, 10, 512, n_layers=1, max_tokens=most) as ctx:
            ctx.synth_layer(0, 5)
            outs.append(ctx.layer_forward(0, x).clone())
            torch.cuda.synchronize()
    assert torch.isfinite(outs[0]).all()
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])

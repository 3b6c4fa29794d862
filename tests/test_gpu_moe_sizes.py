"""The MoE layer's scratch, task lists and choice of kernels over token counts
and expert counts: a call gives the same bits whatever max_tokens its context
was made with, and the oracle's rows (2e-2 max-abs, 1e-3 relative L2)."""
import numpy as np
import pytest

from conftest import load_oracle, load_pkg
from test_gpu_parity import assert_out_close, to_dev

orc = load_oracle()

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_dev(gpu):
    import torch
    return torch, gpu


@pytest.mark.parametrize("n", [2, 17, 64, 65, 300])
def test_call_smaller_than_context(torch_dev, n):
    """calls below the context's max_tokens, whose task lists may have more
    entries than the largest call's"""
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


# (H, E, k, I) and the token counts on both sides of each line between the
# narrow and wide grouped kernels and the two down projections: 64 and 512
# tokens, 4 and 5 or 6 rows an expert, 32 rows, 2400 pairs, inter 512 or not
@pytest.mark.parametrize("shape,counts", [
    ((512, 512, 10, 512), (64, 65, 204, 205, 256, 257, 512, 513)),
    ((512, 64, 8, 512), (256, 257, 512)),
    ((512, 128, 8, 512), (65, 96, 97, 300, 301)),
    ((512, 128, 8, 1024), (65, 96, 97, 300)),
    ((1024, 8, 2, 512), (65, 128, 129, 512, 513)),
])
@pytest.mark.parametrize("bf16,zipf", [(True, 0.0), (False, 1.1)])
def test_kernel_lines(torch_dev, shape, counts, bf16, zipf):
    torch, dev = torch_dev
    pkg = load_pkg()
    H, E, k, I = shape
    rb = orc.zipf_bias(E, zipf, 0.02, 3) if zipf else None
    L = orc.Layer(H, E, k, I, seed=E + I, router_bias=rb)
    most = max(counts)
    x = orc.gen_x(most, H, 41, bf16=bf16)
    xd = to_dev(x, torch, dev)
    with pkg.MoeContext(H, E, k, I, max_tokens=4096) as wide, pkg.MoeContext(H, E, k, I, max_tokens=most) as own:
        for ctx in (wide, own):
            ctx.upload_layer(0, L.arrays())
        for n in counts:
            print(f"case: {shape} n={n} bf16={bf16} zipf={zipf}", flush=True)
            sel = np.unique(np.linspace(0, n - 1, 24).astype(np.int32))
            ref = L.forward(x[:n], bf16, token_sel=sel)
            a = wide.layer_forward(0, xd[:n]).clone()
            b = own.layer_forward(0, xd[:n]).clone()
            torch.cuda.synchronize()
            np.testing.assert_array_equal(own.last_routing(n)["idx"].cpu().numpy(), ref["idx"])
            assert torch.equal(a, b)
            assert_out_close(a.cpu().numpy()[sel], ref["out"], "rows")

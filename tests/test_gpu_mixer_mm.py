"""The mixers' many-token kernels at the edges of their tiles, through the C
ABI against the oracle, with the bars of tests/test_gpu_deltanet.py and
tests/test_gpu_attention.py (outputs 2e-2 max-abs and 1e-3 relative L2,
states and caches 1e-4; the indexer bit for bit)."""
import pytest

import test_gpu_attention as ta
import test_gpu_deltanet as td
import test_gpu_gated_residual as tg

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_dev(gpu):
    import torch
    return torch, gpu


# token counts around the first matrix call, the 32- and 64-row tiles and the
# K-split kernel's last count; hidden 320 and 448 have odd numbers of groups
@pytest.mark.parametrize("shape", [(320, 1, 2, 32, 32, 7), (448, 3, 6, 64, 64, 5), (256, 2, 4, 128, 128, 16)])
@pytest.mark.parametrize("calls", [[5, 6, 31], [32, 33, 1, 64], [65, 1, 129], [320, 1, 321]])
def test_deltanet_token_counts(torch_dev, shape, calls):
    torch, dev = torch_dev
    td.run_steps(torch, dev, shape, calls, seed=8)


@pytest.mark.parametrize("case", [(320, 5, 1, 64, 3, 68, 12, 3, 768, 1.0), (256, 4, 2, 64, 2, 64, 4096, 4, 768, 0.25)])
@pytest.mark.parametrize("calls", [[15, 16, 31], [32, 33, 1, 64], [65, 1, 129], [320, 1, 321]])
def test_attention_token_counts(torch_dev, case, calls):
    torch, dev = torch_dev
    ta.run_calls(torch, dev, case, calls, seed=9)


# hidden sizes past the tiled indexer rows: 17 workgroups of rows with one to
# four tokens each, and 505 workgroups, which take every token
@pytest.mark.parametrize("case", [(2112, 2, 1, 64, 3, 68, 12, 3, 256, 1.0), (2176, 2, 1, 64, 62, 128, 12, 3, 256, 1.0)])
def test_attention_indexer_rows_split(torch_dev, case):
    torch, dev = torch_dev
    ta.run_calls(torch, dev, case, [16, 33, 1, 100], seed=18)


@pytest.mark.parametrize("hd,cap", [(64, 80), (128, 1100), (192, 80), (256, 80)])
def test_attention_head_dims_and_ranges(torch_dev, hd, cap):
    """every head dim of the matrix kernel, 3 query heads per kv head (rows
    of one workgroup from uneven token groups), the last image of a call
    partly filled, several key ranges at 1100 rows"""
    torch, dev = torch_dev
    n = cap - 12
    ta.run_calls(torch, dev, (192, 6, 2, hd, 1, 64, 4096, 4, cap, 0.25), [n, 1, 11], seed=10)
    ta.run_calls(torch, dev, (192, 6, 2, hd, 1, 64, 16, 4, cap, 0.25), [n, 1, 11], seed=11)


@pytest.mark.parametrize("bad", ["nan", "inf", "1e30"])
def test_attention_values_past_the_parts(torch_dev, bad):
    """a token whose value no bf16 parts carry: the tokens before it are
    those of the call without it, and the ones that see it are NaN (nan, inf)
    or the oracle's (1e30: v rows of that size, keys and queries normed)"""
    import numpy as np
    torch, dev = torch_dev
    case = (256, 4, 2, 64, 2, 64, 4096, 4, 64, 0.25)
    n, j = 40, 17
    A = ta.orc.Attention(*case[:8], kv_cap=64, rotary_factor=0.25, seed=12)
    x = ta.orc.gen_attn_x(n, 256, 13)
    outs = []
    for v in (None, float(bad)):
        xi = x.copy()
        if v is not None:
            xi[j, 5] = v
        with ta.load_pkg().AttentionContext(*case[:8], kv_cap=64, rotary_factor=0.25, max_tokens=n) as ctx:
            ctx.upload_layer(0, A.arrays())
            outs.append(ctx.forward(0, torch.from_numpy(xi).to(dev), 0).cpu().numpy())
    clean, got = outs
    assert np.isfinite(clean).all()
    # fp32 sums in another order: 2^-24 per term over 64 dims and 40 keys
    assert ta.rel(got[:j], clean[:j]) < 1e-5
    if bad == "1e30":
        ref = A.forward(xi, A.new_state(), 0)
        for t in range(j, n):
            assert ta.rel(got[t], ref[t]) < ta.REL_L2, t
    else:
        assert np.isnan(got[j:]).all()


# the chunked recurrence: its first count, one token past a chunk, every key
# dim, value dims above its column round, 1 to 16 taps, a call past one
# segment of 2048 tokens
@pytest.mark.parametrize("shape", [(64, 1, 2, 32, 32, 1), (128, 1, 2, 64, 512, 3), (64, 2, 2, 256, 64, 4), (64, 3, 9, 128, 64, 4)])
def test_deltanet_chunks(torch_dev, shape):
    torch, dev = torch_dev
    td.run_steps(torch, dev, shape, [19, 20, 33, 1, 64, 95], seed=14, seed_state=True)


# the first count in chunks of key dim 256 and of wide value dims
@pytest.mark.parametrize("shape,n", [((128, 1, 2, 256, 64, 4), 24), ((128, 1, 1, 32, 512, 4), 32), ((256, 1, 1, 64, 2048, 4), 128)])
def test_deltanet_chunk_lines(torch_dev, shape, n):
    torch, dev = torch_dev
    td.run_steps(torch, dev, shape, [n - 1, n, n + 1], seed=19, seed_state=True)


def test_deltanet_segments(torch_dev):
    torch, dev = torch_dev
    td.run_steps(torch, dev, (64, 1, 2, 64, 64, 4), [2048, 2049, 2100], seed=15)


@pytest.mark.parametrize("bad", ["nan", "inf", "1e30"])
def test_deltanet_values_past_the_products(torch_dev, bad):
    """a token whose values a chunk's products would spread: the tokens before
    it are those of the call without it, and from it on the outputs are NaN
    (nan, inf) or the oracle's (1e30)"""
    import numpy as np
    torch, dev = torch_dev
    shape, n, j = (128, 1, 2, 64, 64, 4), 80, 45
    D = td.orc.DeltaNet(*shape, seed=16)
    x = td.orc.gen_dn_x(n, shape[0], 17)
    outs = []
    for v in (None, float(bad)):
        xi = x.copy()
        if v is not None:
            xi[j, 5] = v
        with td.load_pkg().DeltaNetContext(*shape, max_tokens=n) as ctx:
            ctx.upload_layer(0, D.arrays())
            outs.append(ctx.forward(0, torch.from_numpy(xi).to(dev)).cpu().numpy())
    clean, got = outs
    assert np.isfinite(clean).all()
    # the tokens of j's chunk are stepped one by one: fp32 sums in another order
    assert td.rel(got[:j], clean[:j]) < 1e-5
    if bad == "1e30":
        ref = D.forward(xi, *D.new_state())
        for t in range(j, n):
            assert td.rel(got[t], ref[t]) < td.REL_L2, t
    else:
        assert np.isnan(got[j:]).all()


# the hyper connection's packed planes: the first and last count on them and
# their neighbours, a repeated last token, an odd number of copies and of
# groups, the shapes at the edge of the rule and small ones past it
@pytest.mark.parametrize("hc,d,R", [(4, 256, 128), (3, 192, 64), (8, 64, 64), (1, 2048, 320),
                                    (4, 1024, 256), (3, 1088, 512), (2, 2048, 768), (1, 1024, 64), (5, 1024, 256)])
@pytest.mark.parametrize("n", [256, 257, 1280, 1281])
def test_hyper_token_counts(torch_dev, hc, d, R, n):
    torch, dev = torch_dev
    orc = tg.orc
    hp = orc.Hyper(hc, d, R, seed=21, layer=1, norm_std=0.1)
    hyper = orc.gen_hyper(n, hc, d, seed=n) * 2.0
    with tg.load_pkg().GatedResidualContext(d, hc, R, n_slots=1, max_tokens=1281) as gr:
        gr.upload_slot(0, hp.arrays())
        ht = torch.from_numpy(hyper).to(dev)
        m, i = gr.mix(0, ht)
        m2, _ = gr.mix(0, ht, want_inject=False)
        torch.cuda.synchronize()
        ref = hp.mix(hyper)
        tg.assert_close(m.cpu().numpy(), ref["mixed"], "mixed")
        tg.assert_close(i.cpu().numpy(), ref["inject"], "inject")
        assert torch.equal(m, m2)


# the per-token kernels where x's way through LDS has its edges: one chunk
# pair, a full pass of 2048 columns, one group past one, two and three passes
@pytest.mark.parametrize("d,hv,dk,dv", [(64, 2, 32, 32), (2048, 2, 32, 64), (2112, 33, 64, 64), (4160, 33, 32, 128), (8192, 49, 32, 128)])
def test_deltanet_few_tokens(torch_dev, d, hv, dk, dv):
    torch, dev = torch_dev
    td.run_steps(torch, dev, (d, 1, hv, dk, dv, 4), [1, 5, 2], seed=14)


@pytest.mark.parametrize("d,h,hd", [(64, 1, 64), (2048, 5, 64), (2112, 33, 64), (4160, 12, 64)])
def test_attention_few_tokens(torch_dev, d, h, hd):
    torch, dev = torch_dev
    ta.run_calls(torch, dev, (d, h, 1, hd, 3, 68, 12, 3, 64, 1.0), [1, 15, 2], seed=15)


# hidden sizes on both sides of the line from which chunks are turned in LDS
@pytest.mark.parametrize("hc,d,R", [(8, 64, 64), (1, 2048, 320), (3, 1984, 128), (2, 1088, 64), (4, 1472, 64), (5, 1536, 128)])
@pytest.mark.parametrize("n", [1, 2, 15])
def test_hyper_few_tokens(torch_dev, hc, d, R, n):
    torch, dev = torch_dev
    orc = tg.orc
    hp = orc.Hyper(hc, d, R, seed=22, layer=1, norm_std=0.1)
    hyper = orc.gen_hyper(n, hc, d, seed=n) * 2.0
    with tg.load_pkg().GatedResidualContext(d, hc, R, n_slots=1, max_tokens=n) as gr:
        gr.upload_slot(0, hp.arrays())
        m, i = gr.mix(0, torch.from_numpy(hyper).to(dev))
        torch.cuda.synchronize()
        ref = hp.mix(hyper)
        tg.assert_close(m.cpu().numpy(), ref["mixed"], "mixed")
        tg.assert_close(i.cpu().numpy(), ref["inject"], "inject")

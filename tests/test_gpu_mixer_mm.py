"""The mixers' many-token kernels at the edges of their tiles, through the C
ABI against the oracle, with the bars of tests/test_gpu_deltanet.py and
tests/test_gpu_attention.py (outputs 2e-2 max-abs and 1e-3 relative L2,
states and caches 1e-4; the indexer bit for bit); the precision they keep
against float64, with bars from what a lost bf16 part would cost; and their
large tiles against the small ones."""
import numpy as np
import pytest

import test_gpu_attention as ta
import test_gpu_deltanet as td
import test_gpu_gated_residual as tg

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_dev(gpu):
    import torch
    return torch, gpu


# token counts around the first matrix call and the 32-row tiles of the K-split
# kernel, which every call here takes: the columns are too few for the larger
# tiles at any count; hidden 320 and 448 have odd numbers of groups
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


# ------------------------------------------------------------ large tiles

def one_call_and_many(torch, dev, pkg, shape, n, step):
    """out and states of n tokens in one call and in calls of `step`"""
    D = td.orc.DeltaNet(*shape, seed=30)
    x = torch.from_numpy(td.orc.gen_dn_x(n, shape[0], 31)).to(dev)
    res = []
    with pkg.DeltaNetContext(*shape, n_layers=1, max_tokens=n) as ctx:
        ctx.upload_layer(0, D.arrays())
        for s in (n, step):
            ctx.reset_state(0)
            out = torch.cat([ctx.forward(0, x[t:t + s]).clone() for t in range(0, n, s)])
            torch.cuda.synchronize()
            res.append((out.cpu().numpy(), *td.read_states(ctx, 0)))
    return res


# The 64-row tiles from 321 tokens and the 128-row ones from 1281 on, of qkv | z
# (12288 columns) with the bf16 rows as a launch of their own: ragged last row
# tiles, scales eight at a time (hidden 512) or one (320), an odd number of
# column blocks whose segments share a tile; then of out_proj, at hidden 2048
# the 64-row tiles from 961 tokens on and at 8192 the 128-row ones from 1921.
# Calls of 300 tokens take the K-split kernel.  Both sides stay within 1e-5 of
# float64 (f32 inputs as two bf16 numbers, sums in fp32), so within 2e-5 of each
# other; 4e-5 leaves the factor two that a shape may add.
@pytest.mark.parametrize("shape,counts", [
    ((512, 16, 32, 128, 128, 4), (321, 1281, 1409)), ((320, 16, 32, 128, 128, 4), (321, 1281)),
    ((512, 1, 64, 32, 128, 4), (330, 1409)), ((2048, 1, 16, 32, 32, 4), (961, 1025)),
    ((2048, 1, 2, 32, 32, 4), (1025,)), ((8192, 1, 16, 32, 32, 4), (1921, 2000))])
def test_deltanet_large_tiles(torch_dev, shape, counts):
    torch, dev = torch_dev
    for n in counts:
        one, many = one_call_and_many(torch, dev, td.load_pkg(), shape, n, 300)
        for what, a, b in zip(("out", "conv state", "recurrent state"), one, many):
            e = td.rel(a, b)
            td.say(f"{shape} n={n} {what}: one call against calls of 300 rel-L2 {e:.1e}")
            assert np.isfinite(a).all() and e < 4e-5, (n, what, e)


@pytest.mark.parametrize("kind,d,n", [("dn", 2048, 6), ("dn", 2048, 33), ("dn", 2048, 321), ("dn", 2048, 1025), ("dn", 8192, 1921),
                                      ("attn", 2048, 16), ("attn", 2048, 33), ("attn", 2048, 1025), ("attn", 8192, 1921)])
def test_inject_many_tokens(torch_dev, kind, d, n):
    """the residual's update fused into the output projection, in the K-split
    kernel and in both large tiles: the mixer's bits, each hyper row updated
    once (one fma: half an ulp, and half an ulp of the float64 sum), also with
    no out"""
    torch, dev = torch_dev
    pkg, hc = td.load_pkg(), 3
    g = torch.Generator().manual_seed(n)
    x, h0, inj = (torch.randn(s, generator=g).to(dev) for s in ((n, d), (n, hc * d), (n, hc)))
    if kind == "dn":
        ctx = pkg.DeltaNetContext(d, 1, 16, 32, 32, 4, n_layers=1, max_tokens=n)
        ctx.upload_layer(0, td.orc.DeltaNet(d, 1, 16, 32, 32, 4, seed=32).arrays())
        reset, args = (lambda: ctx.reset_state(0)), (0, x)
    else:
        shape = (d, 8, 1, 64, 1, 64, 4096, 4)
        ctx = pkg.AttentionContext(*shape, kv_cap=n, rotary_factor=0.25, n_layers=1, max_tokens=n)
        ctx.upload_layer(0, ta.orc.Attention(*shape, kv_cap=n, rotary_factor=0.25, seed=32).arrays())
        reset, args = (lambda: ctx.reset(0)), (0, x, 0)
    with ctx:
        reset()
        out = ctx.forward(*args).clone()
        h1, out1 = h0.clone(), torch.empty_like(out)
        reset()
        ctx.forward_inject(*args, h1, inj, out=out1)
        h2 = h0.clone()
        reset()
        ctx.forward_inject(*args, h2, inj)
        torch.cuda.synchronize()
    assert torch.equal(out, out1) and torch.equal(h1, h2)
    ref = h0.view(n, hc, d).double() + inj.double().unsqueeze(-1) * out.double().unsqueeze(1)
    err = (h1.view(n, hc, d).double() - ref).abs()
    assert bool((err <= 2.0 ** -24 * 1.01 * ref.abs() + 1e-38).all()), float((err / ref.abs()).max())


# ------------------------------------------------------------ precision

def bf16(a):
    """round to nearest even, as float64"""
    u = np.asarray(a, np.float32).view(np.uint32)
    return ((u + 0x7FFF + ((u >> 16) & 1)) & 0xFFFF0000).view(np.float32).astype(np.float64)


def bits16(a):
    return (np.asarray(a, np.float32).view(np.uint32) >> 16).astype(np.uint16)


def q4_rows(rng, rows, K):
    """codes, scales, biases of rows around a zero point inside the code range,
    and the float64 matrix"""
    q = rng.integers(0, 16, (rows, K))
    s = bf16(rng.uniform(0.8, 1.2, (rows, K // 64)) / (4.61 * np.sqrt(K)))
    b = bf16(s * rng.normal(-7.5, 0.2, s.shape))
    words = (q.reshape(rows, K // 8, 8).astype(np.uint32) << (4 * np.arange(8, dtype=np.uint32))).sum(-1, dtype=np.uint32)
    return words.ravel(), bits16(s).ravel(), bits16(b).ravel(), q * np.repeat(s, 64, 1) + np.repeat(b, 64, 1), b


@pytest.mark.parametrize("n", [6, 40, 321, 1281])
def test_projection_precision(torch_dev, n):
    """qkv rows of x of mean 1, where the bias term cancels most of the code
    term: the group sums need three bf16 parts (24 bits).  The conv state holds
    the projection's last 15 rows.  Two parts would err by err2, ten times what
    the split of x (2^-17) and the fp32 sums give; the bar is 0.4 of it."""
    torch, dev = torch_dev
    shape = (512, 16, 32, 128, 128, 16)
    rng = np.random.default_rng(n)
    arr = dict(td.orc.DeltaNet(*shape, seed=33).arrays())
    q, s, b, W, bias = q4_rows(rng, 8192, 512)
    arr.update(qkv_q=q, qkv_s=s, qkv_b=b)
    x = (1.0 + 0.05 * rng.standard_normal((n, 512))).astype(np.float32)
    with td.load_pkg().DeltaNetContext(*shape, n_layers=1, max_tokens=n) as ctx:
        ctx.upload_layer(0, arr)
        ctx.forward(0, torch.from_numpy(x).to(dev))
        torch.cuda.synchronize()
        conv, _ = td.read_states(ctx, 0)
    m = min(n, 15)
    xl = x[n - m:].astype(np.float64)
    ref = xl @ W.T
    X = xl.reshape(m, 8, 64).sum(-1)
    hi = bf16(X)
    err2 = np.linalg.norm((X - hi - bf16(X - hi)) @ bias.T) / np.linalg.norm(ref)
    e = td.rel(conv[15 - m:], ref)
    td.say(f"projection n={n}: rel-L2 against float64 {e:.2e}, two parts {err2:.2e}")
    assert e < 0.4 * err2, (e, err2)


@pytest.mark.parametrize("n", [16, 100])
def test_attention_precision(torch_dev, n):
    """scores of one large dim, a thousand and more in size and nearly tied, so
    an error in q or k counts in full: three bf16 parts each.  k takes the first
    32 columns of x, which hardly differ between tokens, v the others.  The
    query rows are the key rows, so q is the cached k; the gate is 1 and o_proj
    the identity, so the output is the softmax over the caches.  Two parts of q
    and k would err by err2 (2^-18 of the scores), the fp32 scores by 2^-24 of
    them; the bar is a quarter of err2."""
    torch, dev = torch_dev
    rng = np.random.default_rng(n)
    shape = (64, 1, 1, 64, 1, 64, 4096, 4)
    A = ta.orc.Attention(*shape, kv_cap=n, rotary_factor=0.01, seed=34)
    arr = dict(A.arrays())
    kc, vc = rng.integers(0, 16, (2, 64, 64))
    kc[:, 32:] = 0
    vc[:, :32] = 0
    kq, vq = (np.sum(c.reshape(64, 8, 8).astype(np.uint32) << (4 * np.arange(8, dtype=np.uint32)), -1, dtype=np.uint32).ravel() for c in (kc, vc))
    one = bits16(np.full(64, 1.0, np.float32))
    zero = np.zeros(64, np.uint16)
    eye = np.zeros((64, 8), np.uint32)
    eye[np.arange(64), np.arange(64) // 8] = 1 << (4 * (np.arange(64, dtype=np.uint32) % 8))
    w = np.full(64, 2.0 ** -6, np.float32)
    w[0] = 128.0
    # gate rows: codes 0, bias 1 per column, so 32 + the sum of the others > 17
    arr.update(q_q=np.concatenate([kq, np.zeros(512, np.uint32)]), q_s=np.concatenate([one, zero]), q_b=np.concatenate([zero, one]),
               k_q=kq, k_s=one, k_b=zero, v_q=vq, v_s=one, v_b=zero, o_q=eye.ravel(), o_s=one, o_b=zero, q_norm=w, k_norm=w)
    x = np.concatenate([1.0 + 0.001 * rng.standard_normal((n, 32)), 0.25 * rng.standard_normal((n, 32))], 1).astype(np.float32)
    with ta.load_pkg().AttentionContext(*shape, kv_cap=n, rotary_factor=0.01, max_tokens=n) as ctx:
        ctx.upload_layer(0, arr)
        out = ctx.forward(0, torch.from_numpy(x).to(dev), 0)
        torch.cuda.synchronize()
        kp, vp, _, ln = ctx.cache(0)
        k, v = ta.d2h(kp, (ln, 64)).astype(np.float64), ta.d2h(vp, (ln, 64)).astype(np.float64)

    def soft(a):
        s = a @ a.T / 8.0
        s = np.where(np.tril(np.ones((n, n), bool)), s, -np.inf)
        p = np.exp(s - s.max(1, keepdims=True))
        return p / p.sum(1, keepdims=True) @ v

    ref = soft(k)
    k2 = bf16(k) + bf16(k - bf16(k))
    err2 = ta.rel(soft(k2), ref)
    e = ta.rel(out.cpu().numpy(), ref)
    ta.say(f"attention n={n}: |score| up to {np.abs(k @ k.T).max() / 8:.0f}, rel-L2 {e:.2e}, two parts {err2:.2e}")
    assert e < 0.25 * err2, (e, err2)


# ------------------------------------------------------------ few tokens, long caches

# calls of 15 tokens in a context for 15: once the cache is past one to three
# 64-key chunks their partials no longer fit the scratch and the 256-key kernel
# runs, without and with the block mask, over one and several chunks and head
# groups
@pytest.mark.parametrize("case", [(256, 2, 1, 64, 2, 64, 4096, 4, 128, 0.25), (64, 9, 1, 64, 1, 64, 16, 4, 600, 0.25),
                                  (128, 4, 2, 256, 2, 64, 32, 4, 320, 0.25)])
def test_attention_256_key_chunks(torch_dev, case):
    torch, dev = torch_dev
    cap = case[8]
    ta.run_calls(torch, dev, case, [15] * (cap // 15 - 1) + [9, 1], seed=35)


# 512 workgroups of 256 keys: 8 tokens, 32 kv heads, two chunks
def test_attention_256_key_grid(torch_dev):
    torch, dev = torch_dev
    ta.run_calls(torch, dev, (64, 32, 32, 64, 1, 64, 4096, 4, 540, 0.25), [500, 8, 15], seed=36)

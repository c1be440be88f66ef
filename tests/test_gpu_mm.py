"""Products of several tokens (sfa_mul_mat_vec, sfa_qkv_rope_kv_append and
sfa_moe_ffn with three or more rows) against float64 and against the one-token
calls, at the edges of their tiles: token counts around 16, 32, 64, 128 and
192, output counts that end inside a tile, one k block and many, operands that
the rule leaves to the one-token kernels.

Tolerances: a sum of n products in f32, in chains of at most 8 roundings whose
results are summed twice more, is within a few 2^-24 of the row's RMS times
sqrt(chain length): 1e-6 of the RMS bounds 16 such roundings.  With F16
weights an expert's activation is rounded to f16 before the down product; a
last-ulp difference moves single roundings by 2^-11 of that activation, so
2e-4 of the largest output there."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _rand(gen, *shape, dtype=torch.float32, std=1.0):
    return (torch.randn(shape, generator=gen, device="cuda") * std).to(dtype)


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _operand(x, w):
    return x.half().double() if w.dtype == torch.float16 else x.double()


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("n_rows,n_in,n_out", [
    (3, 128, 68), (15, 256, 100), (16, 4096, 80), (17, 384, 260), (32, 512, 4096), (33, 128, 68), (65, 256, 1000),
    (128, 2048, 2052), (129, 256, 8192), (257, 4096, 4100), (300, 384, 16384), (9, 128, 8196), (70, 640, 16388), (260, 384, 8196),
    (5, 136, 100), (5, 128, 64), (5, 128, 70), (2, 128, 100)])  # the last four: left to the one-token kernel
def test_products(gpu, dtype, n_rows, n_in, n_out):
    from strataflow_amd import layer
    g = _gen(n_rows * 31 + n_in + n_out)
    w = _rand(g, n_out, n_in, dtype=dtype, std=n_in ** -0.5)
    x, r = _rand(g, n_rows, n_in), _rand(g, n_rows, n_out)
    y = layer.mul_mat_vec(w, x)
    ref = _operand(x, w) @ w.double().t()
    rms = ref.square().mean().sqrt()
    assert float((y.double() - ref).abs().max() / rms) < 3e-6
    assert float((y.double() - ref).norm() / ref.norm()) < 2e-7
    ones = torch.cat([layer.mul_mat_vec(w, x[t:t + 1].contiguous()) for t in (0, n_rows - 1)])
    assert float((y[[0, n_rows - 1]] - ones).abs().max() / rms) < 3e-6
    # the residual after the product, in place; outputs at any float address
    buf = torch.zeros(n_rows * n_out + 1, device="cuda")
    yr = buf[1:].view(n_rows, n_out)
    yr.copy_(r)
    layer.mul_mat_vec(w, x, residual=yr, out=yr)
    assert torch.equal(yr, y + r)
    # a one-hot activation picks a weight column exactly
    cols = torch.randint(0, n_in, (n_rows,), generator=g, device="cuda")
    oh = torch.zeros_like(x)
    oh[torch.arange(n_rows, device="cuda"), cols] = 1.0
    assert torch.equal(layer.mul_mat_vec(w, oh), w[:, cols].t().float())
    # a token whose row is not finite leaves the others alone
    xi = x.clone()
    xi[n_rows // 2] = float("inf")
    keep = [t for t in range(n_rows) if t != n_rows // 2]
    assert torch.equal(layer.mul_mat_vec(w, xi)[keep], y[keep])


@pytest.mark.parametrize("wdtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("kv_type", ["f16", "f32"])
@pytest.mark.parametrize("n_tok,shape", [(2, (8, 4, 32, 256)), (3, (8, 4, 32, 256)), (16, (4, 2, 64, 384)), (40, (16, 4, 128, 512)),
                                         (130, (8, 4, 32, 256)), (300, (32, 8, 128, 1024)),
                                         # few outputs: the one-token kernels, and just past them
                                         (4, (8, 4, 64, 2048)), (4, (16, 4, 128, 2048)), (7, (8, 4, 64, 1024)), (5, (16, 4, 128, 1024)),
                                         (16, (4, 1, 128, 4096)), (32, (4, 2, 64, 2048)), (40, (4, 2, 64, 2048)), (50, (8, 4, 32, 512)), (3, (16, 8, 64, 512)),
                                         # 6144 outputs: F16 tiles of 64 x 32, 64 x 64 and 128 x 128
                                         (64, (32, 8, 128, 256)), (128, (32, 8, 128, 256)), (512, (32, 8, 128, 384))])
def test_qkv_equals_product_then_append(gpu, wdtype, kv_type, n_tok, shape):
    """Bit for bit, with skipped tokens and a page that is not there."""
    from strataflow_amd import layer, synth
    from strataflow_amd.paged_kv import SFA_KV_F16, SFA_KV_F32, PagedKV
    hq, hkv, hd, n_embd = shape
    g = _gen(n_tok + n_embd)
    w = _rand(g, (hq + 2 * hkv) * hd, n_embd, dtype=wdtype, std=n_embd ** -0.5)
    x = _rand(g, n_tok, n_embd)
    page, past = 64, 37
    n_pages = -(-(past + n_tok) // page) + 2
    pt = torch.from_numpy(synth.page_tables(np.random.default_rng(n_tok), [past + n_tok], page, n_pages)).cuda()
    pt[0, -1] = n_pages + 3
    seq = torch.zeros(n_tok, dtype=torch.int32, device="cuda")
    pos = torch.arange(past, past + n_tok, dtype=torch.int32, device="cuda")
    seq[1] = -1
    kt = {"f16": SFA_KV_F16, "f32": SFA_KV_F32}[kv_type]
    a, b = (PagedKV(1, hq, hkv, hd, kt, page, n_pages) for _ in range(2))
    qa = a.qkv_rope_append(0, w, x, seq, pos, pt, 1e6)
    y = layer.mul_mat_vec(w, x)
    q, k, v = (t.contiguous() for t in y.split([hq * hd, hkv * hd, hkv * hd], 1))
    qb = q.view(n_tok, hq, hd)
    b.rope_append(0, qb, k.view(n_tok, hkv, hd), v.view(n_tok, hkv, hd), seq, pos, pt, 1e6)
    assert torch.equal(qa, qb) and torch.equal(a.k, b.k) and torch.equal(a.v, b.v)


@pytest.mark.parametrize("n_rows,n_embd,n_ff,n_expert,k", [
    (3, 128, 384, 4, 2), (13, 256, 1024, 8, 2), (25, 256, 640, 8, 2), (70, 128, 384, 4, 3), (110, 256, 1024, 5, 2), (200, 256, 1024, 5, 2),
    (400, 128, 512, 2, 2), (150, 128, 512, 4, 2), (300, 384, 1152, 3, 2),
    (6, 256, 384, 8, 2), (9, 128, 384, 300, 2), (2, 128, 384, 4, 2),  # no room for the rows; too many experts; two tokens
    (3, 1024, 4096, 4, 2), (13, 512, 2048, 8, 2), (24, 256, 1024, 16, 4), (60, 256, 768, 2, 1), (26, 1024, 2304, 16, 1)])  # grouped, 16 pairs a tile
def test_experts(gpu, n_rows, n_embd, n_ff, n_expert, k):
    """Against float64 and against the tokens one at a time, within 2e-4 of the
    largest output; ids outside the stack add nothing, one expert may hold every
    pair, and the result written over the residual has the same bits."""
    from strataflow_amd import layer
    g = _gen(n_rows + n_embd + n_ff)
    h = torch.float16
    gate = _rand(g, n_expert, n_ff, n_embd, dtype=h, std=n_embd ** -0.5)
    up = _rand(g, n_expert, n_ff, n_embd, dtype=h, std=n_embd ** -0.5)
    down = _rand(g, n_expert, n_embd, n_ff, dtype=h, std=n_ff ** -0.5)
    x, res = _rand(g, n_rows, n_embd), _rand(g, n_rows, n_embd)
    wts = torch.rand((n_rows, k), generator=g, device="cuda") + 0.1
    spread = torch.rand((n_rows, n_expert), generator=g, device="cuda").argsort(-1)[:, :k].int().contiguous()
    out_of = spread.clone()
    out_of[::3, 0] = n_expert + 7
    out_of[1::3, k - 1] = -1
    one = torch.full_like(spread, n_expert - 1)
    for ids in (spread, out_of, one, torch.full_like(spread, -1)):
        ws = torch.full((n_rows * k * n_ff * 4,), 0xff, dtype=torch.uint8, device="cuda")  # NaNs
        y = layer.moe_ffn(x, res, ids, wts, gate, up, down, workspace=ws)
        ref = torch.zeros((n_rows, n_embd), dtype=torch.float64, device="cuda")
        for e in range(n_expert):
            t, j = torch.nonzero(ids == e, as_tuple=True)
            if t.numel():
                xe = x[t].half().double()
                gv, uv = xe @ gate[e].double().t(), xe @ up[e].double().t()
                act = (gv / (1 + torch.exp(-gv)) * uv).float().half().double()
                ref.index_add_(0, t, (act @ down[e].double().t()) * wts[t, j].double()[:, None])
        ref += res.double()
        tol = 2e-4 * max(1.0, float(ref.abs().max()))
        assert float((y.double() - ref).abs().max()) < tol
        rows = [0, n_rows // 2, n_rows - 1]
        single = torch.cat([layer.moe_ffn(x[t:t + 1], res[t:t + 1], ids[t:t + 1], wts[t:t + 1].contiguous(),
                                          gate, up, down) for t in rows])
        assert float((y[rows] - single).abs().max()) < tol
        inplace = res.clone()
        layer.moe_ffn(x, inplace, ids, wts, gate, up, down, out=inplace, workspace=ws)
        assert torch.equal(inplace, y)


@pytest.mark.parametrize("n_in", [128, 256, 384, 512, 768, 1024, 1152])
@pytest.mark.parametrize("n_rows", [3, 17, 40, 300])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_error_is_the_one_token_kernels(gpu, dtype, n_rows, n_in):
    """No further from 64 bits than the one-token call, short rows above all,
    whose one-token sums are chains of eight products in a tree.  The root mean
    squares are over 16384 values or more each: 0.6 % of noise, 3 % allowed."""
    from strataflow_amd import layer
    g = _gen(n_rows + n_in)
    n_out = 4096
    w = _rand(g, n_out, n_in, dtype=dtype, std=n_in ** -0.5)
    x = _rand(g, max(n_rows, 8), n_in)

    def err(y, rows):
        return float((y.double() - _operand(rows, w) @ w.double().t()).square().mean().sqrt())

    several = torch.cat([layer.mul_mat_vec(w, x[i:i + n_rows]) for i in ((0, 3, 5) if n_rows == 3 else (0,))])
    rows = torch.cat([x[i:i + n_rows] for i in ((0, 3, 5) if n_rows == 3 else (0,))])
    ones = torch.cat([layer.mul_mat_vec(w, x[t:t + 1]) for t in range(8)])
    assert err(several, rows) < 1.03 * err(ones, x[:8])


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("n_rows,n_in,n_out", [
    (3, 256, 1024), (3, 8192, 2048), (4, 2048, 2048), (4, 512, 512), (7, 256, 512), (7, 1024, 1024), (5, 14336, 768),
    (8, 2048, 1024), (16, 2048, 1024), (17, 2048, 384), (64, 4096, 128), (128, 4096, 128), (40, 2048, 404)])
def test_few_outputs_stay_with_the_one_token_kernel(gpu, dtype, n_rows, n_in, n_out):
    """A matrix of few outputs, where that kernel is the faster one: the bits of
    the one-token calls."""
    from strataflow_amd import layer
    g = _gen(n_rows + n_in + n_out)
    w = _rand(g, n_out, n_in, dtype=dtype, std=n_in ** -0.5)
    x = _rand(g, n_rows, n_in)
    y = layer.mul_mat_vec(w, x)
    assert torch.equal(y, torch.cat([layer.mul_mat_vec(w, x[t:t + 1]) for t in range(n_rows)]))


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("n_rows,n_in,n_out", [
    (4, 256, 1028), (5, 512, 1024), (8, 1024, 1024), (17, 2048, 1024), (129, 4096, 128), (33, 1024, 1024), (48, 512, 640),
    (64, 1024, 2048), (100, 128, 400), (31, 2048, 2052), (3, 512, 1028), (3, 4096, 2052), (16, 4096, 1028)])
def test_past_few_outputs(gpu, dtype, n_rows, n_in, n_out):
    """The other side of that rule, and the tiles of 16 tokens that F32 weights
    take there, against float64."""
    from strataflow_amd import layer
    g = _gen(n_rows + n_in + n_out)
    w = _rand(g, n_out, n_in, dtype=dtype, std=n_in ** -0.5)
    x, r = _rand(g, n_rows, n_in), _rand(g, n_rows, n_out)
    y = layer.mul_mat_vec(w, x)
    ref = _operand(x, w) @ w.double().t()
    assert float((y.double() - ref).abs().max() / ref.square().mean().sqrt()) < 3e-6
    assert float((y.double() - ref).norm() / ref.norm()) < 2e-7
    assert torch.equal(layer.mul_mat_vec(w, x, residual=r), y + r)


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_rows_past_two_gibibytes(gpu, dtype):
    """Activations of more than 2 GiB: the kernels' 32-bit offsets are unsigned.
    (x lies 2 GiB into its buffer, so an offset taken as signed would read other
    values of it, which the comparison shows.)"""
    from strataflow_amd import layer
    n_rows, n_in, n_out = 133000, 4096, 132
    g = _gen(7)
    w = _rand(g, n_out, n_in, dtype=dtype, std=n_in ** -0.5)
    buf = torch.randn((1 << 29) + n_rows * n_in, generator=g, device="cuda")
    x = buf[1 << 29:].view(n_rows, n_in)
    y = layer.mul_mat_vec(w, x)
    rows = torch.tensor([0, 1, 65535, 65536, 131071, 131072, 131073, 132000, n_rows - 1], device="cuda")
    ref = _operand(x[rows], w) @ w.double().t()
    assert float((y[rows].double() - ref).abs().max() / ref.square().mean().sqrt()) < 3e-6
    some = layer.mul_mat_vec(w, x[-300:].contiguous())
    assert float((y[-300:] - some).abs().max()) < 1e-5


@pytest.mark.parametrize("n_rows", [1, 2, 3, 16, 17, 32, 33, 130])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_infinite_products(gpu, dtype, n_rows):
    """One infinite product in a row's first, a middle or its last k block makes
    that row's result infinite with the weight's sign, whatever is added before
    and after it, and leaves the other rows' bits alone: an infinite activation,
    one beyond f16's range beside F16 weights, an f32 product and an f32 sum that
    overflow."""
    from strataflow_amd import layer
    n_in, n_out = 4096, 2052  # past the one-token kernels' few outputs
    g = _gen(n_rows)
    w = _rand(g, n_out, n_in, dtype=dtype, std=n_in ** -0.5)
    x = _rand(g, n_rows, n_in)
    y, t = layer.mul_mat_vec(w, x), n_rows // 2
    keep = [r for r in range(n_rows) if r != t]
    assert torch.isfinite(y).all()
    for col in (5, 300, 2050, n_in - 1):
        wi = w.clone()
        wi[:, col] = torch.where(wi[:, col] < 0, -2.0, 2.0).to(dtype)
        base = layer.mul_mat_vec(wi, x)
        for value in [float("inf"), -float("inf"), 70000.0 if dtype == torch.float16 else 3e38]:
            xi = x.clone()
            xi[t, col] = value
            got = layer.mul_mat_vec(wi, xi)
            assert torch.equal(got[t], torch.sign(wi[:, col].float()) * np.sign(value) * float("inf")), (col, value)
            assert torch.equal(got[keep], base[keep])
    if dtype == torch.float32:  # terms of one sign whose sum passes f32's range, block after block
        wi, xi = torch.ones_like(w), x.clone()
        xi[t] = 1e35
        got = layer.mul_mat_vec(wi, xi)
        assert torch.equal(got[t], torch.full_like(got[t], float("inf")))
        assert torch.equal(got[keep], layer.mul_mat_vec(wi, x)[keep])


@pytest.mark.parametrize("n_rows", [1, 2, 3, 13, 40, 150, 200])
def test_infinite_expert_activations(gpu, n_rows):
    """An activation beyond f16's range, in the first, a middle and the last k
    block of the down product, in tokens routed to that expert: infinite with
    the sign of the down weight, the other tokens' bits alone."""
    from strataflow_amd import layer
    n_embd, n_ff, n_expert, k = 1024, 2560, 4, 2
    g = _gen(n_rows)
    h = torch.float16
    gate, up = (_rand(g, n_expert, n_ff, n_embd, dtype=h, std=n_embd ** -0.5) for _ in range(2))
    down = _rand(g, n_expert, n_embd, n_ff, dtype=h, std=n_ff ** -0.5)
    x, res = _rand(g, n_rows, n_embd), _rand(g, n_rows, n_embd)
    x[:, 0] = 1.0
    wts = torch.full((n_rows, k), 0.5, device="cuda")
    ids = torch.rand((n_rows, n_expert), generator=g, device="cuda").argsort(-1)[:, :k].int().contiguous()
    ids[0] = torch.tensor([2, 0], device="cuda")
    y = layer.moe_ffn(x, res, ids, wts, gate, up, down)
    assert torch.isfinite(y).all()
    hit = (ids == 2).any(1)
    for col in (3, 1100, n_ff - 1):
        gi, ui = gate.clone(), up.clone()
        gi[2, col] = 0
        ui[2, col] = 0
        gi[2, col, 0] = ui[2, col, 0] = 400.0  # silu(400) * 400 = 160000
        got = layer.moe_ffn(x, res, ids, wts, gi, ui, down)
        want = (torch.sign(down[2, :, col].float()) * float("inf")).expand(int(hit.sum()), -1)
        ok = down[2, :, col] != 0
        assert torch.equal(got[hit][:, ok], want[:, ok]), col
        assert torch.equal(got[~hit], y[~hit])


@pytest.mark.parametrize("n_rows,n_embd,n_ff,n_expert,k", [
    (3, 256, 1024, 8, 2), (13, 256, 1024, 8, 2), (8, 128, 512, 128, 4), (6, 1024, 3072, 8, 1), (3, 512, 2048, 16, 2),
    (4, 2048, 4224, 16, 2)])
def test_experts_that_seldom_share_stay_ungrouped(gpu, n_rows, n_embd, n_ff, n_expert, k):
    """Where grouping would cost more than the weights it reads once less: the
    bits of the tokens one at a time."""
    from strataflow_amd import layer
    g = _gen(n_rows + n_ff)
    h = torch.float16
    gate, up = (_rand(g, n_expert, n_ff, n_embd, dtype=h, std=n_embd ** -0.5) for _ in range(2))
    down = _rand(g, n_expert, n_embd, n_ff, dtype=h, std=n_ff ** -0.5)
    x, res = _rand(g, n_rows, n_embd), _rand(g, n_rows, n_embd)
    wts = torch.rand((n_rows, k), generator=g, device="cuda")
    ids = torch.rand((n_rows, n_expert), generator=g, device="cuda").argsort(-1)[:, :k].int().contiguous()
    y = layer.moe_ffn(x, res, ids, wts, gate, up, down)
    rows = [layer.moe_ffn(x[t:t + 1], res[t:t + 1], ids[t:t + 1], wts[t:t + 1], gate, up, down) for t in range(n_rows)]
    assert torch.equal(y, torch.cat(rows))


def test_several_tokens_in_a_graph(gpu):
    """The calls replay from a captured graph with the bits of eager calls."""
    from strataflow_amd import layer
    g = _gen(5)
    n, n_embd, n_ff, n_expert, k = 40, 256, 1024, 8, 2
    h = torch.float16
    wo = _rand(g, n_embd, n_embd, dtype=h, std=0.06)
    router = _rand(g, n_expert, n_embd, dtype=h, std=0.06)
    gate, up = (_rand(g, n_expert, n_ff, n_embd, dtype=h, std=0.06) for _ in range(2))
    down = _rand(g, n_expert, n_embd, n_ff, dtype=h, std=0.03)
    norm = torch.ones(n_embd, device="cuda")
    x = _rand(g, n, n_embd)
    mid, cur, y = (torch.empty_like(x) for _ in range(3))
    ids = torch.empty((n, k), dtype=torch.int32, device="cuda")
    wts = torch.empty((n, k), device="cuda")
    ws = torch.empty(n * k * n_ff * 4, dtype=torch.uint8, device="cuda")

    def step():
        layer.mul_mat_vec(wo, x, residual=x, out=mid)
        layer.moe_norm_gate(mid, norm, 1e-5, router, k, out=cur, ids=ids, weights=wts)
        layer.moe_ffn(cur, mid, ids, wts, gate, up, down, out=y, workspace=ws)

    step()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step()
    for _ in range(3):
        x.copy_(_rand(g, n, n_embd))
        y.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        got = y.clone()
        step()
        torch.cuda.synchronize()
        assert torch.equal(got, y)

"""The forms of sfa_attn_prefill (the split of a short chunk's history over
waves, two groups of waves, one) against each other: a chunk whose size takes
one form, and the same rows in chunks of 32 tokens, which take the split where they
span 512 positions or more; F16 and F32 caches against float64 too.

Tolerance: the forms cut the positions differently, so a running maximum, and
with it the rounding of a probability to f16 (2^-11), differs: 2^-11 of a
probability each way, averaged over the attended positions, is under 1e-3 of
the row.  F32 caches keep f32 throughout: the sums' order alone, 2e-6."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

# (heads, kv heads, head_dim), cached positions, tokens, page, first attended position
FORMS = [
    ((32, 32, 64), 600, 513, 64, 0),      # two groups (160 workgroups of 128 rows), g = 1, pages of one tile
    ((64, 16, 128), 1000, 300, 64, 130),  # two groups, a window that starts inside a tile
    ((64, 16, 128), 1003, 300, 128, 0),   # two groups, an odd number of tiles
    ((64, 8, 64), 991, 305, 256, 0),      # two groups, g = 8
    ((64, 16, 128), 40, 300, 256, 0),     # a short span: one group for F16
    ((64, 16, 128), 513, 600, 64, 70),    # one group (more workgroups than CUs)
    ((16, 4, 128), 2000, 577, 256, 0),    # the split, three waves' tiles short of a round
    ((8, 8, 64), 600, 100, 64, 500),      # a window of few tiles: one group
    ((8, 8, 64), 700, 100, 64, 280),      # the split, two tiles a wave
    ((32, 8, 128), 0, 1024, 256, 0),      # two groups, nothing for the second one to attend in the first block
    ((32, 8, 128), 0, 777, 64, 0),        # the same for Q8_0 (one group for F16)
    ((16, 4, 128), 4500, 100, 64, 0),     # the split over more pages than the page-id window holds
    ((8, 8, 64), 4700, 64, 64, 300),      # the same, from a window's start
    ((32, 8, 128), 4200, 700, 64, 0),     # two groups over more pages than that
    ((16, 4, 128), 100, 1600, 64, 500),   # two groups, a window that hides everything from the first blocks
    ((8, 2, 128), 100, 1600, 256, 500),   # the split, the same
]


@pytest.mark.parametrize("kv_type", ["f16", "q8_0", "f32"])
@pytest.mark.parametrize("form", FORMS, ids=lambda f: f"h{f[0][0]}kv{f[0][1]}d{f[0][2]}n{f[1]}t{f[2]}p{f[3]}lo{f[4]}")
def test_forms_agree(gpu, kv_type, form):
    from strataflow_amd import synth
    from strataflow_amd.paged_kv import SFA_KV_F16, SFA_KV_F32, SFA_KV_Q8_0, PagedKV
    (hq, hkv, hd), past, n_tok, page, lo = form
    n = past + n_tok
    n_pages = -(-n // page) + 2
    g = torch.Generator(device="cuda")
    g.manual_seed(n + hq)
    kv = PagedKV(1, hq, hkv, hd, {"f16": SFA_KV_F16, "q8_0": SFA_KV_Q8_0, "f32": SFA_KV_F32}[kv_type], page, n_pages)
    pt = torch.from_numpy(synth.page_tables(np.random.default_rng(n), [n], page, n_pages)).cuda()
    k = torch.randn((n, hkv, hd), generator=g, device="cuda")
    k[torch.arange(n, device="cuda") % 61 == 17] *= 5  # maxima that move late in a wave's tiles
    v = torch.randn((n, hkv, hd), generator=g, device="cuda")
    kv.append(0, k, v, torch.zeros(n, dtype=torch.int32, device="cuda"),
              torch.arange(n, dtype=torch.int32, device="cuda"), pt)
    if past > 4 * page:
        pt[0, 2] = -1  # a page that is not there adds nothing
    q = torch.randn((n_tok, hq, hd), generator=g, device="cuda")
    whole = kv.prefill(0, q, pt[0], past, kv_lo=lo)
    assert torch.isfinite(whole).all()
    parts = torch.cat([kv.prefill(0, q[t:t + 32].contiguous(), pt[0], past + t, kv_lo=lo) for t in range(0, n_tok, 32)])
    tol = 2e-6 if kv_type == "f32" else 1e-3
    rel = float((whole.double() - parts.double()).norm() / parts.double().norm())
    assert rel < tol and float((whole - parts).abs().max()) < 20 * tol, rel
    if kv_type == "q8_0":
        return  # the forms quantise Q alike; test_q8_two_groups_vs_oracle and the sweep compare them with the oracle, which does too
    pos = torch.arange(n, device="cuda")
    hidden = (pos[None] > past + torch.arange(n_tok, device="cuda")[:, None]) | (pos[None] < lo)
    if past > 4 * page:
        hidden |= (pos[None] >= 2 * page) & (pos[None] < 3 * page)
    for h in (0, hq // 2 + 1, hq - 1):
        c = (lambda t: t.half().double()) if kv_type == "f16" else (lambda t: t.double())
        kh, vh = c(k[:, h // (hq // hkv)]).contiguous(), c(v[:, h // (hq // hkv)]).contiguous()
        s = (q[:, h].double() @ kh.t()) / hd ** 0.5
        ref = torch.softmax(s.masked_fill(hidden, -float("inf")), -1) @ vh
        ref[hidden.all(1)] = 0.0  # nothing attended
        got = whole.view(n_tok, hq, hd)[:, h].double()
        assert float((got - ref).norm() / ref.norm()) < tol, h


@pytest.mark.parametrize("past,n_tok,page", [(0, 777, 64), (700, 600, 256), (4300, 530, 64)])
def test_q8_two_groups_vs_oracle(gpu, oracle_mod, past, n_tok, page):
    """The Q8_0 kernel with two groups of waves (more than half the CUs), which
    the sweep's sizes do not take."""
    from tests.helpers import assert_close
    from tests.test_gpu_prefill import build, run
    host, dev, pt, q, n_kv = build(oracle_mod, gpu, Hq=32, Hkv=8, hd=128, n_cached=past, T=n_tok, page_size=page,
                                   seed=past + n_tok, kv_type=8)
    out = run(dev, gpu, pt, q, past)
    ref = host.attention(q[None], 32, pt, np.array([n_kv], np.int32), np.array([0], np.int32), T=n_tok,
                         mode=oracle_mod.GGML)[0].reshape(n_tok, -1)
    assert_close(out, ref, what=f"past {past} T {n_tok} page {page}")


@pytest.mark.parametrize("kv_type", ["f32", "q8_0"])
@pytest.mark.parametrize("shape,past,n_tok,lo", [
    ((8, 2, 128), 700, 40, 161), ((8, 8, 64), 700, 100, 95), ((16, 2, 128), 300, 33, 31), ((8, 8, 64), 40, 20, 33),
    ((32, 8, 128), 2000, 64, 1987)])
def test_rows_before_the_window_do_not_reach_the_result(gpu, kv_type, shape, past, n_tok, lo):
    """K and V rows before a window that starts inside a tile may hold anything:
    the bits are those of the call with zeros there.  (The F32 kernel clears such
    V rows in LDS, for other lanes of the wave to read.)"""
    from strataflow_amd import synth
    from strataflow_amd.paged_kv import SFA_KV_F32, SFA_KV_Q8_0, PagedKV
    hq, hkv, hd = shape
    n, page = past + n_tok, 64
    n_pages = -(-n // page) + 2
    g = torch.Generator(device="cuda")
    g.manual_seed(n + lo)
    pt = torch.from_numpy(synth.page_tables(np.random.default_rng(n), [n], page, n_pages)).cuda()
    k, v = (torch.randn((n, hkv, hd), generator=g, device="cuda") for _ in range(2))
    q = torch.randn((n_tok, hq, hd), generator=g, device="cuda")
    seq, pos = torch.zeros(n, dtype=torch.int32, device="cuda"), torch.arange(n, dtype=torch.int32, device="cuda")
    outs = []
    for fill in (0.0, 3e4, float("nan")):
        if kv_type == "q8_0" and fill != fill:
            continue  # a block's quants have no NaN
        kv = PagedKV(1, hq, hkv, hd, {"f32": SFA_KV_F32, "q8_0": SFA_KV_Q8_0}[kv_type], page, n_pages)
        k[:lo], v[:lo] = fill, fill
        kv.append(0, k, v, seq, pos, pt)
        outs.append(kv.prefill(0, q, pt[0], past, kv_lo=lo))
    assert torch.isfinite(outs[0]).all()
    for o in outs[1:]:
        assert torch.equal(o, outs[0])

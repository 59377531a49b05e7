"""Decode-attention and sampler kernels vs the PyTorch references (fp32)."""
import math
import os
import subprocess
import sys

import pytest
import torch

from llm_in_practise_amd.ops.decode import decode_attention_reference, sample_reference

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("hq,hkv,d", [(32, 8, 128), (8, 8, 64), (40, 8, 128), (16, 2, 64)])
@pytest.mark.parametrize("lens", [[1, 300, 4096, 129], [77]])
def test_decode_attention_kernel(native_ext, hq, hkv, d, lens):
    torch.manual_seed(0)
    B, Smax = len(lens), 4096
    kc = torch.randn(B, Smax, hkv * d, device=DEV).to(torch.bfloat16)
    vc = torch.randn(B, Smax, hkv * d, device=DEV).to(torch.bfloat16)
    q = torch.randn(B, hq * d, device=DEV).to(torch.bfloat16)
    L = torch.tensor(lens, device=DEV, dtype=torch.int32)
    o = native_ext.decode_attention(q, kc, vc, L, hq, hkv, d, max(lens), 1 / math.sqrt(d))
    r = decode_attention_reference(q.float(), kc.float(), vc.float(), L, hq, hkv, d)
    assert (o.float() - r).abs().max().item() < 2e-2


def test_sampler_greedy_and_topk1(native_ext):
    torch.manual_seed(0)
    x = torch.randn(8, 151936, device=DEV)
    g = x.argmax(-1)
    assert torch.equal(native_ext.sample(x, None, 0.0, 0, 1.0, 1.0, 1), g)
    assert torch.equal(native_ext.sample(x, None, 0.7, 1, 1.0, 1.0, 2), g)
    assert torch.equal(native_ext.sample(x.to(torch.bfloat16), None, 0.0, 0, 1.0, 1.0, 3),
                       x.to(torch.bfloat16).float().argmax(-1))
    assert torch.equal(native_ext.sample(x, None, 1.0, 0, 1e-6, 1.0, 4), g)


def test_sampler_penalty_matches_reference(native_ext):
    torch.manual_seed(1)
    x = torch.randn(4, 1000, device=DEV)
    hist = torch.randint(0, 1000, (4, 64), device=DEV, dtype=torch.int32)
    hist[:, 50:] = -1
    hist[:, 10] = hist[:, 11]           # duplicates
    want = sample_reference(x, hist, 0.0, penalty=1.3)
    assert torch.equal(native_ext.sample(x, hist, 0.0, 0, 1.0, 1.3, 5), want)


def test_sampler_distribution_top_p(native_ext):
    # probabilities 0.5/0.3/0.15/0.05; top_p 0.7 keeps {0,1} renormalised to 0.625/0.375
    p = torch.tensor([0.5, 0.3, 0.15, 0.05], device=DEV)
    x = torch.log(p)[None].repeat(20000, 1).contiguous()
    s = native_ext.sample(x, None, 1.0, 0, 0.7, 1.0, 12345)
    counts = torch.bincount(s, minlength=4).float() / s.numel()
    assert counts[2] == 0 and counts[3] == 0
    assert abs(counts[0].item() - 0.625) < 0.02
    s2 = native_ext.sample(x, None, 1.0, 3, 1.0, 1.0, 777)   # top-k 3
    c2 = torch.bincount(s2, minlength=4).float() / s2.numel()
    assert c2[3] == 0 and abs(c2[0].item() - 0.5 / 0.95) < 0.02


def test_generate_qwen3_gpu_kv_cache_matches_recompute(native_ext):
    from llm_in_practise_amd.infer.generate import generate
    from llm_in_practise_amd.models.qwen3 import Qwen3ForCausalLM, qwen3_config
    m = Qwen3ForCausalLM.from_config(qwen3_config("qwen3-small"), dtype=torch.bfloat16, device=DEV, seed=0).eval()
    p = torch.randint(0, 4096, (1, 33), device=DEV)
    out = generate(m, p, max_new_tokens=8)
    ids = p.clone()
    with torch.no_grad():
        for _ in range(8):
            ids = torch.cat([ids, m(ids).logits[:, -1].float().argmax(-1, keepdim=True)], 1)
    # bf16 rounding can flip near-ties late in the sequence; the first tokens must agree
    assert torch.equal(out[0, :37], ids[0, :37])


@pytest.mark.parametrize("B,max_len", [(64, 4096), (1, 1024), (7, 3000)])
def test_decode_attention_split_plans(native_ext, B, max_len):
    """Batch sizes that select different split plans (1 split per head up to 64-key chunks)."""
    torch.manual_seed(B)
    hq, hkv, d, Smax = 32, 8, 128, 4096
    kc = torch.randn(B, Smax, hkv * d, device=DEV).to(torch.bfloat16)
    vc = torch.randn(B, Smax, hkv * d, device=DEV).to(torch.bfloat16)
    q = torch.randn(B, hq * d, device=DEV).to(torch.bfloat16)
    L = torch.randint(1, max_len + 1, (B,), device=DEV, dtype=torch.int32)
    L[0] = max_len
    o = native_ext.decode_attention(q, kc, vc, L, hq, hkv, d, max_len, 1 / math.sqrt(d))
    r = decode_attention_reference(q.float(), kc.float(), vc.float(), L, hq, hkv, d)
    assert (o.float() - r).abs().max().item() < 2e-2


@pytest.mark.parametrize("hq,hkv,d", [(32, 8, 128), (8, 8, 64), (40, 8, 128), (16, 1, 64), (64, 4, 128)])
@pytest.mark.parametrize("pos", [[0, 299, 4095, 128], [76], [31, 32, 33, 1000, 1023, 1024, 5, 64]])
def test_decode_attention_append_kernel(native_ext, hq, hkv, d, pos):
    """MFMA decode kernel with the fused KV append: q/k/v are row-strided views of one fused
    qkv projection output; the new rows must land in the caches at pos and take part in the
    attention; no other cache row may change."""
    torch.manual_seed(len(pos) + hq)
    B, Smax = len(pos), 4096
    kc = torch.randn(B, Smax, hkv * d, device=DEV).to(torch.bfloat16)
    vc = torch.randn(B, Smax, hkv * d, device=DEV).to(torch.bfloat16)
    qkv = torch.randn(B, (hq + 2 * hkv) * d, device=DEV).to(torch.bfloat16)
    q, k, v = qkv[:, :hq * d], qkv[:, hq * d:(hq + hkv) * d], qkv[:, (hq + hkv) * d:]
    P = torch.tensor(pos, device=DEV, dtype=torch.long)
    kc0, vc0 = kc.clone(), vc.clone()
    o = native_ext.decode_attention_append(q, k, v, kc, vc, P, hq, hkv, d, max(pos) + 1, 1 / math.sqrt(d))
    rows = torch.arange(B, device=DEV)
    kc0[rows, P] = k
    vc0[rows, P] = v
    assert torch.equal(kc, kc0) and torch.equal(vc, vc0)
    r = decode_attention_reference(q.float(), kc0.float(), vc0.float(), (P + 1).int(), hq, hkv, d)
    assert (o.float() - r).abs().max().item() < 2e-2


@pytest.mark.parametrize("B,max_len", [(256, 1024), (64, 4096), (1, 1024), (7, 3000)])
def test_decode_attention_append_split_plans(native_ext, B, max_len):
    torch.manual_seed(B)
    hq, hkv, d = 32, 8, 128
    kc = torch.randn(B, max_len, hkv * d, device=DEV).to(torch.bfloat16)
    vc = torch.randn(B, max_len, hkv * d, device=DEV).to(torch.bfloat16)
    q = torch.randn(B, hq * d, device=DEV).to(torch.bfloat16)
    k = torch.randn(B, hkv * d, device=DEV).to(torch.bfloat16)
    v = torch.randn(B, hkv * d, device=DEV).to(torch.bfloat16)
    P = torch.randint(0, max_len, (B,), device=DEV)
    P[0] = max_len - 1
    o = native_ext.decode_attention_append(q, k, v, kc, vc, P, hq, hkv, d, max_len, 1 / math.sqrt(d))
    r = decode_attention_reference(q.float(), kc.float(), vc.float(), (P + 1).int(), hq, hkv, d)
    assert (o.float() - r).abs().max().item() < 2e-2


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("max_len", [33, 500, 900, 4097, 9000])
def test_decode_attention_append_merge(native_ext, max_len, d):
    """The merge of fewer splits than it takes in one go, as many, and more, of which few, all or all but one have keys."""
    torch.manual_seed(max_len)
    P = torch.tensor([0, max_len // 3, max_len - 1, 32], device=DEV)
    B, hq, hkv = len(P), 3, 1
    kc, vc = (torch.randn(B, max_len, hkv * d, device=DEV).to(torch.bfloat16) for _ in range(2))
    q, k, v = (torch.randn(B, n * d, device=DEV).to(torch.bfloat16) for n in (hq, hkv, hkv))
    o = native_ext.decode_attention_append(q, k, v, kc, vc, P, hq, hkv, d, max_len, 1 / math.sqrt(d))
    r = decode_attention_reference(q.float(), kc.float(), vc.float(), (P + 1).int(), hq, hkv, d)
    # weights and values in bf16: 2^-8 of the largest value for each, and the output's own rounding
    assert (o.float() - r).abs().max().item() < 3 * 2.0 ** -8 * vc.float().abs().max().item()


@pytest.mark.parametrize("hkv,d", [(1, 128), (3, 64), (8, 128)])
@pytest.mark.parametrize("B", [2, 20, 63, 64, 65, 130])
def test_decode_attention_append_counts_the_splits_that_have_keys(native_ext, B, hkv, d):
    """Rows whose keys end at, behind and in front of tiles and of the splits of one, two and more tiles that a workgroup takes four, two and one of, in
    batches on both sides of 64 rows and of 64 rows x heads; a row's bits are the same among other neighbours."""
    torch.manual_seed(B + hkv)
    hq, max_len = 2 * hkv, 700
    ends = [0, 62, 63, 64, 126, 127, 128, 254, 255, 256, 699, 511, 512]
    P = torch.tensor([ends[(i * 5) % len(ends)] for i in range(B)], device=DEV)
    kc, vc = (torch.randn(B, max_len, hkv * d, device=DEV).to(torch.bfloat16) for _ in range(2))
    q, k, v = (torch.randn(B, n * d, device=DEV).to(torch.bfloat16) for n in (hq, hkv, hkv))
    o = native_ext.decode_attention_append(q, k, v, kc, vc, P, hq, hkv, d, max_len, 1 / math.sqrt(d))
    rows = torch.arange(B, device=DEV)
    assert torch.equal(kc[rows, P], k) and torch.equal(vc[rows, P], v)
    r = decode_attention_reference(q.float(), kc.float(), vc.float(), (P + 1).int(), hq, hkv, d)
    # weights and values in bf16: 2^-8 of the largest value for each, and the output's own rounding
    assert (o.float() - r).abs().max().item() < 3 * 2.0 ** -8 * vc.float().abs().max().item()
    keep = B // 2
    other = torch.full_like(P, 300)
    other[keep] = P[keep]
    again = native_ext.decode_attention_append(q, k, v, kc, vc, other, hq, hkv, d, max_len, 1 / math.sqrt(d))
    assert torch.equal(again[keep], o[keep])


@pytest.mark.parametrize("B,hkv,d", [(8, 8, 128), (11, 8, 128), (16, 4, 64), (22, 3, 128), (66, 1, 64)])
@pytest.mark.parametrize("max_len", [128, 500, 700, 1000])
def test_decode_attention_append_bits_of_counted_splits(native_ext, B, hkv, d, max_len):
    """From 64 rows x heads on a workgroup takes several short splits: the bits are those of a workgroup a split, which fewer rows with as many
    splits (one of every 128 keys on either side) have."""
    torch.manual_seed(B + max_len)
    hq = 4 * hkv
    ends = [0, 5, 31, 32, 33, 62, 63, 64, 95, 126, 127, 128, 191, 255, 256, 257, 383, 499, 511, 512, 699, 767, 999]
    ends = [e for e in ends if e < max_len]
    P = torch.tensor([ends[(i * 7) % len(ends)] for i in range(B - 1)] + [max_len - 1], device=DEV)
    kc, vc = (torch.randn(B, max_len, hkv * d, device=DEV).to(torch.bfloat16) for _ in range(2))
    q, k, v = (torch.randn(B, n * d, device=DEV).to(torch.bfloat16) for n in (hq, hkv, hkv))
    K2, V2 = kc.clone(), vc.clone()
    got = native_ext.decode_attention_append(q, k, v, kc, vc, P, hq, hkv, d, max_len, d ** -0.5)
    n = 63 // hkv                                           # rows of a call below 64 rows x heads
    assert B * hkv >= 64 > n * hkv
    want = torch.cat([native_ext.decode_attention_append(*(t[i:i + n] for t in (q, k, v)), K2[i:i + n], V2[i:i + n], P[i:i + n], hq, hkv, d, max_len,
                                                         d ** -0.5) for i in range(0, B, n)])
    assert torch.equal(got, want) and torch.equal(kc, K2) and torch.equal(vc, V2)


@pytest.mark.parametrize("M", [1, 5, 16, 33, 64])
@pytest.mark.parametrize("N,K", [(6144, 4096), (4096, 12288), (272, 192)])
def test_gemm_skinny_matches_fp32(native_ext, M, N, K):
    """Decode-shaped split-K GEMM (+ residual) vs fp32, incl. N not a multiple of the 128-row block."""
    torch.manual_seed(M)
    w = (torch.randn(N, K, device=DEV) * 0.02).to(torch.bfloat16)
    xb = torch.randn(M, K + 64, device=DEV).to(torch.bfloat16)
    x = xb[:, :K]                                   # row-strided input
    res = torch.randn(M, N, device=DEV).to(torch.bfloat16)
    ref = x.float() @ w.float().t()
    y = native_ext.gemm_skinny(x, w, None)
    assert ((y.float() - ref).abs().max() / ref.abs().max()).item() < 1e-2
    y = native_ext.gemm_skinny(x, w, res)
    want = ref + res.float()
    assert ((y.float() - want).abs().max() / want.abs().max()).item() < 1e-2


@pytest.mark.parametrize("d", [64, 128])
def test_decode_attention_append_rounds_products_before_sums(native_ext, d):
    """The sums over a workgroup's tiles of keys round each product before it is added: a tile whose weighted value is the exact
    negative of the rounded product of the other cancels it to 0 (a fused multiply-add would leave the rounding error)."""
    scale, n = 0.3, 64                                   # two tiles of 32 keys in one split (the cache is too short for more)
    k, v = torch.zeros(1, 2 * n, d), torch.zeros(1, 2 * n, d)
    k[0, 32:n, 0] = -1.0                                 # scores 0 in the first tile, -scale in the second: weights 1 and c
    q = torch.zeros(1, d, device=DEV)
    q[0, 0] = 1.0
    c = torch.exp2(torch.tensor([-1.0], device=DEV) * torch.tensor([scale * 1.4426950408889634], device=DEV)).cpu()
    g = torch.Generator().manual_seed(d)

    def parts(x):                                        # a float as the sum of three bf16
        out = []
        for _ in range(3):
            out.append(x.bfloat16().float())
            x = x - out[-1]
        return torch.stack(out)
    b = parts(torch.rand(d, generator=g) + 0.5)
    product = b.sum(0) * c                               # one float rounding
    assert (product.double() != b.double().sum(0) * c.double()).any()
    v[0, 32:35], v[0, :3] = b, -parts(product)
    kc, vc = k.bfloat16().to(DEV), v.bfloat16().to(DEV)
    o = native_ext.decode_attention_append(q.bfloat16(), kc[:, n - 1].contiguous(), vc[:, n - 1].contiguous(), kc, vc,
                                           torch.tensor([n - 1], device=DEV), 1, 1, d, n, scale)
    assert not o.any()


@pytest.mark.parametrize("M", [1, 3, 16, 17, 40])
@pytest.mark.parametrize("N,K", [(6144, 2560), (4096, 4096), (48, 64), (1040, 576), (6160, 1984), (80, 20480)])
def test_gemm_skinny_pieces(native_ext, M, N, K):
    """The cuts of K (pieces of whole and of partial batches, more pieces than the LDS form takes) and the gated end against 64
    bits: sums of K products in float lie within (K + 1) half-ulps of the absolute sum, then one rounding to bf16."""
    torch.manual_seed(N + M)
    x, w = torch.randn(M, K, device=DEV).to(torch.bfloat16), (torch.randn(N, K, device=DEV) * 0.02).to(torch.bfloat16)
    res = torch.randn(M, N, device=DEV).to(torch.bfloat16)
    exact = x.double() @ w.double().t()
    slack = (K + 1) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())
    for r in (None, res):
        want = exact if r is None else exact + r.double()
        got = native_ext.gemm_skinny(x, w, r).double()
        assert ((got - want).abs() <= 2 * slack + 2.0 ** -8 * want.abs()).all()
    if N % 32 == 0:                                 # both products rounded to bf16, the activation, and rounded again
        F = N // 2
        g, u = exact[:, :F], exact[:, F:]
        eg, eu = 2.0 ** -8 * g.abs() + 2 * slack[:, :F], 2.0 ** -8 * u.abs() + 2 * slack[:, F:]
        want = g * torch.sigmoid(g) * u             # |d silu| <= 1.1
        bound = 1.1 * eg * (u.abs() + eu) + (g * torch.sigmoid(g)).abs() * eu + 2.0 ** -7 * want.abs() + 1e-6
        assert ((native_ext.gemm_skinny_swiglu(x, w).double() - want).abs() <= bound).all()


@pytest.mark.parametrize("M", [1, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("N,K", [(16, 8320), (1040, 8704), (2064, 4608), (3088, 512), (4096, 12288), (2560, 1024)])
def test_narrow_rows(native_ext, M, N, K):
    """The products of few rows and a narrow weight, in four parts of units in turns (whole rounds and not; one to four column tiles a
    workgroup, with and without a remainder; fewer stages than the ring holds and more) and by the rule that picks them, against 64 bits
    (sums of K products in float lie within (K + 1) half-ulps of the absolute sum, then one rounding to bf16), rows of x far apart too.  What
    they do not take stays with the library: a residual whose rows stand apart, or off 16 bytes, and an x off 16 bytes."""
    from llm_in_practise_amd.ops import gemm
    torch.manual_seed(N + M)
    far, w = torch.randn(M, K + 40, device=DEV).to(torch.bfloat16), (torch.randn(N, K, device=DEV) * 0.02).to(torch.bfloat16)
    x, res = far[:, :K].contiguous(), torch.randn(M, N, device=DEV).to(torch.bfloat16)
    exact = x.double() @ w.double().t()
    slack = 2 * (K + 1) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())
    forms = [] if M <= 16 or K % 512 else [lambda a, r, u=u: native_ext.rows_parts(a, w, r, u) for u in (64, 128)]
    if M <= 16:
        forms.append(lambda a, r: native_ext.gemm_skinny(a, w, r))
    forms.append(lambda a, r: gemm._base_gemm(a, w, residual=r))
    for r in (None, res):
        want = exact if r is None else exact + r.double()
        for form in forms:
            got = form(x, r)
            assert ((got.double() - want).abs() <= slack + 2.0 ** -8 * want.abs()).all()
            assert torch.equal(form(far[:, :K], r), got)
    wide, off = torch.randn(M, N + 8, device=DEV).to(torch.bfloat16)[:, :N], torch.randn(M * N + 4, device=DEV).to(torch.bfloat16)[4:].view(M, N)
    xo = torch.zeros(M * K + 4, dtype=torch.bfloat16, device=DEV)[4:].view(M, K).copy_(x)
    for a, r in ((x, wide), (x, off), (xo, None)):
        if M > 16:
            assert gemm._narrow_rows(a, w, r) == 0
            want = exact if r is None else exact + r.double()
            assert ((gemm._base_gemm(a, w, residual=r).double() - want).abs() <= slack + 2.0 ** -8 * want.abs()).all()


@pytest.mark.parametrize("N,K,form", [(4096, 12288, (128, 64)), (1024, 8704, (128, 64)), (4096, 4096, (1, 64)), (2048, 8192, (1, 64)), (1024, 3072, (1, 1)),
                                      (1024, 8320, (0, 0))])
def test_narrow_rows_rule_has_no_row_count_of_its_own(native_ext, N, K, form):
    """One form from 17 to 32 rows and one from 33 to 64, whatever their number (a server's largest batch is any number)."""
    from llm_in_practise_amd.ops import gemm
    w, x = torch.zeros(N, K, dtype=torch.bfloat16, device=DEV), torch.zeros(64, K, dtype=torch.bfloat16, device=DEV)
    assert [gemm._narrow_rows(x[:m], w, None) for m in range(17, 65)] == [form[0]] * 16 + [form[1]] * 32


@pytest.mark.parametrize("M", [33, 40, 48, 63, 64])
@pytest.mark.parametrize("N,K", [(4096, 4096), (2560, 9728), (1024, 4608)])
def test_narrow_rows_round_as_well_as_the_library(native_ext, M, N, K):
    """Results that are not the exact one rounded to bf16: no more than from the library's product, but for the chance of their number (three
    standard deviations of a count)."""
    from llm_in_practise_amd.ops import gemm
    torch.manual_seed(N + M)
    x, r = torch.randn(M, K, device=DEV).to(torch.bfloat16), torch.randn(M, N, device=DEV).to(torch.bfloat16)
    w = (torch.randn(N, K, device=DEV) * 0.02).to(torch.bfloat16)
    right = (x.double() @ w.double().t() + r.double()).to(torch.bfloat16)
    here, there = ((y != right).sum().item() for y in (gemm._base_gemm(x, w, residual=r), torch.addmm(r, x, w.t())))
    assert gemm._narrow_rows(x, w, r) == 64 and here <= there + 3 * (here + there + 1) ** 0.5


@pytest.mark.parametrize("N,K", [(4096, 12288), (1024, 8320)])
def test_no_rows_and_a_deep_narrow_weight(native_ext, N, K):
    """A product of no rows is an empty one, as the library has it."""
    from llm_in_practise_amd.ops import gemm
    x, w = torch.empty(0, K, dtype=torch.bfloat16, device=DEV), torch.zeros(N, K, dtype=torch.bfloat16, device=DEV)
    for r in (None, torch.empty(0, N, dtype=torch.bfloat16, device=DEV)):
        assert gemm._base_gemm(x, w, residual=r).shape == (0, N)


@pytest.mark.parametrize("M", [17, 32, 33, 49, 64])
@pytest.mark.parametrize("F,K", [(16, 128), (80, 640), (4112, 384), (8208, 256), (12320, 256), (14336, 128)])
def test_rows_swiglu(native_ext, M, F, K):
    """The gated product of more rows, one to four column tiles a workgroup with and without a remainder, fewer stages than the ring holds
    and more: against 64 bits (each sum of K products in float within (K + 1) half-ulps of the absolute sum, rounded to bf16, then the
    activation, rounded again; |d silu| <= 1.1), for rows of x side by side and far apart, and a saturated gate."""
    torch.manual_seed(F + M)
    far = torch.randn(M, K + 24, device=DEV).to(torch.bfloat16)
    far[M - 1] = 100.0 * far[M - 1].sign()
    w = (torch.randn(2 * F, K, device=DEV) * 0.02).to(torch.bfloat16)
    w[3] = -1.0 * far[M - 1, :K].sign()                        # gate -100 K: its silu is 0
    x = far[:, :K].contiguous()
    exact = x.double() @ w.double().t()
    slack = 2 * (K + 1) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())
    g, u = exact[:, :F], exact[:, F:]
    eg, eu = 2.0 ** -8 * g.abs() + slack[:, :F], 2.0 ** -8 * u.abs() + slack[:, F:]
    want = g * torch.sigmoid(g) * u
    bound = 1.1 * eg * (u.abs() + eu) + (g * torch.sigmoid(g)).abs() * eu + 2.0 ** -7 * want.abs() + 1e-6
    got = native_ext.rows_swiglu(x, w)
    assert ((got.double() - want).abs() <= bound).all() and got[M - 1, 3] == 0
    assert torch.equal(native_ext.rows_swiglu(far[:, :K], w), got)
    big = x.clone()
    big[:, 5] = float("inf")                                   # infinities and what becomes of them, as from the separate kernels
    h = native_ext.swiglu_fwd(big @ w.t())
    assert torch.equal(torch.isnan(native_ext.rows_swiglu(big, w)), torch.isnan(h))


@pytest.mark.parametrize("M", [1, 16, 33])
@pytest.mark.parametrize("N,K", [(48, 64), (80, 576), (2560, 1216), (96, 4096)])
def test_gemm_skinny_weight_off_lines(native_ext, M, N, K):
    """A weight that starts 16 bytes into a line of memory, its pieces in whole units and ending in half of one: every bit as from
    the weight at a line's start, and nothing of its neighbours."""
    torch.manual_seed(N + M)
    x = torch.randn(M, K, device=DEV).to(torch.bfloat16)
    w = (torch.randn(N, K, device=DEV) * 0.02).to(torch.bfloat16)
    far = torch.full((N * K + 16,), float("nan"), dtype=torch.bfloat16, device=DEV)
    off = far[8:8 + N * K].view(N, K).copy_(w)
    assert w.data_ptr() % 128 == 0 and off.data_ptr() % 128 == 16
    assert torch.equal(native_ext.gemm_skinny(x, off, None), native_ext.gemm_skinny(x, w, None))
    if N % 32 == 0:
        assert torch.equal(native_ext.gemm_skinny_swiglu(x, off), native_ext.gemm_skinny_swiglu(x, w))


@pytest.mark.parametrize("N,K", [(512, 8192), (64, 576), (2048, 1984), (6176, 4096), (96, 64)])
def test_gemm_skinny_rows_do_not_depend_on_their_number(native_ext, N, K):
    """Pieces of 4 units to 32, of half a unit more, of one wave alone: a row's bits are those it has beside 15 others."""
    torch.manual_seed(N)
    xb, w = torch.randn(16, K + 8, device=DEV).to(torch.bfloat16), (torch.randn(N, K, device=DEV) * 0.02).to(torch.bfloat16)
    x, res = xb[:, :K], torch.randn(16, N, device=DEV).to(torch.bfloat16)
    y, h = native_ext.gemm_skinny(x, w, res), native_ext.gemm_skinny_swiglu(x, w)
    assert (y.double() - (x.double() @ w.double().t() + res.double())).norm() <= 2.0 ** -8 * y.double().norm()
    for m in (1, 9):
        assert torch.equal(native_ext.gemm_skinny(x[:m], w, res[:m]), y[:m])
        assert torch.equal(native_ext.gemm_skinny_swiglu(x[:m], w), h[:m])


@pytest.mark.parametrize("M,ld", [(9, 1 << 28), (16, 143165800), (4, 1 << 30), (40, 55063688)])
def test_gemm_skinny_rows_far_apart(native_ext, M, ld):
    """Rows that a 32-bit offset in bytes does not reach: the bits of rows side by side, with a norm and without."""
    torch.manual_seed(M)
    N, K = 64, 512
    near, w = torch.randn(M, K, device=DEV).bfloat16(), (torch.randn(2 * N, K, device=DEV) * K ** -0.5).bfloat16()
    nw = torch.randn(K, device=DEV).bfloat16()
    x = torch.empty((M - 1) * ld + K, dtype=torch.bfloat16, device=DEV).as_strided((M, K), (ld, 1)).copy_(near)
    norms = [(None, 0.0)] + [(nw, 1e-6)] * (M <= 4)
    for norm, eps in norms:
        assert torch.equal(native_ext.gemm_skinny(x, w[:N], None, norm, eps), native_ext.gemm_skinny(near, w[:N], None, norm, eps))
        assert torch.equal(native_ext.gemm_skinny_swiglu(x, w, norm, eps), native_ext.gemm_skinny_swiglu(near, w, norm, eps))


@pytest.mark.parametrize("M", [1, 2, 3, 4])
@pytest.mark.parametrize("N,K", [(16, 512), (6144, 1024), (128, 4096), (4096, 4096), (8192, 1536), (4608, 3584), (9728, 2560), (2560, 2048)])
def test_product_of_rows_in_front_of_their_norm(native_ext, M, N, K):
    """One wave or two a row, W's tiles to 4 and 8 waves in all their cuts: the bits of the norm's own kernel and the product; a row that
    holds an infinity or NaN is NaN and changes no other; rows a stride apart; nothing that does not fit; replays of a captured call."""
    from llm_in_practise_amd.ops.norm import rms_norm
    torch.manual_seed(N + M)
    xb, nw = (3 * torch.randn(M, K + 8, device=DEV)).bfloat16(), torch.randn(K, device=DEV).bfloat16()
    w, x = (torch.randn(2 * N, K, device=DEV) * K ** -0.5).bfloat16(), xb[:, :K]
    forms = [(lambda x: native_ext.gemm_skinny(x, w[:N], None, nw, 1e-6), lambda x: native_ext.gemm_skinny(x, w[:N], None), False),
             (lambda x: native_ext.gemm_skinny_swiglu(x, w, nw, 1e-6), lambda x: native_ext.gemm_skinny_swiglu(x, w), True)]
    for one, product, glu in forms:
        if not native_ext.skinny_norms(M, K, glu):
            with pytest.raises(RuntimeError):
                one(x)
            continue
        assert torch.equal(one(x), product(rms_norm(x.contiguous(), nw, 1e-6)))
        for bad in (float("inf"), float("nan")):
            y = x.clone()
            y[M - 1, K - 1] = bad
            got = one(y)
            assert got[M - 1].isnan().all() and torch.equal(got[:M - 1], one(x)[:M - 1])
        y = x.clone()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            out = one(y)
        for seed in range(3):
            y.copy_(torch.randn(M, K, device=DEV))
            g.replay()
            assert torch.equal(out, product(rms_norm(y, nw, 1e-6)))
    assert not native_ext.skinny_norms(5, K, False) and not native_ext.skinny_norms(1, K + 64, False)


@pytest.mark.parametrize("rows", [1, 3, 4, 5])
def test_decode_layers_norm_their_rows_in_the_products(native_ext, monkeypatch, rows):
    """The same logits as with the norm's own kernel, fused products and separate ones, adapters, a gradient."""
    from llm_in_practise_amd.models import qwen3
    m = qwen3.Qwen3ForCausalLM.from_config(qwen3.qwen3_config("qwen3-small"), dtype=torch.bfloat16, device=DEV, seed=0).eval()
    m.requires_grad_(False)
    ids = torch.randint(0, 4096, (1, rows), device=DEV)
    calls = []
    real = qwen3.normed_rows

    def counted(*a):
        y = real(*a)
        calls.append(y is not None)
        return y
    monkeypatch.setattr(qwen3, "normed_rows", counted)
    for fused in (False, True):
        if fused:
            for layer in m.model.layers:
                layer.self_attn.fuse()
                layer.mlp.fuse()
        calls.clear()
        with torch.no_grad():
            got = m(ids).logits
        assert any(calls) == (fused and rows <= 4)
        with monkeypatch.context() as c, torch.no_grad():
            c.setattr(qwen3.Qwen3Attention, "normed_few_rows", lambda *a: None)
            c.setattr(qwen3.Qwen3MLP, "normed_few_rows", lambda *a: None)
            assert torch.equal(m(ids).logits, got)
    seen = []
    for sub in (m.model.layers[1].self_attn, m.model.layers[1].mlp):    # a hook sees normed rows, whatever their number
        handle = sub.register_forward_pre_hook(lambda mod, args: seen.append(args[0]))
        with torch.no_grad():
            assert torch.equal(m(ids).logits, got)
        handle.remove()
        rms = seen[-1].float().pow(2).mean(-1).sqrt()
        assert (rms - 1).abs().max() < 0.1             # (the norms' weights are ones)
    x = torch.randn(rows, m.config.hidden_size, device=DEV).bfloat16().requires_grad_()
    layer = m.model.layers[0]
    assert layer.self_attn.normed_few_rows(x, layer.input_layernorm) is None        # (the norm's gradient)
    assert layer.mlp.normed_few_rows(x, layer.post_attention_layernorm) is None


@pytest.mark.parametrize("M", [17, 33, 64])
@pytest.mark.parametrize("N,K", [(512, 4096), (1024, 4608), (1536, 512), (2560, 9728), (3584, 4096), (4096, 12288)])
def test_parts_and_the_norm_behind_them(native_ext, M, N, K):
    """The launch that adds up a product's parts and norms the rows: the bits of the sum's launch and the norm's own kernel (one wave or two a
    row), bf16 parts and slices of 4-bit weights (one to many, odd numbers of them); a row that holds an infinity changes no other; a replay."""
    from llm_in_practise_amd.ops.norm import rms_norm
    from llm_in_practise_amd.quant.int4 import int4_linear, int4_normed, quantize_rtn
    torch.manual_seed(N + M)
    x, res, nw = torch.randn(M, K, device=DEV).bfloat16(), torch.randn(M, N, device=DEV).bfloat16(), torch.randn(N, device=DEV).bfloat16()
    w = (torch.randn(N, K, device=DEV) * K ** -0.5).bfloat16()
    forms = [(lambda x, u=u: native_ext.rows_parts_norm(x, w, res, u, nw, 1e-6), lambda x, u=u: native_ext.rows_parts(x, w, res, u)) for u in (64, 128)]
    w4 = quantize_rtn(w, 128)
    forms.append((lambda x: int4_normed(x, w4, res, nw, 1e-6), lambda x: int4_linear(x, w4, None, res)))
    for form, product in forms:
        got = form(x)
        if got is None:                                 # (one launch holds all of K)
            assert M <= 32
            continue
        want = product(x)
        assert torch.equal(got[0], want) and torch.equal(got[1], rms_norm(want, nw, 1e-6))
        y = x.clone()
        y[M - 1, 5] = float("inf")
        bad = form(y)
        assert torch.equal(bad[1][:M - 1], got[1][:M - 1]) and not torch.isfinite(bad[1][M - 1].float()).all()
        y = x.clone()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            out = form(y)
        for _ in range(3):
            y.copy_(torch.randn(M, K, device=DEV))
            g.replay()
            want = product(y)
            assert torch.equal(out[0], want) and torch.equal(out[1], rms_norm(want, nw, 1e-6))
    assert not native_ext.parts_norm_serves(N + 16) and not native_ext.parts_norm_serves(8704)


@pytest.mark.parametrize("M,N,K,served", [(8, 1536, 12288, True), (8, 1024, 17408, False), (17, 4096, 12288, True), (17, 4096, 13824, False),
                                          (8, 5120, 9728, False), (17, 5120, 5120, True), (17, 8192, 5120, False), (40, 8192, 5120, True)])
def test_slices_are_summed_beside_the_norm_only_where_it_is_not_slower(native_ext, M, N, K, served):
    """Sizes on both sides of what one CU brings of a row's slices in the time of two launches, and of the longest chain."""
    from llm_in_practise_amd.ops.norm import rms_norm
    from llm_in_practise_amd.quant.int4 import int4_linear, int4_normed, quantize_rtn
    torch.manual_seed(N + M)
    x, res, nw = torch.randn(M, K, device=DEV).bfloat16(), torch.randn(M, N, device=DEV).bfloat16(), torch.randn(N, device=DEV).bfloat16()
    w4 = quantize_rtn((torch.randn(N, K, device=DEV) * K ** -0.5).bfloat16(), 128)
    got = int4_normed(x, w4, res, nw, 1e-6)
    assert (got is not None) == served
    if served:
        want = int4_linear(x, w4, None, res)
        assert torch.equal(got[0], want) and torch.equal(got[1], rms_norm(want, nw, 1e-6))


@pytest.mark.parametrize("rows", [5, 17, 33, 64])
@pytest.mark.parametrize("weights", ["bf16", "int4"])
def test_decode_steps_norm_rows_where_parts_are_added_up(native_ext, monkeypatch, rows, weights):
    """A decode step's logits are those of the norm's own kernel; a hooked or replaced sublayer, a hooked layer and trainable weights keep it."""
    from llm_in_practise_amd.models import qwen3
    from llm_in_practise_amd.models.common import KVCache
    from llm_in_practise_amd.quant.gptq import replace_with_int4
    from llm_in_practise_amd.quant.int4 import quantize_rtn
    m = qwen3.Qwen3ForCausalLM.from_config(qwen3.qwen3_config("qwen3-small", num_attention_heads=32, intermediate_size=4608),
                                           dtype=torch.bfloat16, device=DEV, seed=0).eval()
    m.requires_grad_(False)
    if weights == "int4":
        replace_with_int4(m, {n: quantize_rtn(mod.weight.detach(), 128) for n, mod in m.named_modules()
                              if isinstance(mod, torch.nn.Linear) and n.startswith("model.layers")})
    m.fuse_projections()
    ids = torch.randint(0, 4096, (rows, 1), device=DEV)
    real, calls = qwen3._with_norm, []

    def counted(*a):
        y = real(*a)
        calls.append(y is not None)
        return y

    def step():
        calls.clear()
        cache = KVCache(m.config.num_hidden_layers, rows, 64, m.config.num_key_value_heads, m.config.head_dim, torch.bfloat16, DEV)
        cache.start_decode(torch.full((rows,), 7, dtype=torch.long, device=DEV))
        with torch.no_grad():
            return m.model(ids, cache=cache)
    monkeypatch.setattr(qwen3, "_with_norm", counted)
    got = step()
    assert len(calls) == 8 and any(calls) == (weights == "int4" or rows > 32)
    with monkeypatch.context() as c:
        c.setattr(qwen3, "_with_norm", lambda *a: None)
        assert torch.equal(step(), got)
    for sub in (m.model.layers[1].self_attn, m.model.layers[1].mlp, m.model.layers[2]):
        seen = []
        handle = sub.register_forward_pre_hook(lambda mod, args: seen.append(args[0]))
        assert torch.equal(step(), got) and len(seen) == 1 and len(calls) < 8
        handle.remove()
    if weights == "bf16":
        m.model.layers[0].mlp.down_proj.weight.requires_grad_()
        step()
        assert not calls[1]


@pytest.mark.parametrize("M", [1, 16, 17, 40])
@pytest.mark.parametrize("N,K", [(32, 64), (1056, 192), (6144, 1088), (64, 1984), (96, 20480)])
def test_gemm_skinny_infinite_weights(native_ext, M, N, K):
    """A partial batch of steps repeats loads: an infinite weight in its last step is an infinite product, not NaN."""
    x, w = torch.ones(M, K, device=DEV).bfloat16(), torch.full((N, K), 2.0 ** -6, device=DEV).bfloat16()
    for j in range(0, K, 32):                           # one infinite weight of every step, in a row of its own
        w[j // 32 % N, j + 31] = float("inf")
    want = x.float() @ w.float().t()
    assert want.isinf().any() and not want.isnan().any()
    y = native_ext.gemm_skinny(x, w, None).float()
    assert torch.equal(y.isinf(), want.isinf()) and not y.isnan().any()
    h = native_ext.gemm_skinny_swiglu(x, w).float()
    assert torch.equal(h.isinf(), want[:, :N // 2].isinf() | want[:, N // 2:].isinf()) and not h.isnan().any()


@pytest.mark.parametrize("M,N,K", [(1, 4096, 12288), (33, 4096, 4096), (64, 2560, 9728), (17, 40, 72), (5, 24, 8)])
def test_product_with_residual_has_addmms_bits(native_ext, M, N, K):
    """Without the copy of the residual; forms that are not taken so (strides, broadcasts, an address off) reach torch.addmm, and
    replays of a captured call see new inputs."""
    torch.manual_seed(M)
    w, x, r = torch.randn(N, K, device=DEV).bfloat16(), torch.randn(M, K, device=DEV).bfloat16(), torch.randn(M, N, device=DEV).bfloat16()
    off = torch.cat([r.new_zeros(1), r.reshape(-1)])[1:].view(M, N)
    for res in (r, off, r[:1].expand(M, N), r.t().contiguous().t(), r[0]):
        before = res.clone()
        assert torch.equal(native_ext.lt_addmm(res, x, w), torch.addmm(res, x, w.t())) and torch.equal(res, before)
    xt = x.t().contiguous().t()
    assert torch.equal(native_ext.lt_addmm(r, xt, w), torch.addmm(r, xt, w.t()))
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        y = native_ext.lt_addmm(r, x, w)
    for seed in range(3):
        torch.manual_seed(seed)
        x.copy_(torch.randn(M, K, device=DEV))
        r.copy_(torch.randn(M, N, device=DEV))
        g.replay()
        assert torch.equal(y, torch.addmm(r, x, w.t()))


def test_products_of_another_workspace_have_plans_of_their_own():
    """lt_linear with a workspace of 1 MiB beside lt_addmm, which asks with more: neither takes the other's candidates."""
    code = """if True:
        import torch
        from llm_in_practise_amd.ops._native import native
        ext, plans = native(), 0
        for M, N, K in ((1, 4096, 12288), (17, 4096, 4096), (64, 2560, 9728)):
            x, w, r = (torch.randn(*s, device="cuda").bfloat16() for s in ((M, K), (N, K), (M, N)))
            want = x.double() @ w.double().t() + r.double()
            for y in (ext.lt_addmm(r, x, w), *(ext.lt_linear(x, w, r, True) for _ in range(6)), ext.lt_addmm(r, x, w)):
                assert (y.double() - want).norm() <= 2.0 ** -8 * want.norm()         # (one rounding to bf16, float sums)
            plans += 2
            assert ext.lt_plans() == plans
    """
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    res = subprocess.run([sys.executable, "-c", code], env={**os.environ, "LIPA_LT_WS_MB": "1"}, cwd=root, capture_output=True, text=True,
                         timeout=110)
    assert res.returncode == 0, res.stderr[-2000:]


def test_product_with_residual_refuses_another_devices_tensors(native_ext):
    x, w, r = torch.zeros(1, 64, device=DEV).bfloat16(), torch.zeros(32, 64, device=DEV).bfloat16(), torch.zeros(1, 32, device=DEV).bfloat16()
    for args in ((r.cpu(), x, w), (r, x.cpu(), w), (r, x, w.cpu())):
        with pytest.raises(RuntimeError):
            native_ext.lt_addmm(*args)


@pytest.mark.parametrize("F,K,own", [(14336, 128, True), (14352, 128, False), (17408, 5120, False), (32, 4096, True), (32, 4160, False)])
def test_gated_product_of_wide_weights_stays_with_the_library(native_ext, F, K, own):
    """One launch for gate, up and activation only up to the widths where it is not the slower form."""
    from llm_in_practise_amd.ops.mlp import skinny_swiglu
    x, w = torch.randn(4, K, device=DEV).bfloat16(), (torch.randn(2 * F, K, device=DEV) * K ** -0.5).bfloat16()
    with torch.no_grad():
        h = skinny_swiglu(x, w)
    assert (h is not None) == own
    if own:
        g, u = (x.float() @ w.float().t()).split(F, 1)
        want = torch.nn.functional.silu(g) * u
        assert (h.float() - want).norm() <= 2.0 ** -7 * want.norm()      # three roundings to bf16 of 2^-9 each

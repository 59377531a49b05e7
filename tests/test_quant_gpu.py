"""W4A16 int4 GEMMs (w4mm, gemm4w W4=2), 4-bit decode GEMV (NF4 + int4), GPTQ/AWQ on the GPU."""
import pytest
import torch

from llm_in_practise_amd.quant.int4 import int4_linear, int4_swiglu, quantize_rtn
from llm_in_practise_amd.quant.nf4 import dequantize_nf4, quantize_nf4

pytestmark = pytest.mark.gpu
DEV = "cuda"


def rel(a, b):
    return ((a.float() - b.float()).norm() / b.float().norm().clamp(min=1e-6)).item()


@pytest.mark.parametrize("M", [1, 3, 8])
@pytest.mark.parametrize("N,K", [(4096, 4096), (1024, 12288), (96, 256)])
def test_gemv_nf4_and_int4(native_ext, M, N, K):
    torch.manual_seed(1)
    x = torch.randn(M, K, device=DEV).to(torch.bfloat16)
    wq = quantize_nf4(torch.randn(N, K, device=DEV).to(torch.bfloat16), 64, True)
    y = native_ext.gemv_w4(x, wq.codes, wq.gemv_scales(), None, N, 64, None)
    assert rel(y, x.float() @ dequantize_nf4(wq, torch.float32).t()) < 1e-2
    w4 = quantize_rtn(torch.randn(N, K, device=DEV), 128, False)
    s, b = w4.gemv_tables()
    res = torch.randn(M, N, device=DEV).to(torch.bfloat16)
    y4 = native_ext.gemv_w4(x, w4.codes, s, b, N, 128, res)
    assert rel(y4, x.float() @ w4.dequantize().t() + res.float()) < 1e-2


@pytest.mark.parametrize("N,K,gs,sym", [(256, 512, 128, False), (384, 1024, 128, True), (96, 256, 64, False)])
def test_int4_linear_dispatch(native_ext, N, K, gs, sym):
    """Every row count through int4_linear's kernel choice — gemv_w4 (M <= 2), w4mm (3..32), w4g (33..64),
    gemm4w W4=2 (65..1023), the expansion + gemm4w prefill (>= 1024), the dequant fallback for shapes no kernel
    takes (N = 96) — against fp32, with residual."""
    torch.manual_seed(4)
    w = quantize_rtn(torch.randn(N, K, device=DEV), gs, sym)
    for M in (1, 2, 3, 8, 32, 33, 64, 100, 256, 300, 2048):
        x = torch.randn(M, K, device=DEV).to(torch.bfloat16)
        res = torch.randn(M, N, device=DEV).to(torch.bfloat16)
        assert rel(int4_linear(x, w), x.float() @ w.dequantize().t()) < 1e-2, M
        assert rel(int4_linear(x, w, residual=res), x.float() @ w.dequantize().t() + res.float()) < 1e-2, M


@pytest.mark.parametrize("M", [33, 48, 64])
@pytest.mark.parametrize("N,K,gs", [(6144, 4096, 128), (4096, 12288, 128), (512, 1024, 256)])
def test_w4g_decode_batches(native_ext, M, N, K, gs):
    """The decode-batch W4A16 GEMM (w4g) at the Qwen3-8B q|k|v / down shapes and a 256-deep group: every
    K-slice count it may pick (1 = bf16 out + residual in-kernel, > 1 = fp32 partials + reduce) against fp32."""
    torch.manual_seed(6)
    w = quantize_rtn(torch.randn(N, K, device=DEV), gs, False)
    x = torch.randn(M, K, device=DEV).to(torch.bfloat16)
    res = torch.randn(M, N, device=DEV).to(torch.bfloat16)
    want = x.float() @ w.dequantize().t() + res.float()
    auto = native_ext.w4g_splits(M, N, K)
    for ks in sorted({1, 2, auto}):
        if (K // 128) % ks:
            continue
        y = native_ext.w4g(x, w.codes, w.w4mm_table(), N, gs, res, ks)
        assert y.shape == (M, N) and rel(y, want) < 1e-2, (ks, rel(y, want))


@pytest.mark.parametrize("M", [3, 8, 12, 16])
@pytest.mark.parametrize("N,K,gs", [(6144, 4096, 128), (24576, 4096, 128), (512, 1024, 256), (4096, 12288, 128), (768, 2560, 128),
                                    (256, 384, 128), (256, 7680, 128)])
def test_w4mm_one_launch_keeps_the_sums(native_ext, M, N, K, gs):
    """All of K in one workgroup (x held by as many waves as slices, or slices in turns; even and ragged shares of tiles) against
    64 bits, and the end in SwiGLU bit for bit the product and the activation."""
    torch.manual_seed(M)
    w = quantize_rtn(torch.randn(N, K, device=DEV), gs, False)
    x, res = torch.randn(M, K, device=DEV).to(torch.bfloat16), torch.randn(M, N, device=DEV).to(torch.bfloat16)
    want = x.double() @ w.dequantize(torch.float32).double().t()
    # the offset form sums 128 + q for q, so its float sums err with (136 |s|) sum |x|
    big = 144 * w.scales.double().abs().max() * x.double().abs().sum(1, keepdim=True)
    y = int4_linear(x, w)
    assert ((y.double() - want).abs() <= (K / 128 + 132) * 2.0 ** -24 * big + 2.0 ** -8 * want.abs()).all()
    wr = want + res.double()
    assert ((int4_linear(x, w, residual=res).double() - wr).abs() <= (K / 128 + 132) * 2.0 ** -24 * big + 2.0 ** -8 * wr.abs()).all()
    h = int4_swiglu(x, w)
    assert h is None or torch.equal(h, native_ext.swiglu_fwd(y))
    assert (h is not None) == (K in (4096, 1024, 2560))


@pytest.mark.parametrize("M,N,K,glu,one", [
    (12, 28672, 512, False, False), (12, 8192, 512, False, True), (3, 1024, 4096, False, False), (12, 1024, 4096, False, True),
    (3, 4096, 4096, True, False), (12, 2048, 4096, True, False), (12, 24576, 4096, True, True), (12, 27648, 5120, False, False),
    (3, 5120, 13824, False, False), (16, 1024, 12288, False, False), (16, 1024, 6144, False, True), (12, 4096, 12288, False, True),
    (24, 24576, 4096, False, True), (24, 4096, 12288, False, False)])
def test_w4mm_one_launch_only_where_it_is_not_slower(native_ext, M, N, K, glu, one):
    """Shapes on both sides of the rule that chooses between one launch and the slices' partial sums."""
    assert native_ext.w4mm_one(M, N, K, glu) == one


@pytest.mark.parametrize("M", [3, 12, 16, 17, 24, 32])
@pytest.mark.parametrize("nkb", [2, 4])
@pytest.mark.parametrize("N,K,gs", [(4096, 1024, 128), (640, 2560, 128), (4096, 4096, 256), (2560, 5120, 128)])
def test_w4mm_one_launch_has_the_bits_of_the_slices(native_ext, M, nkb, N, K, gs):
    assert native_ext.w4mm_one(M, N, K, False, nkb) == (M <= 16 or K <= 4096)      # (else both are the slices' kernel)
    torch.manual_seed(M + nkb)
    w = quantize_rtn(torch.randn(N, K, device=DEV), gs, False)
    x, res = torch.randn(M, K, device=DEV).to(torch.bfloat16), torch.randn(M, N, device=DEV).to(torch.bfloat16)
    for r in (None, res):
        a, b = (native_ext.w4mm(x, w.codes, w.w4mm_table(), N, gs, r, nkb, one) for one in (True, False))
        assert torch.equal(a, b)


@pytest.mark.parametrize("M", [1, 4, 5, 9, 13, 16, 17])
@pytest.mark.parametrize("nkb,N,K,gs", [(4, 4224, 4096, 128), (4, 640, 4608, 512), (4, 128, 5632, 256), (4, 2048, 12288, 128), (4, 128, 6656, 128),
                                        (2, 12416, 768, 384), (2, 256, 5376, 128), (2, 2560, 8192, 256), (4, 128, 512, 512), (4, 16512, 1536, 128)])
def test_w4mm_one_launch_rings(native_ext, nkb, N, K, gs, M):
    """More units than a ring holds and fewer, ragged shares of slices and tiles, groups of several blocks, an odd number of them, a
    table that 16-byte loads cannot take, rows of x that are a slice of wider ones or all the same one: the bits of the slices' kernel."""
    assert native_ext.w4mm_one(M, N, K, False, nkb) == (M <= 16 or K <= 4096)      # (17 rows of a long K: both are the slices' kernel)
    torch.manual_seed(M + K)
    w = quantize_rtn(torch.randn(N, K, device=DEV), gs, False)
    table = w.w4mm_table()
    shifted = torch.empty(table.numel() + 2, device=DEV)[2:].view(table.shape).copy_(table)
    wide, res = torch.randn(M, K + 24, device=DEV).to(torch.bfloat16), torch.randn(M, N, device=DEV).to(torch.bfloat16)
    for x, t, r in ((wide[:, 8:K + 8], table, None), (wide[:, 16:K + 16].contiguous(), shifted, res), (wide[:1, 8:K + 8].expand(M, K), table, res)):
        a, b = (native_ext.w4mm(x, w.codes, t, N, gs, r, nkb, one) for one in (True, False))
        assert torch.equal(a, b)


@pytest.mark.parametrize("N,K,gs,sym", [(256, 512, 128, False), (384, 1024, 64, True)])
def test_int4_dequant_kernel_matches_fp32(native_ext, N, K, gs, sym):
    """The HBM-speed int4 -> bf16 expansion (the W4A16 prefill form) against the fp32 dequantisation."""
    torch.manual_seed(5)
    w = quantize_rtn(torch.randn(N, K, device=DEV), gs, sym)
    s, b = w.gemv_tables()
    got = native_ext.int4_dequant(w.codes, s, b, N, K, gs)
    ref = w.dequantize()
    assert got.dtype == torch.bfloat16 and got.shape == (N, K)
    assert (got.float() - ref).abs().max() <= 1e-2 * ref.abs().max()


def test_awq_gptq_on_gpu_and_quantized_generation(native_ext):
    from llm_in_practise_amd.infer.generate import generate
    from llm_in_practise_amd.models.qwen3 import Qwen3ForCausalLM, qwen3_config
    from llm_in_practise_amd.quant.awq import awq_quantize_model
    from llm_in_practise_amd.quant.eval import dataset_ppl
    from llm_in_practise_amd.quant.gptq import gptq_quantize_model
    calib = [torch.randint(0, 4096, (1, 128), device=DEV) for _ in range(4)]
    held = torch.randint(0, 4096, (1024,), device=DEV)
    base = Qwen3ForCausalLM.from_config(qwen3_config("qwen3-small"), dtype=torch.bfloat16, device=DEV, seed=0).eval()
    p0 = dataset_ppl(base, held)
    for fn in (awq_quantize_model, gptq_quantize_model):
        m = Qwen3ForCausalLM.from_config(qwen3_config("qwen3-small"), dtype=torch.bfloat16, device=DEV, seed=0).eval()
        fn(m, calib)
        p = dataset_ppl(m, held)
        assert abs(p - p0) / p0 < 0.05, (fn.__name__, p, p0)
        out = generate(m, torch.randint(0, 4096, (2, 16), device=DEV), max_new_tokens=8)
        assert out.shape == (2, 24)


def test_nf4_decode_uses_gemv_and_matches_recompute(native_ext):
    from llm_in_practise_amd.infer.generate import generate
    from llm_in_practise_amd.models.qwen3 import Qwen3ForCausalLM, qwen3_config
    from llm_in_practise_amd.peft.lora import quantize_model_nf4
    m = Qwen3ForCausalLM.from_config(qwen3_config("qwen3-small"), dtype=torch.bfloat16, device=DEV, seed=0).eval()
    quantize_model_nf4(m)
    m.fuse_projections()
    p = torch.randint(0, 4096, (1, 40), device=DEV)
    out = generate(m, p, max_new_tokens=4)
    ids = p.clone()
    with torch.no_grad():
        for _ in range(4):
            ids = torch.cat([ids, m(ids).logits[:, -1].float().argmax(-1, keepdim=True)], 1)
    assert torch.equal(out[0, :42], ids[0, :42])

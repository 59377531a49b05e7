"""Routed experts of prompts: the kernels that order pairs by expert and run every expert's products in tiles
(csrc/kernels/seq/seq_moe_gemm.hip), and the routing kernel of prompts, against the reference ops."""
import pytest
import torch

from llm_in_practise_amd.ops import moe as M


@pytest.mark.parametrize("E,F,W,rows,tiles", [
    (8, 4096, 4096, 512, True), (8, 4096, 4096, 1024, False), (8, 14336, 4096, 128, True), (8, 14336, 4096, 512, False),
    (4, 4096, 4096, 1024, True), (4, 4096, 4096, 2048, False), (16, 4096, 2048, 2048, True), (16, 4096, 2048, 4096, False),
    (1, 4096, 4096, 2048, True), (1, 4096, 4096, 8192, False), (8, 2048, 2048, 8192, True), (8, 384, 2048, 30000, True),
    (64, 2048, 4096, 2048, True), (8, 8192, 2048, 512, True), (8, 8192, 2048, 2048, False)])
def test_tiles_only_where_they_are_not_slower(E, F, W, rows, tiles):
    """Timed shapes on both sides of the choice between tiles and a vendor product pair per expert."""
    assert M.expert_tiles_win(rows * E, E, F, W) == tiles


@pytest.mark.gpu
@pytest.mark.parametrize("T,top,E,F,W,kind", [
    (40, 2, 8, 64, 64, "even"), (129, 2, 5, 192, 192, "even"), (300, 4, 8, 128, 320, "identity"), (257, 1, 1, 64, 128, "even"),
    (700, 3, 9, 448, 256, "skewed"), (33, 2, 16, 384, 64, "skewed"), (2100, 2, 3, 64, 64, "even")])
@pytest.mark.parametrize("act,weight_input,gate", [("silu", False, True), ("silu", True, False), ("clipped", False, False)])
def test_expert_tiles(T, top, E, F, W, kind, act, weight_input, gate):
    g = torch.Generator().manual_seed(T + F)
    h = torch.randn(T, W, generator=g).bfloat16()
    gu = (torch.randn(E, 2, F, W, generator=g) * W ** -0.5).bfloat16()
    d = (torch.randn(E, W, F, generator=g) * F ** -0.5).bfloat16()
    n = E + 2 if kind == "identity" else E
    idx = torch.rand(T, max(n, top), generator=g).argsort(1)[:, :top]
    if kind == "skewed":                                # one expert takes nearly all, others nothing
        idx = torch.where(torch.rand(T, top, generator=g) < 0.9, torch.full_like(idx, E - 2), idx)
    idx, w = (idx % n).int().contiguous(), torch.rand(T, top, generator=g)
    sh, sg = torch.randn(T, W, generator=g).bfloat16(), torch.randn(T, generator=g) if gate else None
    on = [t.cuda() for t in (h, gu, d, idx, w)]
    got = M.moe_glu_experts(*on, 7.0, sh.cuda(), False, act=act, shared_gate=None if sg is None else sg.cuda(),
                            weight_input=weight_input)
    want = M.moe_glu_experts(h.float(), gu.float(), d.float(), idx, w, 7.0, sh.float(), False, act=act, shared_gate=sg,
                             weight_input=weight_input)
    # the activation and an expert's output are rounded to bf16 once each: two relative errors of at most 2^-9
    assert torch.isfinite(got).all() and (got.cpu() - want).norm() <= 2.0 ** -8 * want.norm()


@pytest.mark.gpu
@pytest.mark.parametrize("T,E,F,W", [(4000, 8, 256, 128), (4100, 8, 192, 256), (3900, 6, 320, 64), (2200, 4, 640, 192), (1900, 24, 1216, 192)])
def test_expert_tiles_of_many_rows(T, E, F, W):
    """More tiles than CUs: tiles of 128 columns of the activation, the last one half empty at 1216, and of 64 where that pads too much."""
    g = torch.Generator().manual_seed(T)
    top = 3
    h = torch.randn(T, W, generator=g).bfloat16()
    gu, d = (torch.randn(E, 2, F, W, generator=g) * W ** -0.5).bfloat16(), (torch.randn(E, W, F, generator=g) * F ** -0.5).bfloat16()
    idx = torch.rand(T, E, generator=g).argsort(1)[:, :top].int().contiguous()
    w = torch.rand(T, top, generator=g)
    assert (T * top // 128 + E) * -(-F // 64) > 256 and M.expert_tiles_win(T * top, E, F, W)
    got = M.moe_glu_experts(*(t.cuda() for t in (h, gu, d, idx, w)), 7.0, None, False, act="silu")
    want = M.moe_glu_experts(h.float(), gu.float(), d.float(), idx, w, 7.0, None, False, act="silu")
    assert (got.cpu() - want).norm() <= 2.0 ** -8 * want.norm()         # (rounded to bf16 twice, 2^-9 each)


@pytest.mark.gpu
@pytest.mark.parametrize("E", [1, 7, 100, 130, 300])
@pytest.mark.parametrize("pairs", [1, 4095, 4096, 4097, 12291, 36867])
def test_order_of_pairs(E, pairs):
    """Around the turns of 4096 pairs, several to a block where experts are many (100 of them: two parts of five turns); identity experts between the others; ids that start at
    an address of 4 bytes more than a multiple of 16."""
    g = torch.Generator().manual_seed(E + pairs)
    F, W = 64, 64
    h = torch.randn(pairs, W, generator=g).bfloat16()
    gu, d = (torch.randn(E, 2, F, W, generator=g) * W ** -0.5).bfloat16(), (torch.randn(E, W, F, generator=g) * F ** -0.5).bfloat16()
    idx, w = torch.randint(0, E + 2, (pairs, 1), generator=g).int(), torch.rand(pairs, 1, generator=g)
    far = torch.cat([idx.new_zeros(1, 1), idx]).cuda()[1:]
    got = M.moe_glu_experts(h.cuda(), gu.cuda(), d.cuda(), far, w.cuda(), 7.0, None, False, act="silu")
    want = M.moe_glu_experts(h.float(), gu.float(), d.float(), idx, w, 7.0, None, False, act="silu")
    assert M.expert_tiles_win(pairs, E, F, W)
    # every token's row by itself: rounded to bf16 twice, 2^-9 each
    assert ((got.cpu() - want).norm(dim=1) <= 2.0 ** -7 * want.norm(dim=1) + 1e-6).all()
    assert (got.cpu() - want).norm() <= 2.0 ** -8 * want.norm()


@pytest.mark.gpu
@pytest.mark.parametrize("E,T", [(64, 300), (65, 300), (130, 77)])
def test_tiles_of_many_experts(E, T):
    """A tile's expert is found 64 experts at a time; most experts of the last call have no pair."""
    g = torch.Generator().manual_seed(E)
    F, W, top = 64, 128, 2
    h = torch.randn(T, W, generator=g).bfloat16()
    gu, d = (torch.randn(E, 2, F, W, generator=g) * W ** -0.5).bfloat16(), (torch.randn(E, W, F, generator=g) * F ** -0.5).bfloat16()
    idx = torch.rand(T, E, generator=g).argsort(1)[:, :top].int().contiguous()
    idx[:, 0] = E - 1
    w = torch.rand(T, top, generator=g)
    got = M.moe_glu_experts(*(t.cuda() for t in (h, gu, d, idx, w)), 7.0, None, False, act="silu")
    want = M.moe_glu_experts(h.float(), gu.float(), d.float(), idx, w, 7.0, None, False, act="silu")
    assert (got.cpu() - want).norm() <= 2.0 ** -8 * want.norm()         # (rounded to bf16 twice, 2^-9 each)


@pytest.mark.gpu
@pytest.mark.parametrize("act", ["silu", "clipped"])
def test_tiles_activation_of_extreme_values(act):
    """Gates from -3e38 to 3e38, one a token, each beside an up product of 1; infinite and NaN ones reach no other token."""
    gates = [-3e38, -1e4, -200.0, -90.0, -80.0, -20.0, -1.0, -1e-3, 0.0, 1e-3, 1.0, 20.0, 90.0, 1e4, 3e38, float("inf"), -float("inf"), float("nan")]
    E, F, W = 1, 64, 64
    h = torch.zeros(len(gates), W)
    h[:, 0], h[:, 1] = torch.tensor(gates), 1.0
    gu, d = torch.zeros(E, 2, F, W), torch.eye(W)[None].contiguous()
    gu[0, 0, :, 0], gu[0, 1, :, 1] = 1.0, 1.0
    h, gu, d = (t.bfloat16() for t in (h, gu, d))
    idx, w = torch.zeros(len(gates), 1, dtype=torch.int32), torch.ones(len(gates), 1)
    got = M.moe_glu_experts(*(t.cuda() for t in (h, gu, d, idx, w)), 7.0, None, False, act=act).cpu()[:15]
    want = M.moe_glu_experts(h.float(), gu.float(), d.float(), idx, w, 7.0, None, False, act=act)[:15]
    torch.testing.assert_close(got, want, rtol=2.0 ** -8, atol=1e-35)   # (one rounding to bf16; a product below 2^-126 may be 0)


@pytest.mark.gpu
def test_many_rows_of_large_experts():
    """A call past the tiles' range: the vendor's products, the same sums."""
    g = torch.Generator().manual_seed(0)
    T, top, E, F, W = 2100, 1, 1, 8192, 8192
    assert not M.expert_tiles_win(T * top, E, F, W)
    h, w = torch.randn(T, W, generator=g).bfloat16().cuda(), torch.rand(T, top, generator=g).cuda()
    gu = (torch.randn(E, 2, F, W, device="cuda") * W ** -0.5).bfloat16()
    d = (torch.randn(E, W, F, device="cuda") * F ** -0.5).bfloat16()
    got = M.moe_glu_experts(h, gu, d, torch.zeros(T, top, dtype=torch.int32, device="cuda"), w, 7.0, None, False, act="silu")
    z = h.float() @ gu[0].float().reshape(2 * F, W).t()
    want = (torch.nn.functional.silu(z[:, :F]) * z[:, F:]) @ d[0].float().t() * w
    # gate, up, the activation and an expert's output are rounded to bf16 once each: relative errors of at most 2^-9
    assert (got - want).norm() <= 2.0 ** -7 * want.norm()


@pytest.mark.gpu
@pytest.mark.parametrize("T", [256, 259, 1000])
@pytest.mark.parametrize("n,W,top,groups,keep,kw", [
    (8, 2048, 2, 1, 1, dict(normalize=True)), (10, 1024, 4, 2, 1, dict(scale=2.0)), (16, 72, 3, 4, 2, dict(score="sigmoid", group_rank="top2")),
    (3, 64, 1, 1, 1, dict(extra=2)), (7, 516, 7, 1, 1, dict(always=1)), (1, 4, 1, 1, 1, {}), (13, 260, 2, 1, 1, dict(extra=3, always=2))])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
def test_routing_of_prompts(T, n, W, top, groups, keep, kw, dt):
    g = torch.Generator().manual_seed(T + n + W)
    h = torch.randn(T, W, generator=g).to(dt)
    router = torch.randn(n + kw.get("extra", 0), W, generator=g) * W ** -0.5
    corr = 0.1 * torch.randn(n, generator=g)
    got = M.route_tokens(h.cuda(), router.cuda(), corr.cuda(), top, groups, keep, **kw)
    want = M.route_tokens(h, router, corr, top, groups, keep, **kw)
    # float products of W terms in another order; a choice can only differ where two scores are that close
    same = (got[0].cpu() == want[0]).all(1)
    assert same.float().mean() >= 0.995
    assert (got[1].cpu() - want[1])[same].abs().max() <= 1e-5 * max(1.0, kw.get("scale", 1.0))
    if kw.get("extra"):
        torch.testing.assert_close(got[2].cpu(), want[2], rtol=1e-5, atol=1e-5)


@pytest.mark.gpu
@pytest.mark.parametrize("T,W,dt", [(1999, 4160, torch.bfloat16), (2000, 4160, torch.bfloat16), (300, 4096, torch.bfloat16),
                                    (300, 2048, torch.float32), (300, 2052, torch.float32), (2001, 2052, torch.float32)])
def test_routing_of_wide_rows(T, W, dt):
    """On both sides of the width and the number of tokens from which four tokens share a block."""
    g = torch.Generator().manual_seed(T + W)
    h, router = torch.randn(T, W, generator=g).to(dt), torch.randn(12, W, generator=g) * W ** -0.5
    got = M.route_tokens(h.cuda(), router.cuda(), torch.zeros(12).cuda(), 3, 1, 1, normalize=True)
    want = M.route_tokens(h, router, torch.zeros(12), 3, 1, 1, normalize=True)
    same = (got[0].cpu() == want[0]).all(1)             # (a choice can only differ where two scores are that close)
    assert same.float().mean() >= 0.995 and (got[1].cpu() - want[1])[same].abs().max() <= 1e-5


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("top", [1, 2, 3, 4, 5, 8])
@pytest.mark.parametrize("T,W", [(1, 4), (7, 1028), (65, 2048)])
def test_combine_rows_together(T, W, top, dtype):
    """Rows of a token's choices loaded together: choices of no expert (-1) and of the token itself (>= E), a NaN in whatever is read and not
    chosen, a shared expert with and without its gate; against 64 bits (top + 1 products and sums in float)."""
    from llm_in_practise_amd.ops._native import native_seq
    torch.manual_seed(T + top)
    E, dev = 4, "cuda"
    ys, h = torch.randn(T * top, W, device=dev).to(dtype), torch.randn(T, W, device=dev).to(dtype)
    shared, gate, w = torch.randn(T, W, device=dev).to(dtype), torch.randn(T, device=dev), torch.randn(T, top, device=dev)
    idx = torch.randint(-1, E + 2, (T, top), device=dev, dtype=torch.int32)
    pos = torch.randperm(T * top, device=dev).view(T, top)
    h[(idx < E).all(1)] = float("nan")
    ys[pos[(idx < 0) | (idx >= E)]] = float("nan")
    rows = torch.where((idx >= E)[..., None], h[:, None].double(), ys[pos].double())
    terms = torch.where((idx >= 0)[..., None], rows * w[..., None].double(), 0.0)
    for sh, g in ((None, None), (shared, None), (shared, gate)):
        base = torch.zeros(T, W, device=dev, dtype=torch.float64) if sh is None else sh.double() * (1.0 if g is None else torch.sigmoid(g.double())[:, None])
        got = native_seq().moe_combine_sorted(ys, pos, idx, w, h, sh, E, g).double()
        bound = (top + 8) * 2.0 ** -23 * (base.abs() + terms.abs().sum(1))
        assert ((got - base - terms.sum(1)).abs() <= bound).all()


@pytest.mark.gpu
@pytest.mark.parametrize("T,top,E,F,W", [(33, 2, 3, 384, 2048), (8, 2, 8, 512, 2048), (17, 3, 8, 448, 1024), (64, 4, 8, 512, 1024), (128, 4, 16, 96, 640),
                                         (512, 1, 1, 32, 896), (170, 3, 5, 480, 1920)])
@pytest.mark.parametrize("act,weight_input", [("clipped", False), ("silu", False), ("silu", True)])
def test_decode_batches_read_an_expert_once(T, top, E, F, W, act, weight_input):
    """Pairs of an expert that fill no tile of 16, one to four and more than four; identity experts, choices of none, an expert chosen twice;
    depths of few steps, of all and of a number that is no multiple of a load group."""
    from llm_in_practise_amd.ops._native import native_seq
    assert native_seq().moe_few(T, top, E, F, W) and not native_seq().moe_few(T, top, E, F, 4096) and not native_seq().moe_few(513, top, E, F, W)
    g = torch.Generator().manual_seed(T + F)
    h = torch.randn(T, W, generator=g).bfloat16().cuda()
    gu, dn = ((torch.randn(*s, generator=g) * s[-1] ** -0.5).bfloat16().cuda() for s in ((E, 2, F, W), (E, W, F)))
    idx, w = torch.randint(-1, E + 2, (T, top), generator=g).int().cuda(), torch.rand(T, top, generator=g).cuda()
    shared, sg = torch.randn(T, W, generator=g).bfloat16().cuda(), torch.randn(T, generator=g).cuda()
    if weight_input:
        idx = idx.clamp(max=E - 1)
    for extra in ((None, None), (shared, None), (shared, sg)):
        got = M.moe_glu_experts(h, gu, dn, idx, w, 7.0, extra[0], True, act=act, shared_gate=extra[1], weight_input=weight_input)
        want = torch.zeros(T, W, dtype=torch.float64, device="cuda")
        if extra[0] is not None:
            want += shared.double() * (1.0 if extra[1] is None else torch.sigmoid(sg.double())[:, None])
        for j in range(top):
            for e in range(E + 2):
                rows = (idx[:, j] == e).nonzero()[:, 0]
                x, wt = h[rows].double(), w[rows, j, None].double()
                if e < E:
                    gate, up = (x @ gu[e, i].double().t() * (wt if weight_input else 1.0) for i in (0, 1))
                    if act == "silu":
                        a = torch.nn.functional.silu(gate) * up
                    else:
                        gate, up = gate.clamp(max=7.0), up.clamp(-7.0, 7.0)
                        a = gate * torch.sigmoid(1.702 * gate) * (up + 1.0)
                    x = a.float().bfloat16().double() @ dn[e].double().t()
                want[rows] += x * (1.0 if weight_input else wt)
        # float sums of up to 2048 products; of the activations one in a few thousand is rounded to the other bf16 neighbour, 2^-8 of it
        assert ((got.double() - want).norm() / want.norm()).item() < 2e-4


@pytest.mark.gpu
@pytest.mark.parametrize("T,top,E,F,W,few", [
    (8, 4, 16, 512, 1024, False), (9, 4, 16, 512, 1024, True), (12, 4, 16, 448, 640, False), (8, 4, 16, 384, 1536, False), (12, 4, 16, 384, 1536, True),
    (8, 4, 16, 384, 2048, True), (12, 4, 16, 256, 1024, True), (6, 4, 12, 384, 1536, False), (6, 4, 9, 384, 1536, True), (8, 2, 8, 384, 2048, True),
    (7, 2, 8, 384, 2048, False), (512, 1, 1, 64, 512, False), (204, 1, 1, 96, 640, True), (40, 2, 17, 512, 2048, False)])
def test_an_expert_is_read_once_only_where_it_is_not_slower(T, top, E, F, W, few):
    """Timed steps on both sides (in us, a wave a pair / an expert once: 20.7 / 22.9, 26.5 / 22.9, 21.6 / 22.3, 26.7 / 29.6, 34.7 / 30.1, 33.0 / 31.7, 21.8 / 15.1,
    23.8 / 26.4, 23.8 / 18.5, 18.7 / 17.6; 53.9 / 57.7 and 34.5 / 26.9 for a single one), a line nothing was timed at, too many experts."""
    from llm_in_practise_amd.ops._native import native_seq
    assert native_seq().moe_few(T, top, E, F, W) == few

"""The chunked and blocked scans (csrc/kernels/seq/seq_chunk.hip, seq_block.hip) against the token-by-token reference ops, at the
sizes where a chunk, a tile or the choice between two forms ends."""
import pytest
import torch

from llm_in_practise_amd.models.common import SeqBatch, SeqStateCache
from llm_in_practise_amd.ops import recurrent as R

# float sums of up to a few hundred products of order 1, and of decayed states: a few hundred roundings of 2^-24 each, taken
# from both sides and relative to the outputs' norm
TOL = 1e-5


def _batch(spec, lens, starts, device, live=None):
    cache = SeqStateCache([spec], len(lens), max(n + s for n, s in zip(lens, starts)) + 1, torch.bfloat16, device)
    sb = SeqBatch.packed(cache, list(range(len(lens)))[::-1], lens, starts)
    if live is not None:
        sb.live = torch.tensor(live, dtype=torch.int32, device=device)
    return cache.layers[0], sb


def _close(got, want, names):
    for name, a, b in zip(names, got, want):
        a, b = a.detach().cpu().double(), b.detach().cpu().double()
        assert torch.isfinite(a).all(), name
        assert (a - b).norm() <= TOL * b.norm() + 1e-12, (name, ((a - b).norm() / b.norm()).item())


LENS = [([64], [0]), ([128], [0]), ([127, 129, 1, 128, 65], [0, 0, 0, 3, 0]), ([300, 20, 257], [7, 0, 512]), ([63], [5])]


@pytest.mark.gpu
@pytest.mark.parametrize("lens,starts", LENS)
@pytest.mark.parametrize("H,G,dk,dv", [(4, 2, 128, 64), (2, 1, 32, 36), (3, 3, 96, 100), (2, 2, 64, 4), (2, 1, 48, 64)])
def test_ssd_chunks(lens, starts, H, G, dk, dv):
    g = torch.Generator().manual_seed(dk + dv + len(lens))
    T = sum(lens)
    xbc = torch.randn(T, H * dv + 2 * G * dk, generator=g).bfloat16()
    dt, dtb = torch.randn(T, H, generator=g).bfloat16(), torch.randn(H, generator=g) - 2
    a_log, skip = torch.randn(H, generator=g), torch.randn(H, generator=g)
    a_log[-1] = 60.0 if T % 2 else 2.0                  # a head that forgets everything at once
    S0 = 0.3 * torch.randn(len(lens), H, dv, dk, generator=g)
    res = []
    for dev in ("cpu", "cuda"):
        st, sb = _batch({"S": ((H, dv, dk), "f32")}, lens, starts, dev)
        st["S"].copy_(S0)
        x, p = xbc.to(dev), [t.to(dev) for t in (dt, dtb, a_log, skip)]
        y = R.ssd_scan(x[:, H * dv + G * dk:], x[:, H * dv:H * dv + G * dk], x[:, :H * dv], *p, st["S"], H, G, sb)
        res.append((y.view(T, H, dv), st["S"]))
    _close(res[1], res[0], ("y", "state"))


@pytest.mark.gpu
@pytest.mark.parametrize("lens,starts", LENS)
@pytest.mark.parametrize("H,dk,dv", [(2, 128, 192), (2, 64, 96), (3, 32, 36), (1, 96, 4), (2, 160, 32)])
def test_mlstm_chunks(lens, starts, H, dk, dv):
    g = torch.Generator().manual_seed(dk + dv + len(lens))
    T = sum(lens)
    P = torch.randn(T, 2 * H * dk + H * dv, generator=g).bfloat16()
    i, f = 4 * torch.randn(T, H, generator=g), 3 * torch.randn(T, H, generator=g)
    i[::50] += 20.0                                     # the running maximum jumps
    ib, fb = torch.randn(H, generator=g), torch.randn(H, generator=g) + 3
    old = [torch.randn(len(lens), H, dv, dk, generator=g), torch.randn(len(lens), H, dk, generator=g),
           torch.rand(len(lens), H, generator=g)]
    st, sb = _batch({"S": ((H, dv, dk), "f32"), "N": ((H, dk), "f32"), "M": ((H,), "f32")}, lens, starts, "cuda")
    for t, o in zip(st.values(), old):
        t.copy_(o)
    p, gt = P.cuda(), [t.cuda() for t in (i, f, ib, fb)]
    got = R.mlstm_scan(p[:, :H * dk], p[:, H * dk:2 * H * dk], p[:, 2 * H * dk:], *gt, 15.0, dk ** -0.5, st["S"], st["N"],
                       st["M"], H, sb)
    # numerators, normaliser and floor of the reference's recurrence in 64 bits (their quotient is ill-conditioned where the
    # normaliser crosses 0)
    q, k, v = (x.double().view(T, H, -1) for x in P.split([H * dk, H * dk, H * dv], 1))
    ig = 15.0 * torch.tanh((i + ib).double() / 15.0)
    fg = torch.nn.functional.logsigmoid(15.0 * torch.tanh((f + fb).double() / 15.0))
    o, den, floor = torch.empty(T, H, dv).double(), torch.empty(T, H).double(), torch.empty(T, H).double()
    S, N, M = (x.double().clone() for x in old)
    off, slots, pos0 = sb.host()
    for b, slot in enumerate(slots):
        if pos0[b] == 0:
            S[slot], N[slot], M[slot] = 0, 0, 0
        for t in range(off[b], off[b + 1]):
            m = torch.maximum(fg[t] + M[slot], ig[t])
            a, c = torch.exp(fg[t] + M[slot] - m), torch.exp(ig[t] - m)
            M[slot] = m
            S[slot] = a[:, None, None] * S[slot] + c[:, None, None] * v[t][:, :, None] * k[t][:, None, :]
            N[slot] = a[:, None] * N[slot] + c[:, None] * k[t]
            o[t], den[t] = (S[slot] * q[t][:, None]).sum(-1) * dk ** -0.5, (N[slot] * q[t]).sum(-1) * dk ** -0.5
            floor[t] = torch.exp(-m)
    _close((*got, *st.values()), (o, den, floor, S, N, M), ("o", "den", "floor", "S", "N", "M"))


@pytest.mark.gpu
def test_mlstm_chunks_keep_decays_of_a_wide_cap():
    """Caps beyond 512 ln 2: a token may forget more than a float holds while its input weighs still less, or more."""
    lens, H, dk, dv, cap = [131], 3, 32, 32, 2000.0
    g = torch.Generator().manual_seed(0)
    T = sum(lens)
    i, f = torch.zeros(T, H), torch.full((T, H), 5.0)
    f[-2], i[-2] = torch.tensor([-900.0, -900.0, -300.0]), torch.tensor([-500.0, -950.0, -500.0])
    i[-1] = -5000.0
    P = [torch.randn(T, H * n, generator=g).bfloat16().cuda() for n in (dk, dk, dv)]
    st, sb = _batch({"S": ((H, dv, dk), "f32"), "N": ((H, dk), "f32"), "M": ((H,), "f32")}, lens, [0], "cuda")
    zero = torch.zeros(H).cuda()
    R.mlstm_scan(*P, i.cuda(), f.cuda(), zero, zero, cap, dk ** -0.5, st["S"], st["N"], st["M"], H, sb)
    ig, fg = cap * torch.tanh(i.double() / cap), torch.nn.functional.logsigmoid(cap * torch.tanh(f.double() / cap))
    M = torch.zeros(H, dtype=torch.float64)
    for t in range(T):
        M = torch.maximum(fg[t] + M, ig[t])
    torch.testing.assert_close(st["M"][0].cpu().double(), M, rtol=1e-5, atol=1e-3)


@pytest.mark.gpu
@pytest.mark.parametrize("B,H,dk,dv,L", [(1, 8, 128, 192, 1), (30, 8, 128, 192, 1), (96, 8, 64, 96, 1), (200, 4, 128, 64, 1),
                                         (64, 8, 128, 192, 17), (3, 2, 16, 300, 1), (5, 3, 100, 40, 1), (33, 4, 256, 64, 1),
                                         (40, 8, 128, 256, 1), (7, 1, 30, 511, 1)])
def test_mlstm_blocks_of_columns_read_the_old_maximum(B, H, dk, dv, L):
    """More blocks of columns than run at once: those that start after others have ended decay by the maximum from before the step,
    which every step raises here (one block for all columns of a decode step where 1024 threads hold them)."""
    g = torch.Generator().manual_seed(B)
    T = B * L
    q, k, v = (torch.randn(T, H * n, generator=g).bfloat16() for n in (dk, dk, dv))
    i, f = 6.0 + torch.randn(T, H, generator=g), torch.randn(T, H, generator=g)
    st, sb = _batch({"S": ((H, dv, dk), "f32"), "N": ((H, dk), "f32"), "M": ((H,), "f32")}, [L] * B, [5] * B, "cuda",
                    [int(b != 2) for b in range(B)])
    for t in st.values():
        t.fill_(0.25)
    bias = torch.zeros(H, device="cuda")
    got = R.mlstm_scan(q.cuda(), k.cuda(), v.cuda(), i.cuda(), f.cuda(), bias, bias + 3, 15.0, dk ** -0.5, st["S"], st["N"], st["M"],
                       H, sb)
    q, k, v, i, f = (x.double().view(B, L, H, -1) for x in (q, k, v, i, f))
    ig, fg = 15.0 * torch.tanh(i / 15.0), torch.nn.functional.logsigmoid(15.0 * torch.tanh((f + 3) / 15.0))
    S, N, M = (torch.full(s, 0.25, dtype=torch.float64) for s in ((B, H, dv, dk), (B, H, dk), (B, H, 1)))
    want = [torch.empty(B, L, H, dv).double(), torch.empty(B, L, H).double(), torch.empty(B, L, H).double()]
    for t in range(L):
        m = torch.maximum(fg[:, t] + M, ig[:, t])
        a, c, M = torch.exp(fg[:, t] + M - m), torch.exp(ig[:, t] - m), m
        S = a[..., None] * S + (c * v[:, t])[..., None] * k[:, t, :, None]
        N = a * N + c * k[:, t]
        want[0][:, t], want[1][:, t] = (S * q[:, t, :, None]).sum(-1) * dk ** -0.5, (N * q[:, t]).sum(-1) * dk ** -0.5
        want[2][:, t] = torch.exp(-m[..., 0])
    on = torch.arange(B) != 2                           # (an idle row's outputs are nobody's, and its state stays)
    _close([x.view(B, L, *x.shape[1:])[on.cuda()] for x in got], [x[on] for x in want], ("o", "den", "floor"))
    for x, y in zip(st.values(), (S, N, M[..., 0])):    # (slots are the sequences in reverse)
        assert B < 3 or (x.flip(0)[2] == 0.25).all()
        _close([x.flip(0)[on.cuda()]], [y[on]], ["state"])


@pytest.mark.gpu
def test_idle_sequences_keep_their_state():
    lens, H, dk, dv = [130, 200, 70], 2, 64, 32
    g = torch.Generator().manual_seed(0)
    xbc = torch.randn(sum(lens), H * dv + 2 * dk, generator=g).bfloat16().cuda()
    dt, dtb, a_log, skip = (torch.randn(*s, generator=g).cuda() for s in ((sum(lens), H), (H,), (H,), (H,)))
    out = []
    for live in (None, [1, 0, 1]):
        st, sb = _batch({"S": ((H, dv, dk), "f32")}, lens, [0, 0, 0], "cuda", live)
        st["S"].fill_(7.0)
        y = R.ssd_scan(xbc[:, H * dv + dk:], xbc[:, H * dv:H * dv + dk], xbc[:, :H * dv], dt.bfloat16(), dtb, a_log, skip, st["S"],
                       H, 1, sb)
        out.append((y, st["S"]))
    assert (out[1][1][1] == 7.0).all()                  # slot 1 belongs to sequence 1
    assert torch.equal(out[0][1][[0, 2]], out[1][1][[0, 2]])
    assert torch.equal(out[0][0][:130], out[1][0][:130]) and torch.equal(out[0][0][330:], out[1][0][330:])


def _planted(run, inputs, name, t, at, value, lens):
    """Outputs [T, heads, columns] with and without an infinite or NaN entry of one token: every output in front of it, and of the
    other sequences, is what it was; the token's own is no number somewhere."""
    clean = run(inputs)
    x = inputs[name].clone()
    x[t][at] = value
    got = run({**inputs, name: x})
    end = next(e for e in torch.tensor(lens).cumsum(0).tolist() if e > t)
    for a, b in zip(got, clean):
        other = torch.cat([a[:t], a[end:]]), torch.cat([b[:t], b[end:]])
        _close(other[:1], other[1:], (name,))
    assert not torch.isfinite(got[0][t]).all()


@pytest.mark.gpu
@pytest.mark.parametrize("name,value", [("v", float("inf")), ("v", float("nan")), ("k", float("-inf")), ("q", float("nan")),
                                        ("dt", float("nan")), ("dt", float("inf"))])
@pytest.mark.parametrize("t", [150, 203, 268, 383])
def test_ssd_token_that_is_no_number(name, value, t):
    lens, H, dk, dv = [120, 264], 2, 128, 40
    g = torch.Generator().manual_seed(t)
    T = sum(lens)
    inputs = {n: torch.randn(T, w, generator=g).bfloat16().cuda() for n, w in (("q", dk), ("k", dk), ("v", H * dv), ("dt", H))}
    dtb, a_log, skip = (torch.randn(H, generator=g).cuda() for _ in range(3))

    def run(x):
        st, sb = _batch({"S": ((H, dv, dk), "f32")}, lens, [0, 5], "cuda")
        st["S"].fill_(0.5)
        return (R.ssd_scan(x["q"], x["k"], x["v"], x["dt"], dtb, a_log, skip, st["S"], H, 1, sb).view(T, H, dv),)
    _planted(run, inputs, name, t, 1, value, lens)


@pytest.mark.gpu
@pytest.mark.parametrize("name,value", [("v", float("-inf")), ("v", float("nan")), ("k", float("inf")), ("q", float("nan")),
                                        ("i", float("nan")), ("f", float("nan"))])
@pytest.mark.parametrize("t", [129, 204, 299])
def test_mlstm_token_that_is_no_number(name, value, t):
    lens, H, dk, dv = [70, 230], 2, 64, 96
    g = torch.Generator().manual_seed(t)
    T = sum(lens)
    inputs = {n: torch.randn(T, H * w, generator=g).bfloat16().cuda() for n, w in (("q", dk), ("k", dk), ("v", dv))}
    inputs |= {n: 2 * torch.randn(T, H, generator=g).cuda() for n in "if"}
    ib, fb = torch.randn(H, generator=g).cuda(), (torch.randn(H, generator=g) + 3).cuda()

    def run(x):
        st, sb = _batch({"S": ((H, dv, dk), "f32"), "N": ((H, dk), "f32"), "M": ((H,), "f32")}, lens, [9, 0], "cuda")
        for s in st.values():
            s.fill_(0.25)
        return R.mlstm_scan(x["q"], x["k"], x["v"], x["i"], x["f"], ib, fb, 15.0, dk ** -0.5, st["S"], st["N"], st["M"], H, sb)
    _planted(run, inputs, name, t, 1, value, lens)


def _in_chunks(op, lens, H, dk, dv):
    """The step runs in chunks: not walked with the state at hand, not token by token."""
    from llm_in_practise_amd.ops._native import native_seq
    shape = (sum(lens), len(lens), H, dk, dv)
    return native_seq().scan_walk(*shape, max(lens), op) == 0 < native_seq().scan_floats(op, *shape, longest=max(lens))


# keys that have no walk, long sequences; one, two and four chunks a run
CHUNK_LENS = [([120, 264], 2, 1, 96, 40), ([64, 1500], 4, 2, 128, 40), ([3000, 1100], 16, 2, 128, 64), ([1100, 6000], 16, 4, 64, 128)]


@pytest.mark.gpu
@pytest.mark.parametrize("name,value", [("v", float("inf")), ("k", float("-inf")), ("k", float("nan")), ("q", float("nan")), ("q", float("inf")),
                                        ("dt", float("nan")), ("dt", float("inf"))])
@pytest.mark.parametrize("lens,H,G,dk,dv", CHUNK_LENS)
@pytest.mark.parametrize("at", [0, 131, 255])
def test_ssd_chunks_with_a_token_that_is_no_number(name, value, lens, H, G, dk, dv, at):
    assert _in_chunks("ssd", lens, H, dk, dv)
    g = torch.Generator().manual_seed(at)
    T = sum(lens)
    inputs = {n: torch.randn(T, w, generator=g).bfloat16().cuda() for n, w in (("q", G * dk), ("k", G * dk), ("v", H * dv), ("dt", H))}
    dtb, a_log, skip = (torch.randn(H, generator=g).cuda() for _ in range(3))

    def run(x):
        st, sb = _batch({"S": ((H, dv, dk), "f32")}, lens, [0, 5], "cuda")
        st["S"].fill_(0.5)
        return (R.ssd_scan(x["q"], x["k"], x["v"], x["dt"], dtb, a_log, skip, st["S"], H, G, sb).view(T, H, dv),)
    _planted(run, inputs, name, lens[0] + at, 1, value, lens)


@pytest.mark.gpu
@pytest.mark.parametrize("name,value", [("v", float("-inf")), ("k", float("inf")), ("k", float("nan")), ("q", float("nan")), ("i", float("nan")),
                                        ("f", float("nan"))])
@pytest.mark.parametrize("lens,H,G,dk,dv", CHUNK_LENS)
@pytest.mark.parametrize("at", [1, 128, 250])
def test_mlstm_chunks_with_a_token_that_is_no_number(name, value, lens, H, G, dk, dv, at):
    assert _in_chunks("mlstm", lens, H, dk, dv)
    g = torch.Generator().manual_seed(at)
    T = sum(lens)
    inputs = {n: torch.randn(T, H * w, generator=g).bfloat16().cuda() for n, w in (("q", dk), ("k", dk), ("v", dv))}
    inputs |= {n: 2 * torch.randn(T, H, generator=g).cuda() for n in "if"}
    ib, fb = torch.randn(H, generator=g).cuda(), (torch.randn(H, generator=g) + 3).cuda()

    def run(x):
        st, sb = _batch({"S": ((H, dv, dk), "f32"), "N": ((H, dk), "f32"), "M": ((H,), "f32")}, lens, [9, 0], "cuda")
        for s in st.values():
            s.fill_(0.25)
        return R.mlstm_scan(x["q"], x["k"], x["v"], x["i"], x["f"], ib, fb, 15.0, dk ** -0.5, st["S"], st["N"], st["M"], H, sb)
    _planted(run, inputs, name, lens[0] + at, 1, value, lens)


@pytest.mark.gpu
@pytest.mark.parametrize("lens,starts", [([40, 1500], [0, 0]), ([1411, 1, 128], [3, 0, 9])])
@pytest.mark.parametrize("H,G,dk,dv", [(4, 2, 128, 64), (6, 1, 128, 36), (4, 2, 64, 64)])
def test_ssd_chunks_of_long_sequences(lens, starts, H, G, dk, dv):
    """Keys of 64 and 128 that several heads share, sequences long enough to be left to the chunks, against the token-by-token reference."""
    assert _in_chunks("ssd", lens, H, dk, dv)
    g = torch.Generator().manual_seed(dk + dv + len(lens))
    T = sum(lens)
    xbc = torch.randn(T, H * dv + 2 * G * dk, generator=g).bfloat16()
    dt, dtb = torch.randn(T, H, generator=g).bfloat16(), torch.randn(H, generator=g) - 2
    a_log, skip = torch.randn(H, generator=g), torch.randn(H, generator=g)
    S0 = 0.3 * torch.randn(len(lens), H, dv, dk, generator=g)
    res = []
    for dev in ("cpu", "cuda"):
        st, sb = _batch({"S": ((H, dv, dk), "f32")}, lens, starts, dev)
        st["S"].copy_(S0)
        x, p = xbc.to(dev), [t.to(dev) for t in (dt, dtb, a_log, skip)]
        y = R.ssd_scan(x[:, H * dv + G * dk:], x[:, H * dv:H * dv + G * dk], x[:, :H * dv], *p, st["S"], H, G, sb)
        res.append((y.view(T, H, dv), st["S"]))
    _close(res[1], res[0], ("y", "state"))


@pytest.mark.gpu
@pytest.mark.parametrize("op", ["ssd", "mlstm"])
@pytest.mark.parametrize("H,dk,dv", [(2, 128, 32), (3, 96, 20)])
def test_idle_sequences_keep_their_state_in_chunks(op, H, dk, dv):
    lens = [130, 2000, 70]
    assert _in_chunks(op, lens, H, dk, dv)
    g = torch.Generator().manual_seed(0)
    T = sum(lens)
    q, k, v = (torch.randn(T, H * n, generator=g).bfloat16().cuda() for n in (dk, dk, dv))
    i, f = (torch.randn(T, H, generator=g).cuda() for _ in "if")
    a, b, skip = (torch.randn(H, generator=g).cuda() for _ in range(3))
    out = []
    for live in (None, [1, 0, 1]):
        st, sb = _batch({"S": ((H, dv, dk), "f32"), "N": ((H, dk), "f32"), "M": ((H,), "f32")}, lens, [0, 3, 8], "cuda", live)
        for x in st.values():
            x.fill_(7.0)
        if op == "ssd":
            y = [R.ssd_scan(q, k, v, i.bfloat16(), a - 3, b, skip, st["S"], H, H, sb)]
        else:
            y = R.mlstm_scan(q, k, v, i, f, a, b + 3, 15.0, dk ** -0.5, st["S"], st["N"], st["M"], H, sb)
        out.append(([x for x in y], [st["S"]] if op == "ssd" else list(st.values())))
    for x in out[1][1]:
        assert (x[1] == 7.0).all()                      # slot 1 belongs to sequence 1
    for x, y in zip(out[0][1], out[1][1]):
        assert torch.equal(x[[0, 2]], y[[0, 2]])
    for x, y in zip(out[0][0], out[1][0]):
        assert torch.equal(x[:130], y[:130]) and torch.equal(x[2130:], y[2130:])


BLOCK_LENS = [([32], [0]), ([31], [3]), ([48, 15, 1, 128, 65, 33], [0, 0, 9, 5, 0, 0]), ([100, 47], [512, 0])]


@pytest.mark.gpu
@pytest.mark.parametrize("lens,starts", BLOCK_LENS)
@pytest.mark.parametrize("H,G,dk,dv,dt", [(4, 2, 128, 64, torch.float32), (2, 1, 64, 20, torch.bfloat16),
                                          (1, 1, 256, 16, torch.float32), (2, 2, 192, 33, torch.bfloat16),
                                          (2, 1, 96, 32, torch.float32)])
def test_delta_blocks(lens, starts, H, G, dk, dv, dt):
    g = torch.Generator().manual_seed(dk + dv + len(lens))
    T = sum(lens)
    P = torch.randn(T, 2 * G * dk + H * dv, generator=g)
    for j in (0, 1):
        x = P[:, j * G * dk:(j + 1) * G * dk].view(T, G, dk)
        x.copy_(torch.nn.functional.normalize(x, dim=-1))
    P, decay, beta = P.to(dt), torch.rand(T, H * dk, generator=g) ** 0.2, 2 * torch.randn(T, H, generator=g)
    decay[::7, ::3] = 0.0                               # channels that forget everything
    S0 = torch.randn(len(lens), H, dv, dk, generator=g)
    res = []
    for dev in ("cpu", "cuda"):
        st, sb = _batch({"S": ((H, dv, dk), "f32")}, lens, starts, dev)
        st["S"].copy_(S0)
        p = P.to(dev)
        o = R.gated_delta_scan(p[:, :G * dk], p[:, G * dk:2 * G * dk], p[:, 2 * G * dk:], decay.to(dev), beta.to(dev), st["S"], H,
                               G, sb)
        res.append((o, st["S"]))
    _close(res[1], res[0], ("o", "state"))


@pytest.mark.gpu
@pytest.mark.parametrize("lens,starts", BLOCK_LENS)
@pytest.mark.parametrize("H,dk,dv,dt", [(4, 64, 128, torch.bfloat16), (2, 128, 20, torch.float32), (1, 256, 33, torch.bfloat16),
                                        (2, 72, 32, torch.float32)])
def test_gla_blocks(lens, starts, H, dk, dv, dt):
    g = torch.Generator().manual_seed(dk + dv + len(lens))
    T = sum(lens)
    P = torch.randn(T, 2 * H * dk + H * dv, generator=g).to(dt)
    z, zb = 3 * torch.randn(T, H * dk, generator=g), torch.randn(H * dk, generator=g)
    z[::9, ::5] = -4000.0                               # channels that forget everything
    S0 = torch.randn(len(lens), H, dv, dk, generator=g)
    res = []
    for dev in ("cpu", "cuda"):
        st, sb = _batch({"S": ((H, dv, dk), "f32")}, lens, starts, dev)
        st["S"].copy_(S0)
        p = P.to(dev)
        o = R.gated_linear_scan(p[:, :H * dk], p[:, H * dk:2 * H * dk], p[:, 2 * H * dk:], z.to(dev), zb.to(dev), 16.0,
                                dk ** -0.5, st["S"], H, sb)
        res.append((o, st["S"]))
    _close(res[1], res[0], ("o", "state"))


@pytest.mark.gpu
@pytest.mark.parametrize("name,value", [("v", float("inf")), ("v", float("nan")), ("k", float("nan")), ("q", float("inf")),
                                        ("g", float("nan")), ("b", float("nan"))])
@pytest.mark.parametrize("t", [53, 68, 95, 96, 110])
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_delta_token_that_is_no_number(name, value, t, dt):
    lens, H, dk, dv = [50, 70], 2, 128, 20
    g = torch.Generator().manual_seed(t)
    T = sum(lens)
    inputs = {n: torch.nn.functional.normalize(torch.randn(T, dk, generator=g), dim=-1).to(dt).cuda() for n in "qk"}
    inputs |= {"v": torch.randn(T, H * dv, generator=g).to(dt).cuda(), "g": (torch.rand(T, H * dk, generator=g) ** 0.2).cuda(),
               "b": torch.randn(T, H, generator=g).cuda()}

    def run(x):
        st, sb = _batch({"S": ((H, dv, dk), "f32")}, lens, [3, 0], "cuda")
        st["S"].fill_(0.5)
        return (R.gated_delta_scan(x["q"], x["k"], x["v"], x["g"], x["b"], st["S"], H, 1, sb),)
    _planted(run, inputs, name, t, 1, value, lens)


@pytest.mark.gpu
@pytest.mark.parametrize("lens,starts", [([320], [0]), ([351, 1, 640, 209], [0, 3, 0, 9]), ([305, 336], [7, 0]), ([592, 49], [0, 0])])
@pytest.mark.parametrize("H,G,dk,dv,dt", [(3, 1, 64, 36, torch.float32), (2, 2, 128, 20, torch.bfloat16), (4, 2, 128, 64, torch.float32),
                                          (1, 1, 64, 4, torch.bfloat16)])
def test_delta_blocks_of_two_tiles(lens, starts, H, G, dk, dv, dt):
    """Long sequences: a last block of one token, one tile, a tile and a token, all 32; a sequence that does not run."""
    g = torch.Generator().manual_seed(dk + dv + len(lens))
    T, live = sum(lens), [int(b != 3) for b in range(len(lens))]
    P = torch.randn(T, 2 * G * dk + H * dv, generator=g)
    for j in (0, 1):
        x = P[:, j * G * dk:(j + 1) * G * dk].view(T, G, dk)
        x.copy_(torch.nn.functional.normalize(x, dim=-1))
    P, decay, beta = P.to(dt), torch.rand(T, H * dk, generator=g) ** 0.2, 2 * torch.randn(T, H, generator=g)
    decay[::7, ::3] = 0.0                               # channels that forget everything
    S0 = torch.randn(len(lens), H, dv, dk, generator=g)
    tok = torch.cat([torch.full((n,), bool(on)) for n, on in zip(lens, live)])
    res = []
    for dev in ("cpu", "cuda"):
        st, sb = _batch({"S": ((H, dv, dk), "f32")}, lens, starts, dev, live)
        st["S"].copy_(S0)
        p = P.to(dev)
        o = R.gated_delta_scan(p[:, :G * dk], p[:, G * dk:2 * G * dk], p[:, 2 * G * dk:], decay.to(dev), beta.to(dev), st["S"], H,
                               G, sb)
        res.append((o.cpu()[tok], st["S"]))
    _close(res[1], res[0], ("o", "state"))


@pytest.mark.gpu
@pytest.mark.parametrize("lens,starts,live", [([1000], [0], [1]), ([1, 997, 30, 610], [0, 7, 5, 0], [1, 1, 1, 1]),
                                              ([640, 800, 64, 33], [3, 0, 0, 0], [0, 1, 1, 1])])
@pytest.mark.parametrize("H,G,dk,dv,dt", [(2, 1, 128, 20, torch.bfloat16), (3, 3, 64, 36, torch.float32), (1, 1, 128, 132, torch.float32)])
def test_delta_sequences_in_parts(lens, starts, live, H, G, dk, dv, dt):
    """Long sequences in parts that run side by side: a first state, a last part of one token or tile, sequences of one part
    and one that does not run; and a value and a key that are no numbers reach what is behind them, part or not."""
    from llm_in_practise_amd.ops._native import native_seq
    T = sum(lens)
    blocks = native_seq().scan_parts("delta", T, len(lens), H, dk, dv, max(lens))
    assert 0 < 2 * 32 * blocks < max(lens) + 32 * blocks
    g = torch.Generator().manual_seed(dk + dv + len(lens))
    P = torch.randn(T, 2 * G * dk + H * dv, generator=g)
    for j in (0, 1):
        x = P[:, j * G * dk:(j + 1) * G * dk].view(T, G, dk)
        x.copy_(torch.nn.functional.normalize(x, dim=-1))
    P, decay, beta = P.to(dt), torch.rand(T, H * dk, generator=g) ** 0.02, 2 * torch.randn(T, H, generator=g)
    decay[::97, ::3] = 0.0
    S0 = torch.randn(len(lens), H, dv, dk, generator=g)
    tok = torch.cat([torch.full((n,), bool(on)) for n, on in zip(lens, live)])

    def run(dev, p):
        st, sb = _batch({"S": ((H, dv, dk), "f32")}, lens, starts, dev, live)
        st["S"].copy_(S0)
        p = p.to(dev)
        o = R.gated_delta_scan(p[:, :G * dk], p[:, G * dk:2 * G * dk], p[:, 2 * G * dk:], decay.to(dev), beta.to(dev), st["S"], H, G, sb)
        return o.cpu()[tok], st["S"].cpu()
    want, got = run("cpu", P), run("cuda", P)
    _close(got, want, ("o", "state"))
    for column in (2 * G * dk + 5, G * dk + 5):              # a value; a key
        bad, first = P.clone(), sum(lens[:1]) if len(lens) > 1 else 0
        bad[first + 32 * blocks - 3, column] = float("nan")  # near the end of a part
        a, b = run("cpu", bad), run("cuda", bad)
        for x, y in zip(a, b):
            assert torch.equal(x.isnan(), y.isnan())
        _close((b[0].nan_to_num(),), (a[0].nan_to_num(),), ("o",))


@pytest.mark.gpu
@pytest.mark.parametrize("lens,starts,live", [([1025], [0], [1]), ([1, 997, 30, 610], [0, 7, 5, 0], [1, 1, 1, 1]),
                                              ([640, 800, 64, 33], [3, 0, 0, 0], [0, 1, 1, 1])])
@pytest.mark.parametrize("H,dk,dv,dt", [(2, 64, 20, torch.bfloat16), (3, 128, 36, torch.float32), (1, 256, 4, torch.bfloat16)])
def test_gla_sequences_in_parts(lens, starts, live, H, dk, dv, dt):
    from llm_in_practise_amd.ops._native import native_seq
    T = sum(lens)
    blocks = native_seq().scan_parts("gla", T, len(lens), H, dk, dv, max(lens))
    assert 0 < 2 * 16 * blocks < max(lens) + 16 * blocks
    g = torch.Generator().manual_seed(dk + dv + len(lens))
    P, z, zb = torch.randn(T, 2 * H * dk + H * dv, generator=g).to(dt), torch.randn(T, H * dk, generator=g), torch.randn(H * dk, generator=g)
    z[::97, ::3] = -2000.0                               # channels that forget everything
    S0 = torch.randn(len(lens), H, dv, dk, generator=g)
    tok = torch.cat([torch.full((n,), bool(on)) for n, on in zip(lens, live)])

    def run(dev, p):
        st, sb = _batch({"S": ((H, dv, dk), "f32")}, lens, starts, dev, live)
        st["S"].copy_(S0)
        p = p.to(dev)
        o = R.gated_linear_scan(p[:, :H * dk], p[:, H * dk:2 * H * dk], p[:, 2 * H * dk:], z.to(dev), zb.to(dev), 16.0, dk ** -0.5, st["S"], H, sb)
        return o.cpu()[tok], st["S"].cpu()
    _close(run("cuda", P), run("cpu", P), ("o", "state"))
    bad, first = P.clone(), sum(lens[:1]) if len(lens) > 1 else 0
    bad[first + 16 * blocks - 3, 2 * H * dk + 3] = float("nan")            # a value near the end of a part
    a, b = run("cpu", bad), run("cuda", bad)
    for x, y in zip(a, b):
        assert torch.equal(x.isnan(), y.isnan())
    _close((b[0].nan_to_num(),), (a[0].nan_to_num(),), ("o",))


@pytest.mark.gpu
@pytest.mark.parametrize("op,dk", [("delta", 128), ("gla", 64)])
def test_parts_find_room_beside_the_blocks(op, dk):
    from llm_in_practise_amd.ops._native import native_seq
    ext, shape = native_seq(), (4093, 1, 4, dk, 128)
    whole, parts = ext.scan_floats(op, *shape), ext.scan_floats(op, *shape, longest=4093)
    assert whole < parts and ext.scan_parts(op, *shape, longest=4093, most=parts) > 0
    assert ext.scan_parts(op, *shape, longest=4093, most=parts - 1) == 0
    assert ext.scan_floats(op, *shape, most=parts - 1, longest=4093) == whole
    assert ext.scan_parts(op, *shape, longest=0) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("T,B,H,dk,dv,longest,blocks", [
    (10239, 24, 8, 128, 16, 1134, 0), (5073, 8, 32, 128, 16, 2446, 0), (16095, 32, 4, 128, 16, 1065, 0), (8000, 4, 4, 128, 128, 2000, 0),
    (2297, 3, 8, 128, 128, 1500, 12), (700, 1, 8, 128, 128, 700, 8), (4093, 1, 8, 128, 128, 4093, 19), (5120, 4, 4, 128, 128, 5000, 32)])
def test_delta_in_parts_only_where_it_is_not_slower(T, B, H, dk, dv, longest, blocks):
    """Timed shapes, us in one piece / in parts: few long sequences among short ones that fill the chip (122 / 163, 269 / 306, 109 / 121) and long ones that
    do (122 / 121) stay in one piece; (92 / 86, 47 / 43, 208 / 136, 240 / 114) do not."""
    from llm_in_practise_amd.ops._native import native_seq
    assert native_seq().scan_parts("delta", T, B, H, dk, dv, longest) == blocks


@pytest.mark.gpu
@pytest.mark.parametrize("T,B,H,dk,dv,longest,parts", [
    (1396, 1, 16, 192, 192, 1396, False), (3596, 4, 4, 192, 192, 899, False), (9174, 3, 4, 256, 256, 3058, False), (8000, 4, 8, 64, 128, 2000, False),
    (1000, 1, 8, 64, 128, 1000, True), (4093, 1, 16, 64, 128, 4093, True), (6275, 3, 8, 192, 160, 6190, True), (2232, 4, 3, 256, 64, 558, True)])
def test_linear_attention_in_parts_only_where_it_is_not_slower(T, B, H, dk, dv, longest, parts):
    """Timed shapes, us in one piece / in parts: 110 / 147, 79 / 108, 293 / 352, 86 / 91; 40 / 26, 147 / 100, 366 / 241, 66 / 49."""
    from llm_in_practise_amd.ops._native import native_seq
    assert (native_seq().scan_parts("gla", T, B, H, dk, dv, longest) > 0) == parts


@pytest.mark.gpu
def test_parts_that_can_be_counted():
    """Parts are counted in 16 bits: a step that would have more, which takes a longest sequence that is not the longest, has none."""
    from llm_in_practise_amd.ops._native import native_seq
    ext = native_seq()
    part = 16 * ext.scan_parts("gla", 1000, 1, 1, 64, 16, longest=1000)
    assert part > 0
    for T in (32767 * part, 40000 * part, 65537 * part):
        assert ext.scan_parts("gla", T, 1, 1, 64, 16, longest=1000, most=1 << 40) == 0
        assert ext.scan_floats("gla", T, 1, 1, 64, 16, most=1 << 40, longest=1000) == ext.scan_floats("gla", T, 1, 1, 64, 16, most=1 << 40)
    # the delta rule: what a plan holds is no more, whatever the caller says
    assert ext.scan_parts("delta", 2_000_000, 1, 1, 64, 16, longest=2_000_000, most=1 << 40) > 0
    assert ext.scan_parts("delta", 2_100_000, 1, 1, 64, 16, longest=2_100_000, most=1 << 40) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("op,T,dk,most", [("delta", 6000, 64, 262144), ("delta", 3200, 128, 262144), ("gla", 6000, 64, 131072)])
def test_parts_without_room_for_the_blocks(op, T, dk, most):
    """Room for what the parts leave, but for no plan of the blocks they are made of: the step runs as it does with lengths that are not known."""
    from llm_in_practise_amd.ops._native import native_seq
    ext, H, dv, lens = native_seq(), 1, 16, [T - 120, 40, 40, 40]
    floats = ext.scan_floats(op, T, 4, H, dk, dv, most=most)
    assert ext.scan_parts(op, T, 4, H, dk, dv, longest=lens[0]) > 0 == ext.scan_parts(op, T, 4, H, dk, dv, longest=lens[0], most=most)
    assert ext.scan_floats(op, T, 4, H, dk, dv, most=most, longest=lens[0]) == floats <= most
    g = torch.Generator().manual_seed(T + dk)
    P = torch.nn.functional.normalize(torch.randn(T, 2, dk, generator=g), dim=-1).flatten(1).bfloat16().cuda()
    v, z, beta = torch.randn(T, dv, generator=g).bfloat16().cuda(), torch.rand(T, dk, generator=g).cuda() ** 0.02, torch.randn(T, H, generator=g).cuda()
    zb, res = torch.zeros(dk, device="cuda"), []
    for longest in (0, lens[0]):
        st, sb = _batch({"S": ((H, dv, dk), "f32")}, lens, [0] * 4, "cuda")
        st["S"].zero_()
        if op == "delta":
            o = ext.delta_scan(P[:, :dk], P[:, dk:], v, z, beta, st["S"], H, 1, sb.desc, sb.live, longest=longest, most=most)
        else:
            o = ext.gated_linear_scan(P[:, :dk], P[:, dk:], v, z, zb, 16.0, 1.0, st["S"], H, sb.desc, sb.live, longest=longest, most=most)
        res.append((o, st["S"]))
    assert torch.isfinite(res[0][0]).all() and res[0][0].abs().max() > 0
    for a, b in zip(*res):
        assert torch.equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("L,B,H,dk,dv,long", [
    (1000, 1, 8, 128, 128, True), (200, 1, 8, 128, 128, False), (300, 5, 6, 128, 128, True), (299, 5, 6, 128, 128, False),
    (2000, 4, 8, 128, 128, True), (2000, 5, 8, 128, 128, False), (400, 20, 16, 128, 64, True), (400, 20, 16, 128, 68, False),
    (512, 8, 16, 128, 32, True), (600, 4, 32, 64, 64, True), (512, 16, 16, 64, 128, False), (1000, 2, 4, 192, 128, False),
    (1000, 2, 4, 256, 64, False)])
def test_delta_blocks_are_long_only_where_they_are_not_slower(L, B, H, dk, dv, long):
    """Timed shapes on both sides of the choice between blocks of 16 and of 32 tokens."""
    from llm_in_practise_amd.ops._native import native_seq
    assert native_seq().delta_block(L * B, B, H, dk, dv) == (32 if long else 16)


@pytest.mark.gpu
def test_delta_long_blocks_stay_inside_their_grid():
    from llm_in_practise_amd.ops._native import native_seq
    ext, room = native_seq(), 1 << 40
    assert [ext.delta_block(32 * n, 1, 1, 64, 16, room) for n in (65534, 65535)] == [32, 16]       # (a slot more than whole blocks)


@pytest.mark.gpu
@pytest.mark.parametrize("name,value", [("v", float("inf")), ("v", float("nan")), ("k", float("-inf")), ("q", float("nan")),
                                        ("g", float("nan")), ("g", float("inf")), ("b", float("nan"))])
@pytest.mark.parametrize("t", [310, 325, 326, 341, 342, 650, 669])
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_delta_token_that_is_no_number_in_two_tiles(name, value, t, dt):
    """On both sides of a tile (326) and of a block (310, 342), in a block of one tile (650) and at the end."""
    lens, H, dk, dv = [310, 360], 2, 128, 20
    g = torch.Generator().manual_seed(t)
    T = sum(lens)
    inputs = {n: torch.nn.functional.normalize(torch.randn(T, dk, generator=g), dim=-1).to(dt).cuda() for n in "qk"}
    inputs |= {"v": torch.randn(T, H * dv, generator=g).to(dt).cuda(), "g": (torch.rand(T, H * dk, generator=g) ** 0.2).cuda(),
               "b": torch.randn(T, H, generator=g).cuda()}

    def run(x):
        st, sb = _batch({"S": ((H, dv, dk), "f32")}, lens, [3, 0], "cuda")
        st["S"].fill_(0.5)
        return (R.gated_delta_scan(x["q"], x["k"], x["v"], x["g"], x["b"], st["S"], H, 1, sb),)
    _planted(run, inputs, name, t, 1, value, lens)


@pytest.mark.gpu
@pytest.mark.parametrize("name,value", [("v", float("-inf")), ("v", float("nan")), ("k", float("inf")), ("q", float("nan")),
                                        ("z", float("nan"))])
@pytest.mark.parametrize("t", [53, 68, 95, 96, 110])
def test_gla_token_that_is_no_number(name, value, t):
    lens, H, dk, dv = [50, 70], 2, 64, 40
    g = torch.Generator().manual_seed(t)
    T = sum(lens)
    inputs = {n: torch.randn(T, H * w, generator=g).cuda() for n, w in (("q", dk), ("k", dk), ("v", dv), ("z", dk))}
    zb = torch.randn(H * dk, generator=g).cuda()

    def run(x):
        st, sb = _batch({"S": ((H, dv, dk), "f32")}, lens, [0, 4], "cuda")
        st["S"].fill_(0.5)
        return (R.gated_linear_scan(x["q"], x["k"], x["v"], x["z"], zb, 16.0, dk ** -0.5, st["S"], H, sb),)
    _planted(run, inputs, name, t, 1, value, lens)


@pytest.mark.gpu
@pytest.mark.parametrize("lens,starts,C,N,dt,cut", [
    ([2100], [0], 40, 16, torch.bfloat16, True), ([129, 256, 1, 320], [0, 7, 0, 0], 33, 5, torch.float32, True),
    ([127, 130], [0, 3], 130, 40, torch.bfloat16, False), ([200], [0], 64, 200, torch.float32, True),
    ([2305], [0], 2048, 16, torch.bfloat16, True), ([1409, 1, 1500], [5, 0, 0], 64, 16, torch.float32, True),
    ([20, 31], [0, 0], 64, 16, torch.float32, False)])
def test_selective_cut_over_time(lens, starts, C, N, dt, cut):
    from llm_in_practise_amd.ops._native import native_seq
    g = torch.Generator().manual_seed(C + N)
    T = sum(lens)
    assert not native_seq().selective_rows(T, len(lens), C, N) and (native_seq().selective_floats(T, len(lens), C, N) > 0) == cut
    x, z, bc = (torch.randn(T, n, generator=g).to(dt) for n in (C, C, 2 * N))
    dtp, dtb, skip = torch.randn(T, C, generator=g), torch.randn(C, generator=g) - 2, torch.randn(C, generator=g)
    a_log = torch.randn(C, N, generator=g)
    a_log[:, 0], a_log[0] = -30.0, 40.0                 # states that keep everything, a channel that forgets everything
    S0 = torch.randn(len(lens), C, N, generator=g)
    res = []
    for dev in ("cpu", "cuda"):
        st, sb = _batch({"S": ((C, N), "f32")}, lens, starts, dev)
        st["S"].copy_(S0)
        p = [t.to(dev) for t in (x, dtp, dtb, bc[:, :N], bc[:, N:], a_log, skip, z)]
        y = R.selective_scan(*p, st["S"], sb)
        res.append((y.float(), st["S"]))
    # (bf16 outputs: both sides round, to at most one unit of 2^-8 apart)
    (y1, s1), (y0, s0) = res[1], res[0]
    _close((s1,), (s0,), ("state",))
    tol = TOL if dt == torch.float32 else 2.0 ** -8
    assert torch.isfinite(y1).all() and (y1.cpu() - y0).norm() <= tol * y0.norm()


@pytest.mark.gpu
@pytest.mark.parametrize("lens,starts", [([64], [0]), ([63, 65, 16, 1, 129], [0, 3, 0, 0, 7]), ([17, 48, 80], [5, 0, 0]), ([400], [9])])
@pytest.mark.parametrize("C,N,dt", [(16, 16, torch.bfloat16), (129, 16, torch.float32), (130, 9, torch.bfloat16), (40, 13, torch.float32)])
def test_selective_with_a_state_per_lane(lens, starts, C, N, dt):
    """Edges of the 16 and 64 tokens and 16 channels of a block, padded states, column slices, an idle sequence, decays of 0 and 1."""
    from llm_in_practise_amd.ops._native import native_seq
    g = torch.Generator().manual_seed(C + N)
    T, live = sum(lens), [int(b != 2) for b in range(len(lens))]
    assert native_seq().selective_rows(T, len(lens), C, N) or T < 32 * len(lens)
    P, bc = torch.randn(T, 2 * C + 1, generator=g).to(dt), torch.randn(T, 2 * N + 3, generator=g).to(dt)
    dtp, dtb, skip = torch.randn(T, C, generator=g), torch.randn(C, generator=g) - 2, torch.randn(C, generator=g)
    a_log = torch.randn(C, N, generator=g)
    a_log[:, 0], a_log[0] = -30.0, 100.0                # (the second: an infinite rate, a channel that forgets everything)
    S0 = torch.randn(len(lens), C, N, generator=g)
    res = []
    for dev in ("cpu", "cuda"):
        st, sb = _batch({"S": ((C, N), "f32")}, lens, starts, dev, live)
        st["S"].copy_(S0)
        p, q, out = P.to(dev), bc.to(dev), torch.zeros(T, C + 3, dtype=dt, device=dev)
        R.selective_scan(p[:, :C], *[t.to(dev) for t in (dtp, dtb)], q[:, 1:N + 1], q[:, N + 2:2 * N + 2], a_log.to(dev), skip.to(dev),
                         p[:, C + 1:], st["S"], sb, out[:, 1:C + 1], 0.5)
        tok = torch.cat([torch.full((n,), bool(on)) for n, on in zip(lens, live)])
        res.append((out[tok.to(dev)].float().cpu(), st["S"].cpu()))
    (y1, s1), (y0, s0) = res[1], res[0]
    _close((s1,), (s0,), ("state",))
    if len(lens) > 2:
        assert torch.equal(s1[len(lens) - 3], S0[len(lens) - 3])        # (slots run backwards)
    tol = TOL if dt == torch.float32 else 2.0 ** -8      # (bf16 outputs: both sides round, to at most one unit of 2^-8 apart)
    assert torch.isfinite(y1).all() and (y1 - y0).norm() <= tol * y0.norm()
    assert (y1[:, 0] == 0).all() and (y1[:, C + 1:] == 0).all()


@pytest.mark.gpu
@pytest.mark.parametrize("which", ["x", "z", "b", "c"])
@pytest.mark.parametrize("form", ["one", "overlapping", "far"])
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_selective_rows_of_any_stride(which, form, dt):
    """One row for all tokens, rows that share elements, rows too far apart for 32-bit offsets into 64 of them."""
    from llm_in_practise_amd.ops._native import native_seq
    lens, C, N = [70, 33], 40, 16
    g = torch.Generator().manual_seed(len(which + form))
    T, w = sum(lens), C if which in "xz" else N
    p = {k: torch.randn(T, n, generator=g).to(dt) for k, n in (("x", C), ("z", C), ("b", N), ("c", N))}
    flat, ld = torch.randn(T + w, generator=g).to(dt), {"one": 0, "overlapping": 1}.get(form, (1 << 32) // (64 * p["x"].element_size()) + 8)
    dtp, dtb, skip, a_log = (torch.randn(*s, generator=g) for s in ((T, C), (C,), (C,), (C, N)))
    assert native_seq().selective_rows(T, 2, C, N)
    res = []
    for dev in ("cpu", "cuda"):
        st, sb = _batch({"S": ((C, N), "f32")}, lens, [0, 3], dev)
        st["S"].fill_(0.5)
        q = {k: t.to(dev) for k, t in p.items()}
        if form != "far":
            q[which] = flat.to(dev).as_strided((T, w), (ld, 1))
        elif dev == "cuda":
            q[which] = torch.empty((T - 1) * ld + w, dtype=dt, device=dev).as_strided((T, w), (ld, 1)).copy_(p[which])
        y = R.selective_scan(q["x"], dtp.to(dev), dtb.to(dev), q["b"], q["c"], a_log.to(dev), skip.to(dev), q["z"], st["S"], sb)
        res.append((y.float().cpu(), st["S"].cpu()))
    (y1, s1), (y0, s0) = res[1], res[0]
    _close((s1,), (s0,), ("state",))
    tol = TOL if dt == torch.float32 else 2.0 ** -8      # (bf16 outputs: both sides round, to at most one unit of 2^-8 apart)
    assert torch.isfinite(y1).all() and (y1 - y0).norm() <= tol * y0.norm()


@pytest.mark.gpu
@pytest.mark.parametrize("name,value", [("x", float("inf")), ("b", float("nan")), ("b", float("inf")), ("c", float("nan")), ("dt", float("nan"))])
@pytest.mark.parametrize("t", [40, 102, 203])
def test_selective_token_that_is_no_number(name, value, t):
    """At the last token of a sequence too (102, 203): what stands behind it in a block of 64 changes nothing."""
    lens, C, N = [103, 101], 40, 16
    g = torch.Generator().manual_seed(t)
    T = sum(lens)
    inputs = {n: torch.randn(T, w, generator=g).cuda() for n, w in (("x", C), ("dt", C), ("b", N), ("c", N), ("z", C))}
    dtb, a_log, skip = (torch.randn(*s, generator=g).cuda() for s in ((C,), (C, N), (C,)))

    def run(x):
        st, sb = _batch({"S": ((C, N), "f32")}, lens, [0, 5], "cuda")
        st["S"].fill_(0.5)
        y = R.selective_scan(x["x"], x["dt"], dtb, x["b"], x["c"], a_log, skip, x["z"], st["S"], sb)
        run.state = st["S"]
        return (y,)
    _planted(run, inputs, name, t, 1, value, lens)
    if name == "b" and value == float("inf"):
        assert (run.state[0 if t >= 103 else 1, :, 1].abs() == value).all()      # an infinite state is not NaN


@pytest.mark.gpu
@pytest.mark.parametrize("T,B,C,N,rows", [
    (256, 1, 4096, 16, True), (4096, 1, 4096, 16, True), (4096, 1, 2048, 16, False), (3385, 2, 4096, 16, True), (3500, 2, 2048, 16, False),
    (2048, 4, 4096, 16, True), (384, 12, 4096, 16, True), (256, 16, 4096, 16, False), (8192, 16, 8192, 16, False), (1000, 2, 4096, 8, False),
    (1000, 2, 4096, 17, False), (1, 1, 4096, 16, False), (9000, 1, 4096, 16, True), (20000, 1, 4096, 16, True), (9000, 1, 4112, 16, False),
    (1024, 1, 5120, 16, True), (4096, 1, 5120, 16, False), (20000, 1, 5632, 16, False), (9000, 1, 8192, 16, True), (9000, 1, 3072, 16, False),
    (20000, 1, 8208, 16, True), (1024, 1, 1024, 16, False), (2048, 1, 2560, 16, False), (2048, 1, 4112, 16, True), (3072, 1, 4608, 16, False)])
def test_selective_takes_a_state_per_lane_where_that_is_faster(T, B, C, N, rows):
    from llm_in_practise_amd.ops._native import native_seq
    assert native_seq().selective_rows(T, B, C, N) == rows


@pytest.mark.gpu
@pytest.mark.parametrize("T,B,C,N,cut", [
    (4096, 1, 2048, 16, True), (9000, 1, 4112, 16, True), (2048, 1, 4096, 16, False), (6400, 16, 4096, 16, False), (2048, 1, 8192, 32, True),
    (6400, 16, 1024, 32, False), (2048, 1, 4096, 64, True), (2048, 1, 8192, 64, False), (2048, 1, 4096, 128, True),
    (4096, 4, 4096, 128, False), (2048, 1, 1024, 256, True), (6400, 16, 1024, 256, False), (4096, 8, 1024, 256, False),
    (256, 1, 8192, 128, False), (256, 1, 4096, 256, False), (300, 1, 65536, 256, False)])
def test_selective_is_cut_only_where_it_is_not_slower(T, B, C, N, cut):
    """Timed shapes on both sides of the rule: the work of a token grows with its states, what a cut saves does not."""
    from llm_in_practise_amd.ops._native import native_seq
    assert (native_seq().selective_floats(T, B, C, N) > 0) == cut


@pytest.mark.gpu
@pytest.mark.parametrize("N", [17, 32, 64, 100, 256])
def test_selective_cut_with_many_states(N):
    lens, C = [700, 1100], 256
    g = torch.Generator().manual_seed(N)
    T = sum(lens)
    x, z, bc = (torch.randn(T, n, generator=g) for n in (C, C, 2 * N))
    dtp, dtb, skip = torch.randn(T, C, generator=g), torch.randn(C, generator=g) - 2, torch.randn(C, generator=g)
    a_log = torch.randn(C, N, generator=g)
    res = []
    for dev in ("cpu", "cuda"):
        st, sb = _batch({"S": ((C, N), "f32")}, lens, [0, 3], dev)
        st["S"].fill_(0.25)
        p = [t.to(dev) for t in (x, dtp, dtb, bc[:, :N], bc[:, N:], a_log, skip, z)]
        res.append((R.selective_scan(*p, st["S"], sb), st["S"]))
    from llm_in_practise_amd.ops._native import native_seq
    assert native_seq().selective_floats(T, len(lens), C, N) > 0
    _close(res[1], res[0], ("y", "state"))


@pytest.mark.gpu
@pytest.mark.parametrize("op,L,B,H,dk,dv,blocked", [
    ("ssd", 64, 1, 64, 128, 64, True), ("ssd", 63, 1, 64, 128, 64, False), ("ssd", 128, 64, 16, 64, 64, False),
    ("ssd", 192, 64, 16, 64, 64, True), ("ssd", 64, 64, 16, 128, 64, True), ("ssd", 64, 1, 8, 64, 512, False),
    ("ssd", 192, 1, 8, 64, 512, True), ("ssd", 192, 64, 16, 32, 128, False), ("mlstm", 64, 16, 8, 64, 96, True),
    ("mlstm", 72, 8, 8, 128, 192, False), ("mlstm", 80, 8, 8, 128, 192, True), ("mlstm", 80, 64, 4, 64, 128, False),
    ("delta", 32, 1, 8, 128, 128, True), ("delta", 32, 16, 16, 64, 64, False), ("delta", 1024, 64, 16, 64, 64, False),
    ("delta", 1024, 64, 16, 64, 128, False), ("delta", 96, 16, 16, 64, 128, True), ("delta", 512, 64, 16, 128, 32, False),
    ("delta", 128, 16, 16, 128, 32, True), ("delta", 64, 64, 16, 128, 128, True), ("gla", 40, 1, 8, 128, 128, True),
    ("gla", 48, 1, 8, 64, 128, False), ("gla", 64, 4, 16, 64, 128, True), ("gla", 1024, 16, 16, 256, 64, False),
    ("gla", 128, 16, 16, 64, 32, True), ("gla", 256, 24, 16, 64, 128, False)])
def test_chunks_and_blocks_only_where_they_are_not_slower(op, L, B, H, dk, dv, blocked):
    """Timed shapes on both sides of the choice between chunks or blocks and the token-by-token forms."""
    from llm_in_practise_amd.ops._native import native_seq
    assert (native_seq().scan_floats(op, L * B, B, H, dk, dv) > 0) == blocked


def _scans(lens, starts, g):
    """The five scans over one packed step: name -> (run() -> outputs and states, floats of workspace per slot, tokens of a slot)."""
    T, B = sum(lens), len(lens)

    def rand(*s, dt=torch.float32):
        return torch.randn(*s, generator=g).to(dt).cuda()
    H, dk, dv = 3, 64, 32
    bf = torch.bfloat16
    q, k, v = rand(T, H * dk, dt=bf), rand(T, H * dk, dt=bf), rand(T, H * dv, dt=bf)
    dt, dtb, a_log, skip = rand(T, H, dt=bf), rand(H), rand(H), rand(H)
    i, f = 4 * rand(T, H), 3 * rand(T, H)
    decay, z, zb = torch.rand(T, H * dk, generator=g).cuda() ** 0.2, 3 * rand(T, H * dk), rand(H * dk)
    kn = torch.nn.functional.normalize(k.float().view(T, H, dk), dim=-1).view(T, -1).to(bf)
    C, N = 64, 16
    sel = [rand(T, C), rand(T, C), rand(C) - 2, rand(T, N), rand(T, N), rand(C, N), rand(C), rand(T, C)]
    mat = {"S": ((H, dv, dk), "f32")}

    def go(spec, fn):
        def run():
            st, sb = _batch(spec, lens, starts, "cuda")
            for s in st.values():
                s.fill_(0.25)
            out = fn(st, sb)
            return [*(out if isinstance(out, (tuple, list)) else [out]), *st.values()]
        return run
    return {
        "ssd": (go(mat, lambda st, sb: R.ssd_scan(q, k, v, dt, dtb, a_log, skip, st["S"], H, H, sb)), H * (6 + dk * (dv + 1)), 128),
        "mlstm": (go({**mat, "N": ((H, dk), "f32"), "M": ((H,), "f32")}, lambda st, sb: R.mlstm_scan(
            q, k, v, i, f, dtb, dtb + 3, 15.0, dk ** -0.5, st["S"], st["N"], st["M"], H, sb)), H * (6 + dk * (dv + 1)), 128),
        "delta": (go(mat, lambda st, sb: R.gated_delta_scan(q, kn, v, decay, i, st["S"], H, H, sb)), H * (49 * dk + 516), 16),
        "gla": (go(mat, lambda st, sb: R.gated_linear_scan(q, k, v, z, zb, 16.0, dk ** -0.5, st["S"], H, sb)),
                H * (49 * dk + 516), 16),
        "selective": (go({"S": ((C, N), "f32")}, lambda st, sb: R.selective_scan(*sel, st["S"], sb)), C * (N + 1), 32),
    }


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["ssd", "mlstm", "delta", "gla", "selective"])
@pytest.mark.parametrize("lens,starts", [([2100], [0]), ([1500, 1, 900, 640], [0, 0, 3, 512])])
@pytest.mark.parametrize("count", [0, 1, 5, 100])
def test_scans_in_windows_of_a_bounded_workspace(monkeypatch, name, lens, starts, count):
    """Room for `count` slots a sequence: the same outputs and states window after window (or token by token, with no room or too
    many windows), and no more memory than allowed."""
    import functools
    from llm_in_practise_amd.ops import _native
    run, per, _ = _scans(lens, starts, torch.Generator().manual_seed(len(lens)))[name]
    want = run()
    seq, most = _native.native_seq(), count * per * len(lens) + 8
    asked = {"ssd": "ssd_scan", "mlstm": "mlstm_scan", "delta": "delta_scan", "gla": "gated_linear_scan", "selective": "selective_scan"}

    class Bounded:
        def __getattr__(self, a):
            return functools.partial(getattr(seq, a), most=most) if a == asked[name] else getattr(seq, a)
    monkeypatch.setattr(R, "native_seq", Bounded)
    torch.cuda.synchronize()
    base = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    got = run()
    held = 4 * sum(t.numel() for t in got) + 4 * 4 * sum(lens)      # outputs, states, descriptors (rounded up to 512 bytes each)
    assert torch.cuda.max_memory_allocated() - base <= held + 4 * most + 512 * 32
    _close(got, want, [str(j) for j in range(len(got))])


@pytest.mark.gpu
@pytest.mark.parametrize("op", ["ssd", "mlstm", "delta", "gla"])
@pytest.mark.parametrize("which", ["q", "k", "v", "S", "row"])
def test_rows_that_wide_loads_cannot_take(op, which):
    """One operand a single element off, or rows of odd length: the same outputs and states as for aligned copies."""
    lens, H, dk, dv, bf = [200, 90], 2, 64, 32, torch.bfloat16
    g = torch.Generator().manual_seed(len(op))
    T = sum(lens)
    base = {n: torch.randn(T, H * w, generator=g).to(bf).cuda() for n, w in (("q", dk), ("k", dk), ("v", dv))}
    if op == "delta":
        base["k"] = torch.nn.functional.normalize(base["k"].float().view(T, H, dk), dim=-1).view(T, -1).to(bf)
    i, f = torch.randn(T, H, generator=g).cuda(), torch.randn(T, H, generator=g).cuda()
    decay, z, zb = torch.rand(T, H * dk, generator=g).cuda() ** 0.2, torch.randn(T, H * dk, generator=g).cuda(), torch.zeros(H * dk).cuda()
    b = torch.randn(H, generator=g).cuda()

    def off(t, by):                                     # the same values, `by` elements behind an aligned address
        return torch.cat([t.new_zeros(by), t.reshape(-1)])[by:].view(t.shape)

    def run(odd):
        x = dict(base)
        if odd and which == "row":
            x = {n: torch.cat([t, t.new_zeros(T, 1)], 1)[:, :-1] for n, t in x.items()}
        elif odd and which in x:
            x[which] = off(x[which], 1)
        spec = {"S": ((H, dv, dk), "f32")} | ({"N": ((H, dk), "f32"), "M": ((H,), "f32")} if op == "mlstm" else {})
        st, sb = _batch(spec, lens, [0, 3], "cuda")
        for s in st.values():
            s.fill_(0.5)
        if odd and which == "S":
            st["S"] = off(st["S"], 1)
        if op == "ssd":
            o = R.ssd_scan(x["q"], x["k"], x["v"], i.to(bf), b, b, b, st["S"], H, H, sb)
        elif op == "mlstm":
            o = R.mlstm_scan(x["q"], x["k"], x["v"], i, f, b, b + 3, 15.0, dk ** -0.5, st["S"], st["N"], st["M"], H, sb)
        elif op == "delta":
            o = R.gated_delta_scan(x["q"], x["k"], x["v"], decay, i, st["S"], H, H, sb)
        else:
            o = R.gated_linear_scan(x["q"], x["k"], x["v"], z, zb, 16.0, dk ** -0.5, st["S"], H, sb)
        return [*(o if isinstance(o, (tuple, list)) else [o]), *st.values()]
    got, want = run(True), run(False)
    _close(got, want, [str(j) for j in range(len(got))])


@pytest.mark.gpu
@pytest.mark.parametrize("op", ["ssd", "mlstm"])
@pytest.mark.parametrize("lens,H,dk,dv", [([2049, 2175], 48, 128, 64), ([385, 700, 513], 40, 64, 36), ([640, 129, 511], 32, 32, 100),
                                          ([4100], 24, 96, 68), ([1280, 256], 16, 128, 192)])
@pytest.mark.parametrize("bad", [None, 5, 300])
def test_runs_of_chunks(op, lens, H, dk, dv, bad):
    """Runs of two and four chunks, whole and cut off in each of them, against the token-by-token kernel, in one window and in several; with
    an infinite value in the first and in a later chunk: it reaches its own column of the outputs behind it and nothing else."""
    from llm_in_practise_amd.ops._native import native_seq
    ext = native_seq()
    g = torch.Generator().manual_seed(dk + dv)
    T, B = sum(lens), len(lens)
    assert -(-T // 128) * H * -(-dv // 64) >= 512 and T // B >= 384

    def rand(*s, dt=torch.float32):
        return torch.randn(*s, generator=g).to(dt).cuda()
    q, k, v = (rand(T, H * n, dt=torch.bfloat16) for n in (dk, dk, dv))
    if bad is not None:
        v[bad, dv + 1] = float("inf")                   # head 1, column 1 of the first sequence
    i, f, a, b, skip = rand(T, H), rand(T, H), rand(H), rand(H), rand(H)
    S0, N0 = rand(B, H, dv, dk), rand(B, H, dk)
    room = ext.scan_floats(op, T, B, H, dk, dv)
    assert 0 < ext.scan_floats(op, T, B, H, dk, dv, room // 2) <= room // 2        # (several windows)
    res = []
    for most in (room, room // 2, 0):
        st, sb = _batch({"S": ((H, dv, dk), "f32"), "N": ((H, dk), "f32"), "M": ((H,), "f32")}, lens, [7 * (j % 2) for j in range(B)], "cuda")
        st["S"].copy_(S0)
        st["N"].copy_(N0)
        st["M"].fill_(0.5)
        if op == "ssd":
            out = [ext.ssd_scan(q, k, v, i.bfloat16(), a - 3, b, skip, st["S"], H, H, sb.desc, None, most=most).view(T, H, dv)]
        else:
            out = ext.mlstm_scan(q, k, v, i, f, a, b + 3, 15.0, dk ** -0.5, st["S"], st["N"], st["M"], H, sb.desc, None, most=most)
        res.append([*out, st["S"], st["N"], st["M"]])
    for got in res[:2]:
        for x, y in zip(got, res[2]):
            x, y = x.double(), y.double()
            assert torch.equal(torch.isfinite(x), torch.isfinite(y))
            x, y = (torch.nan_to_num(t, 0.0, 0.0, 0.0) for t in (x, y))
            assert (x - y).norm() <= TOL * y.norm(), ((x - y).norm() / y.norm()).item()


@pytest.mark.gpu
@pytest.mark.parametrize("op", ["ssd", "mlstm"])
@pytest.mark.parametrize("lens,H,dk,dv,cols", [([65, 193, 1, 128, 64], 4, 128, 36, 16), ([129, 255], 65, 128, 32, 32), ([384, 320], 33, 128, 100, 48),
                                               ([191, 66, 200], 4, 64, 20, 16), ([130, 90], 90, 64, 24, 32), ([64, 257], 100, 64, 44, 48),
                                               ([300, 128, 63], 80, 64, 52, 64)])
@pytest.mark.parametrize("bad", [None, 40, 64])
@pytest.mark.parametrize("whole", [True, False])
def test_walk_with_the_state_at_hand(op, lens, H, dk, dv, cols, bad, whole):
    """Pieces of 64 tokens cut off everywhere, every width of a block and columns that end inside it, against the token-by-token kernel: in one
    window and in several, with an idle sequence, with an infinite value in a first and in a second piece."""
    from llm_in_practise_amd.ops._native import native_seq
    ext = native_seq()
    g = torch.Generator().manual_seed(dk + dv)
    T, B, longest = sum(lens), len(lens), max(lens)
    assert ext.scan_walk(T, B, H, dk, dv, longest) == cols

    def rand(*s, dt=torch.float32):
        return torch.randn(*s, generator=g).to(dt).cuda()
    q, k, v = (rand(T, H * n, dt=torch.bfloat16) for n in (dk, dk, dv))
    if bad is not None:
        v[bad, dv + 1] = float("inf")                   # head 1, column 1 of the first sequence
    i, f, a, b, skip = 3 * rand(T, H), 3 * rand(T, H), rand(H), rand(H), rand(H)
    S0, N0 = rand(B, H, dv, dk), rand(B, H, dk)
    live = [int(j != 1) for j in range(B)]
    tok = torch.repeat_interleave(torch.tensor(live, dtype=torch.bool), torch.tensor(lens)).cuda()
    room = ext.scan_floats(op, T, B, H, dk, dv, longest=longest)
    res = []
    for most in (room if whole else B * H * 1040, 0):     # (two pieces a sequence at a time; too many windows: token by token)
        st, sb = _batch({"S": ((H, dv, dk), "f32"), "N": ((H, dk), "f32"), "M": ((H,), "f32")}, lens, [7 * (j % 2) for j in range(B)], "cuda", live)
        st["S"].copy_(S0)
        st["N"].copy_(N0)
        st["M"].fill_(0.5)
        if op == "ssd":
            out = [ext.ssd_scan(q, k, v, i.bfloat16(), a - 3, b, skip, st["S"], H, H, sb.desc, sb.live, most=most, longest=longest).view(T, H, dv)]
        else:
            out = ext.mlstm_scan(q, k, v, i, f, a, b + 3, 15.0, dk ** -0.5, st["S"], st["N"], st["M"], H, sb.desc, sb.live, most=most,
                                 longest=longest)
        res.append([*(x[tok] for x in out), st["S"], st["N"], st["M"]])
    for x, y in zip(*res):
        x, y = x.double(), y.double()
        assert torch.equal(torch.isfinite(x), torch.isfinite(y))
        x, y = (torch.nan_to_num(t, 0.0, 0.0, 0.0) for t in (x, y))
        assert (x - y).norm() <= TOL * y.norm(), ((x - y).norm() / y.norm()).item()


@pytest.mark.gpu
@pytest.mark.parametrize("cells", [1, 2, 13 * 33, 64 * 8])
def test_walk_tables_where_vector_loads_take_them(cells):
    """Rows of 8 floats and pairs of doubles at multiples of 16 bytes, doubles at multiples of 8, each behind the one before, odd numbers of cells too."""
    from llm_in_practise_amd.ops._native import native_seq
    tab, loc, m0, end = native_seq().walk_places(cells)
    assert tab % 4 == 0 and loc % 4 == 0 and m0 % 2 == 0
    spans = sorted([(tab, 64 * 8), (loc, 2 * 2), (m0, 2)])
    assert all(a + n * cells <= b for (a, n), b in zip(spans, [spans[1][0], spans[2][0], end]))


@pytest.mark.gpu
@pytest.mark.parametrize("T,B,H,dk,dv,longest,walks", [
    (12, 1, 8, 128, 192, 12, False), (20, 1, 8, 128, 192, 20, True), (63, 1, 8, 128, 192, 0, False), (160, 8, 8, 128, 192, 20, True),
    (240, 12, 8, 128, 192, 20, False), (756, 12, 8, 128, 192, 63, True), (768, 32, 32, 64, 96, 24, False), (192, 8, 8, 64, 96, 24, True),
    (63, 1, 8, 96, 96, 63, False)])
def test_short_mlstm_prompts_walk_where_it_is_not_slower(T, B, H, dk, dv, longest, walks):
    """Timed shapes on both sides of the choice between the walk and tokens one by one; lengths that are not known, keys that have no walk; and
    the state space, which has none of it."""
    from llm_in_practise_amd.ops._native import native_seq
    ext = native_seq()
    assert (ext.scan_walk(T, B, H, dk, dv, longest, "mlstm") > 0) == (ext.scan_floats("mlstm", T, B, H, dk, dv, longest=longest) > 0) == walks
    assert ext.scan_walk(T, B, H, dk, dv, longest) == ext.scan_floats("ssd", T, B, H, dk, dv, longest=longest) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("lens,H,dk,dv", [([20], 2, 128, 192), ([63], 3, 64, 96), ([48, 1, 30, 17, 63], 4, 128, 64), ([40, 33], 2, 64, 36)])
def test_short_mlstm_prompts_walk_as_token_by_token(lens, H, dk, dv):
    from llm_in_practise_amd.ops._native import native_seq
    ext = native_seq()
    g = torch.Generator().manual_seed(dk + dv)
    T, B, longest = sum(lens), len(lens), max(lens)
    assert ext.scan_walk(T, B, H, dk, dv, longest, "mlstm") > 0

    def rand(*s, dt=torch.float32):
        return torch.randn(*s, generator=g).to(dt).cuda()
    q, k, v = (rand(T, H * n, dt=torch.bfloat16) for n in (dk, dk, dv))
    i, f, a, b = 3 * rand(T, H), 3 * rand(T, H), rand(H), rand(H)
    S0, N0, res = rand(B, H, dv, dk), rand(B, H, dk), []
    for most in (1 << 28, 0):                             # (no room: token by token)
        st, sb = _batch({"S": ((H, dv, dk), "f32"), "N": ((H, dk), "f32"), "M": ((H,), "f32")}, lens, [7 * (j % 2) for j in range(B)], "cuda")
        st["S"].copy_(S0)
        st["N"].copy_(N0)
        st["M"].fill_(0.5)
        out = ext.mlstm_scan(q, k, v, i, f, a, b + 3, 15.0, dk ** -0.5, st["S"], st["N"], st["M"], H, sb.desc, sb.live, most=most, longest=longest)
        res.append([*out, st["S"], st["N"], st["M"]])
    _close(res[0], res[1], ("o", "den", "floor", "S", "N", "M"))


@pytest.mark.gpu
@pytest.mark.parametrize("T,B,H,dk,dv,longest,cols", [
    (4093, 1, 64, 128, 64, 4093, 0), (1000, 1, 64, 128, 64, 1000, 16), (2000, 4, 64, 128, 64, 512, 32), (7040, 8, 8, 128, 192, 1024, 48),
    (512, 1, 8, 64, 96, 512, 16), (2048, 1, 8, 64, 96, 2048, 0), (4096, 8, 8, 64, 96, 512, 32), (9060, 12, 8, 64, 96, 9000 - 640, 0),
    (9060, 12, 8, 64, 96, 0, 0), (512, 1, 8, 96, 96, 512, 0)])
def test_walk_only_where_it_is_not_slower(T, B, H, dk, dv, longest, cols):
    """Timed shapes on both sides of the choice between chunks and the walk; one long sequence among short ones, known or not, is not walked."""
    from llm_in_practise_amd.ops._native import native_seq
    assert native_seq().scan_walk(T, B, H, dk, dv, longest) == cols


@pytest.mark.gpu
@pytest.mark.parametrize("op,T,B,H,dk,dv,longest,cols", [
    ("mlstm", 2187, 20, 8, 64, 192, 1126, 0), ("mlstm", 7246, 3, 64, 128, 16, 6732, 0), ("mlstm", 15966, 20, 8, 64, 160, 2517, 0),
    ("ssd", 7884, 16, 32, 64, 96, 7825, 0), ("ssd", 4033, 20, 32, 64, 128, 2724, 0), ("ssd", 12879, 16, 8, 64, 192, 2523, 0),
    ("ssd", 21948, 6, 16, 128, 64, 3658, 32), ("ssd", 2021, 20, 16, 64, 128, 151, 64), ("ssd", 22850, 10, 16, 64, 64, 2285, 64),
    ("mlstm", 7040, 8, 8, 128, 192, 1024, 48), ("mlstm", 1218, 24, 4, 64, 160, 485, 32), ("mlstm", 4480, 64, 24, 64, 16, 2075, 16)])
def test_walk_of_prompts_of_uneven_lengths(op, T, B, H, dk, dv, longest, cols):
    """Timed shapes: more blocks than CUs and a longest sequence far above the mean are left to the chunks (in us, chunks / walk: 43 / 51, 179 / 233, 110 / 160,
    139 / 201, 95 / 122 and 87 / 123), rounds of like blocks are not (150 / 135, 40 / 38, 98 / 93), nor one round (89 / 52), nor what goes token by token
    otherwise (194 / 25, 1073 / 56)."""
    from llm_in_practise_amd.ops._native import native_seq
    assert native_seq().scan_walk(T, B, H, dk, dv, longest, op) == cols


@pytest.mark.gpu
@pytest.mark.parametrize("op", ["ssd", "mlstm", "delta", "delta-16", "gla", "selective"])
@pytest.mark.parametrize("B", [64, 65, 129, 200])
def test_pieces_of_more_sequences_than_a_wave_has_lanes(op, B):
    """Ragged sequences, some of one token, some idle: every block finds the sequence of its piece; against the token-by-token kernels."""
    from llm_in_practise_amd.ops._native import native_seq
    ext = native_seq()
    g = torch.Generator().manual_seed(B)
    lens = [1 if b % 9 == 4 else 250 + 37 * b % 411 for b in range(B)]
    T, H, dk, dv, live = sum(lens), 1, 192 if op == "delta-16" else 64, 32, [int(b % 7 != 3) for b in range(B)]

    def rand(*s, dt=torch.float32):
        return torch.randn(*s, generator=g).to(dt).cuda()
    q, k, v = (rand(T, H * n, dt=torch.bfloat16) for n in (dk, dk, dv))
    k = torch.nn.functional.normalize(k.float().view(T, H, dk), dim=-1).view(T, -1).bfloat16()
    i, f, a, b, z, zb = rand(T, H), rand(T, H), rand(H), rand(H), rand(T, H * dk), rand(H * dk)
    C, N = 16, 32
    sel = [rand(T, C), rand(T, C), rand(C) - 2, rand(T, N), rand(T, N), rand(C, N), rand(C), rand(T, C)]
    if op == "selective":
        assert ext.selective_floats(T, B, C, N) > 0
    elif op.startswith("delta"):
        assert ext.delta_block(T, B, H, dk, dv) == (16 if op == "delta-16" else 32)
    else:
        assert ext.scan_floats(op, T, B, H, dk, dv) > 0
    tok = torch.repeat_interleave(torch.tensor(live, dtype=torch.bool), torch.tensor(lens)).cuda()
    res = []
    for most in (1 << 28, 0):
        spec = {"S": ((C, N) if op == "selective" else (H, dv, dk), "f32"), "N": ((H, dk), "f32"), "M": ((H,), "f32")}
        st, sb = _batch(spec, lens, [3 * (j % 2) for j in range(B)], "cuda", live)
        for s in st.values():
            s.fill_(0.25)
        on = sb.live
        if op == "ssd":
            out = [ext.ssd_scan(q, k, v, i.bfloat16(), a - 3, b, a, st["S"], H, H, sb.desc, on, most=most)]
        elif op == "mlstm":
            out = ext.mlstm_scan(q, k, v, i, f, a, b + 3, 15.0, dk ** -0.5, st["S"], st["N"], st["M"], H, sb.desc, on, most=most)
        elif op == "gla":
            out = [ext.gated_linear_scan(q, k, v, z, zb, 16.0, dk ** -0.5, st["S"], H, sb.desc, on, most=most)]
        elif op == "selective":
            out = [ext.selective_scan(*sel, st["S"], sb.desc, on, None, 1.0, most=most)]
        else:
            out = [ext.delta_scan(q, k, v, torch.sigmoid(z + 3), i, st["S"], H, H, sb.desc, on, most=most)]
        res.append([*(t[tok] for t in out), *st.values()])
    _close(res[0], res[1], [str(j) for j in range(len(res[0]))])

"""The recurrences over portions of prompts at the sizes where their chunks and tiles end: the matrix memory's chunks side by
side on the matrix cores, the selective scan's pieces, against the recurrences token by token in 64 bits."""
import types

import pytest
import torch

pytestmark = pytest.mark.gpu


def ops():
    from lmsf_amd.ops.hip_ops import HipOps
    return HipOps()


def batch(lens):
    starts = [sum(lens[:i]) for i in range(len(lens) + 1)]
    return types.SimpleNamespace(
        aux={}, host_seg_lens=list(lens), host_seg_starts=starts, n_tokens=starts[-1], n_segments=len(lens), replayed=False,
        all_single=False, seg_starts=torch.tensor(starts, dtype=torch.int32, device="cuda"),
        state_slots=torch.arange(len(lens), dtype=torch.int32, device="cuda").flip(0),
        seg_of_token=torch.repeat_interleave(torch.arange(len(lens), dtype=torch.int32), torch.tensor(lens)).cuda())


def memory_by_tokens(q, k, v, gates, og, w, state, lens, H, d, dv, scale, cap, eps):
    """[out, state] in float64; state as [slots, H, d, dv + 1] and the running maximum [slots, H]."""
    S, m = state
    outs, at = [], 0
    for s, n in enumerate(lens):
        slot = len(lens) - 1 - s
        for t in range(at, at + n):
            i, f = cap * torch.tanh(gates[t, :H] / cap), torch.nn.functional.logsigmoid(cap * torch.tanh(gates[t, H:] / cap))
            now = torch.maximum(f + m[slot], i)
            one = torch.cat([v[t].view(H, dv), torch.ones(H, 1, dtype=torch.float64)], 1)
            S[slot] = torch.exp(f + m[slot] - now)[:, None, None] * S[slot] + \
                torch.exp(i - now)[:, None, None] * k[t].view(H, d)[:, :, None] * one[:, None]
            m[slot] = now
            o = (S[slot] * (q[t].view(H, d) * scale)[:, :, None]).sum(1)
            o = o[:, :dv] / (torch.maximum(o[:, dv].abs(), torch.exp(-now)) + 1e-6)[:, None]
            outs.append((o / torch.sqrt((o * o).mean(1, keepdim=True) + eps)).reshape(-1) * w * torch.sigmoid(og[t]))
        at += n
    return torch.stack(outs)


# heads of 16 and 32 entries' multiples and not, values that end inside a block of 16 and of 64 columns, segments of a tile's, a
# chunk's and several chunks' tokens and one more or less, a short one beside them; 200 and 260: more rows of S_0 than a
# wave holds at a time, and smaller chunks; 500 and 700: chunks of 16 where the other form's have 8 and 4
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,d,dv,lens", [(2, 128, 128, (64, 65, 3)), (3, 40, 70, (100, 127)), (1, 17, 5, (65, 192)), (2, 64, 64, (128, 16)),
                                         (2, 200, 24, (33, 47)), (1, 260, 136, (40,)), (2, 128, 65, (32, 33, 1)),
                                         (1, 500, 40, (33, 3)), (1, 700, 20, (16, 17))])
def test_matrix_memory_side_by_side(H, d, dv, lens, dtype):
    o, g = ops(), torch.Generator().manual_seed(d + dv)
    N, scale, cap, eps = sum(lens), d ** -0.5, 15.0, 1e-5
    buf = torch.randn(N, H * (2 * d + 2 * dv), generator=g).to(dtype)
    cut = (H * d, 2 * H * d, 2 * H * d + H * dv)
    gates, w = torch.randn(N, 2 * H, generator=g) * 2, torch.rand(H * dv, generator=g) + 0.5
    floats, copies = o.mlstm_state_floats(H, d, dv), (dv + 31) // 32
    S = torch.randn(len(lens), H, d, dv + 1, generator=g)
    m = torch.rand(len(lens), H, generator=g)
    state = torch.cat([S.reshape(len(lens), -1), m.repeat_interleave(copies, 1)], 1)
    assert state.shape[1] == floats
    dev, st = buf.cuda(), state.cuda()
    q, k, v, og = dev[:, :cut[0]], dev[:, cut[0]:cut[1]], dev[:, cut[1]:cut[2]], dev[:, cut[2]:]
    b = batch(lens)
    o.matrix_memory_parallel_min_tokens = 1
    out = o.mlstm(q, k, v, gates.cuda(), og, w.cuda(), st, b, H, d, dv, scale, cap, eps)
    assert any(key[0] == "mlstm_chunks" for key in b.aux)
    x = buf.double()
    S64, m64 = S.double(), m.double()
    ref = memory_by_tokens(x[:, :cut[0]], x[:, cut[0]:cut[1]], x[:, cut[1]:cut[2]], gates.double(), x[:, cut[2]:], w.double(),
                           (S64, m64), lens, H, d, dv, scale, cap, eps)
    # sums of up to 700 float32 products that partly cancel, against the row's root mean square; a bfloat16 result's own
    # rounding (8 bits) is at most 2^-8 of it
    rel = 2.0 ** -8 if dtype == torch.bfloat16 else 0.0
    err = ((out.cpu().double() - ref).abs() - rel * ref.abs()).amax(1) / ref.pow(2).mean(1).sqrt()
    assert err.max() < 2e-4, float(err.max())
    got = st.cpu().double()
    gs, gm = got[:, :H * d * (dv + 1)].view(S64.shape), got[:, H * d * (dv + 1):].view(len(lens), H, copies)
    assert (gs - S64).abs().max() < 2e-5 * S64.abs().max() and (gm - m64[:, :, None]).abs().max() < 1e-4


# a token in the middle of a tile of 16, at its last place and in a second chunk; columns of two waves and the last one
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("value", [float("inf"), float("nan")])
@pytest.mark.parametrize("token,column", [(5, 0), (47, 37), (70, 69)])
def test_matrix_memory_keeps_a_value_from_earlier_tokens(token, column, value, dtype):
    """A value that is no finite number reaches its own token and later ones of its head, no earlier token and no other head."""
    o, g = ops(), torch.Generator().manual_seed(token)
    H, d, dv, lens = 2, 40, 70, (90, 33)
    N, scale = sum(lens), d ** -0.5
    buf = torch.randn(N, H * (2 * d + 2 * dv), generator=g).to(dtype)
    gates, w = torch.randn(N, 2 * H, generator=g), torch.ones(H * dv)
    state = torch.randn(len(lens), o.mlstm_state_floats(H, d, dv), generator=g)
    cut = (H * d, 2 * H * d, 2 * H * d + H * dv)
    o.matrix_memory_parallel_min_tokens = 1

    def run(buf):
        dev, b = buf.cuda(), batch(lens)
        out = o.mlstm(dev[:, :cut[0]], dev[:, cut[0]:cut[1]], dev[:, cut[1]:cut[2]], gates.cuda(), dev[:, cut[2]:], w.cuda(),
                      state.cuda(), b, H, d, dv, scale, 15.0, 1e-5)
        assert any(key[0] == "mlstm_chunks" for key in b.aux)
        return out.float().cpu()
    plain, odd = run(buf), buf.clone()
    odd[token, cut[1] + column] = value
    out = run(odd)
    assert not out[token:lens[0], :dv].isfinite().all(1).any()
    assert torch.equal(out[:, dv:], plain[:, dv:]) and torch.equal(out[lens[0]:], plain[lens[0]:])
    # (the tile's products are added in another order: 16 float32 sums, and the result's rounding where it has 8 bits)
    rel = 2.0 ** -7 if dtype == torch.bfloat16 else 1e-5
    assert ((out - plain)[:token, :dv].abs() <= rel * plain[:token, :dv].abs() + 1e-5).all()


# one piece and cuts of 16 and of 32 tokens, pieces of fewer than 8, states that the kernel's number of entries is and is not,
# channels that end inside a workgroup; whole segments of more tokens than lie in LDS at a time; states of more entries than a
# lane holds, in chunks of 16 and of 64, and several tiles (of 16 and of 8 tokens) in a chunk of 32
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("inner,n,lens,sizes,chunk", [
    (256, 16, (32,), {}, 64), (300, 16, (65, 7, 1), {}, 16), (260, 5, (97, 130), {}, 16), (512, 32, (33,), {"few_work": 0}, 64),
    (256, 4, (200, 33), {"few_work": 0}, 32), (256, 16, (129, 64), {"few_work": 0}, 32), (302, 8, (70,), {"few_work": 0}, 32),
    (300, 16, (65, 128, 129, 200), {"chunk_tokens": 256, "cut_tokens": 256, "few_work": 0}, 256),
    (48, 33, (65, 33), {}, 16), (48, 33, (65, 130), {"few_work": 0}, 64),
    (40, 72, (150, 31, 1), {"chunk_tokens": 32, "few_work": 0}, 32), (24, 200, (33, 100), {"chunk_tokens": 32, "few_work": 0}, 32)])
def test_selective_scan_in_pieces(inner, n, lens, sizes, chunk, dtype):
    o, g = ops(), torch.Generator().manual_seed(inner + n)
    for name, value in sizes.items():
        setattr(o, "scan_" + name, value)
    N = sum(lens)
    x, z, bc = (torch.randn(N, c, generator=g).to(dtype) for c in (inner, inner, 2 * n))
    dt, al, D = torch.randn(N, inner, generator=g) * 3 - 1, torch.randn(inner, n, generator=g), torch.randn(inner, generator=g)
    st0 = torch.randn(len(lens), inner * n, generator=g)
    st = st0.cuda()
    b = batch(lens)
    y = o.selective_scan(x.cuda(), dt.cuda(), bc.cuda(), 0, n, z.cuda(), al.cuda(), D.cuda(), st, b)
    assert list(b.aux) == [("chunk_plan", chunk)]
    S = st0.double().view(len(lens), inner, n)
    X, Z, B, C = x.double(), z.double(), bc.double()[:, :n], bc.double()[:, n:]
    sp, A, ref, at = torch.nn.functional.softplus(dt.double(), threshold=50), -torch.exp(al.double()), [], 0
    for s, length in enumerate(lens):
        slot = len(lens) - 1 - s
        for t in range(at, at + length):
            S[slot] = torch.exp(sp[t][:, None] * A) * S[slot] + (sp[t] * X[t])[:, None] * B[t]
            ref.append(((S[slot] * C[t]).sum(1) + D.double() * X[t]) * (Z[t] * torch.sigmoid(Z[t])))
        at += length
    ref = torch.stack(ref)
    scale = ref.abs().amax(1, keepdim=True)
    # (a state's exponentials are off by their exponents' 2^-24, and sum up over the tokens that a state remembers)
    rel = 2.0 ** -8 if dtype == torch.bfloat16 else 0.0
    assert (((y.cpu().double() - ref).abs() - rel * ref.abs()) / scale).max() < 5e-6
    assert (st.cpu().double().view(S.shape) - S).abs().max() < 5e-6 * S.abs().max()


# heads whose rows end inside a wave's 16 and beyond them, values that end inside a block of 64, gates of a row of one piece and
# of more columns than the workgroup reads at a time
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("N,H,d,dv,K", [(1, 8, 128, 128, 2048), (9, 3, 40, 70, 8), (2, 1, 200, 24, 4104), (17, 2, 260, 65, 520)])
def test_matrix_memory_of_single_tokens_makes_its_gates(N, H, d, dv, K, dtype):
    o, g = ops(), torch.Generator().manual_seed(d + dv)
    scale, cap, eps = d ** -0.5, 15.0, 1e-5
    buf = torch.randn(N, H * (2 * d + 2 * dv), generator=g).to(dtype)
    x, gw = torch.randn(N, K, generator=g).to(dtype), (torch.randn(2 * H, K, generator=g) * K ** -0.5).to(dtype)
    gb, w = torch.randn(2 * H, generator=g).to(dtype), torch.rand(H * dv, generator=g) + 0.5
    cut, copies = (H * d, 2 * H * d, 2 * H * d + H * dv), (dv + 31) // 32
    S, m = torch.randn(N, H, d, dv + 1, generator=g), torch.rand(N, H, generator=g)
    st = torch.cat([S.reshape(N, -1), m.repeat_interleave(copies, 1)], 1).cuda()
    dev = buf.cuda()
    out = o.mlstm_step(dev[:, :cut[0]], dev[:, cut[0]:cut[1]], dev[:, cut[1]:cut[2]], x.cuda(), gw.cuda(), gb.cuda(),
                       dev[:, cut[2]:], w.cuda(), st, batch([1] * N), H, d, dv, scale, cap, eps)
    b, S64, m64 = buf.double(), S.double(), m.double()
    ref = memory_by_tokens(b[:, :cut[0]], b[:, cut[0]:cut[1]], b[:, cut[1]:cut[2]], x.double() @ gw.double().T + gb.double(),
                           b[:, cut[2]:], w.double(), (S64, m64), [1] * N, H, d, dv, scale, cap, eps)
    rel = 2.0 ** -8 if dtype == torch.bfloat16 else 0.0
    err = ((out.cpu().double() - ref).abs() - rel * ref.abs()).amax(1) / ref.pow(2).mean(1).sqrt()
    assert err.max() < 2e-4, float(err.max())
    got = st.cpu().double()
    gs, gm = got[:, :H * d * (dv + 1)].view(S64.shape), got[:, H * d * (dv + 1):].view(N, H, copies)
    assert (gs - S64).abs().max() < 2e-5 * S64.abs().max() and (gm - m64[:, :, None]).abs().max() < 1e-4


@pytest.mark.parametrize("N,inner,n,rank", [(1, 32, 16, 32), (8, 4096, 16, 128), (9, 96, 8, 160), (17, 64, 32, 64)])
@pytest.mark.parametrize("biased", [True, False])
def test_selective_scan_of_single_tokens_makes_its_steps(N, inner, n, rank, biased):
    o, g, bf = ops(), torch.Generator().manual_seed(inner + n), torch.bfloat16
    x, z, low = (torch.randn(N, c, generator=g).to(bf) for c in (inner, inner, rank + 2 * n))
    W, bias = (torch.randn(inner, rank, generator=g) * rank ** -0.5).to(bf), torch.randn(inner, generator=g).to(bf)
    al, D, st0 = torch.randn(inner, n, generator=g), torch.randn(inner, generator=g), torch.randn(N, inner * n, generator=g)
    st = st0.cuda()
    y = o.selective_scan_step(x.cuda(), low.cuda(), rank, W.cuda(), bias.cuda() if biased else None, rank, rank + n, z.cuda(),
                              al.cuda(), D.cuda(), st, batch([1] * N))
    S = st0.double().view(N, inner, n).flip(0)          # (the slots of ``batch`` run backwards)
    X, Z, L = x.double(), z.double(), low.double()
    dt = torch.nn.functional.softplus(L[:, :rank] @ W.double().T + (bias.double() if biased else 0), threshold=50)
    S = torch.exp(-dt[:, :, None] * torch.exp(al.double())) * S + (dt * X)[:, :, None] * L[:, None, rank:rank + n]
    ref = ((S * L[:, None, rank + n:]).sum(2) + D.double() * X) * (Z * torch.sigmoid(Z))
    assert (((y.cpu().double() - ref).abs() - 2.0 ** -8 * ref.abs()) / ref.abs().amax(1, keepdim=True)).max() < 5e-6
    assert (st.cpu().double().view(S.shape) - S.flip(0)).abs().max() < 5e-6 * S.abs().max()
    assert o.selective_scan_step(x.cuda()[:, :inner - 8], low.cuda(), rank, W.cuda()[:inner - 8], None, rank, rank + n,
                                 z.cuda()[:, :inner - 8], al.cuda()[:inner - 8], D.cuda()[:inner - 8], st, batch([1] * N)) is None


# one piece, chunks, a step of single tokens; a number of entries that the kernel holds and one that it does not
@pytest.mark.parametrize("n", [16, 5])
@pytest.mark.parametrize("lens", [(3,), (70, 2), (1, 1)])
def test_selective_scan_keeps_states_at_the_largest_rates(n, lens):
    """exp(88.5) is a float32 number whose product with log2(e) is none: a step size of zero still leaves the state alone."""
    o, g, bf = ops(), torch.Generator().manual_seed(n), torch.bfloat16
    N, inner, rank = sum(lens), 64, 32
    x, z, low = (torch.randn(N, c, generator=g).to(bf).cuda() for c in (inner, inner, rank + 2 * 16))
    al, D = torch.full((inner, n), 88.5, device="cuda"), torch.ones(inner, device="cuda")
    st0 = torch.randn(len(lens), inner * n, generator=g).cuda()
    st = st0.clone()
    y = o.selective_scan(x, torch.full((N, inner), -200.0, device="cuda"), low, rank, rank + 16, z, al, D, st, batch(lens))
    assert torch.equal(st, st0) and y.isfinite().all()
    if lens == (1, 1) and n == 16:
        W, bias = torch.zeros(inner, rank, dtype=bf, device="cuda"), torch.full((inner,), -200.0, dtype=bf, device="cuda")
        y = o.selective_scan_step(x, low, rank, W, bias, rank, rank + 16, z, al, D, st, batch(lens))
        assert torch.equal(st, st0) and y.isfinite().all()

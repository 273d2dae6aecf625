"""The float32 product split over the waves of a workgroup, and general attention's values read four keys at a time."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from lmsf_amd.ops import get_ops
    return get_ops()


# the edges of its row forms (8, 16, 32 rows a workgroup) and columns (16), K below, at and beyond a step of 32 and a step
# for every wave, K that is no multiple of 4, and many outputs (short K in the 64x64 tiles)
@pytest.mark.parametrize("M,N,K", [(1, 1, 1), (1, 16, 4), (8, 17, 31), (9, 15, 32), (16, 33, 36), (17, 64, 127), (32, 16, 128),
                                   (33, 70, 132), (65, 130, 260), (7, 128, 352), (5, 20, 256), (5, 20, 257), (5, 20, 515), (1024, 1024, 21), (1025, 1024, 21), (1025, 1024, 20),
                                   (2, 20000, 12)])
@pytest.mark.parametrize("types", [(torch.float32, torch.float32, torch.float32), (torch.float32, torch.bfloat16, torch.float32),
                                   (torch.bfloat16, torch.float32, torch.float32), (torch.bfloat16, torch.float32, torch.bfloat16)])
@pytest.mark.parametrize("shift", [0, 1])
def test_product_of_few_outputs(ops, M, N, K, types, shift):
    ta, tw, to = types
    g = torch.Generator().manual_seed(M * 7 + N + K + shift)

    def rows(n, dtype):        # rows that start ``shift`` elements off a 16-byte boundary
        pad = (-K) % 8 + (8 if shift else 0)
        buf = torch.full((n * (K + pad) + 8,), float("nan"), dtype=dtype, device="cuda:0")
        t = buf[shift:shift + n * (K + pad)].view(n, K + pad)[:, :K]
        t.copy_(torch.randn(n, K, generator=g).to(dtype))
        return t
    x, w = rows(M, ta), rows(N, tw)
    b = torch.randn(N, generator=g).to(tw).to("cuda:0")
    y = ops.linear(x, w, b, out_dtype=to).double()
    exact = x.double() @ w.double().T + b.double()
    # a wave adds 16 products of every 256 in turn, two such sums, the waves' eight and the bias come on top; the tiles add
    # all K in turn
    split = M * N <= 1 << 20 or (K % 4 == 0 and shift == 0)
    chain = 16 * -(-K // 256) + 10 if split else K + 1
    bound = (x.double().abs() @ w.double().abs().T + b.double().abs()) * chain * 2.0 ** -24
    if to == torch.bfloat16:
        bound = bound + exact.abs() * 2.0 ** -8
    assert ((y - exact).abs() <= bound + 1e-30).all()


# few rows and many, in both forms of the product: K of one step of 32, of fewer steps than parts, of uneven parts, odd rows
@pytest.mark.parametrize("M,N,K", [(1100, 1001, 21), (1100, 1001, 333), (2100, 1001, 1030), (33, 4100, 15), (24, 9000, 40),
                                   (300, 1000, 16), (9000, 65, 33), (4200, 260, 20), (4200, 260, 36), (4200, 260, 132), (4100, 600, 260), (2100, 2050, 800)])
@pytest.mark.parametrize("types", [(torch.float32, torch.float32), (torch.float32, torch.bfloat16), (torch.bfloat16, torch.float32)])
def test_a_row_does_not_hang_on_the_number_of_rows(ops, M, N, K, types):
    g = torch.Generator(device="cuda:0").manual_seed(M + N + K)
    x, w = (torch.randn(n, K, generator=g, device="cuda:0").to(t) for n, t in zip((M, N), types))
    y = ops.linear(x, w, out_dtype=torch.float32)
    for rows in (1, 9, 40, 700):
        assert torch.equal(ops.linear(x[:rows], w, out_dtype=torch.float32), y[:rows])
    assert torch.equal(ops.linear(x[-33:], w, out_dtype=torch.float32), y[-33:])


# each number of rows a workgroup (8, 16, 32) with more rows than one workgroup's, on either side of where it changes
@pytest.mark.parametrize("M,N", [(17, 16 * 85), (17, 16 * 86), (33, 16 * 102), (33, 16 * 103), (65, 16 * 113), (65, 16 * 114)])
@pytest.mark.parametrize("K", [128, 131, 260])
def test_rows_of_a_workgroup_change_no_bit(ops, M, N, K):
    g = torch.Generator(device="cuda:0").manual_seed(M + N + K)
    x, w = (torch.randn(n, K, generator=g, device="cuda:0") for n in (M, N))
    y = ops.linear(x, w)
    assert torch.equal(torch.cat([ops.linear(x[i:i + 8], w) for i in range(0, M, 8)]), y)
    exact = x.double() @ w.double().T
    bound = (x.double().abs() @ w.double().abs().T) * (16 * -(-K // 256) + 10) * 2.0 ** -24
    assert ((y - exact).abs() <= bound).all()


# as many rows as the grid of the split form takes (32 a workgroup), and one more
@pytest.mark.parametrize("M", [65535 * 32, 65535 * 32 + 1])
def test_product_of_very_many_rows(ops, M):
    g = torch.Generator(device="cuda:0").manual_seed(M)
    x, w = torch.randn(M, 4, generator=g, device="cuda:0"), torch.randn(3, 4, generator=g, device="cuda:0")
    exact = x.double() @ w.double().T
    # four products and their sums in float32
    assert ((ops.linear(x, w).double() - exact).abs() <= 5 * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)).all()


# keys just below, at and beyond four and eight a group (256 / d groups), a second round of 256 keys, pages of odd sizes
@pytest.mark.parametrize("d,ps", [(32, 16), (4, 3), (96, 16), (256, 8), (260, 16)])
@pytest.mark.parametrize("context", [1, 7, 8, 31, 32, 33, 63, 64, 65, 256, 257, 300])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("shift", [0, 1])
def test_general_attention(ops, d, ps, context, dtype, shift):
    nh, nkv, scale = 4, 2, d ** -0.5
    g = torch.Generator().manual_seed(d + context)
    blocks = -(-context // ps)
    pages = blocks + 3

    def cache():                # pages that start ``shift`` elements off a 16-byte boundary
        buf = torch.empty(pages * nkv * ps * d + 8, dtype=dtype, device="cuda:0")
        t = buf[shift:shift + pages * nkv * ps * d]
        t.copy_(torch.randn(t.shape, generator=g).to(dtype))
        return t
    k, v = cache().view(pages, nkv, ps, d), cache().view(pages, nkv, d, ps)
    q = torch.randn(2, nh * d, generator=g).to(dtype).to("cuda:0")
    table = torch.randperm(pages, generator=g)[:blocks].to(torch.int32).view(1, -1).to("cuda:0")
    seg = torch.zeros(2, dtype=torch.int32, device="cuda:0")
    pos = torch.tensor([context - 1, max(0, context - 2)], dtype=torch.int32, device="cuda:0")
    got = ops.paged_attention(q, k, v, table, seg, pos, nh, nkv, d, scale, kernel="generic").double().cpu()
    keys = k[table[0].long()].permute(1, 0, 2, 3).reshape(nkv, -1, d)[:, :context].double().cpu()
    vals = v[table[0].long()].permute(1, 0, 3, 2).reshape(nkv, -1, d)[:, :context].double().cpu()
    for t in range(2):
        n = int(pos[t]) + 1
        for h in range(nh):
            s = keys[h // 2, :n] @ q[t, h * d:(h + 1) * d].double().cpu() * scale
            want = torch.softmax(s, 0) @ vals[h // 2, :n]
            # scores of a few units to 2^-21, weights that add up to one over values of up to 5 units
            tol = 2e-5 + (want.abs() * 2.0 ** -8 if dtype == torch.bfloat16 else 0)
            assert ((got[t, h * d:(h + 1) * d] - want).abs() <= tol).all()


# as many workgroups as the chip takes at once with four on a compute unit, and more: the two register budgets of the form
# without tiles, which pages of 18 tokens, wider heads and unaligned pages run in, and the tiles
@pytest.mark.parametrize("d", [32, 96, 260])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("ps", [16, 18])
def test_general_attention_of_many_tokens_gives_the_bits_of_few(ops, d, dtype, shift, ps):
    nh, nkv = 8, 2
    T = torch.cuda.get_device_properties(0).multi_processor_count * 4 // nh + 3
    g = torch.Generator(device="cuda:0").manual_seed(d)
    pages = -(-T // ps) + 2

    def cache(*shape):
        n = pages * nkv * ps * d
        return torch.randn(n + 8, generator=g, device="cuda:0").to(dtype)[shift:shift + n].view(pages, nkv, *shape)
    k, v = cache(ps, d), cache(d, ps)
    q = torch.randn(T, nh * d, generator=g, device="cuda:0").to(dtype)
    table = torch.randperm(pages, generator=g, device="cuda:0")[:-(-T // ps)].to(torch.int32).view(1, -1)
    seg, pos = torch.zeros(T, dtype=torch.int32, device="cuda:0"), torch.arange(T, dtype=torch.int32, device="cuda:0")

    def run(a, b):
        return ops.paged_attention(q[a:b], k, v, table, seg[a:b], pos[a:b], nh, nkv, d, d ** -0.5, kernel="generic")
    assert torch.equal(run(0, T), torch.cat([run(0, T - 20), run(T - 20, T)]))


# tiles of 64, 32, 16 and 8 keys, eight of them side by side: windows and chunks that begin inside a quad of keys, pages of
# any multiple of 4, and pages whose unwritten places hold NaN
@pytest.mark.parametrize("d,ps", [(4, 4), (32, 12), (36, 16), (64, 8), (100, 16), (128, 20), (256, 16)])
@pytest.mark.parametrize("context", [2, 9, 65, 130, 513, 700])
@pytest.mark.parametrize("mask", [{}, {"window": 1}, {"window": 70}, {"chunk": 50}])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_general_attention_reads_visible_keys_only(ops, d, ps, context, mask, dtype):
    nh, nkv, scale, cap = 4, 2, d ** -0.5, 3.0
    g = torch.Generator().manual_seed(d + context)
    blocks = -(-context // ps)
    keys, vals = (torch.randn(nkv, context, d, generator=g).to(dtype) for _ in range(2))
    k, v = torch.full((blocks + 2, nkv, ps, d), float("nan"), dtype=dtype), torch.full((blocks + 2, nkv, d, ps), float("nan"), dtype=dtype)
    table = torch.randperm(blocks + 2, generator=g)[:blocks].to(torch.int32)
    for j in range(context):
        k[table[j // ps], :, j % ps] = keys[:, j]
        v[table[j // ps], :, :, j % ps] = vals[:, j]
    q = torch.randn(2, nh * d, generator=g).to(dtype)
    pos = torch.tensor([context - 1, context // 2], dtype=torch.int32)
    bias, sink = torch.rand(2, nh, generator=g), torch.randn(nh, generator=g)
    got = ops.paged_attention(q.cuda(), k.cuda(), v.cuda(), table.view(1, -1).cuda(), torch.zeros(2, dtype=torch.int32, device="cuda:0"),
                              pos.cuda(), nh, nkv, d, scale, softcap=cap, distance_bias=bias.cuda(), sink=sink.cuda(),
                              kernel="generic", **mask).double().cpu()
    for t in range(2):
        p = int(pos[t])
        lo = max(0, p - mask["window"] + 1) if "window" in mask else p // mask["chunk"] * mask["chunk"] if "chunk" in mask else 0
        j = torch.arange(lo, p + 1)
        for h in range(nh):
            s = cap * torch.tanh(keys[h // 2, j].double() @ q[t, h * d:(h + 1) * d].double() * scale / cap)
            s = s - bias[0, h].double() * torch.log1p(bias[1, h].double() * (p - j))
            w = torch.softmax(torch.cat([s, sink[h:h + 1].double()]), 0)[:-1]
            want = w @ vals[h // 2, j].double()
            # scores of a few units to 2^-21, weights that add up to at most one over values of up to 5 units
            tol = 2e-5 + (want.abs() * 2.0 ** -8 if dtype == torch.bfloat16 else 0)
            assert ((got[t, h * d:(h + 1) * d] - want).abs() <= tol).all()


# one NaN key: alone in the first tile of a wave (every other key of that tile beyond the token), among the keys of a full
# tile, and every key of a tile; a query of NaN beside a sink
@pytest.mark.parametrize("d", [32, 64, 128, 256])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("context,bad", [(1, [0]), (300, [299]), (300, [5]), (300, list(range(64))), (300, list(range(192, 256)))])
def test_general_attention_keeps_what_is_no_number(ops, d, dtype, context, bad):
    nh, ps, pages = 2, 16, -(-context // 16)
    g = torch.Generator().manual_seed(d + context)
    k, v = torch.randn(pages, 1, ps, d, generator=g).to(dtype), torch.randn(pages, 1, d, ps, generator=g).to(dtype)
    q = torch.randn(2, nh * d, generator=g).to(dtype)
    q[1, :d] = float("nan")                           # the second token: head 0 has no number, head 1 all of them
    table = torch.arange(pages, dtype=torch.int32).view(1, -1).cuda()
    pos = torch.full((2,), context - 1, dtype=torch.int32, device="cuda:0")
    sink = torch.zeros(nh, device="cuda:0")

    def run(keys):
        return ops.paged_attention(q.cuda(), keys.cuda(), v.cuda(), table, torch.zeros(2, dtype=torch.int32, device="cuda:0"), pos,
                                   nh, 1, d, d ** -0.5, kernel="generic", sink=sink).float()
    clean = run(k)
    assert torch.isnan(clean[1, :d]).all() and not torch.isnan(clean[0]).any() and not torch.isnan(clean[1, d:]).any()
    for j in bad:
        k[j // ps, :, j % ps] = float("nan")
    assert torch.isnan(run(k)).all()
    k[k.isnan()] = float("-inf")                      # scores of +-inf and NaN by the query's signs: no number either
    assert torch.isnan(run(k)).all()

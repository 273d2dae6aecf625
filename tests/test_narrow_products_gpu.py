"""The few-rows products whose workgroups own 8 rows of the weight instead of 16: at both sides of the line between the
two every output is added up in the same order, so the same rows give the same bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from lmsf_amd.ops import get_ops
    return get_ops()


def rnd(g, *shape):
    return (torch.randn(*shape, generator=g) * shape[-1] ** -0.5).bfloat16().to("cuda:0")


# 8 compute units' worth of columns more than the line (2,048 on 256 units), odd numbers of columns, one column
@pytest.mark.parametrize("N", [1, 7, 8, 9, 24, 1000, 2041, 2048])
@pytest.mark.parametrize("M", [2, 8, 9, 16])
@pytest.mark.parametrize("K", [8, 64, 1096, 4096])
@pytest.mark.parametrize("out", [torch.bfloat16, torch.float32])
def test_product(ops, M, N, K, out):
    g = torch.Generator().manual_seed(N * K + M)
    w, b, x = rnd(g, 8192, K), rnd(g, 8192), rnd(g, M, K)
    assert torch.equal(ops.linear(x, w[:N], b[:N], out_dtype=out), ops.linear(x, w, b, out_dtype=out)[:, :N])


@pytest.mark.parametrize("I", [1, 8, 23, 2048])
@pytest.mark.parametrize("M", [3, 8, 13])
@pytest.mark.parametrize("kind", ["silu", "gelu", "gelu_tanh"])
def test_gated_product(ops, M, I, kind):
    g = torch.Generator().manual_seed(I + M)
    K, more = 1032, 4096
    gate, up, x = rnd(g, more, K), rnd(g, more, K), rnd(g, M, K)
    few = ops.linear_gated(x, torch.cat([gate[:I], up[:I]]), None, kind)
    assert torch.equal(few, ops.linear_gated(x, torch.cat([gate, up]), None, kind)[:, :I])


@pytest.mark.parametrize("M", [3, 8, 15])
@pytest.mark.parametrize("d,heads", [(32, 2), (96, 5), (64, 62)])
def test_qkv_product_with_rotation(ops, M, d, heads):
    """Few heads beside the same query heads among many: tiles of 8 pairs beside tiles of 16."""
    g = torch.Generator().manual_seed(d + heads + M)
    K, many, ps, pages = 520, 260, 8, 4
    wq, wkv, x = rnd(g, many * d, K), rnd(g, 2 * d, K), rnd(g, M, K)
    pos = torch.randint(0, 40, (M,), generator=g, dtype=torch.int32).to("cuda:0")
    ang = torch.arange(40)[:, None] * torch.rand(d // 2, generator=g)[None, :]
    table = torch.cat([ang.cos(), ang.sin()], 1).contiguous().to("cuda:0")
    slots = torch.randperm(pages * ps, generator=g)[:M].to(torch.int32).to("cuda:0")

    def run(n):
        k = torch.zeros(pages, 1, ps, d, dtype=torch.bfloat16, device="cuda:0")
        v = torch.zeros(pages, 1, d, ps, dtype=torch.bfloat16, device="cuda:0")
        y = ops.qkv_rope_cache(x, torch.cat([wq[:n * d], wkv]), None, n, 1, d, pos, table, d, True, slots, k, v)
        return y, k, v
    (a, ka, va), (b, kb, vb) = run(heads), run(many)
    assert torch.equal(a[:, :heads * d], b[:, :heads * d]) and torch.equal(ka, kb) and torch.equal(va, vb)
    assert ka.abs().sum() > 0


# the widths at which tiles of 8 outputs would fit on the chip, and one beyond; 8 rows and 9
@pytest.mark.parametrize("N", [1008, 1024, 1040, 2048, 2064])
@pytest.mark.parametrize("M", [3, 8, 9])
@pytest.mark.parametrize("K,bias", [(64, False), (4104, True)])
def test_product_before_a_norm(ops, M, N, K, bias):
    g = torch.Generator().manual_seed(N + M + K)
    w, x, b = rnd(g, N, K), rnd(g, M, K), rnd(g, N) if bias else None
    nw = torch.randn(N, generator=g).bfloat16().to("cuda:0")
    before = torch.randn(M, N, generator=g).to("cuda:0") * 3
    stream = before.clone()
    h = ops.add_rms_norm(ops.linear(x, w, b, pending_ok=True), stream, nw, 1e-5, torch.bfloat16, defer_ok=True)
    assert torch.equal(stream, before + ops.linear(x, w, b).float()) and torch.equal(h.xw, (stream * nw.float()).bfloat16())
    # the products that take the norm: their factor rsqrt(sum / N + eps) to the roundings of sums of N squares, the
    # products' own sums of N terms in float32, three roundings to bfloat16 (gate, up, result; silu's slope is below 1.1)
    normed = h.xw.double() * torch.rsqrt(stream.double().pow(2).mean(1, keepdim=True) + 1e-5)
    wg = rnd(g, 2 * 1024, N)
    got = ops.linear_gated(h, wg, None, "silu").double()
    a, u = (normed @ wg.double().T).split(1024, 1)
    want = torch.nn.functional.silu(a) * u
    err = 2.0 ** -8 * (1.1 * a.abs() * u.abs() + want.abs() * 2) + 1e-5
    assert ((got - want).abs() <= err * 1.05).all()


# whole tiles and a last one of 8 columns, widths on both sides of what tiles of 8 outputs would take at once
@pytest.mark.parametrize("N", [1000, 1024, 2048, 2064])
@pytest.mark.parametrize("M", [3, 8, 9, 16])
def test_sums_of_squares_before_a_norm(ops, M, N):
    """A row's sums are those of 16 columns one after the other, whatever the number of rows and the width: the factor, and
    with it every rounding of the layers behind it, hangs on their order."""
    g = torch.Generator().manual_seed(N + M)
    w, x = rnd(g, N, 512), rnd(g, M, 512)
    nw = torch.randn(N, generator=g).bfloat16().to("cuda:0")
    stream = torch.randn(M, N, generator=g).to("cuda:0")
    h = ops.add_rms_norm(ops.linear(x, w, pending_ok=True), stream, nw, 1e-5, torch.bfloat16, defer_ok=True)
    assert h.rows_per_tile == 16 and h.tiles == -(-N // 16)
    squares = torch.zeros(M, 16 * h.tiles)
    squares[:, :N] = stream.cpu() * stream.cpu()
    want = torch.zeros(h.tiles, 16)
    for i in range(16):
        want[:, :M] += squares.view(M, h.tiles, 16)[:, :, i].T
    assert torch.equal(h.sumsq.view(h.tiles, 16).cpu(), want)


@pytest.mark.parametrize("N", [1, 9, 1000, 2048, 2056, 4096])
@pytest.mark.parametrize("M", [1, 2, 8, 9, 16])
@pytest.mark.parametrize("K,bias", [(64, False), (4104, True)])
def test_product_before_dynamic_tanh(ops, M, N, K, bias):
    """One kernel to the bits of the few-rows product and the kernel after it (a separate product of one row would run in the
    one-row kernel, so it is taken from two: rows of the few-rows product hang on nothing else)."""
    from lmsf_amd.ops.handles import DeferredLinear
    g = torch.Generator().manual_seed(N + M + K)
    w, x, b = rnd(g, N, K), rnd(g, max(M, 2), K), rnd(g, N) if bias else None
    tw, tb, alpha = (torch.randn(n, generator=g).to("cuda:0") for n in (N, N, 1))
    before = torch.randn(M, N, generator=g).to("cuda:0") * 2
    s1, s2 = before.clone(), before.clone()
    p = ops.linear(x[:M], w, b, pending_ok=True)
    assert isinstance(p, DeferredLinear)
    got = ops.dyt_norm(p, s1, tw, tb, alpha, torch.bfloat16)
    want = ops.dyt_norm(ops.linear(x, w, b)[:M].contiguous(), s2, tw, tb, alpha, torch.bfloat16)
    assert torch.equal(s1, s2) and torch.equal(got, want) and not torch.equal(s1, before)
    rows = torch.tensor([M - 1], dtype=torch.int32, device="cuda:0")          # wanted rows alone: the kernels one by one
    assert torch.equal(ops.dyt_norm(p, before.clone(), tw, tb, alpha, torch.bfloat16, rows=rows), want[M - 1:])


def test_one_row_before_dynamic_tanh_without_the_few_rows_kernel(ops):
    """With the few-rows kernel switched off the one-row product and the tanh's kernel run one after the other."""
    from lmsf_amd.ops.handles import DeferredLinear
    g = torch.Generator().manual_seed(5)
    N, K = 32768, 8192                                # (so many that a few would round otherwise)
    w, x = rnd(g, N, K), rnd(g, 1, K)
    tw, tb, alpha = (torch.randn(n, generator=g).to("cuda:0") for n in (N, N, 1))
    s1 = torch.randn(1, N, generator=g).to("cuda:0")
    names = ("skinny_max_rows", "mid_max_rows", "large_max_rows")
    s2, before = s1.clone(), [getattr(ops, n) for n in names]
    for n in names:
        setattr(ops, n, 0)
    try:
        p = ops.linear(x, w, pending_ok=True)
        assert isinstance(p, DeferredLinear)
        got = ops.dyt_norm(p, s1, tw, tb, alpha, torch.bfloat16)
        want = ops.dyt_norm(ops.linear(x, w), s2, tw, tb, alpha, torch.bfloat16)
    finally:
        for n, v in zip(names, before):
            setattr(ops, n, v)
    assert torch.equal(s1, s2) and torch.equal(got, want)

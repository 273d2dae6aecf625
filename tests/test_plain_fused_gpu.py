"""The float32 product's forms that do the work of the kernels around it: the addition to the stream, the norm on the way
in, the gated activation, the rotation and cache write. Each gives the bits of the separate kernels (csrc/gemm_plain.hip)."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# rows at the edges of tiles of 8, 16 and 32; K below one step, of one part, of several, and no multiple of a step
ROWS = [1, 7, 8, 9, 16, 17, 33, 100]
COLS = [4, 36, 128, 260, 1000]


@pytest.fixture(scope="module")
def ops():
    from lmsf_amd.ops import get_ops
    return get_ops()


def draw(*shape, seed=0):
    gen = torch.Generator(device="cuda").manual_seed(seed + sum(shape))
    return torch.randn(shape, device="cuda", generator=gen)


def normed_rows(ops, stream, weight, deferred):
    """The norm of the stream: the handle that a product takes (of long rows only few), or the norm kernel's tensor."""
    y = ops.add_rms_norm(None, stream, weight, 1e-6, torch.float32, weight_offset=0.5, defer_ok=deferred)
    assert not isinstance(y, torch.Tensor) if deferred and (len(stream) <= 16 or len(weight) <= 512) else True
    return y


@pytest.mark.parametrize("K", COLS)
@pytest.mark.parametrize("M", ROWS)
def test_product_added_to_the_stream(ops, M, K):
    for N in (4, 20, 128):
        x, w, b, stream, g = draw(M, K), draw(N, K, seed=1), draw(N, seed=2), draw(M, N, seed=3), draw(N, seed=4)
        want = stream.clone()
        y = ops.add_rms_norm(ops.linear(x, w, b), want, g, 1e-6, torch.float32)
        handle = ops.linear(x, w, b, pending_ok=True)
        assert not isinstance(handle, torch.Tensor)
        got = stream.clone()
        rows = ops.add_rms_norm(handle, got, g, 1e-6, torch.float32, defer_ok=True)
        assert torch.equal(got, want) and rows.xw is got
        assert torch.equal(ops.materialize(rows), y)
        got = stream.clone()      # a caller that wants the norm's tensor
        assert torch.equal(ops.add_rms_norm(ops.linear(x, w, b, pending_ok=True), got, g, 1e-6, torch.float32), y)
        assert torch.equal(got, want)


@pytest.mark.parametrize("kind", ["silu", "gelu", "gelu_tanh"])
@pytest.mark.parametrize("K", COLS)
@pytest.mark.parametrize("M", ROWS)
def test_gated_product(ops, M, K, kind):
    for I in (3, 8, 44):
        w, b, stream, g = draw(2 * I, K, seed=1), draw(2 * I, seed=2), draw(M, K, seed=3), draw(K, seed=4)
        x = normed_rows(ops, stream, g, False)
        want = ops.gated_act(ops.linear(x, w, b), kind)
        assert torch.equal(ops.linear_gated(x, w, b, kind), want)
        assert torch.equal(ops.linear_gated(normed_rows(ops, stream, g, True), w, b, kind), want)


@pytest.mark.parametrize("K", COLS)
@pytest.mark.parametrize("M", ROWS)
def test_qkv_product(ops, M, K):
    for nh, nkv, d in ((1, 1, 16), (4, 2, 48)):
        N, ps, pages = (nh + 2 * nkv) * d, 4, 40
        w, b, stream, g = draw(N, K, seed=1), draw(N, seed=2), draw(M, K, seed=3), draw(K, seed=4)
        table = draw(256, d, seed=5)
        pos = torch.arange(M, device="cuda", dtype=torch.int32) * 2
        slots = torch.randperm(pages * ps, device="cuda")[:M].to(torch.int32)
        slots[M // 2] = -1
        x = normed_rows(ops, stream, g, False)

        def pages_of():
            return torch.zeros(pages, nkv, ps, d, device="cuda"), torch.zeros(pages, nkv, d, ps, device="cuda")

        k0, v0 = pages_of()
        want = ops.linear(x, w, b)
        ops.rope_cache_write(want, nh, nkv, d, pos, table, d, True, slots, k0, v0)
        for rows in (x, normed_rows(ops, stream, g, True)):
            k1, v1 = pages_of()
            got = ops.qkv_rope_cache(rows, w, b, nh, nkv, d, pos, table, d, True, slots, k1, v1)
            assert torch.equal(got, want) and torch.equal(k0, k1) and torch.equal(v0, v1)
        # no forms with an epilogue: the norm's handle is finished first
        k2, v2 = pages_of()
        got = ops.qkv_rope_cache(normed_rows(ops, stream, g, True), w, b, nh, nkv, d, pos, table, d, False, slots, k2, v2)
        want = ops.linear(x, w, b)
        ops.rope_cache_write(want, nh, nkv, d, pos, table, d, False, slots, *pages_of())
        assert torch.equal(got, want)


def test_rows_off_a_boundary_and_strided(ops):
    """Operands that no wide load takes run in the separate kernels; strided rows in the fused ones."""
    M, K, I = 5, 64, 24
    w = draw(2 * I, K, seed=1)
    x = draw(M, K + 3, seed=2)[:, 1:1 + K]
    assert torch.equal(ops.linear_gated(x, w, None), ops.gated_act(ops.linear(x, w, None)))
    x = draw(M, K + 8, seed=2)[:, 4:4 + K]
    assert torch.equal(ops.linear_gated(x, w, None), ops.gated_act(ops.linear(x, w, None)))
    half = draw(M, K, seed=2).bfloat16()       # a product of two types
    assert torch.equal(ops.linear_gated(half, w, None), ops.gated_act(ops.linear(half, w, None)))

"""The 17-and-more-rows product with fewer than 64 outputs a workgroup, and with 128: every output is added up in the same
order, so the same rows of the weight give the same bits as among many."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from lmsf_amd.ops import get_ops
    return get_ops()


def rnd(g, *shape):
    return (torch.randn(*shape, generator=g) * shape[-1] ** -0.5).bfloat16().to("cuda:0")


def product(ops, x, w, bias, out, splits, gated):
    from lmsf_amd.ops.hip_ops import _ptr
    M, K, N = x.shape[0], x.shape[1], w.shape[0] // (2 if gated else 1)
    y = torch.full((M, N + 4), float("nan"), dtype=out, device="cuda:0")[:, :N]
    scratch = torch.empty(max(4, ops.lib.lmsf_gemm_mid_scratch_floats(M, N, splits, int(gated))), device="cuda:0")
    ops._check(ops.lib.lmsf_gemm_mid(_ptr(x), x.stride(0), _ptr(w), w.stride(0), _ptr(bias), _ptr(y),
                                     0 if out == torch.float32 else 1, y.stride(0), M, N, K, 1 if gated else 0, splits,
                                     _ptr(scratch), ops._stream()))
    return y


# 32, 40, 48, 56 and 64 outputs a workgroup on 256 units (in one part and in 2), remainders of a workgroup, of 8 and of 4
@pytest.mark.parametrize("N,splits", [(4, 1), (36, 1), (8192, 1), (8196, 1), (10240, 1), (14332, 1), (16380, 1), (4096, 2),
                                      (6144, 2), (6148, 2), (4100, 4)])
@pytest.mark.parametrize("M", [17, 33, 64, 97])
@pytest.mark.parametrize("gated", [False, True])
def test_outputs_a_workgroup(ops, N, splits, M, gated):
    if gated and M > 64:
        pytest.skip("the gated form takes up to 64 rows")
    g = torch.Generator().manual_seed(N + M)
    K, many = 512, 20480               # 320 workgroups of 64 outputs: more than the chip takes at once
    a, b, x = rnd(g, many, K), rnd(g, many, K), rnd(g, M, K)
    ba, bb = rnd(g, many), rnd(g, many)
    w = lambda n: torch.cat([a[:n], b[:n]]) if gated else a[:n]          # noqa: E731
    bias = lambda n: torch.cat([ba[:n], bb[:n]]) if gated else ba[:n].clone()    # noqa: E731
    for out in (torch.bfloat16,) if gated else (torch.bfloat16, torch.float32):
        few = product(ops, x, w(N), bias(N), out, splits, gated)
        assert torch.equal(few, product(ops, x, w(many), bias(many), out, splits, gated)[:, :N])


# both sides of the line to 128 outputs a workgroup (65,408 = 511 such workgroups, 65,412 = 512), remainders
@pytest.mark.parametrize("N", [65412, 65536, 128252])
@pytest.mark.parametrize("M", [17, 64, 65, 128])
def test_float32_output_of_many_columns(ops, N, M):
    g = torch.Generator().manual_seed(N + M)
    K = 64
    w, x = rnd(g, N, K), rnd(g, M, K)
    wide = product(ops, x, w, None, torch.float32, 1, False)
    assert torch.equal(wide[:, :65408], product(ops, x, w[:65408], None, torch.float32, 1, False))
    exact = x.double() @ w.double().T
    # 64 products and their sums in float32
    assert ((wide.double() - exact).abs() <= 66 * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)).all()


# Which kernel a product of up to 16 rows and so many outputs runs in, on 256 compute units: the numbers of rows (of 1, 2, 4, 8,
# 16) that run 64 outputs a workgroup. 191 workgroups of 64 outputs and 192 (the line of 12,288 outputs); a second round nearly
# empty; two rounds 0.98 and 0.88 filled, at short and long rows; one row, of a long K and of a short one, of matrices too large
# for the one-row kernel; rows back to back, 4 KB apart.
MANY = [(12224, 128, 256, ()), (12288, 128, 256, (2, 4, 8, 16)), (16388, 2048, 256, ()), (32000, 2048, 256, (2, 4, 8, 16)),
        (20000, 4096, 256, ()), (32000, 4160, 256, (8, 16)), (28672, 4160, 256, (16,)), (16384, 16448, 256, (2, 4, 8, 16)),
        (32000, 2048, 0, ()), (147456, 2048, 256, (1, 2, 4, 8, 16))]


@pytest.mark.parametrize("N,K,pad,here", MANY)
@pytest.mark.parametrize("out", [torch.bfloat16, torch.float32])
def test_few_rows_and_many_outputs(ops, N, K, pad, here, out):
    from lmsf_amd.ops import dispatch as D
    from lmsf_amd.ops.hip_ops import _ptr
    import ctypes
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the lines are for 256 compute units")
    g = torch.Generator().manual_seed(N + K)
    w, b, xs = rnd(g, N, K + pad)[:, :K], rnd(g, N), rnd(g, 16, K)
    code = 0 if out == torch.float32 else 1
    for M in (1, 2, 4, 8, 16):
        x = xs[:M]
        exact, size = x.double() @ w.double().T + b.double(), x.double().abs() @ w.double().abs().T + b.double().abs()
        for shift in (0, 1):                     # an output that is not aligned stays in the few-rows kernel
            buf = torch.full((M * N + 16,), float("nan"), dtype=out, device="cuda:0")
            y = ops.linear(x, w, b, out_dtype=out, out=buf[shift:shift + M * N].view(M, N))
            assert torch.isnan(buf[:shift]).all() and torch.isnan(buf[shift + M * N:]).all()
            # K products and their sums in float32 in any order, and one rounding where the output is bfloat16
            assert ((y.double() - exact).abs() <= size * (K + 2) * 2.0 ** -24
                    + (exact.abs() * 2.0 ** -8 if out == torch.bfloat16 else 0)).all()
            r = D.Route()
            ops.lib.lmsf_route_linear(ctypes.byref(ops._tun), ctypes.byref(ops._shape(x, w, out, y)), 0, ctypes.byref(r))
            if M == 1 and N * K <= 1 << 28:
                assert r.route == D.GEMV
                continue
            want = torch.empty(M, N, dtype=out, device="cuda:0")
            args = (_ptr(x), K, _ptr(w), w.stride(0), _ptr(b), _ptr(want), code, N, M, N, K)
            if M in here and shift == 0:
                assert r.route == D.MID and r.splits == 1
                ops._check(ops.lib.lmsf_gemm_mid(*args, 0, 1, None, ops._stream()))
            else:
                assert r.route == D.SKINNY
                ops._check(ops.lib.lmsf_gemm_skinny(*args, 0, 0, ops._stream()))
            assert torch.equal(y, want)


# 128 outputs a workgroup from 33 rows on where W's rows lie apart: the last widths before the line and the first beyond it
# (243 workgroups on 256 units), remainders; to the bits of fewer rows, which run 64 outputs a workgroup
@pytest.mark.parametrize("N", [30976, 31104, 31108, 65540])
@pytest.mark.parametrize("M", [33, 48, 64])
@pytest.mark.parametrize("K", [64, 448, 2048])
def test_rows_apart(ops, N, M, K):
    g = torch.Generator().manual_seed(N + M + K)
    w, x, b = rnd(g, N, K + 256)[:, :K], rnd(g, M, K), rnd(g, N)
    many = product(ops, x, w, b, torch.float32, 1, False)
    assert torch.equal(many[:32], product(ops, x[:32], w, b, torch.float32, 1, False))
    assert torch.equal(many[M - 32:], product(ops, x[M - 32:], w, b, torch.float32, 1, False))

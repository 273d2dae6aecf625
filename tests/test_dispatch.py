"""The one table of switch points between the kernels (csrc/dispatch.hip), asked as the step program and the
Python face of the kernels ask it: which kernel a product of Llama-3-8B's shapes runs in at which number of rows,
what the forms around a norm take, and how decode attention splits its keys. Host code only: no GPU needed."""
import ctypes

import pytest

from lmsf_amd.ops import dispatch as D
from lmsf_amd.ops import library

F32, BF16 = 0, 1
H, I, QKV, V = 4096, 14336, 6144, 128256


@pytest.fixture(scope="module")
def lib():
    return library.load_library()


def defaults():
    """The switch points as ``HipOps`` sets them."""
    return D.Tunables(fuse_norm_rows=16, fuse_stream_rows=1, gemv_max_rows=2, skinny_variant=0, mid_wide_max_cols=8192,
                      mid_max_rows=128, skinny_max_rows=16, prefill_attention_variant=0, decode_attention_order=0,
                      decode_attention_splits=0, use_library_gemm=1, large_max_rows=256, large_deep_min_rows=64,
                      mid_scaled_rows=16, large_deep_max_rows=1024, qkv_fused_max_rows=32)


def shape(M, N, K, x=BF16, w=BF16, out=BF16, ld_pad=256, ok16=1):
    return D.ProductShape(M, N, K, x, w, out, K, K + ld_pad, ok16, ok16)


def linear(lib, t, M, N, K, pending_ok=False, **kw):
    r = D.Route()
    lib.lmsf_route_linear(ctypes.byref(t), ctypes.byref(shape(M, N, K, **kw)), 1 if pending_ok else 0, ctypes.byref(r))
    return r


def test_plain_products_change_kernels_with_the_number_of_rows(lib):
    t = defaults()
    o = lambda M, **kw: linear(lib, t, M, H, H, **kw).route          # noqa: E731
    assert [o(M) for M in (1, 2, 16, 17, 64, 128, 129, 256, 257, 4096)] == \
        [D.GEMV, D.SKINNY, D.SKINNY, D.MID, D.MID, D.MID, D.LARGE, D.LARGE, D.BLAS, D.BLAS]
    # a product whose K is at least three times N (down) leaves the 17-and-more-rows kernel at 65 rows and stays
    # with the many-rows kernel up to 1,024
    down = lambda M: linear(lib, t, M, H, I).route                   # noqa: E731
    assert [down(M) for M in (64, 65, 128, 512, 1024, 1025)] == [D.MID, D.LARGE, D.LARGE, D.LARGE, D.LARGE, D.BLAS]
    # beyond 64 rows the wide products (gate_up's 28,672 columns) are the library's
    assert linear(lib, t, 64, 2 * I, H).route == D.MID and linear(lib, t, 65, 2 * I, H).route == D.BLAS
    assert linear(lib, t, 100, 2 * I, H).route == D.BLAS and linear(lib, t, 100, 8192, H).route == D.MID
    # float32 operands, a K that is no multiple of 8, or no library: the float32 multiply-add kernel
    assert linear(lib, t, 8, H, H, x=F32, w=F32, out=F32).route == D.PLAIN
    assert linear(lib, t, 300, H, 4100).route == D.BLAS and linear(lib, t, 8, H, 4100).route == D.PLAIN
    t.use_library_gemm = 0
    assert linear(lib, t, 300, H, H).route == D.PLAIN and linear(lib, t, 300, H, I).route == D.LARGE


def test_logits_in_float32_for_any_number_of_rows(lib):
    t = defaults()
    head = lambda M: linear(lib, t, M, V, H, out=F32)                # noqa: E731
    # (one row of this matrix stays with the few-rows kernel: it is large enough to stream at the same rate there)
    assert head(1).route == D.SKINNY and linear(lib, t, 1, H, H, out=F32).route == D.GEMV
    assert head(8).route == D.SKINNY and head(64).route == D.MID
    r = head(300)
    assert r.route == D.CHUNKS and r.chunk_rows == 128


def test_unfinished_forms_only_where_the_caller_takes_them(lib):
    t = defaults()
    assert linear(lib, t, 8, H, H, pending_ok=True).route == D.DEFERRED       # the norm that follows runs it
    assert linear(lib, t, 8, H, H).route == D.SKINNY
    r = linear(lib, t, 40, H, H, pending_ok=True)
    assert r.route == D.MID and r.splits > 1 and r.pending == 1               # partial sums for the norm to add up
    r = linear(lib, t, 40, H, H)
    assert r.route == D.MID and r.splits > 1 and r.pending == 0               # the product's own reduction kernel
    r = linear(lib, t, 200, H, I, pending_ok=True)
    assert r.route == D.LARGE and r.splits == r.plan % 16 and r.pending == (1 if r.splits > 1 else 0)
    t.fuse_norm_rows = 0
    t.fuse_stream_rows = 0
    assert linear(lib, t, 8, H, H, pending_ok=True).route == D.SKINNY


def test_gated_and_qkv_products(lib):
    t = defaults()

    def gated(M, scaled=0, tiles=0):
        r = D.Route()
        lib.lmsf_route_linear_gated(ctypes.byref(t), ctypes.byref(shape(M, 2 * I, H)), scaled, tiles, ctypes.byref(r))
        return r.route

    assert [gated(M) for M in (1, 2, 3, 16, 17, 64, 65, 256, 257)] == \
        [D.GEMV, D.GEMV, D.SKINNY, D.SKINNY, D.MID, D.MID, D.LARGE, D.LARGE, D.SEPARATE]
    assert gated(1, scaled=1, tiles=8) == D.GEMV_SCALED                       # rows whose norm factor is still to come
    assert gated(8, scaled=16, tiles=H // 16) in (D.SKINNY_SCALED, D.MID_SCALED)

    def qkv(M, fused=1, scaled=0):
        r = D.Route()
        lib.lmsf_route_qkv(ctypes.byref(t), ctypes.byref(shape(M, QKV, H)), fused, scaled, ctypes.byref(r))
        return r

    # (with its rotation and cache write as epilogue the few-rows kernel keeps the QKV product up to 32 rows)
    assert [qkv(M).route for M in (1, 2, 3, 16, 17, 32, 33, 2048)] == [D.GEMV, D.GEMV, D.SKINNY, D.SKINNY, D.SKINNY,
                                                                     D.SKINNY, D.SEPARATE, D.SEPARATE]
    assert qkv(33).pending == 1 and qkv(8, fused=0).route == D.SEPARATE and qkv(8, fused=0).pending == 0
    assert qkv(17, fused=0).route == D.SEPARATE and qkv(17, fused=0).pending == 1
    assert qkv(8, scaled=16).route == D.SKINNY_SCALED and qkv(2, scaled=2).route == D.GEMV_SCALED
    assert qkv(8, fused=0, scaled=16).route == D.MATERIALIZE


def test_a_norm_that_finds_its_branch_unstarted(lib):
    t = defaults()

    def norm(M, fits=1, prepares=1):
        r = D.Route()
        lib.lmsf_route_deferred_norm(ctypes.byref(t), M, H, H, fits, prepares, ctypes.byref(r))
        return r.route

    assert [norm(M) for M in (1, 2, 8, 16)] == [D.GEMV_ADD_NORM, D.SKINNY_ADD_NORM, D.SKINNY_ADD_NORM, D.SKINNY_ADD_NORM]
    assert norm(1, prepares=0) == D.GEMV_ADD and norm(8, prepares=0) == D.MATERIALIZE
    assert norm(1, fits=0, prepares=0) == D.MATERIALIZE               # rows are selected: the product runs first


def test_a_dynamic_tanh_that_finds_its_branch_unstarted(lib):
    t = defaults()
    assert [lib.lmsf_route_deferred_tanh(ctypes.byref(t), M) for M in (1, 2, 16, 17)] == [1, 1, 1, 0]
    t.skinny_max_rows = 0                             # without the few-rows kernel
    assert lib.lmsf_route_deferred_tanh(ctypes.byref(t), 1) == 0


def test_decode_attention_splits(lib):
    t = defaults()

    def split(n, ctx, nh=32, nkv=8):
        c, s = ctypes.c_int(), ctypes.c_int()
        lib.lmsf_route_decode_attention(ctypes.byref(t), n, nh, nkv, ctx, ctypes.byref(c), ctypes.byref(s))
        assert c.value % 128 == 0 and c.value * s.value >= ctx > c.value * (s.value - 1)
        return s.value

    assert split(64, 585) == 1                       # 512 workgroups without a split
    assert split(8, 585) == 5 and split(1, 585) == 5    # one step of 128 keys a workgroup
    assert split(1, 8000) == 63 and split(8, 8000) == 8
    assert split(8, 100000) > split(8, 30000)         # long contexts: more workgroups than the chip holds at once
    t.decode_attention_splits = 2
    assert split(8, 8000) == 2


@pytest.mark.parametrize("lens,inner,n,chunk", [
    ((64,) * 8, 4096, 16, 64), ((64,), 4096, 16, 16), ((41,), 1024, 16, 16), ((40,), 1024, 16, 64), ((1, 512), 4096, 16, 32),
    ((), 64, 16, 64), ((64,) + (1,) * 250, 1024, 32, 16), ((512,), 4096, 17, 32), ((512,), 2048, 17, 16),
    # (many segments of a number of entries that a lane does not read whole)
    ((64,) + (1,) * 15, 1024, 12, 16), ((64,) + (1,) * 16, 1024, 9, 64), ((65,) + (1,) * 16, 1024, 24, 16), ((64,) + (1,) * 16, 1024, 7, 16),
    # (states that a lane does not hold)
    ((64,), 2048, 33, 16), ((64,), 2049, 33, 64), ((48,), 64, 256, 64), ((49,), 64, 256, 16), ((96,), 4096, 256, 16),
    ((97,), 4096, 256, 64), ((65,) + (1,) * 199, 64, 33, 16), ((65,) + (1,) * 200, 64, 33, 64), ((64, 512), 4096, 33, 64),
    # (no more chunks than a launch takes: segments beyond that keep the longer ones)
    ((16 * 65535,), 1, 16, 16), ((16 * 65535 + 1,), 1, 16, 64), ((32 * 65535,), 64, 16, 32), ((3, 32 * 65535 + 1), 64, 16, 64)])
def test_chunks_of_the_selective_scan(lens, inner, n, chunk):
    from lmsf_amd.ops.hip_ops import HipOps
    assert HipOps.__new__(HipOps)._scan_chunk(lens, sum(lens), inner, n) == chunk


@pytest.mark.parametrize("dim,vdim,tokens,many", [
    (512, 512, 24, 24), (256, 256, 32, 32), (255, 64, 48, 48), (128, 128, 48, 48), (127, 64, 64, 64), (64, 64, 64, 64),
    (256, 72, 64, 96), (130, 66, 64, 192), (64, 40, 64, 192), (63, 64, 96, 192), (32, 32, 96, 192), (31, 64, 192, 192)])
def test_the_matrix_memory_goes_side_by_side(lib, dim, vdim, tokens, many):
    """Where every mix of segments that was measured is no slower for it: heads of whole blocks of 64 values beside any
    number of single tokens, others (``many``) later beside many; never later than three of the other form's chunks."""
    from lmsf_amd.ops.hip_ops import HipOps
    o, chunk = HipOps.__new__(HipOps), lib.lmsf_mlstm_chunk_tokens(dim)
    for beside, least in (([], tokens), ([1] * 15, tokens), ([tokens - 1] * 8, tokens), ([1] * 64, many),
                          ([many - 1] * 3 + [1] * 64, many)):
        assert not o._memory_side_by_side([least - 1] + beside, dim, vdim, chunk)
        assert o._memory_side_by_side(beside + [least], dim, vdim, chunk)
    assert lib.lmsf_mlstm_side_tokens(dim) == max(chunk, 16)


def test_the_matrix_memory_goes_side_by_side_sooner_for_many_segments(lib):
    from lmsf_amd.ops.hip_ops import HipOps
    o = HipOps.__new__(HipOps)
    for dim, tokens in ((256, 22), (128, 32), (64, 43)):
        f = lambda lens, vdim: o._memory_side_by_side(lens, dim, vdim, 64)      # noqa: E731
        assert f([tokens] * 16 + [1] * 200, 128) and not f([tokens] * 15 + [tokens - 1], 128) and not f([tokens] * 32, 100)


@pytest.mark.parametrize("inner,rank,most", [(4096, 128, 256), (8192, 256, 64), (16384, 512, 16), (1024, 64, 2048)])
def test_scans_of_single_tokens_with_the_product_inside_end(lib, inner, rank, most):
    """Every 8 tokens read the product's matrix again: beyond 2^27 multiplications the product is a kernel of its own."""
    fits = lambda n: lib.lmsf_selective_scan_step_fits(n, inner, 16, rank, rank, rank + 16, rank + 32, rank, inner * 16, 256, 256,   # noqa: E731
                                                       256, 256)
    assert [fits(n) for n in (1, most, most + 1, 65535)] == [1, 1, 0, 0]


@pytest.mark.parametrize("heads,dim,vdim,size,most", [
    (4, 512, 64, 2, 65535), (16, 64, 64, 2, 256), (32, 127, 65, 2, 64), (32, 32, 32, 2, 48), (16, 63, 64, 2, 96), (4, 16, 16, 2, 128),
    (16, 64, 64, 4, 128), (16, 63, 64, 4, 32), (4, 16, 16, 4, 128)])
def test_the_matrix_memory_of_single_tokens_makes_its_gates_up_to(heads, dim, vdim, size, most):
    from lmsf_amd.ops.hip_ops import HipOps
    assert [HipOps._memory_step(n, heads, dim, vdim, size) for n in (1, most, most + 1)] == [True, True, dim >= 128]
    # (wide heads: in float32 all but just beyond what the chip holds at once)
    assert [HipOps._memory_step(n, 8, 128, 128, size) for n in (64, 65, 80, 81, 4096)] == [True, size == 2, size == 2, True, True]
    assert [HipOps._memory_step(n, 8, 130, 66, size) for n in (64, 65, 81, 4096)] == [True] + [size == 2] * 3


@pytest.mark.parametrize("H,rows", [(512, 1025), (1024, 1025), (1028, 513), (2048, 513), (2052, 341), (508, 8000), (8, 8000), (64, 8000)])
def test_dynamic_tanh_takes_four_rows_a_thread_from(lib, H, rows):
    """Where the chip is full of wide workgroups: narrow rows only once there are very many."""
    assert [lib.lmsf_dyt_norm_many(n, H) for n in (1, rows - 1, rows, rows + 1)] == [0, 0, 1, 1]
    assert not lib.lmsf_dyt_norm_many(100000, H + 2)

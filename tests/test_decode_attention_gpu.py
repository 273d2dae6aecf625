"""Decode attention: the first step's pages are looked up before the position is known, and a key's page is found without a
division. Page sizes that are no power of two, contexts around the ends of pages, steps and splits, stale table entries."""
from types import SimpleNamespace

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from lmsf_amd.ops import get_ops
    return get_ops()


@pytest.mark.parametrize("ps", [4, 12, 16, 20, 28, 32, 96])
@pytest.mark.parametrize("nh,nkv,d", [(16, 1, 256), (8, 2, 128), (3, 3, 48)])
@pytest.mark.parametrize("mask", [{}, {"window": 33}, {"chunk": 40}])
def test_against_the_general_kernel(ops, ps, nh, nkv, d, mask):
    g = torch.Generator().manual_seed(ps * d)
    contexts = [1, 2, ps, ps + 1, 31, 32, 33, 97, 127, 128, 129, 255, 256, 257, 300]
    width = -(-max(contexts) // ps)
    pages = len(contexts) * width + 1
    k, v = torch.randn(pages, nkv, ps, d, generator=g).bfloat16(), torch.randn(pages, nkv, d, ps, generator=g).bfloat16()
    table = torch.randperm(pages - 1, generator=g).to(torch.int32).view(len(contexts), width)
    for i, n in enumerate(contexts):
        table[i, -(-n // ps):] = pages - 1            # what lies beyond a request: a page of NaN
    k[pages - 1], v[pages - 1] = float("nan"), float("nan")
    q = torch.randn(len(contexts), nh * d, generator=g).bfloat16()
    pos = torch.tensor(contexts, dtype=torch.int32) - 1
    args = [t.cuda() for t in (q, k, v, table, torch.arange(len(contexts), dtype=torch.int32), pos)]
    run = lambda kernel: ops.paged_attention(*args, nh, nkv, d, d ** -0.5, kernel=kernel, **mask).float()
    got, want = run("mfma"), run("generic")
    # weights rounded to bfloat16 (2^-9 of values of up to 5 units, averaged) and both results rounded to it
    assert not torch.isnan(got).any() and float((got - want).abs().max()) <= 5 * 2.0 ** -8


# 2, 3, 4, 5 and 16 splits, tokens in order and (16 and more) in order of their contexts as a step lists them, last tiles of one
# token, windows that leave the first splits without keys
@pytest.mark.parametrize("n,longest,splits", [(1, 256, 2), (8, 300, 3), (8, 512, 4), (17, 600, 5), (33, 300, 3), (3, 2000, 16)])
@pytest.mark.parametrize("H,R,D,O", [(4, 32, 48, 5), (16, 224, 256, 64), (3, 160, 176, 80)])
@pytest.mark.parametrize("window", [0, 150])
@pytest.mark.parametrize("wide", [False, True])
def test_product_that_adds_up_the_splits(ops, n, longest, splits, H, R, D, O, window, wide):
    from lmsf_amd.ops.handles import SplitAttention
    g = torch.Generator().manual_seed(n * D + longest)
    ps, width = 16, longest // 16 + 1
    pages = n * width
    k, v = (torch.randn(pages, 1, *s, generator=g).bfloat16().cuda() for s in ((ps, D), (D, ps)))
    table = torch.randperm(pages, generator=g).to(torch.int32).view(n, width).cuda()
    pos = torch.randint(0, longest, (n,), generator=g, dtype=torch.int32)
    pos[0] = longest - 1
    q, w = torch.randn(n, H * D, generator=g).bfloat16().cuda(), torch.randn(H, O, R, generator=g).bfloat16().cuda()
    gate = torch.randn(n, (H * O if wide else H) + 3, generator=g).bfloat16().cuda()
    before = ops.decode_attention_splits
    ops.decode_attention_splits = splits
    try:
        args = (q, k, v, table, torch.arange(n, dtype=torch.int32).cuda(), pos.cuda(), H, 1, D, D ** -0.5, window)
        batch = SimpleNamespace(aux={}, host_seg_lens=[1] * n, host_seg_starts=list(range(n + 1)), host_seg_first_pos=pos.tolist(),
                                max_context=longest, replayed=False, all_single=True, n_tokens=n,
                                longest_first=torch.argsort(pos, descending=True, stable=True).to(torch.int32).cuda())
        kept, whole = ops.paged_attention(*args, batch=batch, keep_parts=True), ops.paged_attention(*args, batch=batch)
        assert torch.equal(whole, ops.paged_attention(*args))
    finally:
        ops.decode_attention_splits = before
    assert isinstance(kept, SplitAttention) and kept.shape == whole.shape and kept.splits > 1
    assert (kept.tokens is not None) == (n >= 16)
    outs = [torch.zeros(n, H * O, dtype=torch.bfloat16, device="cuda:0") for _ in range(2)]
    for x, out in zip((kept, whole), outs):
        ops.head_linear(x, D, w, out, O, gate=gate, gate_wide=wide)
    assert torch.equal(*outs) and outs[0].abs().sum() > 0

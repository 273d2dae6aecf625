"""Decode attention: the first step's pages are looked up before the position is known, and a key's page is found without a
division. Page sizes that are no power of two, contexts around the ends of pages, steps and splits, stale table entries."""
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

"""The few-row kernels that read their rows with wide loads, beside the general ones (the same rows off the boundaries)."""
from types import SimpleNamespace

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from lmsf_amd.ops import get_ops
    return get_ops()


def off(t, elements=1):
    """The same tensor ``elements`` off a 16-byte boundary."""
    buf = torch.empty(t.numel() + elements, dtype=t.dtype, device=t.device)[elements:].view(t.shape)
    return buf.copy_(t)


# widths below, at and beyond a workgroup's 1,024 entries, odd ones (the general kernel), ids outside the table
@pytest.mark.parametrize("H", [4, 6, 1020, 1024, 1028, 4096, 5000])
@pytest.mark.parametrize("N", [1, 9])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_embedding(ops, H, N, dtype):
    g = torch.Generator().manual_seed(H + N)
    table = torch.randn(50, H, generator=g).to(dtype).to("cuda:0")
    ids = torch.randint(0, 50, (N,), generator=g, dtype=torch.int32).to("cuda:0")
    want = table[ids.long()].float() * 1.25
    assert torch.equal(ops.embedding(ids, table, 1.25), want)
    assert torch.equal(ops.embedding(ids, off(table), 1.25), want)
    assert not ops.bad_token_seen()
    ids[-1] = 50
    out = ops.embedding(ids, table, 1.25)
    assert ops.bad_token_seen() and torch.equal(out[:-1], want[:-1]) and not out[-1].any()


# one, two and four pieces a thread and one beyond (8,192 entries in bfloat16, 4,096 in float32), remainders of a piece
@pytest.mark.parametrize("W", [8, 12, 13, 2040, 2048, 2056, 4096, 4104, 8192, 8200])
@pytest.mark.parametrize("N", [1, 5])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_rms_pair(ops, W, N, dtype):
    g = torch.Generator().manual_seed(W + N)
    a, b = (torch.randn(N, W + 24, generator=g).to(dtype).to("cuda:0")[:, :W] for _ in range(2))
    wa, wb = (torch.randn(W, generator=g).to("cuda:0") for _ in range(2))
    got = ops.rms_pair(a, b, wa, wb, 1e-5, 0.5).double()
    rms = lambda t: t.double() / torch.sqrt((t.double() ** 2).mean(-1, keepdim=True) + 1e-5)    # noqa: E731
    x, y = rms(a) * wa.double(), rms(b) * wb.double()
    want = 0.5 * (x + y)
    # float32 throughout, each term to a few 2^-24 and the sums of squares to 2^-21; the result rounded to its type
    tol = 2e-6 * (x.abs() + y.abs()) + (want.abs() * 2.0 ** -8 if dtype == torch.bfloat16 else 0)
    assert ((got - want).abs() <= tol + 1e-30).all()


# every number of entries that the lane kernel holds exactly, one it does not (12), segments of single tokens, of several and of
# more than a chunk of 64
@pytest.mark.parametrize("n", [4, 8, 12, 16, 32])
@pytest.mark.parametrize("lens", [[1, 1, 1], [1], [3, 70, 1, 200]])
def test_selective_scan_state_on_and_off_the_boundary(ops, n, lens):
    g = torch.Generator().manual_seed(n + sum(lens))
    inner, N, S = 300, sum(lens), len(lens)
    r = lambda *s: torch.randn(*s, generator=g).to("cuda:0")         # noqa: E731
    x, z, bc, dt = r(N, inner).bfloat16(), r(N, inner).bfloat16(), r(N, 2 * n).bfloat16(), r(N, inner)
    a_log, d = r(inner, n), r(inner)
    starts = [sum(lens[:i]) for i in range(S + 1)]
    seg_of = torch.repeat_interleave(torch.arange(S), torch.tensor(lens)).to(torch.int32).to("cuda:0")
    batch = SimpleNamespace(seg_of_token=seg_of, seg_starts=torch.tensor(starts, dtype=torch.int32, device="cuda:0"), n_segments=S,
                            state_slots=torch.arange(S, dtype=torch.int32, device="cuda:0"), host_seg_lens=lens, aux={},
                            all_single=max(lens) == 1)
    first = r(S, inner * n)

    def run(width):
        state = torch.zeros(S, width, device="cuda:0")
        state[:, :inner * n] = first
        y = ops.selective_scan(x, dt, bc, 0, n, z, a_log, d, state, batch)
        return y, state[:, :inner * n].clone()
    (ya, sa), (yb, sb) = run(inner * n), run(inner * n + 1)       # (the second one's rows start off 16-byte boundaries)
    assert torch.equal(ya, yb) and torch.equal(sa, sb) and not torch.equal(sa, first)


@pytest.mark.parametrize("W", [8, 12, 248, 2048, 2056, 4096, 8192])
@pytest.mark.parametrize("N", [1, 300])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_rms_pair_on_and_off_the_boundary(ops, W, N, dtype):
    g = torch.Generator().manual_seed(W + N)
    a, b = (torch.randn(N, W, generator=g).to(dtype).to("cuda:0") for _ in range(2))
    wa, wb = (torch.randn(W, generator=g).to("cuda:0") for _ in range(2))
    assert torch.equal(ops.rms_pair(a, b, wa, wb, 1e-5, 0.5), ops.rms_pair(a, b, off(wa), wb, 1e-5, 0.5))

"""The group norm that keeps its row in registers, beside the one that keeps it in LDS, against float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from lmsf_amd.ops import get_ops
    return get_ops()


def gn(v, w, groups, eps):
    p = v.view(v.shape[0], groups, -1)
    return (p / torch.sqrt((p * p).mean(-1, keepdim=True) + eps)).view(v.shape) * w


# widths below, at and beyond a wave's 256 columns, groups of whole parts of 256 and others, 1, 2 and 4 groups of four a
# thread, nearly the widest row that is taken (13,632: three rows of LDS, 12 * W bytes)
@pytest.mark.parametrize("W,groups", [(4, 1), (252, 1), (256, 1), (260, 1), (512, 2), (768, 3), (768, 2), (1023, 1),
                                      (2048, 2), (2048, 8), (4096, 4), (4100, 1), (8192, 2), (13312, 4)])
@pytest.mark.parametrize("rows", [1, 3, 513])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("form", ["branch", "add", "add to out", "rows", "average", "average first", "off the boundary"])
def test_group_norm(ops, W, groups, rows, dtype, form):
    g = torch.Generator().manual_seed(W + rows)
    r = lambda *s: torch.randn(*s, generator=g).to("cuda:0")      # noqa: E731
    shift = 1 if form == "off the boundary" else 0
    x = r(rows, W + 16).to(dtype)[:, shift:shift + W]
    wa, wb, res = r(W), r(W), r(rows, W)
    eps = 1e-5
    xd, rd = x.double(), res.double()
    rel = 2.0 ** -8 if dtype == torch.bfloat16 else 0.0

    def close(got, want, rounded):
        # float32: sums of squares of up to 13,312 terms, a square root, two roundings; all of about unit size
        assert ((got.double() - want).abs() <= 2e-6 * (1 + want.abs()) + (rel * want.abs() if rounded else 0)).all()
    if form in ("branch", "off the boundary"):
        close(ops.group_norm(x=x, x_weight=wa, groups=groups, x_eps=eps, out_dtype=dtype), gn(xd, wa.double(), groups, eps), True)
    elif form in ("add", "add to out"):
        out = ops.group_norm(x=x, x_weight=wa, residual=res, out_weight=wb if form == "add" else None, groups=groups, x_eps=eps,
                             out_eps=eps, out_dtype=dtype)
        stream = rd + gn(xd, wa.double(), groups, eps)
        close(res, stream, False)
        close(out, gn(stream, wb.double(), groups, eps) if form == "add" else stream, True)
    elif form == "rows":
        pick = torch.tensor([rows - 1, 0], dtype=torch.int32, device="cuda:0")
        out = ops.group_norm(residual=res, out_weight=wb, groups=groups, out_eps=eps, out_dtype=dtype, rows=pick)
        close(out, gn(rd[pick.long()], wb.double(), groups, eps), True)
        assert torch.equal(res.double(), rd)
    else:
        index = 0 if form == "average first" else 3
        hist, mix = r(5, rows, W), r(index + 1)
        hd = hist.double()
        out = ops.group_norm(x=x, x_weight=wa, residual=res, groups=groups, x_eps=eps, history=hist, index=index, mix=mix,
                             out_weight=wb, out_eps=eps, out_dtype=dtype)
        new = rd + gn(xd, wa.double(), groups, eps)
        mixed = (mix.double()[:index, None, None] * hd[:index]).sum(0) + mix[index].double() * new
        close(hist[index], new, False)
        assert torch.equal(hist[index + 1:].double(), hd[index + 1:])
        scale = 1 + (mix.double().abs()[:index, None, None] * hd[:index].abs()).sum(0) + (mix[index].double() * new).abs()
        assert ((res.double() - mixed).abs() <= 2e-6 * scale).all()
        # (what the average's cancellation leaves is divided by the same root mean square)
        want = gn(mixed, wb.double(), groups, eps)
        grow = gn(scale, wb.double().abs(), groups, eps) * (scale.view(rows, groups, -1).pow(2).mean(-1) /
                                                            mixed.view(rows, groups, -1).pow(2).mean(-1)).sqrt().amax(-1, keepdim=True)
        assert ((out.double() - want).abs() <= 4e-6 * (1 + grow) + rel * want.abs()).all()


# rows below and from 1,024 on (other numbers of threads), one to sixteen groups of four a thread, several groups a thread
@pytest.mark.parametrize("W,groups", [(4, 1), (252, 1), (260, 1), (512, 2), (768, 3), (1024, 1), (1020, 1), (2048, 2), (2048, 1),
                                      (2048, 8), (3072, 3), (4096, 1), (4100, 1), (8192, 1), (8192, 8), (13312, 52), (13312, 4),
                                      (12800, 5), (13632, 1)])
@pytest.mark.parametrize("rows", [1, 9, 1024])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_same_bits_in_registers_and_in_lds(ops, W, groups, rows, dtype):
    """Weights off a 16-byte boundary keep the row in LDS; the results are the same bits either way."""
    g = torch.Generator(device="cuda:0").manual_seed(W + rows)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda:0")      # noqa: E731
    x, res, hist, mix = r(rows, W).to(dtype), r(rows, W), r(4, rows, W), r(4)
    wa, wb = r(W), r(W)
    off = lambda t: torch.empty(t.numel() + 1, device="cuda:0")[1:].copy_(t)      # noqa: E731

    def run(a, b):
        args = dict(groups=groups, x_eps=1e-5, out_eps=1e-6, out_dtype=dtype)
        out = [ops.group_norm(x=x, x_weight=a, **args), ops.group_norm(residual=res.clone(), out_weight=b, **args)]
        for more in ({}, dict(history=hist.clone(), index=3, mix=mix)):
            s = res.clone()
            out += [ops.group_norm(x=x, x_weight=a, residual=s, out_weight=b, **args, **more), s, more.get("history", s)]
        return out
    for got, want in zip(run(wa, wb), run(off(wa), off(wb))):
        assert torch.equal(got, want)

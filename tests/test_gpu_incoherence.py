"""The block-128 transforms with the channel scales folded into their passes
against the same arithmetic on the CPU (torch's sgemm sums every output as one
fp32 multiply-add chain in ascending order), bit for bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def xq():
    import quantize
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    return quantize


@pytest.mark.parametrize("k,n", [(128, 128), (256, 128), (128, 384), (640, 1152)])
def test_scaled_transforms_match_cpu(xq, k, n):
    """to_inner and from_inner with magnitudes whose quotients round, and the
    forms that keep their separate passes: a transposed view, fp64 scales."""
    g = torch.Generator().manual_seed(k + n)
    w = torch.randn(k, n, generator=g)
    su = (torch.randn(k, generator=g).abs() + 0.1).half()
    sv = (torch.randn(n, generator=g) + 3.0).half()
    h = xq.hadamard128(None, torch.float32)
    want_in = xq.to_inner(w, su, sv, h)
    want_out = xq.from_inner(w, su, sv, h)
    sud, svd, hd = su.cuda(), sv.cuda(), h.cuda()
    for wd in (w.cuda(), w.t().contiguous().cuda().t()):
        assert torch.equal(xq.to_inner(wd, sud, svd, hd).cpu(), want_in)
        assert torch.equal(xq.from_inner(wd, sud, svd, hd).cpu(), want_out)
    assert torch.equal(xq.to_inner(w.cuda(), sud.double(), svd.double(), hd).cpu(), want_in)


def test_from_inner_follows_column_scales(xq):
    """from_inner's product with the column scales stays torch's where torch
    follows them: a gradient, a tangent and a batch of scales equal the CPU's."""
    g = torch.Generator().manual_seed(5)
    w = torch.randn(128, 256, generator=g)
    su = torch.randn(128, generator=g) + 3.0
    sv = torch.randn(256, generator=g) + 3.0
    svs = torch.randn(3, 256, generator=g) + 3.0
    h = xq.hadamard128(None, torch.float32)
    res = {}
    for dev in ("cpu", "cuda"):
        a = [t.to(dev) for t in (w, su, sv, svs, h)]
        v = a[2].clone().requires_grad_()
        out = xq.from_inner(a[0], a[1], v, a[4])
        assert out.requires_grad
        # one term per column: no sum whose order could differ
        grad, = torch.autograd.grad(out[7].sum(), v)
        with torch.autograd.forward_ad.dual_level():
            dual = torch.autograd.forward_ad.make_dual(a[2], a[3][0])
            tan = torch.autograd.forward_ad.unpack_dual(xq.from_inner(a[0], a[1], dual, a[4]))[1]
        batch = torch.vmap(lambda s: xq.from_inner(a[0], a[1], s, a[4]))(a[3])
        with torch.no_grad():
            assert not xq.from_inner(a[0], a[1], v, a[4]).requires_grad
        res[dev] = [t.detach().cpu() for t in (out, grad, tan, batch)]
    for got, want in zip(res["cuda"], res["cpu"]):
        assert torch.equal(got, want)


def test_scaled_transforms_more_blocks_than_workgroups(xq):
    """17 x 17 blocks (a second round for 33 of the 256 workgroups) and
    multipliers that are not symmetric."""
    k = n = 17 * 128
    g = torch.Generator().manual_seed(17)
    w = torch.randn(k, n, generator=g)
    su = torch.randn(k, generator=g) + 3.0
    sv = torch.randn(n, generator=g) + 3.0
    h = torch.randn(128, 128, generator=g) / 11.0
    dev = [t.cuda() for t in (w, su, sv, h)]
    assert torch.equal(xq.to_inner(*dev).cpu(), xq.to_inner(w, su, sv, h))
    assert torch.equal(xq.from_inner(*dev).cpu(), xq.from_inner(w, su, sv, h))


@pytest.mark.parametrize("cols", (1, 63, 64, 65, 200))
def test_had_left_ragged_columns(xq, cols):
    """Column counts around the kernel's 64-column tiles, and more tiles than
    workgroups of one launch."""
    rows = 128 * (600 if cols == 1 else 2)
    w = torch.randn(rows, cols, generator=torch.Generator().manual_seed(cols))
    h = xq.hadamard128(None, torch.float32)
    # the CPU product of the padded matrix: torch sums narrow ones otherwise
    pad = torch.cat([w, torch.zeros(rows, 256 - cols)], 1)
    want = xq.had_left(pad, h)[:, :cols]
    assert torch.equal(xq.had_left(w.cuda(), h.cuda()).cpu(), want)

"""The block-128 transforms, alone and with the channel scales folded into their
passes, against the same arithmetic on the CPU (torch's sgemm sums every output
as one fp32 multiply-add chain in ascending order), bit for bit."""
import ctypes
import subprocess

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
    """to_inner and from_inner with magnitudes whose quotients round; also from a
    transposed view and with fp64 scales."""
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


@pytest.mark.parametrize("rows,cols", [(63, 256), (64, 256), (65, 256), (127, 128), (2113, 2048)])
def test_had_right_row_tiles(xq, rows, cols):
    """Row counts around the kernel's 64-row tiles, and a ragged one with more
    tiles (34 x 16) than workgroups of a launch."""
    w = torch.randn(rows, cols, generator=torch.Generator().manual_seed(rows))
    h = xq.hadamard128(None, torch.float32)
    # the CPU product of the padded matrix: torch sums few rows otherwise
    pad = torch.cat([w, torch.zeros(max(0, 1024 - rows), cols)])
    assert torch.equal(xq.had_right(w.cuda(), h.cuda()).cpu(), xq.had_right(pad, h)[:rows])


def test_scales_of_half_weights_keep_their_passes(xq):
    """fp16 and fp64 weights: torch's own divisions and products around the
    transforms."""
    g = torch.Generator().manual_seed(9)
    w = torch.randn(256, 128, generator=g)
    su = torch.randn(256, generator=g) + 3.0
    sv = torch.randn(128, generator=g) + 3.0
    h = xq.hadamard128(None, torch.float32)
    wh = w.half().cuda()
    # fp16 weights are divided in fp32: the transforms then run on fp32
    assert torch.equal(xq.to_inner(wh, su.cuda(), sv.cuda(), h.cuda()).cpu(),
                       xq.to_inner(w.half().float(), su, sv, h))
    # fp64: 256 products and two scales a result, each side's roundings at most
    # 2^-53 of the sum of the magnitudes
    wd, hd = w.double(), h.double()
    for f in (xq.to_inner, xq.from_inner):
        bound = 2 * 259 * 2.0 ** -53 * f(wd.abs(), su.abs(), sv.abs(), hd.abs())
        got = f(wd.cuda(), su.cuda(), sv.cuda(), hd.cuda()).cpu()
        assert ((got - f(wd, su, sv, hd)).abs() <= bound).all()


CHAIN = r"""
#include <math.h>
#include <stddef.h>
// out[r][c] = fma chain over t of h[r][t] * x[t][c], 128 rows, from zero
extern "C" void left(const float* h, const float* x, float* out, int cols) {
    for (int r = 0; r < 128; ++r)
        for (int c = 0; c < cols; ++c) {
            float a = 0.0f;
            for (int t = 0; t < 128; ++t) a = fmaf(h[r * 128 + t], x[(size_t)t * cols + c], a);
            out[(size_t)r * cols + c] = a;
        }
}
// out[r][c] = fma chain over t of x[r][t] * h[t][c], 128 columns, from zero
extern "C" void right(const float* h, const float* x, float* out, int rows) {
    for (int r = 0; r < rows; ++r)
        for (int c = 0; c < 128; ++c) {
            float a = 0.0f;
            for (int t = 0; t < 128; ++t) a = fmaf(x[r * 128 + t], h[t * 128 + c], a);
            out[r * 128 + c] = a;
        }
}
"""


@pytest.fixture(scope="module")
def chain(tmp_path_factory):
    """One 128x128 block's transforms as fp32 multiply-add chains in C."""
    tmp = tmp_path_factory.mktemp("chain")
    (tmp / "chain.cpp").write_text(CHAIN)
    subprocess.run(["g++", "-O2", "-ffp-contract=off", "-shared", "-fPIC", str(tmp / "chain.cpp"),
                    "-o", str(tmp / "chain.so")], check=True)
    lib = ctypes.CDLL(str(tmp / "chain.so"))

    def run(name, h, x):
        h, x = h.contiguous(), x.contiguous()
        out = torch.empty(128, 128)
        getattr(lib, name)(*(ctypes.c_void_p(t.data_ptr()) for t in (h, x, out)), 128)
        return out

    return run


def _same_bits(got, want):
    nan = want.isnan()
    assert torch.equal(got.isnan(), nan)
    assert torch.equal(got[~nan].view(torch.int32), want[~nan].view(torch.int32))


@pytest.mark.parametrize("kind", ("subnormal", "mixed", "zeros", "inf", "nan", "overflow"))
def test_transforms_of_special_values(xq, chain, kind):
    """The matrix cores' chains equal fmaf's where inputs, products or sums are
    subnormal, zero of either sign, infinite, NaN or overflow."""
    g = torch.Generator().manual_seed(len(kind))
    w = torch.randn(128, 128, generator=g)
    h = torch.randn(128, 128, generator=g)
    if kind == "subnormal":                 # sums of a few units of 2^-149
        w = w * 2.0 ** -140
        h = h * 0.5
    elif kind == "mixed":                   # from subnormal to normal, multipliers too
        w = w * 2.0 ** torch.randint(-145, -110, (128, 128), generator=g).float()
        h = h * 2.0 ** torch.randint(-20, 4, (128, 128), generator=g).float()
    elif kind == "zeros":
        w = torch.where(torch.rand(128, 128, generator=g) < 0.5, 0.0, -0.0)
        w[5] = 1.0
    elif kind == "inf":
        w[3, 7], w[60, 90], w[61, 90] = float("inf"), float("inf"), -float("inf")
    elif kind == "nan":
        w[17, 33] = float("nan")
    else:
        w = w * 2.0 ** 126
    if kind in ("inf", "nan"):
        h[:, 40] = 0.0
    su = torch.rand(128, generator=g) + 0.5
    sv = torch.rand(128, generator=g) + 0.5
    wd, hd, sud, svd = w.cuda(), h.cuda(), su.cuda(), sv.cuda()
    _same_bits(xq.had_left(wd, hd).cpu(), chain("left", h, w))
    _same_bits(xq.had_right(wd, hd).cpu(), chain("right", h, w))
    _same_bits(xq.to_inner(wd, sud, svd, hd).cpu(),
               chain("right", h, chain("left", h, w / su[:, None] / sv)))
    _same_bits(xq.from_inner(wd, sud, svd, hd).cpu(),
               chain("right", h, chain("left", h, w) * su[:, None]) * sv)

"""MFMA tensor_linear against the oracle (plain matmul): rel 1e-5 / abs 1e-6 against the float64 evaluation, widened
only by twice the distance of the float32 evaluation of the same formula from it (tests/parity.py)."""
import ctypes
import importlib

import pytest
import torch

from oracle import products as OP
from parity import assert_parity_of

pytestmark = pytest.mark.gpu


def _check(y, formula, what="tensor_linear"):
    """formula(dtype): the reference on the CPU in that dtype."""
    assert_parity_of(y, formula, what)


@pytest.mark.parametrize("inds", [0, 1, 2])
@pytest.mark.parametrize("dims", [(64, 64), (117, 210), (16, 512), (128, 32), (8, 128), (20, 256), (1, 64), (64, 1)])
def test_tensor_linear(ops, inds, dims):
    dim_in, dim_out = dims
    g = torch.Generator().manual_seed(100 + inds)
    W = torch.randn(dim_out, dim_in, generator=g) * dim_in ** -0.5
    x = torch.randn(10, 37, dim_in, *([3] * inds), generator=g)
    y = ops.tensor_linear_fwd(inds, W.cuda(), x.cuda())
    assert tuple(y.shape) == (10, 37, dim_out) + (3,) * inds
    _check(y, lambda dt: OP.tensor_linear(inds, W.to(dt), x.to(dt)))


@pytest.mark.parametrize("inds", [0, 1, 2])
def test_tensor_linear_transposed_weight(ops, inds):
    g = torch.Generator().manual_seed(7)
    W = torch.randn(96, 48, generator=g)
    x = torch.randn(50, 96, *([3] * inds), generator=g)
    y = ops.tensor_linear_fwd(inds, W.cuda().t(), x.cuda())
    _check(y, lambda dt: OP.tensor_linear(inds, W.t().to(dt), x.to(dt)))


def test_tensor_linear_large_rows(ops):
    g = torch.Generator().manual_seed(8)
    W = torch.randn(512, 512, generator=g) / 512 ** 0.5
    x = torch.randn(3000, 512, generator=g)
    b = torch.randn(512, generator=g)
    y = ops.tensor_linear_fwd(0, W.cuda(), x.cuda(), bias=b.cuda(), act=ops.ACT_SILU)
    lin = lambda dt: torch.nn.functional.linear(x.to(dt), W.to(dt), b.to(dt))
    _check(y, lambda dt: torch.nn.functional.silu(lin(dt)))
    y2 = ops.tensor_linear_fwd(0, W.cuda(), x.cuda(), bias=b.cuda(), act=ops.ACT_LEAKY)
    _check(y2, lambda dt: torch.nn.functional.leaky_relu(lin(dt), 0.1))


def test_tensor_linear_accumulate(ops):
    g = torch.Generator().manual_seed(9)
    W = torch.randn(40, 24, generator=g)
    x = torch.randn(33, 24, 3, generator=g)
    base = torch.randn(33, 40, 3, generator=g)
    out = base.cuda().clone()
    ops.tensor_linear_fwd(1, W.cuda(), x.cuda(), out=out, accumulate=True)
    _check(out, lambda dt: base.to(dt) + OP.tensor_linear(1, W.to(dt), x.to(dt)))


@pytest.mark.parametrize("inds", [0, 1, 2])
@pytest.mark.parametrize("rows,dim_in,dim_out", [(4096, 128, 1), (77, 16, 3), (1001, 132, 4), (5, 1280, 2), (1, 64, 1)])
def test_tensor_linear_with_a_few_output_channels(ops, inds, rows, dim_in, dim_out):
    """Readout shapes (at most four output channels) have a kernel of their own: every layout, weight stride,
    bias / activation and the accumulating form against float64."""
    g = torch.Generator().manual_seed(300 + 10 * inds + dim_out)
    T = 3 ** inds
    W = torch.randn(dim_out, dim_in, generator=g) * dim_in ** -0.5
    x = torch.randn(rows, dim_in, *([3] * inds), generator=g)
    ref = lambda dt: torch.einsum("oi,ri...->ro...", W.to(dt), x.to(dt))
    y = ops.tensor_linear_fwd(inds, W.cuda(), x.cuda())
    assert tuple(y.shape) == (rows, dim_out) + (3,) * inds
    _check(y, ref)
    # a weight with strides (the transposed view the input gradient of an n -> few linear would pass is the other
    # shape; this is the forward of a layer whose weight is stored transposed)
    Wt = W.t().contiguous().cuda().t()
    assert dim_out == 1 or Wt.stride() == (1, dim_out)
    _check(ops.tensor_linear_fwd(inds, Wt, x.cuda()), ref)
    # component-major output
    ycm = ops.tensor_linear_fwd(inds, W.cuda(), x.cuda(), y_layout=ops.LAYOUT_COMP_CHAN)
    _check(ycm.reshape(rows, T, dim_out), lambda dt: ref(dt).reshape(rows, dim_out, T).transpose(1, 2))
    # accumulate
    base = torch.randn(rows, dim_out, *([3] * inds), generator=g)
    out = base.cuda().clone()
    ops.tensor_linear_fwd(inds, W.cuda(), x.cuda(), out=out, accumulate=True)
    _check(out, lambda dt: base.to(dt) + ref(dt))
    if inds == 0:
        b = torch.randn(dim_out, generator=g)
        yb = ops.tensor_linear_fwd(0, W.cuda(), x.cuda(), bias=b.cuda(), act=ops.ACT_SILU)
        _check(yb, lambda dt: torch.nn.functional.silu(ref(dt) + b.to(dt)))


def test_tensor_linear_empty_and_errors(ops):
    W = torch.randn(8, 4).cuda()
    y = ops.tensor_linear_fwd(1, W, torch.empty(0, 4, 3).cuda())
    assert tuple(y.shape) == (0, 8, 3)
    with pytest.raises(RuntimeError, match="channel dim size mismatch"):
        ops.tensor_linear_fwd(0, W, torch.randn(3, 5).cuda())
    with pytest.raises(RuntimeError, match="3d"):
        ops.tensor_linear_fwd(1, W, torch.randn(3, 4, 2).cuda())
    with pytest.raises(RuntimeError, match="contiguous"):
        ops.tensor_linear_fwd(0, W, torch.randn(4, 3).cuda().t())
    with pytest.raises(RuntimeError, match="up to 2"):
        ops.tensor_linear_fwd(3, W, torch.randn(2, 4, 3, 3, 3).cuda())


@pytest.mark.parametrize("inds", [0, 1, 2])
def test_tensor_linear_autograd(pkg, inds):
    tp = importlib.import_module("learned-dynamics_amd.tensor_products")
    g = torch.Generator().manual_seed(10)
    W = torch.randn(70, 50, generator=g)
    x = torch.randn(6, 21, 50, *([3] * inds), generator=g)
    dy = torch.randn(6, 21, 70, *([3] * inds), generator=g)
    Wr, xr = W.clone().requires_grad_(True), x.clone().requires_grad_(True)
    OP.tensor_linear(inds, Wr, xr).backward(dy)
    Wg, xg = W.cuda().requires_grad_(True), x.cuda().requires_grad_(True)
    tp.tensor_linear(inds, Wg, xg).backward(dy.cuda())
    torch.testing.assert_close(xg.grad.cpu(), xr.grad, rtol=1e-5, atol=1e-5)
    torch.testing.assert_close(Wg.grad.cpu(), Wr.grad, rtol=1e-5, atol=1e-4)


@pytest.mark.parametrize("mode", [0, 1, 2])
@pytest.mark.parametrize("shape", [(5000, 512, 512, 0), (3000, 96, 200, 0), (2000, 64, 128, 1), (1500, 160, 72, 2),
                                   (1024, 64, 64, 0), (4096, 768, 256, 0),
                                   # large enough for the 256x256-tile kernel (ragged last tile; transposed output)
                                   (140001, 64, 512, 0), (90001, 32, 256, 1)])
def test_linear_modes_agree_with_float64(ops, mode, shape):
    """fp32 MFMA (mode 0), bf16x3-split MFMA (mode 1) and two-piece fp16 split (mode 2) against a float64
    product: all must sit at fp32 rounding level; the split paths use pre-packed weights and may
    transpose (row, comp) outputs."""
    rows, dim_in, dim_out, inds = shape
    T = 3 ** inds
    g = torch.Generator().manual_seed(77)
    W = torch.randn(dim_out, dim_in, generator=g) / dim_in ** 0.5
    b = torch.randn(dim_out, generator=g)
    x_cm = torch.randn(rows, T, dim_in, generator=g)                   # component-major rows
    def ref_aos(dt):
        ref = torch.nn.functional.silu(x_cm.to(dt) @ W.to(dt).t() + b.to(dt))            # (rows, T, O)
        return ref.transpose(1, 2).reshape(rows, dim_out, *([3] * inds))

    prev = ops.get_linear_mode()
    try:
        ops.set_linear_mode(mode)
        C = ops.LAYOUT_COMP_CHAN
        y = ops.tensor_linear_fwd(inds, W.cuda(), x_cm.cuda() if inds else x_cm[:, 0].contiguous().cuda(),
                                  bias=b.cuda(), act=ops.ACT_SILU, x_layout=C if inds else 0)
    finally:
        ops.set_linear_mode(prev)
    _check(y, ref_aos, f"tensor_linear mode {mode} {shape}")


@pytest.mark.parametrize("shape", [(70000, 512, 512, 1), (3001, 256, 192, 0), (1500, 96, 16, 2), (2048, 1280, 64, 0),
                                   (1024, 64, 8, 0), (40000, 160, 130, 1), (140001, 64, 256, 2),
                                   # column tiles chosen to divide the width and narrowed for few rows
                                   (49152, 128, 384, 1), (16384, 256, 384, 0), (512, 512, 512, 1), (300, 64, 96, 2),
                                   (700, 64, 2080, 0), (2048, 64, 1056, 0),
                                   # few rows, at most 64 columns, long K: the waves of a workgroup split K
                                   (18432, 1280, 16, 0), (6144, 1280, 64, 2), (33, 512, 32, 1), (1000, 544, 40, 0),
                                   (8192, 768, 64, 1), (32768, 768, 16, 1), (1, 2048, 3, 0)])
def test_linear_f16x2_rows_of_very_different_size(ops, shape):
    """mg_tensor_linear_f16x2 through the C ABI.  Rows spanning twelve orders of magnitude: the per-row
    power-of-two scales keep the error relative to EACH row's own scale at fp32 rounding level (a single
    scale for the tensor would not); weight rows of different size likewise.  Also: accumulate, the row
    maxima the epilogue emits, and their use as the next call's bounds."""
    rows, dim_in, dim_out, act = shape
    g = torch.Generator().manual_seed(rows + dim_out)
    W = torch.randn(dim_out, dim_in, generator=g) / dim_in ** 0.5
    W[::3] *= 1e-4
    W[1::5] *= 300.0
    b = torch.randn(dim_out, generator=g) * 1e-3
    x = torch.randn(rows, dim_in, generator=g)
    x *= 10.0 ** torch.randint(-6, 7, (rows, 1), generator=g).float()
    pre = x.double() @ W.double().t() + b.double()
    ref = {0: pre, 1: torch.nn.functional.silu(pre), 2: torch.where(pre > 0, pre, 0.1 * pre)}[act]
    # error budget per entry: fp32-level rounding of a length-K dot product whose terms are bounded by
    # |x row| * |W row|, plus rel 2e-6 of the result (rounding, hardware exp2 / reciprocal in SiLU)
    budget = (x.abs().amax(1, keepdim=True).double() * W.abs().amax(1).double() * 4e-7 * dim_in ** 0.5
              + 2e-6 * ref.abs() + 1e-30)
    y, ymax = ops.tensor_linear_f16x2(W.cuda(), x.cuda(), bias=b.cuda(), act=act, want_rowmax=True)
    assert bool(((y.cpu().double() - ref).abs() <= budget).all())
    assert torch.equal(ymax.amax(dim=1), y.abs().amax(dim=1))
    # explicit bounds: exact maxima, and a loose shared bound (accuracy must not depend on tightness)
    y2 = ops.tensor_linear_f16x2(W.cuda(), x.cuda(), ops.row_absmax(x.cuda()) * 100.0, bias=b.cuda(), act=act)
    assert bool(((y2.cpu().double() - ref).abs() <= budget).all())
    # accumulate into an existing result, bounds taken from the previous call's emitted maxima
    W2 = torch.randn(dim_in, dim_out, generator=g) / dim_out ** 0.5
    if dim_out % 32 == 0 and dim_out >= 64:
        base = torch.randn(rows, dim_in, generator=g)
        out = base.cuda().clone()
        ops.tensor_linear_f16x2(W2.cuda(), y, ymax, out=out, accumulate=True)
        ref2 = base.double() + y.cpu().double() @ W2.double().t()
        budget2 = (y.cpu().abs().amax(1, keepdim=True).double() * W2.abs().amax(1).double() * 4e-7 * dim_out ** 0.5
                   + 2e-6 * ref2.abs() + 4e-7 * base.abs().double() + 1e-30)
        assert bool(((out.cpu().double() - ref2).abs() <= budget2).all())


@pytest.mark.parametrize("nodes,T,dim_in,dim_out", [(700, 9, 320, 16), (2048, 9, 1280, 16), (2048, 3, 1280, 64),
                                                    (37, 3, 640, 24)])
def test_linear_f16x2_component_outputs_and_node_bounds(ops, nodes, T, dim_in, dim_out):
    """Rows that are (node, comp) pairs with one bound per node, output stored (node, chan, comp); the shapes with
    K >= 512 take the kernel whose waves split K."""
    g = torch.Generator().manual_seed(4)
    W = torch.randn(dim_out, dim_in, generator=g) / dim_in ** 0.5
    x = torch.randn(nodes, T, dim_in, generator=g)
    bound = x.abs().amax(dim=(1, 2)).reshape(nodes, 1)
    y = ops.tensor_linear_f16x2(W.cuda(), x.reshape(nodes * T, dim_in).cuda(), bound.cuda(), out_comps=T,
                                rows_per_bound=T)
    ref = lambda dt: (x.to(dt) @ W.to(dt).t()).transpose(1, 2)
    assert y.shape == (nodes, dim_out, T)
    _check(y, ref, "f16x2, component outputs, one bound per node")
    base = torch.randn(nodes, dim_out, T, generator=g)
    out = base.cuda().clone()
    ops.tensor_linear_f16x2(W.cuda(), x.reshape(nodes * T, dim_in).cuda(), bound.cuda(), out=out, accumulate=True,
                            out_comps=T, rows_per_bound=T)
    _check(out, lambda dt: base.to(dt) + ref(dt), "f16x2, component outputs, accumulate")


@pytest.mark.parametrize("inds,rows,dim_in,dim_out", [(1, 12000, 64, 256), (2, 4000, 16, 128), (1, 11000, 40, 64)])
def test_rows_per_component_formed_once_for_several_weights(ops, inds, rows, dim_in, dim_out):
    """components_as_rows + x_rows=: two weights applied to the same x give, bit for bit, what two plain calls give;
    None (and the plain route) when the input would not take that path."""
    g = torch.Generator().manual_seed(inds + rows)
    x = torch.randn(rows, dim_in, *([3] * inds), generator=g).cuda()
    shared = ops.components_as_rows(inds, x)
    assert shared is not None and shared[0].shape[0] == rows * 3 ** inds and shared[0].shape[1] % 32 == 0
    for k in range(2):
        W = (torch.randn(dim_out, dim_in, generator=g) / dim_in ** 0.5).cuda()
        y0 = ops.tensor_linear_fwd(inds, W, x, y_layout=ops.LAYOUT_COMP_CHAN)
        y1 = ops.tensor_linear_fwd(inds, W, x, y_layout=ops.LAYOUT_COMP_CHAN, x_rows=shared)
        assert torch.equal(y0, y1)
        _check(y1, lambda dt: OP.tensor_linear(inds, W.cpu().to(dt), x.cpu().to(dt)).reshape(
            rows, dim_out, 3 ** inds).transpose(1, 2), "shared rows per component")
    assert ops.components_as_rows(inds, x[:100].contiguous()) is None
    assert ops.components_as_rows(0, x) is None


def test_row_bounds_carried_as_factor_and_offset(ops):
    """ScaledBound: a chain of three layers that hands the first layer's row maxima on as (array, factor, offset)
    gives the float64 chain at the layer tolerance, the factors are upper bounds of what they stand for, and a
    negative factor is refused by the library."""
    g = torch.Generator().manual_seed(21)
    x = (torch.randn(3000, 128, generator=g) * 10.0 ** torch.randint(-3, 4, (3000, 1), generator=g).float()).cuda()
    Ws = [(torch.randn(256, 128, generator=g) / 128 ** 0.5).cuda(), (torch.randn(256, 256, generator=g) / 16).cuda(),
          (torch.randn(192, 256, generator=g) / 16).cuda()]
    bs = [torch.randn(256, generator=g).cuda() * 0.1, torch.randn(256, generator=g).cuda() * 0.1, None]
    bound = ops.ScaledBound(ops.row_absmax(x))
    h = x
    for k, (W, b) in enumerate(zip(Ws, bs)):
        l1, bmax = ops.linear_out_bound_factors(W, b)
        assert l1 >= float(W.abs().sum(1).amax()) and bmax >= (float(b.abs().amax()) if b is not None else 0.0)
        h_next = ops.tensor_linear_f16x2(W, h, bound, bias=b, act=ops.ACT_SILU if k < 2 else ops.ACT_NONE)
        assert bool((h_next.abs().amax(1, keepdim=True) <= bound.through(l1, bmax).tensor() * (1 + 1e-6)).all())
        h, bound = h_next, bound.through(l1, bmax)

    def chain(dt):
        t = x.cpu().to(dt)
        for k, (W, b) in enumerate(zip(Ws, bs)):
            t = torch.nn.functional.linear(t, W.cpu().to(dt), None if b is None else b.cpu().to(dt))
            t = torch.nn.functional.silu(t) if k < 2 else t
        return t
    _check(h, chain, "three layers on one array of row maxima")
    assert ops.linear_out_bound_factors(Ws[0], bs[0]) == ops.linear_out_bound_factors(Ws[0], bs[0])
    with torch.no_grad():
        Ws[0].mul_(3.0)
    assert ops.linear_out_bound_factors(Ws[0], bs[0])[0] > 2.9 * l1 * 0 + float(Ws[0].abs().sum(1).amax()) * 0.999
    with pytest.raises(RuntimeError, match="non-negative"):
        ops.tensor_linear_f16x2(Ws[1], h.new_zeros(300, 256), ops.ScaledBound(h.new_ones(300, 1), -1.0, 0.0))


def test_linear_out_bound_is_an_upper_bound(ops):
    g = torch.Generator().manual_seed(5)
    W = torch.randn(96, 64, generator=g).cuda()
    b = torch.randn(96, generator=g).cuda()
    x = torch.randn(500, 64, generator=g).cuda() * 3
    xb = ops.row_absmax(x)
    assert torch.equal(xb[:, 0], x.abs().amax(1))
    yb = ops.linear_out_bound(W, b, xb)
    y = torch.nn.functional.silu(torch.nn.functional.linear(x, W, b))
    assert bool((y.abs().amax(1, keepdim=True) <= yb).all())
    unit = ops.linear_out_bound(W, b, None)                      # inputs bounded by 1
    y1 = torch.nn.functional.linear(torch.rand(100, 64, device="cuda") * 2 - 1, W, b)
    assert unit.shape == (1, 1) and bool((y1.abs().amax() <= unit).all())
    assert ops.linear_out_bound(W, b, None) is unit                # cached per parameter version
    with torch.no_grad():
        W.mul_(2.0)
    assert float(ops.linear_out_bound(W, b, None)) > float(unit)  # recomputed after an in-place update


def test_packed_weight_cache_tracks_in_place_updates(ops):
    prev = ops.get_linear_mode()
    try:
        ops.set_linear_mode(1)
        W = torch.randn(128, 128, device="cuda")
        x = torch.randn(2048, 128, device="cuda")
        y1 = ops.tensor_linear_fwd(0, W, x)
        with torch.no_grad():
            W.mul_(2.0)
        y2 = ops.tensor_linear_fwd(0, W, x)
        torch.testing.assert_close(y2, 2 * y1, rtol=1e-5, atol=1e-5)
    finally:
        ops.set_linear_mode(prev)


def test_weight_written_behind_the_version_counter(pkg, ops):
    """`param.data.mul_()` changes a weight without touching its version counter: the caches cannot see it, and
    ops.invalidate_weight_caches() is the documented remedy (layer caches included)."""
    painn = importlib.import_module("learned-dynamics_amd.painn")
    torch.manual_seed(5)
    upd = painn.Update(64).cuda().eval()
    x_a, x_v = torch.randn(1, 700, 64).cuda(), torch.randn(1, 700, 64, 3).cuda()
    with torch.no_grad():
        upd(x_a, x_v)                                            # fills the caches
        for p in upd.parameters():
            p.data.mul_(1.25)
        ops.invalidate_weight_caches()
        got = upd(x_a, x_v)
        fresh = painn.Update(64).cuda().eval()
        fresh.load_state_dict(upd.state_dict())
        ref = fresh(x_a, x_v)
    for a, b in zip(got, ref):
        torch.testing.assert_close(a, b, rtol=0, atol=0)


def _segment_lengths(kind, n, g):
    if kind == "long":
        return torch.randint(40, 140, (n,), generator=g)
    if kind == "short":
        return torch.randint(0, 9, (n,), generator=g)
    if kind == "aligned":
        return torch.tensor([32, 64, 1, 31, 32, 0, 0, 96, 33, 31] * (n // 10))
    return torch.cat([torch.randint(0, 5, (n // 2,), generator=g), torch.randint(20, 300, (n - n // 2,), generator=g)])[
        torch.randperm(n, generator=g)]


@pytest.mark.parametrize("dim_in,dim_out,act,kind,want_rows", [(512, 512, 2, "long", False), (96, 256, 0, "short", True),
                                                               (256, 256, 1, "aligned", True), (64, 768, 2, "mixed", False)])
def test_linear_with_row_sums_in_the_epilogue(ops, dim_in, dim_out, act, kind, want_rows):
    """out[s] = scale * sum over the rows of segment s of act(x W^T + b), against the plain GEMM followed by
    the segment sum, and against float64; segments placed in every way relative to the kernel's 32-row blocks."""
    g = torch.Generator().manual_seed(dim_in + dim_out)
    n_seg = 300
    lengths = _segment_lengths(kind, n_seg, g)
    seg = torch.repeat_interleave(torch.arange(n_seg), lengths)
    rows = int(seg.numel())
    x = (torch.randn(rows, dim_in, generator=g) * (torch.rand(rows, 1, generator=g) * 3)).cuda()
    W = (torch.randn(dim_out, dim_in, generator=g) / dim_in ** 0.5).cuda()
    b = torch.randn(dim_out, generator=g).cuda()
    row_ptr = ops.segment_row_ptr(seg.int().cuda(), n_seg)
    bound = ops.row_absmax(x)
    out, y = ops.tensor_linear_f16x2_rowsum(W, x, bound, row_ptr, seg.int().cuda(), n_seg, bias=b, act=act, scale=0.5,
                                            want_rows=want_rows)
    y_ref = ops.tensor_linear_f16x2(W, x, bound, bias=b, act=act)
    if want_rows:
        assert torch.equal(y, y_ref)          # the same accumulators through another epilogue
    else:
        assert y is None
    two_step = 0.5 * ops.segment_sum_csr(y_ref, row_ptr, n_seg)
    def ref(dt):
        z = x.cpu().to(dt) @ W.cpu().to(dt).T + b.cpu().to(dt)
        z = torch.nn.functional.silu(z) if act == 1 else (torch.nn.functional.leaky_relu(z, 0.1) if act == 2 else z)
        return 0.5 * torch.zeros(n_seg, dim_out, dtype=dt).index_add_(0, seg, z)

    _check(out, ref, f"row sums in the epilogue {dim_in}->{dim_out} {kind}")
    _check(two_step, ref, f"GEMM then segment sum {dim_in}->{dim_out} {kind}")
    assert not bool(out[(lengths == 0).cuda()].any())


@pytest.mark.parametrize("rows,dim_in,dim_out", [(4500, 96, 512), (20001, 64, 256), (70000, 64, 256)])
def test_row_sums_in_the_epilogue_at_every_tile_width(ops, rows, dim_in, dim_out):
    """Row counts for which the rule takes tiles of 64, 128 and 256 columns: the rows bit for bit those of the plain linear (an
    element's order of summation does not depend on the tile), the sums to fp32 rounding."""
    g = torch.Generator().manual_seed(rows)
    n_seg = rows // 16
    seg = torch.sort(torch.randint(0, n_seg, (rows,), generator=g)).values
    x = torch.randn(rows, dim_in, generator=g).cuda()
    W, b = (torch.randn(dim_out, dim_in, generator=g) / dim_in ** 0.5).cuda(), torch.randn(dim_out, generator=g).cuda()
    row_ptr, bound = ops.segment_row_ptr(seg.int().cuda(), n_seg), ops.row_absmax(x)
    args = (W, x, bound, row_ptr, seg.int().cuda(), n_seg)
    out, y = ops.tensor_linear_f16x2_rowsum(*args, bias=b, act=2, want_rows=True)
    assert torch.equal(y, ops.tensor_linear_f16x2(W, x, bound, bias=b, act=2))
    assert torch.equal(ops.tensor_linear_f16x2_rowsum(*args, bias=b, act=2)[0], out)
    z = torch.nn.functional.leaky_relu(x.cpu().double() @ W.cpu().double().T + b.cpu().double(), 0.1)
    _check(out, lambda dt: torch.zeros(n_seg, dim_out, dtype=dt).index_add_(0, seg, z.to(dt)), f"row sums, {rows} rows")


@pytest.mark.parametrize("inds,rows,dim_in,dim_out", [(2, 8000, 16, 64), (1, 22000, 40, 96), (1, 30000, 64, 256), (1, 25000, 70, 64)])
def test_component_major_output_from_reference_layout_at_many_rows(ops, inds, rows, dim_in, dim_out):
    """x in the reference layout (rows, chan, 3..), y component-major (rows, 3^inds, chan_out): at many rows
    the dispatcher transposes x and uses the plain-row matrix path (K zero-padded to a multiple of 32).
    Against the einsum of extensions/tensor_ops/test.py:9-15 in float64, with accumulate."""
    T = 3 ** inds
    assert rows * T >= 65536
    g = torch.Generator().manual_seed(rows)
    x = torch.randn(rows, dim_in, *([3] * inds), generator=g).cuda()
    W = (torch.randn(dim_out, dim_in, generator=g) / dim_in ** 0.5).cuda()
    y = ops.tensor_linear_fwd(inds, W, x, y_layout=ops.LAYOUT_COMP_CHAN)
    ref = lambda dt: torch.einsum("oi,bit->bto", W.cpu().to(dt), x.cpu().to(dt).reshape(rows, dim_in, T))
    assert y.shape == (rows, T, dim_out)
    _check(y, ref, f"component-major output, {rows} rows")
    y2 = ops.tensor_linear_fwd(inds, W, x, y_layout=ops.LAYOUT_COMP_CHAN, out=y.clone(), accumulate=True)
    _check(y2, lambda dt: y.cpu().to(dt) + ref(dt), f"component-major output, accumulate, {rows} rows")
    # the generic kernel, which serves fewer rows, on the first rows
    small = ops.tensor_linear_fwd(inds, W, x[:500].contiguous(), y_layout=ops.LAYOUT_COMP_CHAN)
    _check(small, lambda dt: ref(dt)[:500], "component-major output, generic kernel")


@pytest.mark.parametrize("rows,dim,comps,pad", [(1, 5, 3, 32), (3, 40, 9, 64), (1030, 256, 9, 256), (4100, 16, 9, 32), (5000, 128, 3, 128),
                                                (2, 250, 70, 256)])
def test_components_to_rows(pkg, rows, dim, comps, pad):
    """One plain row per (row, component), zero-padded, and its largest magnitude, bit for bit: rows of half a wave to four
    pieces, channel counts that are no multiple of four, a last workgroup that is not full."""
    L = importlib.import_module("learned-dynamics_amd._lib")
    x = torch.randn(rows, dim, comps, generator=torch.Generator().manual_seed(rows + dim)).cuda()
    y, m = torch.full((rows * comps, pad), 7., device="cuda"), torch.full((rows * comps,), 7., device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    L.check(L.load().mg_components_to_rows(x.data_ptr(), rows, dim, comps, pad, y.data_ptr(), m.data_ptr(), stream))
    want = torch.nn.functional.pad(x.transpose(1, 2), (0, pad - dim)).reshape(rows * comps, pad)
    assert torch.equal(y, want) and torch.equal(m, want.abs().amax(1))


@pytest.mark.parametrize("inds,rows,dim_in,dim_out", [(1, 321, 64, 256), (1, 1000, 40, 128), (2, 117, 32, 256), (2, 8200, 16, 256), (2, 300, 64, 96)])
def test_component_output_in_runs(ops, inds, rows, dim_in, dim_out):
    """Reference layout in and out through the plain-row kernels: tiles that begin and end inside a row's components, nine of
    them in runs (short reductions, whole tiles of 64 columns) and otherwise, and accumulation, against float64."""
    g = torch.Generator().manual_seed(rows)
    x = torch.randn(rows, dim_in, *([3] * inds), generator=g).cuda()
    W = (torch.randn(dim_out, dim_in, generator=g) / dim_in ** 0.5).cuda()
    ref = lambda dt: torch.einsum("oi,bit->bot", W.cpu().to(dt), x.cpu().to(dt).reshape(rows, dim_in, -1)).reshape(rows, dim_out, *([3] * inds))
    y = ops.tensor_linear_fwd(inds, W, x)
    _check(y, ref, f"components {rows} x {dim_in} -> {dim_out}")
    rows2 = x.reshape(rows, dim_in, -1).transpose(1, 2).reshape(-1, dim_in).contiguous()
    if dim_in % 32 == 0 and dim_in >= 64:
        y2 = ops.tensor_linear_f16x2(W, rows2, ops.row_absmax(rows2), out_comps=3 ** inds, out=y.clone(), accumulate=True)
        _check(y2.reshape(y.shape), lambda dt: y.cpu().to(dt) + ref(dt), "accumulated")


def test_linear_with_row_sums_edge_cases(ops):
    W = torch.randn(256, 64).cuda()
    row_ptr = torch.zeros(11, dtype=torch.int32, device="cuda")
    seg = torch.empty(0, dtype=torch.int32, device="cuda")
    out, y = ops.tensor_linear_f16x2_rowsum(W, torch.empty(0, 64, device="cuda"), torch.ones(1, 1, device="cuda"), row_ptr, seg,
                                            10, want_rows=True)
    assert out.shape == (10, 256) and not bool(out.any()) and y.shape == (0, 256)
    # one segment holding every row, fewer rows than a tile
    x = torch.randn(77, 64).cuda()
    seg = torch.zeros(77, dtype=torch.int32, device="cuda")
    row_ptr = torch.tensor([0, 77], dtype=torch.int32, device="cuda")
    out, _ = ops.tensor_linear_f16x2_rowsum(W, x, ops.row_absmax(x), row_ptr, seg, 1)
    _check(out, lambda dt: (x.cpu().to(dt) @ W.cpu().to(dt).T).sum(0, keepdim=True), "one segment of 77 rows")
    with pytest.raises(RuntimeError, match="multiple of 256"):
        ops.tensor_linear_f16x2_rowsum(W[:128].contiguous(), x, ops.row_absmax(x), row_ptr, seg, 1)


@pytest.mark.parametrize("inds", [0, 1, 2])
def test_plain_entry_point_through_ctypes(pkg, inds):
    """mg_tensor_linear called as a foreign caller would (raw pointers, element strides of W, the current stream):
    the transposed view of W, bias + SiLU for inds = 0, accumulation into y, and zero rows."""
    import ctypes
    L = importlib.import_module("learned-dynamics_amd._lib")
    lib = L.load()
    g = torch.Generator().manual_seed(40 + inds)
    Wt = torch.randn(48, 96, generator=g)                      # stored (dim_in, dim_out): W = Wt.t()
    x = torch.randn(33, 48, *([3] * inds), generator=g)
    bias = torch.randn(96, generator=g) if inds == 0 else None
    y0 = torch.randn(33, 96, *([3] * inds), generator=g)
    Wd, xd, yd = Wt.cuda(), x.cuda(), y0.cuda()
    bd = bias.cuda() if bias is not None else None
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    act = 1 if inds == 0 else 0
    L.check(lib.mg_tensor_linear(inds, Wd.data_ptr(), Wd.stride(1), Wd.stride(0), xd.data_ptr(), 33, 48, 96,
                                 bd.data_ptr() if bd is not None else None, act, 0, yd.data_ptr(), st))
    def ref(dt):
        lin = OP.tensor_linear(inds, Wt.t().to(dt), x.to(dt))
        return torch.nn.functional.silu(lin + bias.to(dt)) if inds == 0 else lin

    _check(yd, ref)
    L.check(lib.mg_tensor_linear(inds, Wd.data_ptr(), Wd.stride(1), Wd.stride(0), xd.data_ptr(), 33, 48, 96,
                                 None, 0, 1, yd.data_ptr(), st))
    _check(yd, lambda dt: ref(dt) + OP.tensor_linear(inds, Wt.t().to(dt), x.to(dt)))
    before = yd.clone()
    L.check(lib.mg_tensor_linear(inds, Wd.data_ptr(), Wd.stride(1), Wd.stride(0), xd.data_ptr(), 0, 48, 96,
                                 None, 0, 0, yd.data_ptr(), st))
    assert torch.equal(yd, before)


@pytest.mark.parametrize("span", [1e4, 1e6])
def test_linear_f16x2_in_row_dynamic_range_meeting_zero_weights(ops, span):
    """Inside ONE row: a few entries `span` times larger than the rest, and weights that are exactly zero on those
    entries, so the result is made of the small entries alone.  The row scale puts the row maximum M at 2^14..2^15
    and every entry is carried by two fp16 pieces with an absolute error of at most 2^-25 in scaled units, i.e.
    2^-39 M per term whatever the term's own size: the error bound is relative to the ROW, not to the term.
      span 1e4: the small terms still carry about 2^-26 relative error each: the rel 1e-5 / abs 1e-6 contract holds
                on the result itself;
      span 1e6: the bound 2^-39 M |w| sqrt(K) is about 1e-5 of a result of order one: the edge of the contract, and
                what this test pins is that bound (rows of the models carry activations and products of order one,
                their in-row spans stay far below 1e4)."""
    g = torch.Generator().manual_seed(int(span) % 97)
    rows, dim_in, dim_out = 4096, 512, 256
    x = torch.randn(rows, dim_in, generator=g)
    big = torch.zeros(dim_in, dtype=torch.bool)
    big[::37] = True
    x[:, big] *= span
    W = torch.randn(dim_out, dim_in, generator=g) / dim_in ** 0.5
    W[:, big] = 0.0
    ref = x.double() @ W.double().t()
    y = ops.tensor_linear_f16x2(W.cuda(), x.cuda())
    small = x.clone()
    small[:, big] = 0.0
    ref32 = (small @ W.t()).double()                          # fp32 evaluation of the same sum (the zeros drop out exactly)
    e_ref = float((ref32 - ref).abs().max())
    err = (y.cpu().double() - ref).abs()
    contract = 1e-6 + 1e-5 * ref.abs() + 2 * e_ref            # the tolerance on the result, as everywhere else
    row_scale = (3 * 2.0 ** -39 * dim_in ** 0.5) * x.abs().amax(1, keepdim=True).double() * W.abs().amax(1).double()
    print(f"[f16x2 in-row span {span:g}] max err {float(err.max()):.3g}  e_ref {e_ref:.3g}  max row-scale bound "
          f"{float(row_scale.max()):.3g}  |ref| max {float(ref.abs().max()):.3g}")
    if span <= 1e4:
        assert bool((err <= contract).all()), (float(err.max()), e_ref)
    else:
        assert bool((err <= contract + row_scale).all()), (float(err.max()), e_ref)
        assert float(err.max()) < 3e-5 * float(ref.abs().max())


@pytest.mark.parametrize("inds,rows,dim_in,dim_out", [(0, 5000, 117, 210), (0, 70, 16, 512), (0, 1, 33, 31),
                                                      (0, 100003, 512, 384), (1, 3000, 48, 70), (2, 900, 20, 130),
                                                      (1, 300, 48, 70), (2, 100, 20, 130), (1, 8192, 64, 256),
                                                      (2, 4001, 16, 16), (1, 2000, 300, 64)])
def test_weight_gradient_against_float64(ops, inds, rows, dim_in, dim_out):
    """dW[o, i] = sum over rows and components of dy[r, o, t] x[r, i, t]: plain rows through the matrix cores (fp32
    ones where a dimension is not a multiple of 4 or the rows are few, else split fp16; tiles of 128 x 128 with ragged
    edges, row slices that do not divide the rows), tensor components transposed to plain rows for the matrix cores
    when there are at least 4096 of them and the channels fit 256, else through the vector kernel; slices are summed
    in a fixed order, so two runs agree bit for bit."""
    g = torch.Generator().manual_seed(rows + dim_in)
    comps = (3,) * inds
    x = torch.randn(rows, dim_in, *comps, generator=g).cuda()
    dy = torch.randn(rows, dim_out, *comps, generator=g).cuda()
    got = ops.tensor_linear_wgrad(inds, dy, x)
    want = torch.einsum("ro...,ri...->oi", dy.double(), x.double())
    fp32 = torch.einsum("ro...,ri...->oi", dy, x).double()
    scale = float(want.abs().max())
    err, err_ref = float((got.double() - want).abs().max()), float((fp32 - want).abs().max())
    assert err <= 1e-6 + 1e-5 * scale + 2 * err_ref, (err, err_ref, scale)
    assert torch.equal(ops.tensor_linear_wgrad(inds, dy, x), got)


@pytest.mark.parametrize("rows,dim_in,dim_out", [(4096, 64, 64), (5000, 68, 132), (40001, 512, 512), (33333, 128, 512),
                                                 (9000, 260, 64), (20011, 16, 512), (4100, 4, 8)])
@pytest.mark.parametrize("bounds", ["scanned", "row maxima", "loose"])
def test_weight_gradient_split_fp16(ops, rows, dim_in, dim_out, bounds):
    """Plain rows on the fp16 matrix cores with hi + lo operands: tiles with ragged edges, row slices that do not
    divide the rows, rows whose magnitudes span 2^12, the scales taken from the operands themselves, from row maxima
    or from a bound 1000 times too large; to the tolerance of the fp32 kernels, and the same bits on every run."""
    g = torch.Generator().manual_seed(rows + 3 * dim_in + dim_out)
    spread = torch.exp2(torch.randint(-12, 1, (rows, 1), generator=g).float())
    x = (torch.randn(rows, dim_in, generator=g) * spread).cuda()
    dy = (torch.randn(rows, dim_out, generator=g) * spread.flip(0) * 37.0).cuda()
    assert ops.get_linear_mode() == ops.LINEAR_F16X2
    kw = {}
    if bounds == "row maxima":
        kw = dict(dy_bound=ops.row_absmax(dy), x_bound=ops.row_absmax(x))
    elif bounds == "loose":
        kw = dict(dy_bound=dy.abs().max().reshape(1) * 1000.0, x_bound=x.abs().max().reshape(1) * 1000.0)
    got, got_b = ops.tensor_linear_wgrad(0, dy, x, want_bias=True, **kw)
    want_b = dy.double().sum(0)
    err_b, ref_b = float((got_b.double() - want_b).abs().max()), float((dy.sum(0).double() - want_b).abs().max())
    assert err_b <= 1e-6 + 1e-5 * float(want_b.abs().max()) + 2 * ref_b, (err_b, ref_b)
    want = dy.double().t() @ x.double()
    fp32 = (dy.t() @ x).double()
    scale = float(want.abs().max())
    err, err_ref = float((got.double() - want).abs().max()), float((fp32 - want).abs().max())
    print(f"[wgrad f16x2 {rows}x{dim_in}x{dim_out} {bounds}] err {err:.3g} fp32 err {err_ref:.3g} scale {scale:.3g}")
    assert err <= 1e-6 + 1e-5 * scale + 2 * err_ref, (err, err_ref, scale)
    assert torch.equal(ops.tensor_linear_wgrad(0, dy, x, **kw), got)
    # the fp32 matrix-core kernel on the same operands
    ops.set_linear_mode(ops.LINEAR_FP32_MFMA)
    try:
        plain = ops.tensor_linear_wgrad(0, dy, x)
    finally:
        ops.set_linear_mode(ops.LINEAR_F16X2)
    assert float((plain.double() - want).abs().max()) <= 1e-6 + 1e-5 * scale + 2 * err_ref
    assert not torch.equal(plain, got)          # (another kernel, another summation order)


@pytest.mark.parametrize("rows, dim_in, dim_out", [(4096, 4, 4), (4097, 260, 132), (4127, 132, 388), (5000, 640, 128), (70001, 36, 260)])
def test_wgrad_slices_and_tiles_over_the_chip(ops, rows, dim_in, dim_out):
    """One tile and several, as many (slice, tile) pairs as no eighth of them is whole, a last stage that overlaps the one before: against
    float64, the weights' gradient in its 2-norm (sums of runs of 256 rows: 2^-22 a product, random) and the bias row sums."""
    g = torch.Generator().manual_seed(rows)
    dy, x = torch.randn(rows, dim_out, generator=g).cuda(), torch.randn(rows, dim_in, generator=g).cuda()
    dW, db = ops.tensor_linear_wgrad(0, dy, x, want_bias=True)
    ref = dy.double().t() @ x.double()
    assert float((dW.double() - ref).norm()) <= 1e-6 * float(ref.norm())
    assert float((db.double() - dy.double().sum(0)).abs().max()) <= 2.0 ** -24 * rows ** 0.5 * 64
    assert torch.equal(ops.tensor_linear_wgrad(0, dy, x), dW)


@pytest.mark.parametrize("inds,rows,dims", [(0, 4096, (64, 1)), (0, 4097, (16, 260)), (0, 70001, (1280, 13)), (0, 5000, (3, 64)),
                                            (1, 1366, (1, 128)), (1, 9001, (128, 16)), (1, 3000, (76, 5)), (2, 456, (64, 1)),
                                            (2, 2001, (4, 100)), (2, 2001, (300, 5))])
def test_weight_gradient_with_one_narrow_dimension(ops, inds, rows, dims):
    """One dimension of at most 16: lanes without channels, slices and chunks cut short, every width the kernel is compiled for and both
    operands narrow.  float32 products and sums of few rows each: 2^-24 a product and addition, in the 2-norm; rows with infinities
    reach the entries that they reach in the formula and no others."""
    lib = importlib.import_module("learned-dynamics_amd._lib").load()
    dim_in, dim_out = dims
    assert lib.mg_tensor_linear_wgrad_narrow_supported(inds, rows, dim_in, dim_out)
    g, T = torch.Generator().manual_seed(rows), 3 ** inds
    dy, x = (torch.randn(rows, d, *[3] * inds, generator=g).cuda() for d in (dim_out, dim_in))
    plain = lambda t: t.double().reshape(rows, -1, T).transpose(1, 2).reshape(rows * T, -1)
    dW = ops.tensor_linear_wgrad(inds, dy, x)
    ref = plain(dy).t() @ plain(x)
    assert float((dW.double() - ref).norm()) <= 4e-7 * float(ref.norm())
    assert torch.equal(ops.tensor_linear_wgrad(inds, dy, x), dW)
    if inds == 0:
        with_bias, db = ops.tensor_linear_wgrad(0, dy, x, want_bias=True)
        assert torch.equal(with_bias, dW)
        assert float((db.double() - dy.double().sum(0)).abs().max()) <= 2.0 ** -24 * rows ** 0.5 * 64
    dy[-1, 0] = float("inf")
    marked = ops.tensor_linear_wgrad(inds, dy, x)
    assert not marked[0].isfinite().any() and torch.equal(marked[1:], dW[1:])


@pytest.mark.parametrize("rows,dim_in,dim_out", [(1, 64, 64), (33, 128, 512), (337, 512, 512), (300, 1280, 96), (2048, 256, 256),
                                                 (40, 96, 40), (60000, 64, 128)])
def test_linear_that_finds_its_own_row_maxima(ops, rows, dim_in, dim_out):
    """Without bounds the results are those with the exact row maxima to the bit, on either side of the line to reductions split over
    waves, fewer pieces of a row than waves and more; the maxima are those of a pass of its own, and a layer behind it scales by them.
    Rows of zeros, of small numbers, with infinities and NaN."""
    L = importlib.import_module("learned-dynamics_amd._lib")
    lib = L.load()
    g = torch.Generator().manual_seed(rows + dim_in)
    W, b = (torch.randn(dim_out, dim_in, generator=g) * dim_in ** -0.5).cuda(), torch.randn(dim_out, generator=g).cuda()
    W2, b2 = (torch.randn(dim_out, dim_out, generator=g) * dim_out ** -0.5).cuda(), torch.randn(dim_out, generator=g).cuda()
    x = torch.randn(rows, dim_in, generator=g) * torch.randint(-20, 20, (rows, 1), generator=g).float().exp2()
    if rows > 30:
        x[3], x[5, 7], x[9, dim_in - 1], x[11] = 0.0, float("inf"), float("nan"), x[11] * 2.0 ** -120
    x = x.cuda()
    bound = ops.row_absmax(x)
    same = lambda a, b: torch.equal(a.nan_to_num(1.5), b.nan_to_num(1.5))
    planes, (y, maxima) = ops.packed_weight_f16x2(W), (torch.full((rows, n), -1.0, device="cuda") for n in (dim_out, 1))
    args = _F16x2Linear(packed_W=planes.data_ptr(), x=x.data_ptr(), rows=rows, dim_in=dim_in, dim_out=dim_out, bias=b.data_ptr(), bias_rows=rows,
                        out_comps=1, y=y.data_ptr())
    L.check(lib.mg_tensor_linear_f16x2_run_unbounded(ctypes.byref(args), ctypes.c_void_p(maxima.data_ptr()),
                                                     ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
    assert torch.equal(maxima, bound)
    given = y.clone()
    args.x_rowmax, args.x_rowmax_parts, args.x_rowmax_stride, args.x_rows_per_bound, args.bound_mul = bound.data_ptr(), 1, 1, 1, 1.0
    args.y = given.data_ptr()
    L.check(lib.mg_tensor_linear_f16x2_run(ctypes.byref(args), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
    assert same(y, given) and torch.isfinite(y).any()
    assert same(ops.tensor_linear_fwd(0, W, x, bias=b), ops.tensor_linear_fwd(0, W, x, bias=b, row_bound=bound))
    acts = [ops.ACT_SILU, ops.ACT_NONE]
    assert same(ops._ext.linear_chain(x, [W, W2], [b, b2], acts, None, 1.0, 0.0), ops._ext.linear_chain(x, [W, W2], [b, b2], acts, bound, 1.0, 0.0))


class _F16x2Linear(ctypes.Structure):
    _fields_ = [("packed_W", ctypes.c_void_p), ("x", ctypes.c_void_p), ("x_rowmax", ctypes.c_void_p), ("x_rowmax_parts", ctypes.c_int),
                ("x_rowmax_stride", ctypes.c_long), ("x_rows_per_bound", ctypes.c_long), ("bound_mul", ctypes.c_float),
                ("bound_add", ctypes.c_float), ("rows", ctypes.c_long), ("dim_in", ctypes.c_int), ("dim_out", ctypes.c_int),
                ("bias", ctypes.c_void_p), ("bias_rows", ctypes.c_long), ("act", ctypes.c_int), ("accumulate", ctypes.c_int),
                ("out_comps", ctypes.c_int), ("sequential", ctypes.c_int), ("y", ctypes.c_void_p), ("y_rowmax", ctypes.c_void_p)]


class _WgradJob(ctypes.Structure):
    _fields_ = [("dy", ctypes.c_void_p), ("x", ctypes.c_void_p), ("dy_bound", ctypes.c_void_p), ("n_dy_bound", ctypes.c_long),
                ("x_bound", ctypes.c_void_p), ("n_x_bound", ctypes.c_long), ("bias_rows", ctypes.c_long), ("dim_in", ctypes.c_int),
                ("dim_out", ctypes.c_int), ("dW", ctypes.c_void_p), ("db", ctypes.c_void_p)]


@pytest.mark.parametrize("rows,dims", [(4096, [(4, 4)]), (4097, [(128, 132), (256, 128), (4, 300)]), (20011, [(64, 64)] * 6),
                                       (5000, [(1024, 640), (1024, 1024), (512, 512)]), (40003, [(128, 256), (256, 256), (256, 256), (128, 256)])])
def test_weight_gradients_of_several_layers_in_one_launch(ops, rows, dims):
    """Products that share a launch, more than one launch holds and more tiles than it takes, with and without bias, with bounds given
    (short and long arrays, two products with one of them), from the data, biases of a part of the rows, an output off the 16-byte
    grid: float64 as for one product, and the same products taken singly to the order of their slices."""
    L = importlib.import_module("learned-dynamics_amd._lib")
    lib, g = L.load(), torch.Generator(device="cuda").manual_seed(rows)
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    jobs, held = (_WgradJob * len(dims))(), []
    shared = torch.randn(rows, max(k for k, _ in dims), device="cuda", generator=g)
    for k, (dim_in, dim_out) in enumerate(dims):
        x = shared if dim_in == shared.shape[1] else torch.randn(rows, dim_in, device="cuda", generator=g)
        dy = torch.randn(rows, dim_out, device="cuda", generator=g)
        bounds = [None, None] if k % 3 == 2 else [dy.abs().amax(1), x.abs().amax(1)]
        out = torch.full((dim_in * dim_out + 8,), float("nan"), device="cuda")
        dW, db = out[k % 2:][:dim_in * dim_out], torch.full((dim_out,), float("nan"), device="cuda")
        bias_rows = rows if k % 2 else rows // 2 + 1
        jobs[k] = _WgradJob(dy.data_ptr(), x.data_ptr(), *(v for b in bounds for v in (None if b is None else b.data_ptr(), rows)), bias_rows,
                            dim_in, dim_out, dW.data_ptr(), None if k == 3 else db.data_ptr())
        held.append((x, dy, bounds, out, dW, db, bias_rows))
    size = ctypes.c_size_t()
    L.check(lib.mg_tensor_linear_wgrad_f16x2_many_workspace_bytes(ctypes.byref(jobs), len(dims), rows, ctypes.byref(size)))
    ws = torch.empty(size.value, dtype=torch.uint8, device="cuda")
    L.check(lib.mg_tensor_linear_wgrad_f16x2_many(ctypes.byref(jobs), len(dims), rows, ws.data_ptr(), stream))
    for k, (x, dy, bounds, out, dW, db, bias_rows) in enumerate(held):
        ref = dy.double().t() @ x.double()
        assert float((dW.reshape(ref.shape).double() - ref).norm()) <= 1e-6 * float(ref.norm()), k
        one = ops.tensor_linear_wgrad(0, dy, x, *(None if b is None else b[:, None] for b in bounds))
        assert float((dW.reshape(ref.shape) - one).norm()) <= 1e-6 * float(ref.norm()), k
        assert int(out.isnan().sum()) == 8, k
        if k == 3:
            assert db.isnan().all()
        else:
            assert float((db.double() - dy[:bias_rows].double().sum(0)).abs().max()) <= 2.0 ** -24 * rows ** 0.5 * 64, k
    assert lib.mg_tensor_linear_wgrad_f16x2_many(ctypes.byref(jobs), len(dims), 4095, ws.data_ptr(), stream) != 0



@pytest.mark.parametrize("rows", [4096, 78000])
def test_gradients_of_several_layers_in_one_launch_in_short_chains(ops, rows):
    """The three layers of an MLP of 512 columns: together the slices of rows are longer, the chains in which they are summed are not.
    Column sums: chains of 32 numbers, of as many runs as a slice has (44 at most here) and of 14 slices in eights, which for random
    numbers are off by 2^-24 (32 / 6 + 44 / 6 + 3)^(1/2) = 4 x 2^-24 of their 2-norm: 5 x 2^-24.  Products: within a
    fifth of the error that they have singly in shorter slices (a chain twice as long is off by a fifth more where half of the
    error is the pieces')."""
    L = importlib.import_module("learned-dynamics_amd._lib")
    lib, g = L.load(), torch.Generator(device="cuda").manual_seed(rows)
    dims, jobs, held = [(128, 512), (512, 512), (512, 512)], (_WgradJob * 3)(), []
    for k, (dim_in, dim_out) in enumerate(dims):
        x, dy = (torch.randn(rows, d, device="cuda", generator=g) for d in (dim_in, dim_out))
        dW, db = torch.empty(dim_out, dim_in, device="cuda"), torch.empty(dim_out, device="cuda")
        jobs[k] = _WgradJob(dy.data_ptr(), x.data_ptr(), None, 0, None, 0, rows, dim_in, dim_out, dW.data_ptr(), db.data_ptr())
        held.append((x, dy, dW, db))
    size = ctypes.c_size_t()
    L.check(lib.mg_tensor_linear_wgrad_f16x2_many_workspace_bytes(ctypes.byref(jobs), 3, rows, ctypes.byref(size)))
    ws = torch.empty(size.value, dtype=torch.uint8, device="cuda")
    L.check(lib.mg_tensor_linear_wgrad_f16x2_many(ctypes.byref(jobs), 3, rows, ws.data_ptr(), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
    off = lambda t, ref: float((t.double() - ref).norm() / ref.norm())
    for x, dy, dW, db in held:
        one, one_b = ops.tensor_linear_wgrad(0, dy, x, want_bias=True)
        ref, ref_b = dy.double().t() @ x.double(), dy.double().sum(0)
        print(f"[together / singly] {rows}: dW {off(dW, ref):.3g} / {off(one, ref):.3g}, db {off(db, ref_b):.3g} / {off(one_b, ref_b):.3g}")
        assert off(db, ref_b) <= 5 * 2.0 ** -24 and off(one_b, ref_b) <= 5 * 2.0 ** -24
        assert off(dW, ref) <= 1.2 * off(one, ref)


def test_weight_gradient_at_the_edge_count_of_configs2(ops):
    """The split-fp16 weight gradient at the size training runs it at (1592454 edge rows, 512 x 512): against float64
    accumulated over row chunks on the device, with the error of torch's own fp32 product of the same operands as
    the yardstick; the bias gradient from the same pass; and the same bits on a second run."""
    rows, dim = 1592454, 512
    g = torch.Generator(device="cuda").manual_seed(5)
    x = torch.randn(rows, dim, device="cuda", generator=g)
    dy = torch.randn(rows, dim, device="cuda", generator=g) * torch.rand(rows, 1, device="cuda", generator=g)
    got, got_b = ops.tensor_linear_wgrad(0, dy, x, want_bias=True)
    want = torch.zeros(dim, dim, dtype=torch.float64, device="cuda")
    want_b = torch.zeros(dim, dtype=torch.float64, device="cuda")
    fp32 = torch.zeros(dim, dim, dtype=torch.float64, device="cuda")
    for lo in range(0, rows, 65536):
        a, b = dy[lo:lo + 65536], x[lo:lo + 65536]
        want += a.double().t() @ b.double()
        want_b += a.double().sum(0)
        fp32 += (a.t() @ b).double()
    scale = float(want.abs().max())
    err, err_ref = float((got.double() - want).abs().max()), float((fp32 - want).abs().max())
    print(f"[wgrad f16x2 {rows}x{dim}x{dim}] err {err:.3g}  chunked fp32 err {err_ref:.3g}  scale {scale:.3g}")
    assert err <= 1e-6 + 1e-5 * scale + 2 * err_ref, (err, err_ref, scale)
    assert float((got_b.double() - want_b).abs().max()) <= 1e-6 + 1e-5 * float(want_b.abs().max())
    again, again_b = ops.tensor_linear_wgrad(0, dy, x, want_bias=True)
    assert torch.equal(again, got) and torch.equal(again_b, got_b)


# around the crossovers of the split-K kernel (256 / 512 / 1536 blocks of 32 x 32, four and eight waves, partial row and
# column blocks) and one problem past them; dim_in 96 leaves one of its four waves without a chunk
@pytest.mark.parametrize("rows,dim_in,dim_out", [(1, 512, 512), (31, 64, 40), (33, 96, 512), (512, 256, 512), (544, 256, 512),
                                                 (1025, 512, 512), (3072, 512, 512), (3105, 512, 512), (6145, 1280, 64),
                                                 (700, 768, 100)])
@pytest.mark.parametrize("act", [0, 1, 2])
def test_linear_f16x2_split_reduction(ops, rows, dim_in, dim_out, act):
    """Few rows: the reduction split over the waves of a workgroup, with the row maxima it emits; sequential=True gives every
    row the bits it has in a batch too large to split."""
    g = torch.Generator().manual_seed(rows + dim_in)
    x = (torch.randn(rows, dim_in, generator=g) * (torch.rand(rows, 1, generator=g) * 3)).cuda()
    W = (torch.randn(dim_out, dim_in, generator=g) / dim_in ** 0.5).cuda()
    b = torch.randn(dim_out, generator=g).cuda()
    y, ymax = ops.tensor_linear_f16x2(W, x, ops.row_absmax(x), bias=b, act=act, want_rowmax=True)

    def ref(dt):
        z = x.cpu().to(dt) @ W.cpu().to(dt).T + b.cpu().to(dt)
        return torch.nn.functional.silu(z) if act == 1 else (torch.nn.functional.leaky_relu(z, 0.1) if act == 2 else z)
    _check(y, ref, f"split reduction {rows} x {dim_in} -> {dim_out}")
    assert torch.equal(ymax.amax(1), y.abs().amax(1))
    if rows >= 256:
        many = x.repeat(60, 1)[:60000]
        a = ops.tensor_linear_fwd(0, W, x, bias=b, act=act, sequential=True)
        assert torch.equal(a, ops.tensor_linear_fwd(0, W, many, bias=b, act=act)[:rows])


@pytest.mark.parametrize("inds,dim_in", [(0, 1), (0, 8), (0, 20), (0, 32), (1, 1), (1, 8), (2, 3), (1, 9), (1, 16), (2, 13), (2, 16)])
@pytest.mark.parametrize("rows,dim_out", [(1, 5), (63, 256), (700, 300)])
def test_linear_few_inputs(ops, inds, dim_in, rows, dim_out):
    g = torch.Generator().manual_seed(rows + dim_in)
    x = torch.randn(rows, dim_in, *([3] * inds), generator=g)
    W, b = torch.randn(dim_out, dim_in, generator=g), torch.randn(dim_out, generator=g)
    T = 3 ** inds
    y = ops.tensor_linear_fwd(inds, W.cuda(), x.cuda())
    _check(y, lambda dt: OP.tensor_linear(inds, W.to(dt), x.to(dt)), "few inputs")
    if inds == 0:
        y2 = ops.tensor_linear_fwd(0, W.cuda(), x.cuda(), bias=b.cuda(), act=ops.ACT_SILU, out=y.clone(), accumulate=True)
        _check(y2, lambda dt: y.cpu().to(dt) + torch.nn.functional.silu(x.to(dt) @ W.to(dt).T + b.to(dt)), "few inputs, accumulated")
    else:
        y2 = ops.tensor_linear_fwd(inds, W.cuda(), x.cuda(), y_layout=ops.LAYOUT_COMP_CHAN)
        assert torch.equal(y2.reshape(rows, T, dim_out).transpose(1, 2), y.reshape(rows, dim_out, T))


# few rows (the split reduction: one, two column blocks, four and eight waves), many (row streaming, with a partial column
# tile, with the epilogue in runs of nine components)
@pytest.mark.parametrize("inds,rows,dim_in,dim_out", [(0, 1, 64, 8), (0, 40, 128, 512), (0, 200, 1280, 16), (0, 255, 256, 256),
                                                      (0, 9000, 64, 300), (0, 9000, 128, 256), (1, 330, 128, 384),
                                                      (1, 9000, 64, 192), (2, 120, 64, 64), (2, 3001, 64, 256)])
def test_rows_and_columns_the_fp16_pieces_cannot_carry(ops, inds, rows, dim_in, dim_out):
    """Infinite and very large entries of x, and infinite weights, through the split-fp16 kernels: infinities and NaN where
    float64 arithmetic has them, finite results to the tolerance of a sum in fp32, other rows and columns bit for bit as without them.
    Then the same with bias, activation and accumulation, and through the row maxima into a second layer."""
    assert ops.get_linear_mode() == ops.LINEAR_F16X2
    g = torch.Generator().manual_seed(rows + dim_in)
    T = 3 ** inds
    x = torch.randn(rows, dim_in, *([3] * inds), generator=g)
    W = torch.randn(dim_out, dim_in, generator=g) / dim_in ** 0.5
    W[dim_out // 3] = torch.randint(1, 5, (dim_in,), generator=g).float() / 4     # (its low pieces are zeros)
    W[dim_out // 2, 1] = 0.0
    inf = float("inf")
    odd = sorted({0, rows // 2, rows - 1})
    bad = x.clone().reshape(rows, dim_in, T)
    bad[odd[0], 1, 0] = inf
    bad[odd[-1], dim_in - 1, T - 1] = -inf
    bad[odd[len(odd) // 2], :, T // 2] *= 1e30                                    # (one component only: a row of its own)
    bad = bad.reshape(x.shape)

    def close(y, want, what):
        y, want = y.cpu().double(), want.cpu()
        assert torch.equal(torch.isnan(y), torch.isnan(want)), what
        assert torch.equal(torch.where(torch.isinf(y), y, 0.0), torch.where(torch.isinf(want), want, 0.0)), what
        y, want = (torch.where(torch.isfinite(t), t, 0.0).reshape(rows, -1, T) for t in (y, want))
        scale = want.abs().amax(1, keepdim=True).clamp_min(1e-30)
        assert float(((y - want).abs() / scale).max()) <= dim_in * 2 ** -23, what       # the chain's bound, K roundings of half an ulp, twice

    def product(x_, W_):
        return OP.tensor_linear(inds, W_.double(), x_.double())

    plain = ops.tensor_linear_fwd(inds, W.cuda(), x.cuda())
    y = ops.tensor_linear_fwd(inds, W.cuda(), bad.cuda())
    close(y, product(bad, W), "infinite entries")
    same = (bad == x).reshape(rows, dim_in, T).all(1)                                    # (rows, components) left as they were
    keep = same[:, None].expand(rows, dim_out, T)
    assert torch.equal(y.cpu().reshape(rows, dim_out, T)[keep], plain.cpu().reshape(rows, dim_out, T)[keep])
    Wi = W.clone()
    Wi[dim_out - 1, 0], Wi[1, dim_in - 1] = inf, -inf
    yw = ops.tensor_linear_fwd(inds, Wi.cuda(), x.cuda())
    close(yw, product(x, Wi), "infinite weights")
    cols = [o for o in range(dim_out) if o not in (1, dim_out - 1)]
    assert torch.equal(yw.cpu().reshape(rows, dim_out, T)[:, cols], plain.cpu().reshape(rows, dim_out, T)[:, cols])
    if inds > 0:
        base = torch.randn(y.shape, generator=g)
        rows_ = ops.components_as_rows(inds, bad.cuda())
        out = ops.tensor_linear_f16x2(W.cuda(), rows_[0][:, :dim_in].contiguous(), rows_[1], out=base.cuda(), accumulate=True, out_comps=T)
        assert torch.equal(torch.nan_to_num(out), torch.nan_to_num(y + base.cuda()))
        return
    b = torch.randn(dim_out, generator=g)
    base = torch.randn(rows, dim_out, generator=g)
    z = product(bad, W) + b.double()
    for act, f in ((ops.ACT_NONE, lambda t: t), (ops.ACT_LEAKY, lambda t: torch.nn.functional.leaky_relu(t, 0.1))):
        out = ops.tensor_linear_fwd(0, W.cuda(), bad.cuda(), bias=b.cuda(), act=act, out=base.cuda(), accumulate=True)
        close(out, f(z) + base.double(), "bias, activation, accumulated")
    h, hmax = ops.tensor_linear_f16x2(W.cuda(), bad.cuda(), ops.row_absmax(bad.cuda()), bias=b.cuda(), want_rowmax=True)
    assert bool((hmax.amax(1) >= torch.nan_to_num(h, nan=0.0, posinf=inf, neginf=-inf).abs().amax(1)).all())
    if dim_out % 32 == 0 and dim_out >= 64:
        W2 = torch.randn(64, dim_out, generator=g) / dim_out ** 0.5
        y2 = ops.tensor_linear_f16x2(W2.cuda(), h, hmax)
        want = h.cpu().double() @ W2.double().T
        finite = torch.isfinite(want).all(1)
        assert torch.equal(torch.isfinite(y2.cpu()).all(1), finite)
        err = (y2.cpu().double() - want)[finite].abs() / want[finite].abs().amax(1, keepdim=True)
        assert float(err.max()) <= dim_out * 2 ** -23


@pytest.mark.parametrize("inds,rows,dim_in,dim_out", [(1, 2048, 16, 64), (2, 2048, 16, 256), (2, 1000, 24, 64), (1, 1000, 32, 64),
                                                      (2, 500, 64, 64), (1, 337, 128, 384), (0, 1, 64, 256), (0, 200, 64, 8),
                                                      (0, 100, 256, 768), (0, 18432, 1280, 16)])
def test_small_problems_are_no_less_precise_than_fp32(ops, inds, rows, dim_in, dim_out):
    """Whatever kernel these sizes take by default is as close to float64 as products and sums in fp32 are (2-norms)."""
    g = torch.Generator().manual_seed(rows + dim_in)
    x = torch.randn(rows, dim_in, *([3] * inds), generator=g)
    x = x * torch.exp(0.5 * torch.randn(rows, dim_in, *([1] * inds), generator=g))
    W = torch.randn(dim_out, dim_in, generator=g) / dim_in ** 0.5
    ref = OP.tensor_linear(inds, W.double(), x.double())
    err = lambda: float((ops.tensor_linear_fwd(inds, W.cuda(), x.cuda()).cpu().double() - ref).norm() / ref.norm())
    default = err()
    ops.set_linear_mode(ops.LINEAR_FP32_MFMA)
    try:
        fp32 = err()
    finally:
        ops.set_linear_mode(ops.LINEAR_F16X2)
    assert default <= 1.01 * fp32, (default, fp32)               # (where both run the same kernel they are equal)


def test_packed_weight_of_any_multiple_of_eight(ops):
    """A reduction of 8, 40 or 72 packs as with zero columns up to the next multiple of 32; 12 is refused."""
    for dim_in in (8, 40, 72):
        W = torch.randn(50, dim_in, device="cuda")
        padded = torch.nn.functional.pad(W, (0, -dim_in % 32))
        assert torch.equal(ops.packed_weight_f16x2(W), ops.packed_weight_f16x2(padded))
    with pytest.raises(RuntimeError, match="multiple of 8"):
        ops.packed_weight_f16x2(torch.randn(50, 12, device="cuda"))


@pytest.mark.parametrize("rows", [10, 400])
@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
def test_mlp_with_a_weight_that_is_no_number(pkg, rows, bad):
    """An MLP whose first layer holds a NaN or an infinity evaluates (its bounds are infinite) and gives no numbers where float64
    arithmetic gives none; with the weight set again it is what it was (three sums of at most 128 terms: 24 sqrt(128) 2^-24)."""
    painn = importlib.import_module("learned-dynamics_amd.painn")
    torch.manual_seed(rows)
    mlp = painn.MLP(64, 128).cuda().requires_grad_(False)
    mlp.layers[0].weight[3, 5] = bad
    x = torch.randn(rows, 64)
    double = lambda: [p.cpu().double() for k in (0, 2, 4) for p in (mlp.layers[k].weight, mlp.layers[k].bias)]

    def want():
        W0, b0, W1, b1, W2, b2 = double()
        silu = torch.nn.functional.silu
        return silu(silu(x.double() @ W0.T + b0) @ W1.T + b1) @ W2.T + b2
    y = mlp(x.cuda()).cpu()
    assert torch.equal(torch.isfinite(y), torch.isfinite(want()))
    mlp.layers[0].weight[3, 5] = 0.25
    y = mlp(x.cuda()).cpu().double()
    assert float((y - want()).abs().max() / want().abs().max()) <= 1.7e-5


@pytest.mark.parametrize("rows,dim_in,dim_out", [(1, 16, 256), (15, 1, 5), (17, 3, 257), (33, 4, 64), (300, 5, 40), (514, 8, 256),
                                                 (1030, 12, 300), (40, 16, 1000)])
def test_few_inputs_of_rank_two_by_component_and_by_channel(rows, dim_in, dim_out):
    """Nine components of a handful of channels: the kernel whose lanes own channels (component-major outputs) and the one whose threads
    own (channel, component) form every sum in the same order, so they agree bit for bit; weights in rows, as a transposed view and
    one float off 16-byte alignment, with and without accumulation."""
    ops = importlib.import_module("learned-dynamics_amd.ops")
    g = torch.Generator().manual_seed(rows)
    x = torch.randn(rows, dim_in, 3, 3, generator=g).cuda()
    flat = torch.randn(dim_out * dim_in + 1, generator=g).cuda()
    for W in (flat[:-1].view(dim_out, dim_in), flat[:-1].view(dim_in, dim_out).t(), flat[1:].view(dim_out, dim_in)):
        by_channel = ops.tensor_linear_fwd(2, W, x)
        y = ops.tensor_linear_fwd(2, W, x, y_layout=ops.LAYOUT_COMP_CHAN)
        y = y[0] if isinstance(y, tuple) else y
        assert torch.equal(y.reshape(rows, 9, dim_out).transpose(1, 2), by_channel.reshape(rows, dim_out, 9))
        base = torch.randn(y.shape, generator=g).cuda()
        assert torch.equal(ops.tensor_linear_fwd(2, W, x, out=base.clone(), accumulate=True, y_layout=ops.LAYOUT_COMP_CHAN), y + base)
        ref = torch.einsum("oi,nixy->noxy", W.double().cpu(), x.double().cpu()).reshape(rows, dim_out, 9)
        torch.testing.assert_close(by_channel.cpu().double().reshape(rows, dim_out, 9), ref, rtol=1e-5, atol=1e-6 * dim_in)


@pytest.mark.parametrize("rows,dim_in,dim_out", [(1, 16, 63), (1, 16, 64), (767, 8, 128), (768, 8, 128), (900, 12, 127), (769, 12, 128),
                                                 (5, 16, 513)])
def test_few_inputs_of_rank_two_beside_the_line_between_their_kernels(rows, dim_in, dim_out):
    """Channels and sums on either side of where a lane takes a channel of its own: the same bits from both."""
    test_few_inputs_of_rank_two_by_component_and_by_channel(rows, dim_in, dim_out)


@pytest.mark.parametrize("rows, dim_in, dim_out, comps", [
    (1, 288, 64, 1), (33, 256, 256, 1), (95, 544, 40, 1), (31, 1280, 16, 1), (333, 1280, 64, 3), (2050, 160, 70, 1), (1800, 320, 96, 9)])
def test_reductions_split_over_waves_with_one_chunk_and_several(ops, rows, dim_in, dim_out, comps):
    """Onto values that are there, row bounds in one part, four and seven (the bound is their maximum: the same bits), rows and columns
    that end inside a tile, components.  22-bit pieces and fp32 sums: 2^-21 of the norms of the rows that are multiplied."""
    g = torch.Generator().manual_seed(rows)
    W = torch.randn(dim_out, dim_in, generator=g).cuda()
    x = (torch.randn(rows, dim_in, generator=g) * torch.exp(torch.randn(rows, 1, generator=g))).cuda()
    nodes = -(-rows // comps)
    x = torch.cat([x, x[:nodes * comps - rows]])
    base = torch.randn((nodes, dim_out, comps) if comps > 1 else (nodes, dim_out), generator=g).cuda()
    bound = ops.row_absmax(x)
    low = torch.zeros_like(bound)

    def onto(b):
        return ops.tensor_linear_f16x2(W, x, b, out=base.clone(), accumulate=True, out_comps=comps)
    y = onto(bound)
    ref = (x.double() @ W.double().t()).view(nodes, comps, dim_out).transpose(1, 2).reshape(base.shape) + base.double()
    size = (x.double().norm(dim=1)[:, None] * W.double().norm(dim=1)).view(nodes, comps, dim_out).transpose(1, 2).reshape(base.shape)
    assert float(((y.double() - ref).abs() / (size + base.abs())).max()) <= 2.0 ** -21
    for parts in ([low, low, bound, low], [low, low, low, low, low, low, bound], [low, low, low, low, bound]):
        assert torch.equal(onto(torch.cat(parts, 1)), y)
    # a row without a bound that the pieces can carry, in every tile but its own the same bits
    x[rows // 2, 1] = 2.0 ** 100
    z = onto(ops.row_absmax(x))
    ref = (x.double() @ W.double().t()).view(nodes, comps, dim_out)[rows // 2 // comps, rows // 2 % comps]
    pick = lambda t: t.view(nodes, dim_out, comps)[rows // 2 // comps, :, rows // 2 % comps]
    assert float(((pick(z).double() - ref) / ref).abs().max()) <= 1e-6
    keep = torch.ones(nodes, dtype=torch.bool, device="cuda")
    keep[rows // 2 // comps] = False
    assert torch.equal(z[keep], y[keep])


@pytest.mark.parametrize("rows, products, dim_in, dim_out", [
    (1, 1, 32, 1), (33, 5, 64, 16), (64, 2, 96, 17), (95, 8, 32, 32), (31, 3, 160, 33), (2049, 5, 256, 64), (65, 4, 64, 65), (130, 2, 32, 130)])
def test_linears_side_by_side_at_the_edges_of_their_tiles(ops, rows, products, dim_in, dim_out):
    """Both block sizes and each tile: rows and columns that end inside one, an odd number of slabs.  In fp32: every addition of a chain of
    dim_in products, and of the products' sums, rounds by 2^-24 of at most the norms of what is multiplied.  Row maxima are exact, and a
    row does not depend on those beside it."""
    g = torch.Generator().manual_seed(rows + dim_out)
    x = torch.randn(rows, products * dim_in, generator=g).cuda()
    W = [torch.randn(dim_out, dim_in, generator=g).cuda() for _ in range(products)]
    y, m = ops.row_linears_fwd(x, W, 9, True)
    parts = x.double().view(rows, products, dim_in)
    ref = sum(parts[:, k] @ W[k].double().t() for k in range(products))
    size = sum(parts[:, k].norm(dim=1)[:, None] * W[k].double().norm(dim=1) for k in range(products))
    assert float(((y.double() - ref).abs() / size).max()) <= (dim_in + products) * 2.0 ** -24
    assert torch.equal(m, x.view(rows, products, dim_in).abs().amax(2))
    x[0] = float("inf")
    z, _ = ops.row_linears_fwd(x, W, 9, True)
    assert torch.equal(z[1:], y[1:]) and not bool(z[0].isfinite().any())


@pytest.mark.parametrize("rows, dim_out", [(40960, 40), (40961, 33), (41001, 64)])
def test_linears_side_by_side_of_many_rows(ops, rows, dim_out):
    """Either side of the rows from which 33 to 64 columns go in larger blocks."""
    test_linears_side_by_side_at_the_edges_of_their_tiles(ops, rows, 2, 32, dim_out)

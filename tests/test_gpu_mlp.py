"""Linear, SiLU, Linear, SiLU, Linear as one kernel (csrc/mlp_f16x2.hip) against the same formula in float64."""
import importlib

import pytest
import torch

pytestmark = pytest.mark.gpu

ACTS = (1, 1, 0)
INF, NAN = float("inf"), float("nan")


@pytest.fixture
def bee(pkg):
    return importlib.import_module("learned-dynamics_amd.bee_layers")


def _weights(dim_in, dim, seed=3):
    g = torch.Generator().manual_seed(seed)
    W = [torch.randn(dim, k, generator=g) * k ** -0.5 for k in (dim_in, dim, dim)]
    return [w.cuda() for w in W], [torch.randn(dim, generator=g).cuda() * 0.1 for _ in W]


def _formula(x, W, b):
    h = x
    for k in range(3):
        h = h @ W[k].to(x.dtype).t() + b[k].to(x.dtype)
        h = torch.nn.functional.silu(h) if k < 2 else h
    return h


def _assert_rows(y, ref, what, f32=None):
    """2-norm of a row's difference against the row's: three layers, each rounding its operands to 22 bits and its sums and
    activation to 24, err by 5e-7 at most; measured 2e-7 .. 3e-7 over all rows.  f32: the formula in float32, where a row's terms may
    cancel (the adjoint's g f' + g_t z_t f''): twice its distance is what the row's conditioning adds."""
    def error(t):
        return (t.double() - ref).norm(dim=1) / ref.norm(dim=1)
    err = error(y) - (0 if f32 is None else 2 * error(f32))
    assert float(err.max()) <= 1.5e-6, (what, float(err.max()))


# (rows at the edges of the 32- and 64-row tiles; 512 columns of few rows go layer by layer, of 16 500 rows in tiles of 64)
@pytest.mark.parametrize("rows, dim_in, dim", [(1, 64, 64), (31, 96, 96), (33, 512, 64), (65, 128, 256), (40, 512, 256), (700, 96, 224),
                                               (1024, 128, 512), (1057, 256, 384), (8193, 64, 512), (16500, 160, 288), (66000, 64, 64)])
def test_mlp_in_one_kernel(ops, rows, dim_in, dim):
    W, b = _weights(dim_in, dim)
    g = torch.Generator().manual_seed(rows)
    x = (torch.randn(rows, dim_in, generator=g) * torch.exp(2 * torch.randn(rows, 1, generator=g))).cuda()
    x[rows // 2] = 0
    y = ops.linear_chain(x, W, b, ACTS, None)
    _assert_rows(y, _formula(x.double(), W, b), (rows, dim_in, dim))


@pytest.mark.parametrize("rows, dim_in, dim", [(70, 64, 64), (1100, 128, 512), (16500, 64, 320)])
def test_mlp_rows_and_weights_beyond_the_pieces(ops, rows, dim_in, dim):
    W, b = _weights(dim_in, dim)
    x = torch.randn(rows, dim_in, generator=torch.Generator().manual_seed(1)).cuda()
    clean = ops.linear_chain(x, W, b, ACTS, None)
    x[3, 1], x[rows - 1, dim_in - 1], x[17, 5] = INF, -INF, NAN
    x[40] *= 2.0 ** 110
    y = ops.linear_chain(x, W, b, ACTS, None)
    odd = torch.zeros(rows, dtype=torch.bool, device="cuda")
    odd[[3, 17, 40, rows - 1]] = True
    assert torch.equal(y[~odd], clean[~odd])                     # (no other row notices)
    for r in (3, 17, rows - 1):
        assert not bool(torch.isfinite(y[r]).any())              # (an infinite or undefined h in every sum)
    _assert_rows(y[40:41], _formula(x[40:41].double(), W, b), "2^110")
    x = torch.randn(rows, dim_in, generator=torch.Generator().manual_seed(1)).cuda()
    W[2][5, 3] = INF
    y = ops.linear_chain(x, W, b, ACTS, None)
    h = torch.nn.functional.silu(x.double() @ W[0].double().t() + b[0].double())
    h = torch.nn.functional.silu(h @ W[1].double().t() + b[1].double())
    assert torch.equal(y[:, 5].double(), INF * torch.sign(h[:, 3]))
    keep = [k for k in range(dim) if k != 5]
    _assert_rows(y[:, keep], (h @ W[2].double().t() + b[2].double())[:, keep], "beside an infinite weight")
    W[2][5, 3] = 0.5
    W[0][7, 2] = NAN
    assert bool(torch.isnan(ops.linear_chain(x, W, b, ACTS, None)).all())


def _dual_formula(x, x_t, W, b):
    """y and its tangent in float64, differentiable."""
    h, h_t = x, x_t
    for k in range(3):
        z, z_t = h @ W[k].t() + b[k], None if h_t is None else h_t @ W[k].t()
        if k < 2:
            s = torch.sigmoid(z)
            h, h_t = z * s, None if z_t is None else (s + z * s * (1 - s)) * z_t
        else:
            h, h_t = z, z_t
    return h, h_t


# (rows at the edges of the tiles of 32 rows, 16 with tangents, and on both sides of one workgroup per CU)
@pytest.mark.parametrize("rows, dim_in, dim, dual", [(1, 64, 64, False), (33, 128, 256, False), (1025, 96, 512, False), (8300, 64, 320, False),
                                                     (1, 64, 96, True), (17, 512, 128, True), (1000, 256, 192, True), (2300, 128, 512, True),
                                                     (4200, 64, 384, True), (4100, 64, 288, True)])
def test_mlp_adjoint_in_one_kernel(ops, rows, dim_in, dim, dual):
    W, b = _weights(dim_in, dim)
    g = torch.Generator().manual_seed(rows)
    S = (torch.randn(2 * rows, dim_in, generator=g) * torch.exp(torch.randn(2 * rows, 1, generator=g))).cuda()
    G = torch.randn(2 * rows, dim, generator=g).cuda()
    x, x_t, gy, gy_t = S[:rows], S[rows:] if dual else None, G[:rows], G[rows:] if dual else None
    y, y_t, saved = ops.mlp_silu_fwd(x, x_t, None, W, b, True)
    g_x, g_xt, params = ops.mlp_silu_bwd(gy, gy_t, x, x_t, W, saved, True, True)

    def formula(dt):
        leaves = [t.detach().clone().to(dt).requires_grad_() for t in (x, *W, *b)] + ([x_t.clone().to(dt).requires_grad_()] if dual else [])
        ref, ref_t = _dual_formula(leaves[0], leaves[7] if dual else None, leaves[1:4], leaves[4:7])
        loss = (ref * gy.to(dt)).sum() + ((ref_t * gy_t.to(dt)).sum() if dual else 0)
        grads = torch.autograd.grad(loss, leaves)
        return [ref.detach(), grads[0]] + ([ref_t.detach(), grads[7]] if dual else []), grads

    (ref, grads), (ref32, _) = formula(torch.float64), formula(torch.float32)
    for what, a, r, r32 in zip(("y", "g_x", "y_t", "g_xt"), (y, g_x, y_t, g_xt), ref, ref32):
        _assert_rows(a, r, (what, rows, dim_in, dim, dual), r32)
    for k in range(3):                                           # (sums over rows: the whole matrix against its norm)
        for a, r in ((params[2 * k], grads[1 + k]), (params[2 * k + 1], grads[4 + k])):
            assert float((a.double() - r).norm() / r.norm()) <= 4e-6, (k, rows, dim_in, dim, dual)
    no_x, _, _ = ops.mlp_silu_bwd(gy, gy_t, x, x_t, W, saved, False, True)
    assert no_x is None


@pytest.mark.parametrize("spread", [0.3, 1.0, 4.0])
def test_silu_between_the_layers(ops, spread):
    """The hidden rows h = SiLU(z) that the training kernel keeps beside z, entry by entry in float64, against the same from float32
    exp and a division: no further off.  And the ends of the range: four roundings of 2^-24 and an exponential good to one more."""
    W, b = _weights(64, 256)
    x = spread * 1.4 * torch.randn(4000, 64, generator=torch.Generator().manual_seed(3)).cuda()
    _, _, saved = ops.mlp_silu_fwd(x, None, None, W, b, True)
    z, h = saved[1], saved[3]
    ref = torch.nn.functional.silu(z.double())
    rms = lambda y: float((((y.double() - ref) / ref) ** 2).mean().sqrt())
    assert rms(h) <= rms(z * (1.0 / (1.0 + torch.exp(-z)))), spread
    bias = torch.tensor([200.0, 87.0, 0.0, -87.0, -89.0, -200.0, -1e30, 1e30]).repeat(8).cuda()
    _, _, saved = ops.mlp_silu_fwd(torch.zeros(64, 64).cuda(), None, None, [W[0][:64]] + [w[:64, :64].contiguous() for w in W[1:]],
                                   [bias] + [t[:64].contiguous() for t in b[1:]], True)
    ref = torch.nn.functional.silu(bias.double())
    # (where the sigmoid is below the smallest normal number, 2^-126, the result is 0: off by 89 * 2^-126 = 1e-36 at most)
    assert bool(((saved[3].double() - ref).abs() <= 3e-7 * ref.abs() + 1.1e-36).all())


@pytest.mark.parametrize("rows, dim", [(50, 64), (1100, 512), (8300, 512)])
def test_mlp_adjoint_of_a_row_beyond_the_pieces(ops, rows, dim):
    W, b = _weights(64, dim)
    g = torch.Generator().manual_seed(2)
    x, gy = torch.randn(rows, 64, generator=g).cuda(), torch.randn(rows, dim, generator=g).cuda()
    y, _, saved = ops.mlp_silu_fwd(x, None, None, W, b, True)
    clean, _, _ = ops.mlp_silu_bwd(gy, None, x, None, W, saved, True, False)
    gy[rows - 2, 3], gy[5] = INF, gy[5] * 2.0 ** 100
    g_x, _, _ = ops.mlp_silu_bwd(gy, None, x, None, W, saved, True, False)
    same = torch.ones(rows, dtype=torch.bool, device="cuda")
    same[[5, rows - 2]] = False
    assert torch.equal(g_x[same], clean[same])
    assert not bool(torch.isfinite(g_x[rows - 2]).any())
    assert float((g_x[5].double() * 2.0 ** -100 - clean[5].double()).norm() / clean[5].double().norm()) <= 1.5e-6


def _segments(rows, seed):
    """Segments that begin and end anywhere in the blocks of 32 rows: empty ones, ones of one row, of a block, of several."""
    g = torch.Generator().manual_seed(seed)
    deg = torch.tensor([0, 32, 1, 31, 0, 0, 33, 30, 1, 64, 200, 2, 29, 3, 95, 1])
    deg = torch.cat([deg, torch.randint(0, 40, (rows // 10 + 8,), generator=g)])
    ends = deg.cumsum(0).clamp(max=rows)
    ends[-1] = rows
    row_ptr = torch.cat([torch.zeros(1, dtype=torch.long), ends])
    return row_ptr, torch.repeat_interleave(torch.arange(ends.numel()), row_ptr[1:] - row_ptr[:-1])


def _layers_and_sum(x, W, b, seg, n_out):
    f = torch.nn.functional
    h = x
    for k in range(2):
        h = f.leaky_relu(h @ W[k].to(x.dtype).t() + b[k].to(x.dtype), 0.1)
    zero = torch.zeros(n_out, h.shape[1], dtype=x.dtype, device=x.device)
    return zero.index_add(0, seg, h), torch.zeros(n_out, dtype=x.dtype, device=x.device).index_add(0, seg, h.norm(dim=1))


@pytest.mark.parametrize("rows, dim_in, dim", [(1, 64, 64), (33, 512, 32), (64, 96, 288), (700, 160, 512), (4161, 256, 512), (5000, 32, 96)])
def test_mlp_summed_over_segments(ops, rows, dim_in, dim):
    """Against the formula in float64, relative to the sum of the segment's row norms: two layers of rows as above and sums of
    up to 200 rows of which each addition rounds by 6e-8."""
    W, b = (t[:2] for t in _weights(dim_in, dim))
    g = torch.Generator().manual_seed(rows)
    x = (torch.randn(rows, dim_in, generator=g) * torch.exp(2 * torch.randn(rows, 1, generator=g))).cuda()
    row_ptr, seg = (t.cuda() for t in _segments(rows, rows))
    n_out = row_ptr.numel() - 1
    args = (row_ptr.int(), seg.int(), n_out)
    out = ops.mlp_leaky_rowsum(W[0], b[0], W[1], b[1], x, *args)
    ref, size = _layers_and_sum(x.double(), W, b, seg, n_out)
    assert float(((out.double() - ref).norm(dim=1) / size.clamp_min(1e-30)).max()) <= 1.5e-6
    assert not bool(out[row_ptr[1:] == row_ptr[:-1]].any())
    assert torch.equal(ops.mlp_leaky_rowsum(W[0], b[0], W[1], b[1], x, *args), out)
    # rows that the pieces cannot carry stay in their segments
    x[rows // 2] *= 2.0 ** 110
    x[0, 1] = INF
    odd = ops.mlp_leaky_rowsum(W[0], b[0], W[1], b[1], x, *args)
    hit = torch.zeros(n_out, dtype=torch.bool, device="cuda")
    hit[seg[[0, rows // 2]]] = True
    assert torch.equal(odd[~hit], out[~hit]) and not bool(torch.isfinite(odd[seg[0]]).any())
    if int(seg[rows // 2]) != int(seg[0]):
        big, size = _layers_and_sum(x.double(), W, b, seg, n_out)
        k = seg[rows // 2]
        assert float((odd[k].double() - big[k]).norm() / size[k]) <= 1.5e-6


def _summed(pkg, dim, rows, bias_offset=0):
    """bee_layers.MLP of `dim` columns, rows and their segments, and the sum of the MLP's rows in float32 and float64."""
    torch.manual_seed(dim)
    mlp = pkg.MLP(dim).cuda()
    for k in (0, 2):
        layer = mlp.layers[k]
        flat = torch.zeros(bias_offset + layer.out_features, device="cuda")
        flat[bias_offset:] = layer.bias.detach()
        layer.bias = torch.nn.Parameter(flat[bias_offset:])
    x = torch.randn(rows, dim, generator=torch.Generator().manual_seed(rows)).cuda()
    row_ptr, seg = (t.int().cuda() for t in _segments(rows, dim))
    n_out = row_ptr.numel() - 1

    def reference(dt):
        w = lambda t: t.detach().to(dt)
        W, b = [w(mlp.layers[k].weight) for k in (0, 2, 4)], [w(mlp.layers[k].bias) for k in (0, 2, 4)]
        s_h, _ = _layers_and_sum(x.to(dt), W, b, seg.long(), n_out)
        s_x = torch.zeros(n_out, dim, dtype=dt, device="cuda").index_add(0, seg.long(), x.to(dt))
        count = (row_ptr[1:] - row_ptr[:-1]).to(dt)[:, None]
        return s_x @ w(mlp.lin_direct.weight).t() + s_h @ W[2].t() + count * b[2]

    with torch.no_grad():
        got = mlp.summed_over_rows(x, row_ptr, n_out, seg=seg)
    ref = reference(torch.float64)
    error = lambda y: float((y.double() - ref).norm() / ref.norm())
    return error(got), error(reference(torch.float32))


@pytest.mark.parametrize("rows, dim_in, in_place", [(6177, 96, True), (7001, 64, False)])
def test_linear_and_mlp_summed_over_segments_as_one_matrix(bee, ops, rows, dim_in, in_place):
    """The sums of a linear's rows and of the MLP's hidden rows as blocks of one matrix, against the same sums apart: the hidden rows'
    sums to the bit, their maxima exact, the result as close to float64 (rounding of 768 products and of the additions to the base, with
    empty segments and segments of one row to hundreds)."""
    torch.manual_seed(rows)
    mlp = bee.MLP(256).cuda()
    g = torch.Generator().manual_seed(rows)
    W = (torch.randn(256, dim_in, generator=g) * dim_in ** -0.5).cuda()
    x = torch.randn(rows, dim_in, generator=g).cuda()
    row_ptr, seg = (t.int().cuda() for t in _segments(rows, 7))
    n_out = row_ptr.numel() - 1
    base = torch.randn(n_out, 256, generator=g).cuda() if in_place else None
    with torch.no_grad():
        mlp.layers[4].bias.normal_()
        bound = ops.row_absmax(x)
        assert mlp.takes_linear_summed_over_rows(rows, x, base)
        out = mlp.of_linear_summed_over_rows(W, x, bound, row_ptr, n_out, seg, 0.1, base.clone() if in_place else None)
        s_psi, psi = ops.tensor_linear_f16x2_rowsum(W, x, bound, row_ptr, seg, n_out, want_rows=True)
        apart = mlp.summed_over_rows(psi, row_ptr, n_out, plus_identity=True, seg=seg, s_x=s_psi, scale=0.1,
                                     add_to=base.clone() if in_place else None)
        L = mlp.layers
        s_h = ops.mlp_leaky_rowsum(L[0].weight, L[0].bias, L[2].weight, L[2].bias, psi, row_ptr, seg, n_out)
        S, maxima = torch.full((n_out, 1024), 7., device="cuda"), torch.full((n_out, 4), 7., device="cuda")
        count = torch.empty(n_out, 256, device="cuda")
        ops.tensor_linear_f16x2_rowsum(W, x, bound, row_ptr, seg, n_out, into=(S, maxima, 0), count_bias=L[4].bias, base=count)
        ops.mlp_leaky_rowsum(L[0].weight, L[0].bias, L[2].weight, L[2].bias, psi, row_ptr, seg, n_out, (S, maxima, 256))
    assert torch.equal(S[:, :256], s_psi) and torch.equal(S[:, 256:768], s_h) and bool((S[:, 768:] == 7).all())
    assert torch.equal(maxima, S.view(n_out, 4, 256).abs().amax(2))
    n = (row_ptr[1:] - row_ptr[:-1]).double()[:, None]
    assert torch.equal(count, (n * L[4].bias.double()).float())
    w = lambda t: t.detach().double()
    ref = 0.1 * (s_psi.double() @ w(mlp.lin_direct.weight).t() + s_psi.double() + s_h.double() @ w(L[4].weight).t() + n * w(L[4].bias))
    ref = ref + base.double() if in_place else ref
    error = lambda y: float((y.double() - ref).norm() / ref.norm())
    assert error(out) <= 3e-7 and error(out) <= 1.2 * error(apart)
    # an unaligned base keeps the general path; sizes and columns that do not fit are refused
    assert not mlp.takes_linear_summed_over_rows(rows, x, torch.zeros(n_out * 256 + 1, device="cuda")[1:].view(n_out, 256))
    with pytest.raises(RuntimeError):
        ops.tensor_linear_f16x2_rowsum(W, x, bound, row_ptr, seg, n_out, into=(S, maxima, 800))


def test_messages_whose_hidden_layers_are_no_blocks_of_columns(pkg, bee):
    """Hidden layers of 320 columns, put in the place of the 512 of an MLP on 256: their sums are no block of a matrix whose maxima are
    taken over 256 columns, and the messages sum them by themselves.  Against the layers in float64: products of 768 and fewer terms
    in 22-bit pieces, four layers deep."""
    gl = importlib.import_module("learned-dynamics_amd.graph_layers")
    torch.manual_seed(8)
    N, r0, side = 1024, 5.0, 20.0
    mod = bee.Messages(r0, 256, 16, 8, 64)
    for k, (i, o) in {0: (256, 320), 2: (320, 320), 4: (320, 256)}.items():
        mod.mlp_a.layers[k] = torch.nn.Linear(i, o)
    mod = mod.cuda()
    x = torch.randn(1, N, 256).cuda(), torch.randn(1, N, 16, 3).cuda(), torch.randn(1, N, 8, 3, 3).cuda()
    graph, r_ij = gl.graph_setup(r0, (side,) * 3, (torch.rand(1, N, 3) * side).cuda(), neighbours_max=256, celllist_max=64)
    assert graph.src.numel() >= 4096
    with torch.no_grad():
        got = mod(graph, r_ij, *x)[0]
    x[0].requires_grad_()                                     # the differentiable path runs every layer on every edge
    want = mod(graph, r_ij, *x)[0]
    assert float((got - want.detach()).norm() / want.detach().norm()) <= 2e-6


def test_narrow_layers_summed_over_segments_stay_in_fp32(bee, ops, monkeypatch):
    """A linear of 32 columns has fp32 arithmetic: the kernel of 22-bit pieces takes a layer from 64 columns on."""
    x = torch.zeros(5000, 64).cuda()
    assert ops.mlp_rowsum_supported(5000, 64, 64, x)
    assert not ops.mlp_rowsum_supported(5000, 32, 64, x) and not ops.mlp_rowsum_supported(5000, 64, 32, x)
    monkeypatch.setattr(ops, "mlp_leaky_rowsum", None)
    err, f32 = _summed(bee, 32, 5000)
    assert err <= 2 * f32                                        # (two fp32 sums of the same terms in different orders)


def test_biases_at_any_offset_summed_over_segments(bee, ops, monkeypatch):
    """Biases that are views of a flat buffer: layer by layer, as before there was a kernel for both; that kernel takes the others."""
    rows = 4200
    called, kernel = [], ops.mlp_leaky_rowsum
    monkeypatch.setattr(ops, "mlp_leaky_rowsum", lambda *a: (called.append(1), kernel(*a))[1])
    for offset in (0, 1, 4):
        err, f32 = _summed(bee, 96, rows, bias_offset=offset)
        assert err <= 1.5e-6
        assert len(called) == (0 if offset % 4 else 1), offset
        called.clear()


@pytest.mark.parametrize("rows, dim_in, dim", [(256, 64, 64), (300, 96, 160), (5000, 256, 256)])
def test_leaky_mlp_that_adds_its_input(ops, rows, dim_in, dim):
    """x + mlp(x) and its gradients against the same kernels with the addition outside: one rounding more or less; a row that the pieces
    cannot carry; sizes that differ are refused."""
    g = torch.Generator().manual_seed(rows)
    W = [(torch.randn(o, k, generator=g) * k ** -0.5).cuda() for o, k in ((dim, dim_in), (dim, dim), (dim_in, dim), (dim_in, dim_in))]
    b = [(torch.randn(w.shape[0], generator=g) * 0.1).cuda() for w in W[:3]]
    x, dy = (torch.randn(rows, dim_in, generator=g).cuda() for _ in range(2))
    x[5] *= 2.0 ** -100
    dy[7] *= 2.0 ** -100
    y, saved = ops.mlp_leaky_fwd(x, W, b)
    both, saved_both = ops.mlp_leaky_fwd(x, W, b, True)
    _assert_rows(both, x.double() + y.double(), "x + y")
    assert all(torch.equal(s, t) for s, t in zip(saved, saved_both))
    g_x, params = ops.mlp_leaky_bwd(dy, x, W, saved, True, True)
    g_both, params_both = ops.mlp_leaky_bwd(dy, x, W, saved, True, True, True)
    _assert_rows(g_both, dy.double() + g_x.double(), "g_x")
    assert all(torch.equal(s, t) for s, t in zip(params, params_both))
    narrow = [W[0], W[1], W[2][:32].contiguous(), W[3][:32].contiguous()]
    with pytest.raises(RuntimeError):
        ops.mlp_leaky_fwd(x, narrow, [b[0], b[1], b[2][:32].contiguous()], True)


@pytest.mark.parametrize("rows, dim_in, dim, dim_out", [(256, 64, 64, 32), (257, 96, 96, 160), (700, 256, 512, 256),
                                                         (5000, 64, 128, 64)])
def test_leaky_mlp_and_its_adjoint(ops, rows, dim_in, dim, dim_out):
    """Values, hidden rows and all gradients against float64 (its slopes at the kernel's signs, which may differ from its own only
    where z is within the rounding of a layer of zero); rows as above, weights' gradients in their 2-norm; a row has the
    same bits among fewer rows."""
    g = torch.Generator().manual_seed(rows)
    W = [(torch.randn(o, k, generator=g) * k ** -0.5).cuda() for o, k in ((dim, dim_in), (dim, dim), (dim_out, dim), (dim_out, dim_in))]
    b = [(torch.randn(w.shape[0], generator=g) * 0.1).cuda() for w in W[:3]]
    x, dy = (torch.randn(rows, k, generator=g).cuda() for k in (dim_in, dim_out))
    assert ops.mlp_leaky_takes(x, W, b)
    y, saved = ops.mlp_leaky_fwd(x, W, b)
    Wd, bd, h, slopes, hs = [w.double() for w in W], [t.double() for t in b], x.double(), [], [x.double()]
    for k in range(2):
        z = h @ Wd[k].t() + bd[k]
        kernel = saved[1 + 2 * k]
        assert not bool((((z > 0) != (kernel > 0)) & (z.abs() > 2e-6 * z.norm(dim=1, keepdim=True))).any())
        slopes.append(torch.where(kernel > 0, 1.0, 0.1).double())
        h = z * slopes[-1]
        hs.append(h)
        _assert_rows(kernel, h, ("h", k))
        assert torch.equal(saved[2 + 2 * k][:, 0], kernel.abs().amax(1))
    assert torch.equal(saved[0][:, 0], x.abs().amax(1))
    _assert_rows(y, h @ Wd[2].t() + bd[2] + hs[0] @ Wd[3].t(), "y")
    g_x, params = ops.mlp_leaky_bwd(dy, x, W, saved, True, True)
    d = dy.double()
    dz2 = (d @ Wd[2]) * slopes[1]
    dz1 = (dz2 @ Wd[1]) * slopes[0]
    _assert_rows(g_x, dz1 @ Wd[0] + d @ Wd[3], "g_x")
    refs = dz1.t() @ hs[0], dz1.sum(0), dz2.t() @ hs[1], dz2.sum(0), d.t() @ hs[2], d.sum(0), d.t() @ hs[0]
    for k, (p, r) in enumerate(zip(params, refs)):
        assert p.shape == r.shape and float((p.double() - r).norm() / r.norm()) <= 1.5e-6, k
    assert ops.mlp_leaky_bwd(dy, x, W, saved, False, True)[0] is None
    assert torch.equal(ops.mlp_leaky_fwd(x[:256].contiguous(), W, b)[0], y[:256])
    x[3, 1] = INF
    odd, _ = ops.mlp_leaky_fwd(x, W, b)
    keep = torch.arange(rows, device="cuda") != 3
    assert torch.equal(odd[keep], y[keep]) and not bool(torch.isfinite(odd[3]).any())


@pytest.mark.parametrize("rows, dim_in, dim", [((1, 33), (64, 96), 64), ((512, 4096), (64, 64), 512), ((4096, 700), (64, 160), 256),
                                               ((9000, 8000), (64, 128), 512)])
def test_two_mlps_in_one_launch(ops, rows, dim_in, dim):
    """The grids of two filters of one width together, on either side of the line to 64 rows a workgroup."""
    unit = torch.ones(1, 1).cuda()
    jobs = []
    for k in range(2):
        W, b = _weights(dim_in[k], dim, seed=k)
        x = torch.rand(rows[k], dim_in[k], generator=torch.Generator().manual_seed(k)).cuda() * 2 - 1
        jobs.append((x, unit, W, b))
    for y, (x, _, W, b) in zip(ops.filter_grids(*jobs), jobs):
        _assert_rows(y, _formula(x.double(), W, b), (rows, dim_in, dim))
    # layers of two widths, and encodings that end in zero columns
    (x, _, W, b), other = jobs[0], _weights(64, 96)
    alone = ops.filter_grid(x, unit, W, b), ops.filter_grid(x[:, :64].contiguous(), unit, *other)
    assert all(torch.equal(p, q) for p, q in zip(ops.filter_grids((x, unit, W, b), (x[:, :64].contiguous(), unit, *other)), alone))
    narrow = [W[0][:, :48].contiguous(), *W[1:]]
    padded = torch.cat([x[:, :48], torch.zeros_like(x[:, 48:])], dim=1)
    for y in ops.filter_grids((padded, unit, narrow, b), (padded, unit, narrow, b)):
        _assert_rows(y, _formula(x[:, :48].double(), narrow, b), "zero columns")


@pytest.mark.parametrize("rows, dim", [((700, 1, 33, 4096), 128), ((672,) * 5 + (6100,) * 5, 512), ((64,) * 17 + (3000,), 256), ((5, 0, 9), 512)])
def test_many_mlps_in_one_launch(ops, rows, dim):
    """As many as sixteen and more, one set of rows under several weights, none at all: each as by itself."""
    unit = torch.ones(1, 1).cuda()
    x = torch.rand(max(rows), 64, generator=torch.Generator().manual_seed(dim)).cuda() * 2 - 1
    jobs = [(x[:r], unit, *_weights(64, dim, seed=k)) for k, r in enumerate(rows)]
    for r, y, (x_k, _, W, b) in zip(rows, ops.filter_grids(*jobs), jobs):
        assert y.shape == (r, dim)
        if r:
            _assert_rows(y, _formula(x_k.double(), W, b), (r, dim))
    assert len(ops.filter_grids()) == 0


@pytest.mark.parametrize("rows, dim_in, dim", [(1024, 64, 512), (1025, 64, 512), (1344, 256, 384), (1345, 256, 384), (1023, 64, 320), (1024, 64, 320)])
def test_wide_mlp_on_either_side_of_the_line(ops, rows, dim_in, dim):
    """Three launches that split their reductions up to one round of the chip, one kernel beyond: the same tolerance."""
    W, b = _weights(dim_in, dim)
    x = torch.randn(rows, dim_in, generator=torch.Generator().manual_seed(rows)).cuda()
    _assert_rows(ops.linear_chain(x, W, b, ACTS, None), _formula(x.double(), W, b), (rows, dim))


BAD = [(0, INF), (0, NAN), (1, INF), (1, NAN), (2, INF), (2, NAN), (2, 2.0 ** 110)]


def _with(W, layer, value):
    """The weights with one entry that the pieces cannot carry."""
    W = [w.clone() for w in W]
    W[layer][5, 3] = value
    return W


def _assert_like(y, ref, what):
    """Finite where the formula in float64 is (which does not overflow where float32 would: larger than it holds counts as infinite).
    There, row by row over the columns of ordinary size, as exact as any other result; a column made of ONE hidden value times 2^110
    has that value's error, which is in proportion to its row and not to itself: relative to the column."""
    finite = torch.isfinite(ref.float())
    assert torch.equal(torch.isfinite(y), finite), what
    large = finite.all(0) & (ref.abs().amax(0) > 2.0 ** 60)
    cols = finite.all(0) & ~large
    if bool(cols.any()):
        _assert_rows(y[:, cols], ref[:, cols], what)
    if bool(large.any()):
        assert float(((y[:, large].double() - ref[:, large]).norm(dim=0) / ref[:, large].norm(dim=0)).max()) <= 1.5e-6, what


@pytest.mark.parametrize("layer, value", [t for t in BAD if t[0] < 2])
@pytest.mark.parametrize("rows, dim_in, dim", [(300, 64, 64), (4161, 128, 512)])
def test_weights_beyond_the_pieces_summed_over_segments(ops, rows, dim_in, dim, layer, value):
    W, b = (t[:2] for t in _weights(dim_in, dim))
    W = _with(W, layer, value)
    x = torch.randn(rows, dim_in, generator=torch.Generator().manual_seed(rows)).cuda()
    row_ptr, seg = (t.cuda() for t in _segments(rows, rows))
    n_out = row_ptr.numel() - 1
    out = ops.mlp_leaky_rowsum(W[0], b[0], W[1], b[1], x, row_ptr.int(), seg.int(), n_out)
    ref, _ = _layers_and_sum(x.double(), W, b, seg, n_out)
    filled = row_ptr[1:] > row_ptr[:-1]
    assert torch.equal(torch.isfinite(out), torch.isfinite(ref)) and not bool(out[~filled].any())
    cols = [k for k in range(dim) if k != 5]
    if layer == 1:
        _, size = _layers_and_sum(x.double(), [W[0], W[1][cols]], [b[0], b[1][cols]], seg, n_out)
        assert float(((out[:, cols].double() - ref[:, cols]).norm(dim=1) / size.clamp_min(1e-30)).max()) <= 1.5e-6
        assert not bool(torch.isfinite(out[filled][:, 5]).any())
    else:
        assert not bool(torch.isfinite(out[filled]).any())


@pytest.mark.parametrize("layer, value", BAD)
@pytest.mark.parametrize("leaky", [False, True])
@pytest.mark.parametrize("rows, dim", [(300, 64), (1400, 512), (8300, 512)])
def test_weights_beyond_the_pieces_under_differentiation(ops, rows, dim, leaky, layer, value):
    """One weight of each layer that is infinite, undefined or beyond the pieces, forward and in the gradient of x (whose hidden rows
    are those of the finite weights, so that it is the adjoint's own products that meet it)."""
    W, b = _weights(64, dim)
    x = torch.randn(rows, 64, generator=torch.Generator().manual_seed(1)).cuda()
    gy = torch.randn(rows, dim, generator=torch.Generator().manual_seed(2)).cuda()
    Wd = torch.randn(dim, 64, generator=torch.Generator().manual_seed(3)).cuda() / 8
    act = (lambda z: torch.nn.functional.leaky_relu(z, 0.1)) if leaky else torch.nn.functional.silu
    bad = _with(W, layer, value)
    h = x.double()
    for k in range(3):
        h = h @ bad[k].double().t() + b[k].double()
        h = act(h) if k < 2 else h
    if leaky:
        y, _ = ops.mlp_leaky_fwd(x, bad + [Wd], b)
        h = h + x.double() @ Wd.double().t()
        _, saved = ops.mlp_leaky_fwd(x, W + [Wd], b)
        g_x, _ = ops.mlp_leaky_bwd(gy, x, bad + [Wd], saved, True, False)
        slopes = [torch.where(saved[1 + 2 * k] > 0, 1.0, 0.1).double() for k in range(2)]
    else:
        y, _, _ = ops.mlp_silu_fwd(x, None, None, bad, b, True)
        _, _, saved = ops.mlp_silu_fwd(x, None, None, W, b, True)
        g_x, _, _ = ops.mlp_silu_bwd(gy, None, x, None, bad, saved, True, False)
        s = [torch.sigmoid(saved[1 + 3 * k].double()) for k in range(2)]
        slopes = [s[k] * (1 + saved[1 + 3 * k].double() * (1 - s[k])) for k in range(2)]
    _assert_like(y, h, "y")
    d = gy.double() @ bad[2].double() * slopes[1]
    d = d @ bad[1].double() * slopes[0]
    _assert_like(g_x, d @ bad[0].double() + (gy.double() @ Wd.double() if leaky else 0), "g_x")


@pytest.mark.parametrize("rows, dim", [(300, 64), (4200, 512)])
def test_tangents_and_gradients_of_a_row_beyond_the_pieces(ops, rows, dim):
    """A tangent row of the dual kernel and a gradient row of the LeakyReLU adjoint: linear in them, and no other row notices."""
    W, b = _weights(64, dim)
    g = torch.Generator().manual_seed(4)
    x, x_t = torch.randn(rows, 64, generator=g).cuda(), torch.randn(rows, 64, generator=g).cuda()
    y, y_t, _ = ops.mlp_silu_fwd(x, x_t, None, W, b, True)
    odd = x_t.clone()
    odd[5] *= 2.0 ** 110
    odd[rows - 2, 3] = INF
    same = torch.ones(rows, dtype=torch.bool, device="cuda")
    same[[5, rows - 2]] = False
    z, z_t, _ = ops.mlp_silu_fwd(x, odd, None, W, b, True)
    assert torch.equal(z, y) and torch.equal(z_t[same], y_t[same]) and not bool(torch.isfinite(z_t[rows - 2]).any())
    assert float((z_t[5].double() * 2.0 ** -110 - y_t[5].double()).norm() / y_t[5].double().norm()) <= 1.5e-6
    Wd = torch.randn(dim, 64, generator=g).cuda() / 8
    gy = torch.randn(rows, dim, generator=g).cuda()
    _, saved = ops.mlp_leaky_fwd(x, W + [Wd], b)
    clean, _ = ops.mlp_leaky_bwd(gy, x, W + [Wd], saved, True, False)
    gy[5] *= 2.0 ** 100
    gy[rows - 2, 3] = INF
    g_x, _ = ops.mlp_leaky_bwd(gy, x, W + [Wd], saved, True, False)
    assert torch.equal(g_x[same], clean[same]) and not bool(torch.isfinite(g_x[rows - 2]).any())
    assert float((g_x[5].double() * 2.0 ** -100 - clean[5].double()).norm() / clean[5].double().norm()) <= 1.5e-6


@pytest.mark.parametrize("layer, value", BAD)
def test_a_weight_beyond_the_pieces_in_one_of_two_mlps(ops, layer, value):
    unit = torch.ones(1, 1).cuda()
    W, b = _weights(64, 96)
    x = torch.rand(500, 64, generator=torch.Generator().manual_seed(3)).cuda()
    bad = _with(W, layer, value)
    one, other = ops.filter_grids((x, unit, W, b), (x, unit, bad, b))
    assert torch.equal(one, ops.filter_grid(x, unit, W, b))
    _assert_like(other, _formula(x.double(), bad, b), (layer, value))


@pytest.mark.parametrize("n, rows", [(128, [6000] * 6), (128, [1100, 16000, 2000, 9000, 5000]), (64, [300, 20000, 5000, 7000]), (64, [700] * 33)])
def test_filters_evaluated_together_are_those_evaluated_alone(pkg, ops, n, rows):
    """More rows together than the chip holds in tiles of 32, some of them more by themselves, more MLPs than a launch takes: every one
    the bits that it has alone."""
    painn = importlib.import_module("learned-dynamics_amd.painn")
    torch.manual_seed(n + len(rows))
    jobs = []
    with torch.no_grad():
        for E in rows:
            msg = painn.Message(5.0, n).cuda()
            enc = ops.painn_radial_encode(torch.randn(E, 3, device="cuda") * 2, msg.n_rbf, 5.0)
            jobs.append((enc, ops.linear_in_unit_bound(enc.device), *painn._plain_params(msg.mlp_dist)))
        for y, job in zip(ops.filter_grids(*jobs), jobs):
            assert torch.equal(y, ops.filter_grid(*job)), job[0].shape

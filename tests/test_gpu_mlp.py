"""Linear, SiLU, Linear, SiLU, Linear as one kernel (csrc/mlp_f16x2.hip) against the same formula in float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu

ACTS = (1, 1, 0)
INF, NAN = float("inf"), float("nan")


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


def _assert_rows(y, ref, what):
    """2-norm of a row's difference against the row's: three layers, each rounding its operands to 22 bits and its sums and
    activation to 24, err by 5e-7 at most; measured 2e-7 .. 3e-7 over all rows."""
    err = (y.double() - ref).norm(dim=1) / ref.norm(dim=1)
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

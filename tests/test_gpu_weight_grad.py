"""Parameter gradients of Linear layers (weight_grad) against float64, and the training Linear that uses them."""
import pytest
import torch

pytestmark = pytest.mark.gpu

EPS = {torch.float32: 2.0 ** -23, torch.float16: 2.0 ** -10, torch.bfloat16: 2.0 ** -7}


def _native():
    from clusten import _native as nat
    return nat


def _bound(d_y, x):
    """Products of 16-bit values are exact in fp32 and fp32 ones round once; a sum of `rows` of them in fp32, in any order,
    is off by at most rows * 2^-24 of the sum of magnitudes (far less in practice: 8 * sqrt(rows) of them is used)."""
    rows = d_y.shape[0]
    return 2.0 ** -24 * 8 * (rows ** 0.5 + 2) * (d_y.abs().t().double() @ x.abs().double()) + 1e-30


# tiles of 64 and 128, stages of 32 to 128 rows: one row, edges of a stage and of four, the longest of AFF-Tiny's first stage / 8
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16], ids=str)
@pytest.mark.parametrize("rows", [1, 31, 64, 127, 129, 513, 25089])
def test_weight_grad_against_float64(dtype, rows):
    nat = _native()
    gen = torch.Generator(device="cuda").manual_seed(rows)
    for shapes in ([(8, 8)], [(96, 32), (32, 32), (64, 32), (32, 64)], [(192, 64), (72, 200)], [(384, 128), (128, 256), (128, 384)]):
        pairs = []
        for i, (n, k) in enumerate(shapes):
            d_y = torch.randn(rows, n + 8, generator=gen, device="cuda").to(dtype)[:, :n]      # rows apart from each other
            pairs.append((d_y, torch.randn(rows, k, generator=gen, device="cuda").to(dtype), i != 1))
        for (d_w, d_b), (d_y, x, with_bias) in zip(nat.weight_grad(pairs), pairs):
            want = d_y.double().t() @ x.double()
            assert bool(((d_w.double() - want).abs() <= _bound(d_y, x)).all())
            assert (d_b is not None) == with_bias
            if with_bias:
                one = torch.ones(rows, 1, device="cuda", dtype=dtype)
                assert bool(((d_b.double() - d_y.double().sum(0)).abs() <= _bound(d_y, one)[:, 0]).all())
        again = nat.weight_grad(pairs)
        first = nat.weight_grad(pairs)
        assert all(torch.equal(a[0], b[0]) for a, b in zip(again, first))


# ranges of 512 rows: 1 to 12 of them are added up by one thread, 13 to 48 by four, more by sixteen
@pytest.mark.parametrize("splits", [1, 12, 13, 48, 49, 65])
def test_sums_of_the_splits(splits):
    nat = _native()
    gen = torch.Generator(device="cuda").manual_seed(splits)
    d_y, x = (torch.randn(512 * splits, 64, generator=gen, device="cuda").half() for _ in range(2))
    (d_w, d_b), = nat.weight_grad([(d_y, x, True)])
    assert bool(((d_w.double() - d_y.double().t() @ x.double()).abs() <= _bound(d_y, x)).all())
    one = torch.ones(512 * splits, 1, device="cuda").half()
    assert bool(((d_b.double() - d_y.double().sum(0)).abs() <= _bound(d_y, one)[:, 0]).all())


def test_an_infinity_stays_in_its_row_and_column():
    nat = _native()
    d_y, x = torch.ones(130, 64, device="cuda").half(), torch.ones(130, 64, device="cuda").half()
    d_y[129, 5], x[3, 7] = float("inf"), float("nan")
    (d_w, d_b), = nat.weight_grad([(d_y, x, True)])
    assert bool(d_w[:, 7].isnan().all()) and bool(d_w[5, :7].isinf().all()) and bool(d_b[5].isinf())
    d_w[5], d_w[:, 7], d_b[5] = 130, 130, 130
    assert bool((d_w == 130).all()) and bool((d_b == 130).all())


@pytest.mark.parametrize("amp", [None, torch.float16])
def test_training_linear(amp):
    """Against the layer itself: the value bit for bit, gradients to the storage type's rounding; a second derivative too."""
    from aff.model import _linear, default_ops
    torch.manual_seed(3)
    lin = torch.nn.Linear(64, 192).cuda()
    x = torch.randn(5, 77, 64, device="cuda", requires_grad=True)
    g = torch.randn(5, 77, 192, device="cuda")

    def grads(fn):
        with torch.autocast("cuda", dtype=amp or torch.float16, enabled=amp is not None):
            y = fn(x)
        return y, torch.autograd.grad(y, [x, lin.weight, lin.bias], g.to(y.dtype), create_graph=True)

    (y, got), (want_y, want) = grads(lambda t: _linear(lin, t, default_ops())), grads(lin)
    assert torch.equal(y, want_y)
    torch.autograd.grad(got[1].float().square().sum(), x)       # the recorded backward is differentiable
    y = _run(lin, x, amp)
    got = torch.autograd.grad(y, [x, lin.weight, lin.bias], g.to(y.dtype))
    tol = 4 * EPS[amp or torch.float32]
    for a, b in zip(got, want):
        assert a.dtype == b.dtype and float((a - b).norm() / b.norm()) < tol


def _run(lin, x, amp):
    from aff.model import _linear, default_ops
    with torch.autocast("cuda", dtype=amp or torch.float16, enabled=amp is not None):
        return _linear(lin, x, default_ops())

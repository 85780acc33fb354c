"""Products of few rows by workgroups of more than 64 rows of weights."""
import pytest
import torch

from aurora_amd import ops

pytestmark = pytest.mark.gpu


def _check(got, want):
    """64 bits rounded to bf16, but for fp32 sums whose error is far below 2^-16 of the largest."""
    slack = 2 ** -16 * want.abs().max()
    assert ((got.double() - want).abs() <= want.abs() * 2 ** -8 + slack).all()


def _inputs(m, n, k):
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    x, w = (torch.randn(r, k, generator=g, device="cuda").bfloat16() for r in (m, n))
    return x, w * k ** -0.5


@pytest.mark.parametrize("m", [1, 32, 33, 64, 65, 96, 97, 128])
@pytest.mark.parametrize("n,k", [(8, 64), (95, 128), (97, 192), (129, 448), (1000, 576)])
@pytest.mark.parametrize("width", [96, 128])
def test_wide_tiles(m, n, k, width):
    x, w = _inputs(m, n, k)
    want = x.double() @ w.double().t()
    for parts in (1, 3, 16):
        _check(ops._hip.few_rows(x, w, False, parts, width), want)
        raw = ops._hip.few_rows(x, w, True, parts, width)
        _check((raw.sum(0) if raw.dim() == 3 else raw).bfloat16(), want)


@pytest.mark.parametrize("m", [33, 65, 97, 128])
@pytest.mark.parametrize("n", [14336, 14344])  # a tile of 112 for every CU, and one too many
def test_silu_tiles(m, n):
    x, w = _inputs(m, 2 * n, 192)
    y = x.double() @ w.double().t()
    _check(ops._hip.silu_few_rows(x, w), torch.nn.functional.silu(y[:, :n]) * y[:, n:])


@pytest.mark.parametrize("m", [52, 53])
@pytest.mark.parametrize("n", [13056, 13064])
def test_silu_rows_far_apart(m, n):
    """Tiles of 64 and 112 on either side of their line."""
    x, w = _inputs(m, 2 * n, 2048)
    y = x.double() @ w.double().t()
    _check(ops._hip.silu_few_rows(x, w), torch.nn.functional.silu(y[:, :n]) * y[:, n:])


@pytest.mark.parametrize("m", [1, 2, 40, 70, 128])
@pytest.mark.parametrize("n,k", [(6144, 4096), (8576, 4160), (3584, 18944)])
def test_chosen_cuts(m, n, k):
    """Sizes whose cuts are wide, and weights beyond 128 MB in parts."""
    x, w = _inputs(m, n, k)
    want = x.double() @ w.double().t()
    y = ops.linear_parts(x, w)
    _check((y.sum(0) if y.dim() == 3 else y).bfloat16(), want)
    _check(ops.linear(x, w), want)
    if n <= 8192 and k > 4096:
        assert y.dim() == 3


@pytest.mark.parametrize("m", [2, 40, 70, 128])
@pytest.mark.parametrize("n", [64, 512, 768, 1024, 1536, 2048])
def test_steps_that_do_not_divide(m, n):
    """Every number of steps is cut, into parts that use at least half of what 64 rows of weights
    leave room for."""
    for steps in (20, 24, 25, 31, 36, 40, 55, 56, 64, 81):
        x, w = _inputs(m, n, steps * 64)
        y = ops.linear_parts(x, w)
        room = min(256 // (-(-n // 64)), steps // 2, 16)
        assert y.dim() == 3 and y.shape[0] >= room / 2
        _check(y.sum(0).bfloat16(), x.double() @ w.double().t())


@pytest.mark.parametrize("m", [65, 97, 129, 192, 193, 300, 1000])
@pytest.mark.parametrize("n,k", [(512, 576), (768, 3072), (2048, 2048), (2120, 4160), (72, 64),
                                 (3400, 1024)])
def test_blocks_of_rows(m, n, k):
    """65 to 1000 rows: every form, whole and in parts, rows past a block's end."""
    x, w = _inputs(m, n, k)
    want = x.double() @ w.double().t()
    for rows in (64, 96, 128):
        for width, parts in ((64, 1), (64, 3), (128, 1), (128, 2)):
            _check(ops._hip.few_rows(x, w, False, parts, width, rows), want)
            raw = ops._hip.few_rows(x, w, True, parts, width, rows)
            _check((raw.sum(0) if raw.dim() == 3 else raw).bfloat16(), want)
    _check(ops.linear(x, w), want)
    y = ops.linear_parts(x, w)
    _check((y.sum(0) if y.dim() == 3 else y).bfloat16(), want)


@pytest.mark.parametrize("m", [129, 192, 300])
def test_blocks_whose_steps_do_not_divide(m):
    """44 steps in 15 parts of three and less, where 16 were asked for."""
    x, w = _inputs(m, 512, 44 * 64)
    y = ops.linear_parts(x, w)
    assert y.dim() == 3 and y.shape[0] >= 5
    _check(y.sum(0).bfloat16(), x.double() @ w.double().t())


@pytest.mark.parametrize("m,n,experts,parts", [(256, 4096, False, True), (257, 4096, False, False),
                                               (257, 4096, True, True), (300, 2048, False, True),
                                               (300, 2064, False, False)])
def test_parts_that_a_norm_holds(m, n, experts, parts):
    x, w = _inputs(m, n, 14336)
    assert ops.linear_parts(x, w).dim() == 3
    y = ops.linear_norm_parts(x, w, experts)
    assert (y.dim() == 3) == parts
    _check((y.sum(0) if parts else y).bfloat16(), x.double() @ w.double().t())


@pytest.mark.parametrize("m,n,k,own", [
    (512, 4096, 4096, True), (1000, 2048, 576, True), (1000, 512, 576, True),
    (513, 4096, 640, False), (1001, 2048, 576, False), (300, 504, 1024, False),
    (300, 1024, 512, True), (300, 1456, 512, False), (300, 2824, 256, True), (128, 8192, 64, True),
    (129, 64, 320, True), (128, 56, 256, False), (65, 2816, 2048, True), (65, 2816, 2112, False),
    (100, 2808, 576, False), (128, 8192, 1024, True), (64, 64, 64, True)])
def test_line_to_the_library(m, n, k, own):
    x, w = _inputs(m, n, k)
    got = ops._hip.own_product(x, w, 0)
    assert (got is not None) == own
    strided = torch.cat([x, x], 1)[:, :k]  # rows apart
    _check(ops.linear(strided, w), x.double() @ w.double().t())


@pytest.mark.parametrize("m,n,k,own", [
    (512, 3584, 2048, True), (512, 2816, 4096, False), (512, 2816, 2048, True),
    (384, 3584, 4096, True), (512, 3328, 4096, False), (512, 3584, 4096, True),
    (300, 4608, 3584, False), (1000, 1536, 5632, False), (256, 8192, 4096, True)])
def test_line_of_long_rows(m, n, k, own):
    """Workgroups of one round and more, blocks of a tile on few XCDs and many."""
    x, w = _inputs(m, n, k)
    assert (ops._hip.own_product(x, w, 0) is not None) == own
    _check(ops.linear(x, w), x.double() @ w.double().t())


@pytest.mark.parametrize("m", [2, 33, 65, 128])
@pytest.mark.parametrize("n,k,parts", [(6144, 4096, 2), (4096, 14336, 4), (4608, 3584, 3),
                                       (2048, 2048, 8), (64, 8192, 16)])
def test_steady(m, n, k, parts):
    """What fills an 8-bit cache: K in the parts that 64 rows of weights want."""
    x, w = _inputs(m, n, k)
    y = ops.linear_parts(x, w, True)
    assert torch.equal(y, ops._hip.few_rows(x, w, True, parts, 64))
    whole = ops._hip.own_product(x, w, 4)
    if whole is not None:
        cut = k * (2 if m > 32 else 1) >= 4096
        assert torch.equal(whole, ops._hip.few_rows(x, w, False, parts if cut else 1, 64))


def test_steady_leaves_the_library_its_own():
    for m, n, k in ((16, 3584, 18944), (96, 9216, 4096)):
        x, w = _inputs(m, n, k)
        assert ops._hip.own_product(x, w, 5) is None and ops._hip.own_product(x, w, 1) is not None
        assert torch.equal(ops.linear_parts(x, w, True), torch.nn.functional.linear(x, w))

"""The grouped product of 256-row tiles: stages, ragged tiles of rows and columns."""
import pytest
import torch

from aurora_amd.ops.sequence import _hip

pytestmark = pytest.mark.gpu


def _rows_of(E, top, least):
    """Rows of experts at the edges of a tile, the rest evenly, ``least`` each on average."""
    edges = [0, 1, 255, 256, 257, 600, 16, 0]
    left = least * E - sum(edges)
    rows = edges + [left // (E - len(edges))] * (E - len(edges))
    rows[-1] += -sum(rows) % top
    return rows


#: width, ff, experts: 1, 2 and 3, 5 and 7, 16 and 9 stages; columns of a tile and less
@pytest.mark.parametrize("W,F,E,top", [(64, 64, 128, 1), (128, 192, 100, 2), (320, 448, 48, 1),
                                       (1024, 576, 24, 3)])
@pytest.mark.parametrize("kind", ["glu", "relu2"])
def test_tiles(W, F, E, top, kind):
    g = torch.Generator(device="cuda").manual_seed(W)
    rows = torch.tensor(_rows_of(E, top, 84), device="cuda")
    sel = torch.repeat_interleave(torch.arange(E, device="cuda"), rows)
    sel = sel[torch.randperm(len(sel), generator=g, device="cuda")].int().view(-1, top).contiguous()
    T = len(sel)
    n = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    h, dn = n(T, W).bfloat16(), (n(E, W, F) * F ** -0.5).bfloat16()
    up = (n(E, (2 if kind == "glu" else 1) * F, W) * W ** -0.5).bfloat16()
    if kind == "glu":
        y, place = _hip("moe_clamped_glu").moe_clamped_glu(h, sel, up, dn, 0.9, 1.702, 1.0)
    else:
        y, place = _hip("moe_relu2").moe_relu2(h, sel, up, dn)
    assert sorted(place.flatten().tolist()) == list(range(T * top))
    for e in range(E):
        t, k = (sel == e).nonzero(as_tuple=True)
        z = h[t].double() @ up[e].double().t()
        if kind == "glu":
            a, b = z[:, :F].clamp(max=0.9), z[:, F:].clamp(-0.9, 0.9)
            z = a * torch.sigmoid(1.702 * a) * (b + 1)
        else:
            z = z.clamp(min=0) ** 2
        want = z @ dn[e].double().t()
        # activations and then results are rounded, each by up to 2^-8 of itself
        err = (y[place[t, k].long()].double() - want).norm(dim=-1)
        through = torch.linalg.matrix_norm(dn[e].double(), 2) * z.norm(dim=-1)
        assert (err <= 2 ** -8 * (want.norm(dim=-1) + through) + 1e-9).all()


@pytest.mark.parametrize("T", [1, 129, 255, 256, 257, 2100])
@pytest.mark.parametrize("N,K", [(16, 64), (200, 128), (258, 192), (1000, 448), (2080, 1024)])
@pytest.mark.parametrize("silu", [False, True])
def test_dense(T, N, K, silu):
    """The same tiles without experts; 2100 rows of 2080 columns make a second band."""
    g = torch.Generator(device="cuda").manual_seed(T + N)
    x = torch.randn(T, K, generator=g, device="cuda").bfloat16()
    w = (torch.randn(N * (1 + silu), K, generator=g, device="cuda") * K ** -0.5).bfloat16()
    got = _hip("many_rows").many_rows(x, w, silu).double()
    want = x.double() @ w.double().t()
    if silu:
        want = torch.nn.functional.silu(want[:, :N]) * want[:, N:]
    # rounded by up to 2^-8 of itself; fp32 sums of K terms stay below 2^-16 of the largest
    assert ((got - want).abs() <= 2 ** -8 * want.abs() + 2 ** -16 * want.abs().max()).all()


#: rows at the edges of 32 and of the tiles that a product is cut into; K of two and three stages
@pytest.mark.parametrize("T", [31, 33, 64, 65, 128, 160, 161, 192, 224, 225, 513, 1057, 5000])
@pytest.mark.parametrize("N,K", [(264, 128), (1032, 192), (2048, 512)])
@pytest.mark.parametrize("silu", [False, True])
def test_rows_of_a_tile(T, N, K, silu):
    """Tiles of every height, strided rows of x, and nothing written past the last row."""
    g = torch.Generator(device="cuda").manual_seed(T + N)
    x = torch.randn(T, K + 136, generator=g, device="cuda").bfloat16()[:, 64:64 + K]
    w = (torch.randn(N * (1 + silu), K, generator=g, device="cuda") * K ** -0.5).bfloat16()
    got = _hip("many_rows").many_rows(x, w, silu)
    assert got.equal(_hip("many_rows").many_rows(x.contiguous(), w, silu))
    want = x.double() @ w.double().t()
    if silu:
        want = torch.nn.functional.silu(want[:, :N]) * want[:, N:]
    # rounded by up to 2^-8 of itself; fp32 sums of K terms stay below 2^-16 of the largest
    assert ((got.double() - want).abs() <= 2 ** -8 * want.abs() + 2 ** -16 * want.abs().max()).all()


@pytest.mark.parametrize("W,F,E,top", [(128, 256, 180, 1), (192, 320, 180, 2), (520, 448, 64, 1)])
@pytest.mark.parametrize("kind", ["glu", "relu2"])
def test_tiles_of_uneven_experts(W, F, E, top, kind):
    """Enough experts of 36 rows and more for tiles of up to 256: experts cut into two to five
    alike, those of no and of one row, and the two products' tables."""
    W = W // 64 * 64
    g = torch.Generator(device="cuda").manual_seed(E + W)
    rows = [0, 1, 31, 32, 33, 255, 256, 257, 289, 600, 1100, 16, 0] + [45] * (E - 13)
    rows[-1] += -sum(rows) % top
    A = sum(rows)
    assert A >= 36 * E and (A // 128 + E) * min(-(-F // 256), -(-W // 256)) >= 170
    sel = torch.repeat_interleave(torch.arange(E, device="cuda"), torch.tensor(rows, device="cuda"))
    sel = sel[torch.randperm(A, generator=g, device="cuda")].int().view(-1, top).contiguous()
    n = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    h, dn = n(len(sel), W).bfloat16(), (n(E, W, F) * F ** -0.5).bfloat16()
    up = (n(E, (2 if kind == "glu" else 1) * F, W) * W ** -0.5).bfloat16()
    if kind == "glu":
        y, place = _hip("moe_silu_glu").moe_silu_glu(h, sel, up, dn)
    else:
        y, place = _hip("moe_relu2").moe_relu2(h, sel, up, dn)
    assert sorted(place.flatten().tolist()) == list(range(A))
    for e in range(E):
        t, k = (sel == e).nonzero(as_tuple=True)
        z = h[t].double() @ up[e].double().t()
        z = torch.nn.functional.silu(z[:, :F]) * z[:, F:] if kind == "glu" else z.clamp(min=0) ** 2
        want = z @ dn[e].double().t()
        # activations and then results are rounded, each by up to 2^-8 of itself
        err = (y[place[t, k].long()].double() - want).norm(dim=-1)
        through = torch.linalg.matrix_norm(dn[e].double(), 2) * z.norm(dim=-1)
        assert (err <= 2 ** -8 * (want.norm(dim=-1) + through) + 1e-9).all()

"""The fp16 GEMMs of the diffusion transformer at the row counts where their tile rule changes (640 and 1536 rows), with
rows and columns that end inside a tile, against float64 from the fp16 operands."""

import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

ROWS = [1, 63, 639, 641, 1535, 1537]


def _half(*shape, scale=1.0):
    return (torch.randn(shape, device="cuda") * scale).half()


@pytest.mark.parametrize("R", ROWS)
@pytest.mark.parametrize("K,M", [(768, 2048), (768, 2052), (832, 3072)])
def test_wide_projection(R, K, M):
    """fp16 out: an fp16 rounding of an fp32 sum over K products (2^-24 sqrt(K) of their size)."""
    from boltz_mlx_amd import kernels as Kn

    torch.manual_seed(R + K + M)
    x, w, b = _half(R, K), _half(M, K, scale=K ** -0.5), torch.randn(M, device="cuda")
    ref = x.double() @ w.double().T + b.double()
    got = Kn.linear(x, w, bias=b).double()
    assert ((got - ref).abs() <= ref.abs() * 2.0 ** -11 + 1e-5).all()


@pytest.mark.parametrize("R", ROWS)
@pytest.mark.parametrize("K,M", [(768, 768), (1536, 100), (64, 2048)])
def test_gated(R, K, M):
    """fp32 out: the sum's error and the fast sigmoid's (1e-6 of the product)."""
    from boltz_mlx_amd import kernels as Kn

    torch.manual_seed(R + K + M)
    x, w = _half(R, K), _half(M, K, scale=K ** -0.5)
    gate, y = torch.randn((max(R // 5, 1), M), device="cuda"), torch.randn((R, M), device="cuda")
    g = torch.sigmoid(gate.double())[torch.arange(R, device="cuda") % gate.shape[0]]
    ref = y.double() + g * (x.double() @ w.double().T)
    Kn.linear_gated(x, w, gate, y)
    assert (y.double() - ref).abs().max() < 2e-5


@pytest.mark.parametrize("R", ROWS)
@pytest.mark.parametrize("K,H", [(768, 1536), (64, 64), (128, 96)])
def test_swiglu3(R, K, H):
    """fp16 out of three fp32 sums' product: the rounding, and each factor's error on the product (5e-6 of its largest)."""
    from boltz_mlx_amd import kernels as Kn

    torch.manual_seed(R + K + H)
    x, w = _half(R, K), _half(3 * H, K, scale=K ** -0.5)
    a, b, c = (x.double() @ w.double().T).split(H, -1)
    ref = torch.nn.functional.silu(a) * b * c
    got = Kn.linear_swiglu3(x, Kn.group_swiglu3_rows(w[:H], w[H:2 * H], w[2 * H:])).double()
    assert ((got - ref).abs() <= ref.abs() * 2.0 ** -11 + ref.abs().max() * 5e-6 + 2.0 ** -25).all()

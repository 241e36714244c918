"""The fp32 kernels that run on the bf16 matrix cores with every operand split into three exact parts, against plain
torch in float64 at the sizes where their tiles, stages and masks end, and against the kernels they stand beside.

Tolerance: fp32 sums over up to N terms of softmax weights or products err by a few 1e-7 of the output's norm (the
float32 VALU kernels measure 2e-7 .. 4e-7 here); 1e-6 leaves two to four times that, and a dropped part product (2^-8 of
a part, 2^-16 of the value) would show as 1e-5."""

import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

LOG2E = 1.4426950408889634


@pytest.fixture(autouse=True)
def _fp32():
    from boltz_mlx_amd import kernels as K

    before = K.PRECISION
    K.set_precision("fp32")
    yield
    K.set_precision(before)


def _rel(a, ref):
    return ((a.double() - ref).norm() / ref.norm()).item()


def _core_ref(qkg, vt, tb, mask, inf, N, H, C):
    """The attention core in float64 from the projection's buffers; where the mask term is not zero it is added in 32
    bits, the model's definition of a row whose keys are all masked."""
    from boltz_mlx_amd import kernels as K

    b = tb.double()[torch.from_numpy(K.tri_bias_offsets(N, H)).cuda()]
    q, k, g = (qkg[H * x:H * (x + 1)].double().view(H, N, N, C) for x in range(3))
    out = torch.empty((N, N, H, C), dtype=torch.float64, device="cuda")
    for i in range(N):
        s = q[:, i] @ k[:, i].transpose(1, 2).contiguous()
        mb = inf * (mask[i] - 1) * LOG2E
        s = torch.where(mb == 0, s + b, ((s.float() + mb).float() + b.float()).double())
        p = torch.softmax(s / LOG2E, -1)
        out[i] = ((p @ vt[:, i, :, :N].double().transpose(1, 2).contiguous()) * torch.sigmoid(g[:, i])).transpose(0, 1)
    return out.view(N * N, H * C)


# query tiles of 32 (128 a workgroup), key stages of 32: their edges, one token, padding inside and past a stage, rows
# with every key masked, a strided (ending-node) mask, and an inf small enough that no stage may be skipped
@pytest.mark.parametrize("N,pad,holes,trans,inf", [
    (1, 0, False, False, 1e9), (31, 0, False, False, 1e9), (32, 1, False, True, 1e9), (33, 0, True, False, 1e9),
    (64, 33, False, False, 1e9), (97, 5, False, False, 5e5), (129, 6, True, True, 1e9), (130, 64, True, False, 1e4)])
def test_triattn_core_f32(N, pad, holes, trans, inf):
    from boltz_mlx_amd import kernels as K

    H, C = 4, 32
    g = torch.Generator(device="cuda").manual_seed(N)
    xn = torch.randn((N * N, H * C), generator=g, device="cuda")
    w = torch.randn((4 * H * C + H, H * C), generator=g, device="cuda") * (H * C) ** -0.5
    mask = torch.ones((N, N), device="cuda")
    mask[N - pad:] = 0
    mask[:, N - pad:] = 0
    if holes:
        mask *= (torch.rand((N, N), generator=g, device="cuda") > 0.3).float()
    bufs = K.triattn_proj(xn, w, trans, N, H, C)
    ref = _core_ref(*bufs, mask.T if trans else mask, inf, N, H, C)
    got = K.triattn_core(*bufs, mask, trans, inf, N, H, C)
    valu = K.triattn_core(*bufs, mask, trans, inf, N, H, C, impl=1)
    if inf < 1e6:
        # a row with every key masked by a small inf keeps logits rounded to 2^-10 (inf = 1e4) or 2^-4 (5e5): one that
        # rounds the other way moves its weight by that much, so only its finiteness is looked at
        live = ((mask.T if trans else mask) != 0).any(1)
        assert torch.isfinite(got).all()
        got, valu, ref = (t.view(N, N, H * C)[live] for t in (got, valu, ref))
    assert _rel(got, ref) <= 1e-6
    assert _rel(got, valu.double()) <= 2e-6


# tile edges of the two tile shapes (128 and 192), the k extent, one token
@pytest.mark.parametrize("N,k_len", [(1, 0), (29, 0), (64, 40), (128, 0), (129, 0), (192, 100), (193, 0), (333, 320)])
def test_trimul_contract_f32(N, k_len):
    from boltz_mlx_amd import kernels as K

    D, ld = 16, K.row_pitch(N)
    g = torch.Generator(device="cuda").manual_seed(N)
    ab = torch.zeros((2 * D, N, ld), device="cuda")
    ab[:, :, :k_len or N] = torch.randn((2 * D, N, k_len or N), generator=g, device="cuda")
    o = K.trimul_contract(ab, N, k_len)
    ref = ab[:D].double() @ ab[D:].double().transpose(1, 2).contiguous()
    assert _rel(o[:, :, :N], ref) <= 1e-6

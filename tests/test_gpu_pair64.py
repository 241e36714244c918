"""The fused pair kernels at 64 channels (the template stack) against plain torch in float64 on the same operands, at the
edges of their position tiles. Tolerance (relative, 2-norm): an fp16 output is rounded once (2^-11 at most, 2.8e-4 rms);
the tail's LayerNorm output and folded weight are fp16 operands too, three such roundings in all: 1e-3. fp32: 1e-6."""

import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu
CASES = [(dt, n) for dt in (torch.float32, torch.float16) for n in (1, 29, 64, 65, 130)]


def _rel(a, ref):
    return ((a.double() - ref).norm() / ref.norm()).item()


def _rand(g, dt, *shape):
    return torch.randn(shape, generator=g, device="cuda").to(dt)


class _Ln:
    def __init__(self, g, n):
        self.weight = 1 + 0.1 * torch.randn(n, generator=g, device="cuda")
        self.bias = 0.1 * torch.randn(n, generator=g, device="cuda")
        self.eps = 1e-5

    def __call__(self, x, eps=1e-5):
        return torch.nn.functional.layer_norm(x, x.shape[-1:], self.weight.double(), self.bias.double(), eps)


@pytest.mark.parametrize("dt,N", CASES)
def test_trimul64(dt, N):
    from boltz_mlx_amd import kernels as K

    g = torch.Generator(device="cuda").manual_seed(N)
    xn = _rand(g, dt, N * N, 64)
    w = _rand(g, torch.float32, 256, 64).mul(0.125).to(dt)
    mask = (torch.rand((N, N), generator=g, device="cuda") > 0.2).float()
    mask[0, 0] = 1.0
    tol = 1e-6 if dt == torch.float32 else 5e-4
    x2 = xn.double().view(N, N, 64)
    for incoming in (False, True):
        ab = K.trimul_proj64(xn, w, mask, 0.25, incoming, N)
        ref = (x2 @ w[:128].double().T) * torch.sigmoid(x2 @ w[128:].double().T) * mask[..., None].double() * 0.25
        ref = ref.permute(2, 1, 0) if incoming else ref.permute(2, 0, 1)
        assert _rel(ab[..., :N], ref) <= tol
        assert torch.all(ab[..., N:] == 0)
    o = _rand(g, dt, 64, N, K.row_pitch(N))
    no, nx = _Ln(g, 64), _Ln(g, 64)
    w_po, w_go = (_rand(g, torch.float32, 64, 64).mul(0.125).to(dt) for _ in range(2))
    z = torch.randn((N, N, 64), generator=g, device="cuda")
    up = (no(o[..., :N].double().permute(1, 2, 0), 1e-4) @ w_po.double().T) * torch.sigmoid(x2 @ w_go.double().T)
    for accumulate in (False, True):
        got = z.clone()
        nxt = K.trimul_tail64(o, no, 1e-4, w_po, xn, w_go, got, accumulate, nx, N)
        ref = up + z.double() if accumulate else up
        assert _rel(got, ref) <= (1e-6 if dt == torch.float32 else 1e-3)
        assert _rel(nxt.view(N, N, 64), nx(got.double())) <= tol


def test_half_layernorm_parameters():
    """LayerNorm parameters held in fp16 give what the same values in fp32 give, bit for bit."""
    from boltz_mlx_amd import kernels as K

    N = 37
    g = torch.Generator(device="cuda").manual_seed(N)

    class Half:
        eps = 1e-5

        def __init__(self, ln):
            self.weight, self.bias = ln.weight.half(), ln.bias.half()

    class Full(Half):
        def __init__(self, ln):
            super().__init__(ln)
            self.weight, self.bias = self.weight.float(), self.bias.float()

    no, nx = _Ln(g, 64), _Ln(g, 64)
    o, xn = _rand(g, torch.float16, 64, N, K.row_pitch(N)), _rand(g, torch.float16, N * N, 64)
    w_po, w_go = (_rand(g, torch.float32, 64, 64).mul(0.125).half() for _ in range(2))
    z = torch.randn((N, N, 64), generator=g, device="cuda")
    out = []
    for kind in (Full, Half):
        got = z.clone()
        out.append((got, K.trimul_tail64(o, kind(no), 1e-4, w_po, xn, w_go, got, True, kind(nx), N)))
    assert all(torch.equal(a, b) for a, b in zip(*out))
    z, w = torch.randn((N, N, 128), generator=g, device="cuda"), _rand(g, torch.float16, 16, 128)
    ln = _Ln(g, 128)
    assert torch.equal(K.pair_bias(z, Full(ln), w), K.pair_bias(z, Half(ln), w))


@pytest.mark.parametrize("dt,N", CASES)
def test_triattn64(dt, N):
    from boltz_mlx_amd import kernels as K

    H, C = 4, 32
    g = torch.Generator(device="cuda").manual_seed(N)
    xn = _rand(g, dt, N * N, 64)
    w = _rand(g, torch.float32, 4 * H * C + H, 64).mul(0.125).to(dt)
    idx = torch.from_numpy(K.tri_bias_offsets(N, H)).cuda()
    tol = 1e-6 if dt == torch.float32 else 5e-4
    for trans in (False, True):
        qkg, vt, tb = K.triattn_proj64(xn, w, trans, N, H, C)
        p = xn.double().view(N, N, 64) @ w.double().T
        p = p.transpose(0, 1) if trans else p
        q, k, v, gt = (p[..., 128 * i:128 * (i + 1)].reshape(N * N, H, C).transpose(0, 1) for i in range(4))
        assert _rel(qkg, torch.cat([q * (K.LOG2E / C ** 0.5), k, gt])) <= tol
        assert _rel(vt[..., :N], v.reshape(H, N, N, C).transpose(2, 3)) <= tol
        assert torch.all(vt[..., N:] == 0)
        assert _rel(tb[idx], p[..., 512:].permute(2, 0, 1) * K.LOG2E) <= tol
        x, wo, nx = _rand(g, dt, N * N, 128), _rand(g, torch.float32, 64, 128).mul(0.1).to(dt), _Ln(g, 64)
        z = torch.randn((N, N, 64), generator=g, device="cuda")
        y = (x.double() @ wo.double().T).view(N, N, 64)
        y = y.transpose(0, 1) if trans else y
        for accumulate in (False, True):
            got = z.clone()
            nxt = K.linear_resid_ln64(x, wo, trans, got, accumulate, nx, N)
            assert _rel(got, y + z.double() if accumulate else y) <= 1e-6  # exact fp16 products, fp32 sums
            assert _rel(nxt.view(N, N, 64), nx(got.double())) <= tol

"""The fp32 kernels on split operands where an operand has no parts (an infinity, or a finite value that rounds to a bf16
infinity) or a product ends close to the largest fp32 value: they give what fp32 products give.

Reference: the same sums in float64, taken back to fp32 (an overflow there is the infinity). Infinities and NaNs must be at
the same places with the same signs; finite values within 1e-6 of the sum of the terms' sizes (fp32 sums of up to 512
terms err by 1e-7 .. 3e-7 of it)."""

import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

INF, HUGE = float("inf"), 3.4e38  # HUGE rounds to a bf16 infinity


@pytest.fixture(autouse=True)
def _fp32():
    from boltz_mlx_amd import kernels as K

    before = K.PRECISION
    K.set_precision("fp32")
    yield
    K.set_precision(before)


def _dot(x, w):
    """(x w^T in fp32, the sum of its terms' sizes) for x [R, K], w [M, K]: every product formed, 0 inf among them."""
    out, size = [], []
    for r in x.double().split(64):
        t = r[:, None, :] * w.double()
        out.append(t.sum(-1).float())
        size.append(t.abs().sum(-1))
    return torch.cat(out), torch.cat(size)


def _same(got, ref, size=None):
    size = torch.zeros_like(ref) if size is None else size
    assert torch.equal(torch.isnan(got), torch.isnan(ref))
    inf = torch.isinf(ref)
    assert torch.equal(torch.isinf(got), inf) and torch.equal(got[inf], ref[inf])
    ok = torch.isfinite(ref)
    assert ((got.double() - ref.double())[ok].abs() <= 1e-6 * size[ok] + 1e-30).all()


def _rand(seed, *shape):
    return torch.randn(shape, generator=torch.Generator(device="cuda").manual_seed(seed), device="cuda")


def _spoil(x):
    """Infinities of both signs, a row with both, a NaN, finite values without parts and a row near the fp32 limit."""
    x[1 % len(x), 3] = INF
    x[2 % len(x), 40] = -INF
    x[5 % len(x), 7], x[5 % len(x), 9] = INF, -INF
    x[7 % len(x), 0] = float("nan")
    x[9 % len(x), 11] = HUGE
    x[11 % len(x), 30] = -HUGE
    return x


class _Ln:
    def __init__(self, seed, n):
        self.weight, self.bias, self.eps = 1 + 0.1 * _rand(seed, n), 0.1 * _rand(seed + 1, n), 1e-5

    def __call__(self, x):
        return torch.nn.functional.layer_norm(x.double(), x.shape[-1:], self.weight.double(), self.bias.double(), self.eps)


@pytest.mark.parametrize("R,k,M", [(13, 96, 20), (70, 384, 132), (40, 1536, 36)])
def test_linear_few_rows(R, k, M):
    from boltz_mlx_amd import kernels as K

    x, w = _spoil(_rand(R, R, k)), _rand(k, M, k) * k ** -0.5
    w[3, 17] = 0.0
    w[4, 3] = INF
    _same(K.linear(x, w), *_dot(x, w))
    y = _rand(3, R, M)
    ref, size = _dot(x, w)
    _same(K.linear(x, w, out=y.clone(), accumulate=True), y + ref, size + y.abs())


def test_linear_near_the_limit():
    """1.999 * 1.7e38 is finite; its rounded parts' product is not."""
    from boltz_mlx_amd import kernels as K

    x, w = torch.zeros(4, 64, device="cuda"), torch.zeros(8, 64, device="cuda")
    x[:, 5], w[:, 5] = 1.9999, 1.7e38
    assert torch.equal(K.linear(x, w), (x[:, 5:6].double() * w[:, 5].double()).float())


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("incoming", [False, True])
def test_trimul_proj(D, incoming):
    from boltz_mlx_amd import kernels as K

    N = 37
    xn, w = _spoil(_rand(N, N * N, D)), _rand(D, 4 * D, D) * D ** -0.5
    mask = torch.ones(N, N, device="cuda")
    proj = K.trimul_proj if D == 128 else K.trimul_proj64
    ab = proj(xn, w, mask, 1.0, incoming, N)
    (p, size), (gt, _) = _dot(xn, w[:2 * D]), _dot(xn, w[2 * D:])
    ref = (p * torch.sigmoid(gt)).view(N, N, 2 * D)
    size = size.view(N, N, 2 * D) * 4  # the gate's own error beside the product's
    turn = (lambda t: t.permute(2, 1, 0)) if incoming else (lambda t: t.permute(2, 0, 1))
    _same(ab[..., :N].contiguous(), turn(ref).contiguous(), turn(size).contiguous())


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("trans", [False, True])
def test_triattn_proj(D, trans):
    from boltz_mlx_amd import kernels as K

    N, H, C = 37, 4, 32
    xn, w = _spoil(_rand(N, N * N, D)), _rand(D, 4 * H * C + H, D) * D ** -0.5
    qkg, vt, tb = (K.triattn_proj if D == 128 else K.triattn_proj64)(xn, w, trans, N, H, C)
    y, size = _dot(xn, w)

    def turn(t, scale=1.0):
        t = (t * scale).view(N, N, -1)
        return t.transpose(0, 1) if trans else t

    def heads(t):
        return t.reshape(N * N, H, C).transpose(0, 1)

    for got, lo, scale in ((qkg[:H], 0, K.LOG2E / C ** 0.5), (qkg[H:2 * H], 128, 1.0), (qkg[2 * H:], 384, 1.0)):
        _same(got, heads(turn(y[:, lo:lo + 128], scale)), heads(turn(size[:, lo:lo + 128])))
    v, sv = (turn(t[:, 256:384]).reshape(N, N, H, C).permute(2, 0, 3, 1) for t in (y, size))
    _same(vt[..., :N].contiguous(), v.contiguous(), sv.contiguous())
    b, sb = (turn(t[:, 512:], s).permute(2, 0, 1) for t, s in ((y, K.LOG2E), (size, 2.0)))
    idx = torch.from_numpy(K.tri_bias_offsets(N, H)).cuda()
    _same(tb[idx], b.contiguous(), sb.contiguous())


@pytest.mark.parametrize("D", [64, 128])
def test_trimul_tail(D):
    from boltz_mlx_amd import kernels as K

    N = 37
    o = torch.zeros((D, N, K.row_pitch(N)), device="cuda")
    o[..., :N] = _rand(1, D, N, N)
    xn, ln = _spoil(_rand(2, N * N, D)), _Ln(3, D)
    w_po, w_go = _rand(4, D, D) * D ** -0.5, _rand(5, D, D) * D ** -0.5
    w_po[6, 8] = INF
    w_po[7, 8] = HUGE
    z = torch.zeros(N, N, D, device="cuda")
    (K.trimul_tail if D == 128 else K.trimul_tail64)(o, ln, ln.eps, w_po, xn, w_go, z, False, None, N)
    x = ln(o[..., :N].permute(1, 2, 0).reshape(N * N, D)).float()
    (p, size), (gt, _) = _dot(x, w_po), _dot(xn, w_go)
    ref = p * torch.sigmoid(gt)
    near = ref.abs().double() > 1e30  # the HUGE weight's column: LN_out near 0 may lose its sign beside fp32's rounding
    _same(z.view(N * N, D)[~near], ref[~near], 4 * size[~near])
    rel = (z.view(N * N, D)[near].double() / ref[near].double() - 1).abs()
    assert (rel[torch.isfinite(ref[near])] < 1e-2).all()


@pytest.mark.parametrize("DO", [64, 128])
@pytest.mark.parametrize("trans", [False, True])
def test_linear_resid(DO, trans):
    from boltz_mlx_amd import kernels as K

    N = 21
    x, w = _spoil(_rand(DO, N * N, 128)), _rand(1, DO, 128) * 128 ** -0.5
    w[2, 40] = 0.0
    z0 = _rand(2, N, N, DO)
    z = z0.clone()
    (K.linear_resid_ln if DO == 128 else K.linear_resid_ln64)(x, w, trans, z, True, None, N)
    y, size = (t.view(N, N, DO) for t in _dot(x, w))
    y, size = (t.transpose(0, 1) if trans else t for t in (y, size))
    _same(z, z0 + y, size + z0.abs())


def test_pair_bias():
    from boltz_mlx_amd import kernels as K

    N, H = 21, 16
    z, ln, w = _rand(1, N, N, 128), _Ln(2, 128), _rand(3, H, 128) * 128 ** -0.5
    z[3, 4] = float("nan")
    w[2, 8], w[5, 9], w[7, 60] = INF, -INF, 3.4e37
    got = K.pair_bias(z, ln, w)
    y, size = _dot(ln(z).float().view(N * N, 128), w)
    size[:, 7] += 3.4e37  # LN(z)'s own rounding where it is close to 0
    ref, size = (t.view(N, N, H).permute(2, 0, 1).contiguous() for t in (y, size))
    _same(got, ref, 4 * size)


@pytest.mark.parametrize("rows", [40, 5000, 20000, 65536 + 300])  # each form of the kernel
def test_transition(rows):
    from boltz_mlx_amd import kernels as K

    hidden, unit = 512, 77
    xn, w12, w3 = _rand(1, rows, 128), _rand(2, 2 * hidden, 128) * 128 ** -0.5, _rand(3, 128, hidden) * hidden ** -0.5
    w3[3, unit] = 0.0
    xn[:, 50] = 0.0
    w12[:, 50] = 0.0
    w12[unit, 50] = w12[hidden + unit, 50] = 1e15
    bad = torch.tensor([0, 3, 17, 30, rows // 2, rows - 1], device="cuda")
    xn[0, 5] = INF
    xn[3] *= 1e22  # hidden units overflow
    xn[17, 9] = HUGE
    xn[30, 50] = 1e15  # one hidden unit overflows: every output is its infinity, but where its weight is 0
    xn[rows // 2, 2] = float("nan")
    xn[rows - 1, 60] = -INF
    z = torch.zeros(rows, 1, 128, device="cuda")
    K.transition(xn, w12, w3, z, False)
    near = torch.unique(torch.cat([bad, (bad + 1).clamp(max=rows - 1), (bad - 1).clamp(min=0)]))  # their tiles too
    h, hs = _dot(xn[near], w12)
    h1, h2 = h[:, :hidden], h[:, hidden:]
    a = torch.nn.functional.silu(h1) * h2
    ref, size = _dot(a, w3)
    got = z.view(rows, 128)[near]
    finite = torch.isfinite(a).all(1) & (a.abs().amax(1) < 1e30)
    assert finite.any() and not finite.all()
    _same(got[finite], ref[finite], 10 * size[finite])
    # infinite hidden units: the same infinities and NaNs
    rest = ~torch.isfinite(a).all(1)
    assert torch.isinf(ref[rest]).sum() == 127
    _same(got[rest], ref[rest])
    assert torch.isfinite(z.view(rows, 128)).all(1).sum() >= rows - len(bad)


@pytest.mark.parametrize("N", [70, 190])  # both tile widths
def test_contraction(N):
    from boltz_mlx_amd import kernels as K

    D, ld = 8, K.row_pitch(N)
    ab = torch.zeros((2 * D, N, ld), device="cuda")
    ab[..., :N] = _rand(N, 2 * D, N, N)
    ab[0, 3, 5], ab[0, 9, 5] = INF, -INF
    ab[D, 7, 5] = 0.0
    ab[D + 1, 2, 60] = HUGE
    ab[2, 1, 1] = float("nan")
    ab[3, N - 1, N - 1], ab[D + 3, 4, N - 1] = INF, -INF
    o = K.trimul_contract(ab, N)
    for c in range(D):
        _same(o[c, :, :N].contiguous(), *_dot(ab[c, :, :N], ab[D + c, :, :N]))


@pytest.mark.parametrize("N", [37, 150])
def test_attention_core(N):
    """K and V with infinities: a key at a logit of -inf has no weight, one at +inf makes the query's row NaN, an infinite
    value reaches the queries that see it. Values near the fp32 limit stay finite (the weights of a row sum to 1)."""
    from boltz_mlx_amd import kernels as K

    H, C, D = 4, 32, 128
    xn = _rand(N, N * N, D)
    w = _rand(1, 4 * H * C + H, D) * D ** -0.5
    mask = torch.ones(N, N, device="cuda")
    mask[:, N - 3:] = 0
    qkg, vt, tb = K.triattn_proj(xn, w, False, N, H, C)
    idx = torch.from_numpy(K.tri_bias_offsets(N, H)).cuda()
    q4, k4, g4 = (t.view(H, N, N, C) for t in qkg.split(H))
    k4[0, 2, 9, 3] = INF      # head 0, row 2, key 9
    k4[1, 4, 0, 5] = -INF     # the first key
    k4[1, 5, 20, 7] = HUGE
    vt[2, 6, 3, 11] = INF     # head 2, row 6, channel 3, key 11
    vt[3, 7, :, :N] *= 1e37   # a whole row of large values
    vt[3, 8, 0, 2] = HUGE
    out = K.triattn_core(qkg, vt, tb, mask, False, 1e9, N, H, C).view(N, N, H, C)
    for h, i in ((0, 2), (1, 4), (1, 5), (2, 6), (3, 7), (3, 8), (0, 3)):
        q, k, g, v = q4[h, i].double(), k4[h, i].double(), g4[h, i].double(), vt[h, i, :, :N].double().T
        s = ((q[:, None] * k).sum(-1).float() + 1e9 * (mask[i] - 1) * K.LOG2E + tb[idx[h]]).double()
        p = torch.softmax(s * 0.6931471805599453, -1)
        t = p[..., None] * v
        gate = torch.sigmoid(g)
        got, ref = out[i, :, h], (t.sum(1) * gate).float()
        size = t.abs().sum(1) * 20  # the weights' own error: 1e-6 of a logit of some units
        if i == 5:  # logits of 1e38: all weight on one key
            assert torch.isfinite(got).all() and ((got - ref).abs() < 1e-4 * (1 + ref.abs())).float().mean() > 0.99
        else:
            _same(got, ref, size)

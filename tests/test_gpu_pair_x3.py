"""The fp32 row kernels of the pair track (split operands on the bf16 matrix cores) against float64, at the sizes where
their tiles of 16, 32, 64 and 256 rows end, and at the row counts where the transition changes its form.

Tolerance: fp32 sums over 128 to 512 terms err by 1e-7 .. 3e-7 of the result's norm; 1e-6 leaves a factor of three, and a
dropped part product (2^-16 of the value) would show as 1e-5."""

import pytest

from conftest import mask_key_extent

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

LOG2E = 1.4426950408889634
TOL = 1e-6


@pytest.fixture(autouse=True)
def _fp32():
    from boltz_mlx_amd import kernels as K

    before = K.PRECISION
    K.set_precision("fp32")
    yield
    K.set_precision(before)


def _rel(a, ref):
    return ((a.double() - ref).norm() / ref.norm()).item()


def _ln(x, ln):
    return torch.nn.functional.layer_norm(x, x.shape[-1:], ln.weight.double(), ln.bias.double(), ln.eps)


def _make(N, D, DO=None):
    from boltz_mlx_amd.layers.norm import LayerNorm

    g = torch.Generator(device="cuda").manual_seed(1000 * D + N)
    randn = lambda *s: torch.randn(s, generator=g, device="cuda")
    ln = LayerNorm(DO or D).cuda()
    with torch.no_grad():
        ln.weight.copy_(1 + 0.1 * randn(DO or D))
        ln.bias.copy_(0.1 * randn(DO or D))
    return randn, ln


SIZES = [1, 5, 16, 33, 64, 95]


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("N", SIZES)
def test_trimul_proj_and_tail(N, D):
    from boltz_mlx_amd import kernels as K

    randn, ln = _make(N, D)
    proj, tail = (K.trimul_proj64, K.trimul_tail64) if D == 64 else (K.trimul_proj, K.trimul_tail)
    xn, w = randn(N * N, D), randn(4 * D, D) * D ** -0.5
    mask = (torch.rand((N, N), device="cuda") > 0.2).float()
    p, gate = (xn.double() @ w.double().T).view(N, N, 4 * D).split(2 * D, -1)
    ref = (p * torch.sigmoid(gate) * mask.double()[..., None]).permute(2, 0, 1)
    for incoming in (False, True):
        ab = proj(xn, w, mask, 0.5, incoming, N)
        want = 0.5 * (ref.transpose(1, 2) if incoming else ref)
        assert _rel(ab[..., :N], want) < TOL if want.norm() > 0 else not ab[..., :N].any()
        assert not ab[..., N:].any()
    with torch.no_grad():
        norm_out = type(ln)(D).cuda()
        norm_out.weight.copy_(1 + 0.1 * randn(D))
        norm_out.bias.copy_(0.1 * randn(D))
        o = torch.full((D, N, K.row_pitch(N)), float("nan"), device="cuda")  # columns past N may hold anything
        o[..., :N] = randn(D, N, N) * 3 + 1
        w_po, w_go, z0 = randn(D, D) * D ** -0.5, randn(D, D) * D ** -0.5, randn(N, N, D)
        y = (_ln(o[..., :N].double().permute(1, 2, 0), norm_out) @ w_po.double().T) * torch.sigmoid(
            xn.double() @ w_go.double().T).view(N, N, D)
        for acc, nxt in ((False, None), (True, ln)):
            z = z0.clone() if acc else torch.full_like(z0, float("nan"))
            xo = tail(o, norm_out, norm_out.eps, w_po, xn, w_go, z, acc, nxt, N)
            want = y + z0.double() if acc else y
            assert _rel(z, want) < TOL
            if nxt is not None:
                assert _rel(xo.view(N, N, D), _ln(want, ln)) < TOL


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("N,H,C", [(1, 4, 32), (5, 8, 16), (16, 2, 64), (33, 4, 32), (64, 4, 32), (95, 4, 32)])
def test_triattn_proj(N, H, C, D):
    from boltz_mlx_amd import kernels as K

    randn, _ = _make(N, D)
    xn, w = randn(N * N, D), randn(4 * H * C + H, D) * D ** -0.5
    for trans in (False, True):
        qkg, vt, tb = (K.triattn_proj64 if D == 64 else K.triattn_proj)(xn, w, trans, N, H, C)
        y = (xn.double() @ w.double().T).view(N, N, -1)
        y = y.transpose(0, 1) if trans else y
        q, k, v, g, b = y.split([H * C] * 4 + [H], -1)
        heads = lambda t: t.reshape(N * N, H, C).transpose(0, 1)
        want = torch.cat([heads(q) * LOG2E / C ** 0.5, heads(k), heads(g)])
        assert _rel(qkg, want) < TOL
        assert _rel(vt[..., :N], v.reshape(N, N, H, C).permute(2, 0, 3, 1)) < TOL and not vt[..., N:].any()
        off = torch.from_numpy(K.tri_bias_offsets(N, H)).cuda()
        assert _rel(tb[off], b.permute(2, 0, 1) * LOG2E) < TOL


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("N", SIZES)
def test_linear_resid_ln(N, D):
    from boltz_mlx_amd import kernels as K

    randn, ln = _make(N, D)
    x, w, z0 = randn(N * N, 128), randn(D, 128) * 128 ** -0.5, randn(N, N, D)
    y = (x.double() @ w.double().T).view(N, N, D)
    with torch.no_grad():
        for trans, acc, nxt in ((False, True, ln), (True, True, ln), (True, False, None)):
            z = z0.clone() if acc else torch.full_like(z0, float("nan"))
            xo = (K.linear_resid_ln64 if D == 64 else K.linear_resid_ln)(x, w, trans, z, acc, nxt, N)
            want = (y.transpose(0, 1) if trans else y) + (z0.double() if acc else 0.0)
            assert _rel(z, want) < TOL
            if nxt is not None:
                assert _rel(xo.view(N, N, D), _ln(want, ln)) < TOL


# the fp16 projections with 4, 2 and 1 weight groups: both sides of the tile counts where each form ends (512 and 1,024
# tiles of 32 positions on 2,048 waves, 768 and 1,536 on 3,072), and the fp16 tail with and without empty tiles
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("N", [3, 100, 128, 129, 150, 170, 171, 203])
def test_f16_projections_and_tail(N, D):
    """Against float64 from the fp16 operands. The largest error of an fp16 store is 2^-11 of the value; 2^-9 of the largest
    value leaves room for the fp16 LayerNorm output and gates inside the tail."""
    from boltz_mlx_amd import kernels as K

    K.set_precision("f16")
    randn, ln = _make(N, D)
    half = lambda *s: (randn(*s) * (s[-1] ** -0.5 if s[0] != N * N else 1.0)).half()
    close = lambda a, ref: ((a.double() - ref).abs().max() <= ref.abs().max() * 2.0 ** -9).item()
    proj, attn, tail = (K.trimul_proj64, K.triattn_proj64, K.trimul_tail64) if D == 64 else (
        K.trimul_proj, K.triattn_proj, K.trimul_tail)
    xn, w, wq = half(N * N, D), half(4 * D, D), half(4 * 128 + 4, D)
    mask = (torch.rand((N, N), device="cuda") > 0.2).float()
    p, gate = (xn.double() @ w.double().T).view(N, N, 4 * D).split(2 * D, -1)
    ref = (p * torch.sigmoid(gate) * mask.double()[..., None]).permute(2, 0, 1)
    q, k, v, g, b = (xn.double() @ wq.double().T).view(N, N, -1).split([128] * 4 + [4], -1)
    off = torch.from_numpy(K.tri_bias_offsets(N, 4)).cuda()
    for flip in (False, True):
        turn = (lambda t: t.transpose(0, 1)) if flip else (lambda t: t)
        ab = proj(xn, w, mask, 1.0, flip, N)
        assert close(ab[..., :N], ref.transpose(1, 2) if flip else ref) and not ab[..., N:].any()
        qkg, vt, tb = attn(xn, wq, flip, N, 4, 32)
        heads = lambda t: turn(t).reshape(N * N, 4, 32).transpose(0, 1)
        assert close(qkg, torch.cat([heads(q) * LOG2E / 32 ** 0.5, heads(k), heads(g)]))
        assert close(vt[..., :N], turn(v).reshape(N, N, 4, 32).permute(2, 0, 3, 1)) and not vt[..., N:].any()
        assert close(tb[off], turn(b).permute(2, 0, 1) * LOG2E)
    with torch.no_grad():
        o = torch.zeros((D, N, K.row_pitch(N)), device="cuda", dtype=torch.float16)
        o[..., :N] = (randn(D, N, N) * 3).half()
        w_po, w_go, z = half(D, D), half(D, D), torch.full((N, N, D), float("nan"), device="cuda")
        y = (_ln(o[..., :N].double().permute(1, 2, 0), ln) @ w_po.double().T) * torch.sigmoid(
            xn.double() @ w_go.double().T).view(N, N, D)
        tail(o, ln, ln.eps, w_po, xn, w_go, z, False, None, N)
        assert close(z, y)


# masks whose last live column and row fall inside, at and past a 64-lane step; no live entry; one live entry
@pytest.mark.parametrize("N,rows,cols", [(1, 1, 1), (5, 0, 0), (64, 40, 64), (65, 65, 1), (130, 64, 65), (200, 129, 70)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_key_extent_device(N, rows, cols, dtype):
    """The extents against the host's count, and the contraction that reads one against the same contraction told it."""
    from boltz_mlx_amd import kernels as K

    mask = torch.zeros((N, N), device="cuda")
    if rows and cols:
        mask[rows - 1, 0] = mask[0, cols - 1] = 1.0
    ab = torch.randn((16, N, K.row_pitch(N)), device="cuda", dtype=dtype)
    with K.pair_mask_scope():
        for incoming, want in ((False, cols), (True, rows)):
            ext = K.key_extent_device(mask, N, incoming)
            assert int(ext.item()) == want == mask_key_extent(mask, incoming)
            masked = ab.clone()
            masked[:, :, want or N:] = 0
            got, ref = K.trimul_contract(masked, N, ext), K.trimul_contract(masked, N, want or N)
            assert torch.equal(got[..., :N], ref[..., :N])
    assert K.key_extent_device(mask, N, False) == 0


def test_mask_scope_around_a_capture():
    """Triangle multiplication and ending-node attention captured inside a scope that is older than the capture: replays
    follow the mask that they find, not the one of the warm-up."""
    from boltz_mlx_amd import kernels as K
    from boltz_mlx_amd.layers.triangular_attention.attention import TriangleAttentionEndingNode
    from boltz_mlx_amd.layers.triangular_mult import TriangleMultiplicationOutgoing

    N = 150
    torch.manual_seed(2)
    old = K.PRECISION
    K.set_precision("f16")
    try:
        with torch.no_grad(), torch.device("cuda"):
            mods = [TriangleMultiplicationOutgoing(128), TriangleAttentionEndingNode(128, 32, 4)]
            z = torch.randn(1, N, N, 128)
            mask = torch.zeros(1, N, N)
            mask[:, :40, :40] = 1
            run = lambda: [mod(z, mask) for mod in mods]  # noqa: E731
            with K.pair_mask_scope():
                run()
                graph = torch.cuda.CUDAGraph()
                torch.cuda.synchronize()
                with torch.cuda.graph(graph):
                    out = run()
            for live in (150, 90, 20, 150):
                mask.zero_()
                mask[:, :live, :live] = 1
                want = run()
                graph.replay()
                torch.cuda.synchronize()
                assert all(torch.equal(a, b) for a, b in zip(out, want)), live
    finally:
        K.set_precision(old)


# one row, the end of a 16-row tile, more tiles than resident waves (65,536 rows and more), few and all 16 heads
@pytest.mark.parametrize("N,H", [(1, 16), (3, 4), (16, 8), (37, 16), (270, 16), (333, 1)])
def test_pair_bias(N, H):
    from boltz_mlx_amd import kernels as K

    randn, ln = _make(N, 128)
    z, w = randn(N, N, 128) * 2 + 1, randn(H, 128) * 128 ** -0.5
    with torch.no_grad():
        ref = (_ln(z.double(), ln) @ w.double().T).permute(2, 0, 1)
        assert _rel(K.pair_bias(z, ln, w), ref) < TOL


# rows: ends of the 16-, 32-, 128- and 256-row tiles, both sides of the row counts where the form changes, and whole
# rounds of 65,536 rows with a remainder in each form
@pytest.mark.parametrize("rows,hidden", [(1, 64), (15, 512), (17, 320), (4096, 512), (4097, 64), (16384, 64),
                                         (16385, 512), (32768, 64), (32769, 512), (65536, 64), (65537, 192),
                                         (70001, 64), (90000, 128), (100000, 64)])
def test_transition(rows, hidden):
    from boltz_mlx_amd import kernels as K

    randn, ln = _make(rows, 128)
    xn, z0 = randn(rows, 128), randn(rows, 1, 128)
    w12, w3 = randn(2 * hidden, 128) * 128 ** -0.5, randn(128, hidden) * hidden ** -0.5
    h1, h2 = (xn.double() @ w12.double().T).split(hidden, -1)
    y = ((torch.nn.functional.silu(h1) * h2) @ w3.double().T).view(rows, 1, 128)
    with torch.no_grad():
        for acc, nxt in ((True, ln), (False, None)):
            z = z0.clone() if acc else torch.full_like(z0, float("nan"))
            xo = K.transition(xn, w12, w3, z, acc, nxt)
            want = y + z0.double() if acc else y
            assert _rel(z, want) < TOL
            if nxt is not None:
                assert _rel(xo.view(rows, 1, 128), _ln(want, ln)) < TOL


# fp32 Linear over few rows: one row, ends of its 16- and 32-row tiles, a column count that ends inside a tile, fewer steps of
# 32 k than waves and more, and both sides of its largest grid (768 tiles of 16 columns x 32 rows)
@pytest.mark.parametrize("R,k,M", [(1, 384, 1536), (16, 32, 4), (17, 64, 20), (33, 288, 36), (128, 1536, 384),
                                   (128, 384, 3072), (129, 384, 3072), (1024, 384, 384), (1025, 384, 384)])
def test_linear_few_rows(R, k, M):
    from boltz_mlx_amd import kernels as K

    g = torch.Generator(device="cuda").manual_seed(R + k + M)
    randn = lambda *s: torch.randn(s, generator=g, device="cuda")
    x, w, b, y0 = randn(R, k), randn(M, k) * k ** -0.5, randn(M), randn(R, M)
    ref = x.double() @ w.double().T + b.double()
    assert _rel(K.linear(x, w, bias=b), ref) < TOL
    assert _rel(K.linear(x, w, bias=b, out_dtype=torch.float16), ref) < 2.0 ** -11
    assert _rel(K.linear(x, w, bias=b, out=y0.clone(), accumulate=True), y0.double() + ref) < TOL
    gate = randn((R + 2) // 3, M)
    sig = torch.sigmoid(gate.double())[torch.arange(R, device="cuda") % gate.shape[0]]
    assert _rel(K.linear_gated(x, w, gate, y0.clone(), bias=b), y0.double() + sig * ref) < TOL
    assert _rel(K.linear_residual(x, w, y0, torch.empty_like(y0), bias=b), y0.double() + ref) < TOL

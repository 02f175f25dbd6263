"""Few-token products on row-major weights (expert_skinny.hip) at the edges of
their tiles: rows off 16 and 64, widths whose last chunk overlaps the one
before, one to eight chunks, token counts around the 16- and 32-token tiles.

Tolerance: activations carry 22 significant bits (2^-22 of a chunk's largest
value per piece), sums are f32 over at most 4096 terms: both leave errors
below 1e-6 of the largest output; TOL (5e-6) is the bar of every product."""
import numpy as np
import pytest

from gpu_util import TOL

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from moe_amd.layer import Context

    return Context(0)


def stored(dt, rows, cols, seed=0):
    """Quantised bytes of N(0, 0.02) rows and their float64 values."""
    import ctypes as C

    from moe_amd import _lib as L
    from moe_amd.layer import row_bytes

    w = (np.random.default_rng(seed).standard_normal((rows, cols)) * 0.02).astype(np.float32)
    raw = np.zeros(rows * row_bytes(dt, cols), dtype=np.uint8)
    p = lambda a: a.ctypes.data_as(C.c_void_p)  # noqa: E731
    L.check(L.lib().moe_quantize_rows(dt, p(w), rows, cols, p(raw)))
    back = np.empty_like(w)
    L.check(L.lib().moe_dequant_rows(dt, p(raw), rows, cols, p(back)))
    return raw, back.astype(np.float64)


def linear(ctx, dt, rows, cols, raw):
    from moe_amd.layer import View
    from moe_amd.model import Linear

    region = ctx.upload(raw)
    lin = Linear(ctx, View(dt, rows, cols, region.id, 0))
    lin.region = region
    return lin


def path(lin, t):
    from moe_amd import _lib as L

    return L.lib().moe_debug_linear_path(lin.handle, t)


def apply(lin, x, residual=None):
    import torch

    from moe_amd.layer import MoeLayer

    xd = torch.from_numpy(np.ascontiguousarray(x)).cuda()
    y = torch.full((x.shape[0], lin.n), float("nan"), device="cuda")
    r = torch.from_numpy(residual.copy()).cuda() if residual is not None else None
    lin(xd, y, MoeLayer.new_workspace(lin.workspace_size(x.shape[0])), residual=r)
    torch.cuda.synchronize()
    return y.cpu().numpy(), None if r is None else r.cpu().numpy()


@pytest.mark.parametrize("dt", [2, 6, 8])
@pytest.mark.parametrize("rows,cols", [(16, 256), (17, 320), (64, 512), (200, 704), (129, 768), (576, 1408),
                                       (2050, 2048), (100, 2112), (96, 4096), (5000, 2048), (4112, 1088)])
def test_linear_edges(ctx, dt, rows, cols):
    raw, w = stored(dt, rows, cols)
    lin = linear(ctx, dt, rows, cols, raw)
    g = np.random.default_rng(1)
    for t in (1, 2, 7, 16, 17, 31, 33, 64):
        # A token or two on few rows wider than 2048 stay on the GEMV.
        assert path(lin, t) == (GEMV if t <= 2 and cols > 2048 else STREAM), t
        x = g.standard_normal((t, cols)).astype(np.float32)
        x *= (10.0 ** g.integers(-3, 4, size=(t, 1))).astype(np.float32)
        res = g.standard_normal((t, rows)).astype(np.float32)
        y, r = apply(lin, x, res)
        want = x.astype(np.float64) @ w.T
        err = (np.abs(y - want).max(1) / np.abs(want).max(1)).max()
        assert err < TOL, (t, err)
        assert np.array_equal(r, res + y), t


@pytest.mark.parametrize("dt", [2, 6, 8])
@pytest.mark.parametrize("cols,bar", [(512, 8.8e-8), (2048, 1.09e-7), (4096, 1.15e-7)])
def test_linear_error_against_64_bits(ctx, dt, cols, bar):
    """No further from 64 bits (2-norm) than the MFMA kernel these calls ran
    on before: the bar is what that one measures (8.84e-8 to 9.0e-8, 1.10e-7 to
    1.11e-7, 1.155e-7 to 1.17e-7 over formats and token counts)."""
    rows = 1 << 21 >> (cols.bit_length() - 1)
    raw, w = stored(dt, rows, cols)
    lin = linear(ctx, dt, rows, cols, raw)
    for t in (4, 9, 32):
        assert path(lin, t) == STREAM
        x = np.random.default_rng(t).standard_normal((t, cols)).astype(np.float32)
        y, _ = apply(lin, x)
        want = x.astype(np.float64) @ w.T
        err = np.linalg.norm(y - want) / np.linalg.norm(want)
        assert err < bar, (t, err)


@pytest.mark.parametrize("dt", [2, 8])
def test_linear_non_finite_tokens(ctx, dt):
    """A token that holds an infinity or a NaN gives what f32 products give
    (infinities of the products' signs, NaN where they cancel or multiply a
    zero), and leaves the other tokens alone."""
    rows, cols = 64, 1408
    raw, w = stored(dt, rows, cols)
    lin = linear(ctx, dt, rows, cols, raw)
    x = np.random.default_rng(2).standard_normal((9, cols)).astype(np.float32)
    assert path(lin, 9) == STREAM
    clean, _ = apply(lin, x)
    x[1, 5], x[4, 1400], x[6, 700] = np.inf, -np.inf, np.nan
    x[7] = 0.0
    y, _ = apply(lin, x)
    for t in (0, 2, 3, 5, 8):
        assert np.array_equal(y[t], clean[t])
    assert (y[7] == 0).all()
    for t, c, v in ((1, 5, np.inf), (4, 1400, -np.inf)):
        q = w[:, c]
        assert np.array_equal(y[t][q > 0], np.full((q > 0).sum(), v, np.float32))
        assert np.array_equal(y[t][q < 0], np.full((q < 0).sum(), -v, np.float32))
        assert np.isnan(y[t][q == 0]).all()
    assert np.isnan(y[6]).all()


@pytest.mark.parametrize("dt", [2, 6, 8])
def test_linear_infinity_beside_large_values(ctx, dt):
    """Finite values too large for f16 in the chunk that holds an infinity
    (or in the last chunk, which re-reads units of the one before, when the
    infinity lies there) stay finite: the sums are the infinity's, as f32
    products give them, and never NaN from a made-up opposite one."""
    rows, cols = 64, 1408
    raw, w = stored(dt, rows, cols)
    lin = linear(ctx, dt, rows, cols, raw)
    g = np.random.default_rng(3)
    cases = [(c, big, v) for c, big in ((5, 9), (1200, 1300), (1400, 1290)) for v in (1e5, -1e5, 3e30)]
    x = g.standard_normal((len(cases), cols)).astype(np.float32)
    for t, (c, big, v) in enumerate(cases):
        x[t, c], x[t, big:big + 3] = np.inf, v
    for n in (1, 7, len(cases)):
        assert path(lin, n) == STREAM
        y, _ = apply(lin, x[:n])
        for t in range(n):
            q = w[:, cases[t][0]]
            want = np.where(q > 0, np.inf, np.where(q < 0, -np.inf, np.nan)).astype(np.float32)
            assert np.array_equal(y[t], want, equal_nan=True), cases[t]


@pytest.mark.parametrize("dt", [2, 6, 8])
@pytest.mark.parametrize("n", [512, 2048, 4096])
def test_linear_in_place(ctx, dt, n):
    """x += W x with the residual in x's own memory (whole, or a shifted
    range of it) gives what a separate residual gives, bit for bit; y in x's
    memory from 9 tokens on gives the product of the old x."""
    import torch

    from moe_amd.layer import MoeLayer

    raw, w = stored(dt, n, n)
    lin = linear(ctx, dt, n, n, raw)
    for t in (1, 2, 8, 17, 32, 64, 96):
        x = np.random.default_rng(t).standard_normal((t, n)).astype(np.float32)
        y, r = apply(lin, x, x)
        ws = MoeLayer.new_workspace(lin.workspace_size(t))
        for shift in (0, 64):  # floats between x and the residual
            mem = torch.zeros(t * n + shift, device="cuda")
            xd, res = mem[:t * n].view(t, n), mem[shift:].view(t, n)
            xd.copy_(torch.from_numpy(x))
            before = res.clone()
            yd = torch.full((t, n), float("nan"), device="cuda")
            lin(xd, yd, ws, residual=res)
            assert np.array_equal(yd.cpu().numpy(), y), (t, shift)
            assert torch.equal(res, before + yd), (t, shift)
            assert shift or np.array_equal(res.cpu().numpy(), r), t
        if t > 8:
            xd = torch.from_numpy(x).cuda()
            lin(xd, xd, ws)
            want = x.astype(np.float64) @ w.T
            assert np.abs(xd.cpu().numpy() - want).max() < TOL * np.abs(want).max(), t


def test_linear_past_4_gib_needs_no_workspace(ctx):
    """Matrices of 4 GiB and more, which no MFMA kernel takes, run without a
    workspace at any token count; rows at both ends and beside the 4 GiB line
    come out right."""
    import ctypes as C

    import torch

    from moe_amd import _lib as L

    cols, rows = 4096, 987200  # 4352 bytes a row: the last 304 lie past 2^32
    pick = np.r_[0:16, (1 << 32) // 4352 - 8:(1 << 32) // 4352 + 8, rows - 16:rows]
    part, w = stored(8, len(pick), cols)
    raw = np.zeros(rows * 4352, dtype=np.uint8)
    raw.reshape(rows, 4352)[pick] = part.reshape(len(pick), 4352)
    lin = linear(ctx, 8, rows, cols, raw)
    x = np.random.default_rng(9).standard_normal((9, cols)).astype(np.float32)
    xd, y = torch.from_numpy(x).cuda(), torch.full((9, rows), float("nan"), device="cuda")
    for t in (1, 8, 9):
        y.fill_(float("nan"))
        L.check(L.lib().moe_linear_forward(lin.handle, C.c_void_p(xd.data_ptr()), t, C.c_void_p(y.data_ptr()), None,
                                           None, 0, C.c_void_p(torch.cuda.current_stream().cuda_stream)))
        got, want = y[:t].cpu().numpy(), x[:t].astype(np.float64) @ w.T
        assert np.abs(got[:, pick] - want).max() < TOL * np.abs(want).max()
        rest = np.ones(rows, bool)
        rest[pick] = False
        assert (got[:, rest] == 0).all()
    lin.close()


# What moe_debug_layer_path and moe_debug_linear_path call the kernels.
GEMV, MFMA, FEW, TILED, STREAM = 2, 3, 5, 6, 7

LAYERS = [
    # 16- and 32-token tiles (t k / E above 14), shared experts whose down rows split K, rows off 16
    ("v2_lite", dict(n_experts=8, top_k=3, inter=704, shared_inter=2816), (6, 33, 64)),
    ("v2_lite", dict(n_experts=4, top_k=2, hidden=768, inter=320, shared_inter=1344), (8, 40)),
    ("qwen2_moe", dict(n_experts=6, inter=1408, shared_inter=5632), (5, 36)),
    ("qwen3", dict(n_experts=16, top_k=8, inter=768), (2, 3, 31, 48)),
    # eight-unit chunks on both sides, K parts, 4- and 5-bit codes
    ("mixtral", dict(inter=4480), (6, 16, 60)),
    ("mixtral", dict(inter=14336, n_experts=2, expert_dt=6), (2, 17, 16)),
    ("qwen3", dict(n_experts=16, inter=832, expert_dt=2), (3, 32)),
    ("tiny_mixtral", dict(hidden=320, inter=256), (5, 16, 100)),
    # 5-bit codes in four-unit chunks, both tiles; 8-bit ones in eight-unit chunks
    ("v2_lite", dict(n_experts=8, top_k=3, inter=704, shared_inter=2816, expert_dt=6, shared_dt=6), (6, 20, 40)),
    ("qwen3", dict(n_experts=8, inter=768, expert_dt=6), (3, 15, 16)),
    ("qwen3", dict(n_experts=4, top_k=2, inter=2304, expert_dt=8), (9, 40)),
    # a shared expert in another format
    ("v2_lite", dict(n_experts=4, top_k=2, inter=320, shared_inter=1344, expert_dt=2, shared_dt=8), (5, 17, 31)),
    ("qwen2_moe", dict(n_experts=6, inter=1408, shared_inter=2816, expert_dt=8, shared_dt=6), (7, 22, 36)),
    ("qwen2_moe", dict(n_experts=6, inter=704, shared_inter=4480, expert_dt=6, shared_dt=2), (4, 23)),
    # a dense MLP
    ("mixtral", dict(n_experts=1, top_k=1, inter=2112, expert_dt=2), (2, 16)),
    ("qwen3", dict(n_experts=1, top_k=1, inter=768, expert_dt=8), (16, 24)),
]
# The token counts above that lie outside the rule.
OUTSIDE = {("mixtral", 17): MFMA, ("tiny_mixtral", 5): FEW, ("tiny_mixtral", 100): MFMA}


@pytest.mark.parametrize("name,scale,ts", LAYERS, ids=str)
@pytest.mark.parametrize("tiled", [False, True])
def test_layer_few_tokens(ctx, oracle, name, scale, ts, tiled):
    """Layers at token counts the few-token kernels serve, against the
    oracle, on the kernels they are meant to test; a tiled layer (which takes
    the tiled kernel for 4- and 5-bit codes) agrees too."""
    from gpu_util import assert_routing_equal, rel_err, run_gpu
    from moe_amd import _lib as L
    from moe_amd import synth

    host = synth.build_host_layer(synth.scaled(synth.SHAPES[name], **scale), 3)
    layer, ref = synth.make_layer(ctx, host), oracle.from_host_layer(host)
    if tiled:
        layer.set_tiled(True)
    for t in ts:
        path = L.lib().moe_debug_layer_path(layer.handle, t)
        if tiled and host.shape.expert_dt != 8:
            assert path == TILED, (t, path)
        elif not tiled:
            assert path == OUTSIDE.get((name, t), STREAM), (t, path)
        x = synth.activations(5, t, host.shape.hidden)
        out, sel, w, _, _ = ref.forward(x)
        res = synth.normal(7, t, x.size).reshape(x.shape)
        got = run_gpu(layer, x, residual=res)
        assert_routing_equal(got, sel, w, f"{name} T={t}")
        err = rel_err(got["out"], out)
        assert err < TOL, (t, err)
        assert np.array_equal(got["residual"], res + got["out"])
    layer.close()

"""moe_attention (src/model.rs:790-831) against float64: one prompt, many
sequences, mixed groups of rows, grouped and single key/value heads, windows,
head widths on and off the kernels' tiles, values no row may see.

Tolerance: a score is a sum of qd f32 products of N(0, 1) values times
qd^-0.5; its rounding error is a random walk of qd steps of 2^-24 times
partial sums of up to qd^0.5, so about qd 2^-24 qd^-0.5 = qd^0.5 2^-24, below
1e-6 up to qd = 256.  A weight carries its score's error as a relative one,
and an output averages values of order 1 under such weights: 5e-6 of the
largest output (the bar of the other kernels) leaves a factor of five."""
import ctypes as C
import math

import numpy as np
import pytest

from gpu_util import TOL

pytestmark = pytest.mark.gpu


def attend64(q, kc, vc, seq, pos, heads, n_kv, qd, vd, scale, window):
    out = np.zeros((len(seq), heads, vd))
    rep = heads // n_kv
    for r, (s, p) in enumerate(zip(seq, pos)):
        lo = max(0, p + 1 - window) if window else 0
        for h in range(heads):
            kvh = h // rep if rep > 1 else min(h, n_kv - 1)
            k = kc[s, lo:p + 1, kvh * qd:(kvh + 1) * qd].astype(np.float64)
            v = vc[s, lo:p + 1, kvh * vd:(kvh + 1) * vd].astype(np.float64)
            w = k @ q[r, h * qd:(h + 1) * qd].astype(np.float64) * scale
            w = np.exp(w - w.max())
            out[r, h] = (w / w.sum()) @ v
    return out.reshape(len(seq), heads * vd)


def run(q, kc, vc, seq, pos, heads, n_kv, qd, vd, scale, window):
    import torch

    from moe_amd import _lib as L

    d = [torch.from_numpy(np.ascontiguousarray(v)).cuda() for v in (q, kc, vc)]
    ids = [torch.tensor(v, dtype=torch.int32, device="cuda") for v in (seq, pos)]
    out = torch.full((len(seq), heads * vd), float("nan"), device="cuda")
    p = lambda t: C.c_void_p(t.data_ptr())  # noqa: E731
    rc = L.lib().moe_attention(p(d[0]), q.shape[1], len(seq), heads, n_kv, qd, vd, scale, p(d[1]), p(d[2]),
                               kc.shape[1], p(ids[0]), p(ids[1]), max(pos), window, p(out), out.shape[1],
                               C.c_void_p(torch.cuda.current_stream().cuda_stream))
    L.check(rc, "moe_attention")
    torch.cuda.synchronize()
    return out.cpu().numpy()


def inputs(seqs, ctx, rows, heads, n_kv, qd, vd, seed=0):
    g = np.random.default_rng(seed)
    f = lambda *s: g.standard_normal(s).astype(np.float32)  # noqa: E731
    return f(rows, heads * qd), f(seqs, ctx, n_kv * qd), f(seqs, ctx, n_kv * vd)


ROWS = {
    # one row per sequence, lengths around the 16-position tiles
    "decode": [(s, p) for s, p in enumerate([0, 15, 16, 17, 130, 63, 64, 1, 299])],
    "one_row": [(0, 200)],
    "prompt": [(0, p) for p in range(37)],
    "chunk": [(0, 100 + p) for p in range(70)],
    # two prompts, single rows and a run of the first sequence again, in one call
    "mixed": [(0, p) for p in range(9)] + [(1, 40 + p) for p in range(21)] + [(2, 5), (3, 77)] +
             [(0, 9 + p) for p in range(13)],
    # positions in no order
    "shuffled": [(0, p) for p in (90, 3, 50, 51, 7, 0, 128)],
}
HEADS = [(8, 2, 64, 64), (16, 16, 192, 128), (32, 8, 128, 128), (6, 2, 80, 80), (4, 4, 40, 24), (40, 1, 64, 32),
         (4, 2, 256, 256), (3, 3, 20, 200), (2, 2, 30, 30)]


@pytest.mark.parametrize("rows", list(ROWS))
@pytest.mark.parametrize("shape", HEADS, ids=str)
def test_attention_shapes(rows, shape):
    heads, n_kv, qd, vd = shape
    seq, pos = zip(*ROWS[rows])
    q, kc, vc = inputs(max(seq) + 1, 300, len(seq), heads, n_kv, qd, vd)
    for window in (0, 21):
        args = (seq, pos, heads, n_kv, qd, vd, 1.0 / math.sqrt(qd), window)
        got, want = run(q, kc, vc, *args), attend64(q, kc, vc, *args)
        err = np.abs(got - want).max() / np.abs(want).max()
        assert err < TOL, (window, err)


@pytest.mark.parametrize("rows,shape", [(1000, (16, 16, 64, 64)), (700, (32, 8, 128, 128)), (520, (32, 32, 192, 128))],
                         ids=str)
def test_attention_wide_groups(rows, shape):
    """Enough rows for the 32-column tiles: a prompt with a second one and
    single rows at its end, every kind of group in one call."""
    heads, n_kv, qd, vd = shape
    cut = rows - 60
    seq = [0] * cut + [1] * 40 + list(range(20))
    pos = list(range(cut)) + list(range(40)) + [cut + i for i in range(20)]
    q, kc, vc = inputs(20, cut + 30, rows, heads, n_kv, qd, vd)
    pick = np.r_[0:20, cut - 9:cut + 60]
    for window in (0, 100):
        args = (heads, n_kv, qd, vd, 1.0 / math.sqrt(qd), window)
        got = run(q, kc, vc, seq, pos, *args)[pick]
        want = attend64(q[pick], kc, vc, [seq[i] for i in pick], [pos[i] for i in pick], *args)
        assert np.abs(got - want).max() < TOL * np.abs(want).max()


@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
@pytest.mark.parametrize("shape", [(8, 2, 64, 64), (16, 16, 192, 128), (4, 4, 40, 24)], ids=str)
def test_attention_ignores_unseen_values(shape, bad):
    """Keys and values a row may not see (later positions, positions before
    the window, the cache past the end) leave it unchanged whatever they hold."""
    heads, n_kv, qd, vd = shape
    seq, pos = [0] * 30, list(range(50, 80))
    q, kc, vc = inputs(1, 100, 30, heads, n_kv, qd, vd)
    args = (seq, pos, heads, n_kv, qd, vd, 1.0 / math.sqrt(qd), 25)
    want = attend64(q, kc, vc, *args)
    kb, vb = kc.copy(), vc.copy()
    for p in (0, 10, 25, 26, 65, 66, 79, 80, 99):
        kb[0, p], vb[0, p] = bad, bad
    got = run(q, kb, vb, *args)
    sees = np.array([any(max(0, p - 24) <= b <= p for b in (26, 65, 66, 79)) for p in pos])
    assert (~sees).sum() >= 3
    assert np.abs(got[~sees] - want[~sees]).max() < TOL * np.abs(want).max()
    assert not np.isfinite(got[sees]).all(axis=1).any()


def test_attention_large_scores():
    """Scores hundreds apart: the running maximum moves at every step, the
    far weights vanish, nothing overflows."""
    heads, n_kv, qd, vd = 8, 2, 64, 64
    q, kc, vc = inputs(2, 200, 40, heads, n_kv, qd, vd)
    kc *= np.linspace(-40, 40, 200, dtype=np.float32)[None, :, None]
    seq, pos = [0] * 39 + [1], list(range(160, 199)) + [199]
    args = (seq, pos, heads, n_kv, qd, vd, 1.0, 0)
    got, want = run(q, kc, vc, *args), attend64(q, kc, vc, *args)
    assert np.isfinite(got).all()
    # A score of up to ~1000 carries an error of 1000 2^-24 = 6e-5, which is
    # its weight's relative error.
    assert np.abs(got - want).max() < 4 * 6e-5 * np.abs(want).max()


@pytest.mark.parametrize("shape", [(8, 2, 64, 64), (16, 16, 192, 128), (4, 4, 40, 24), (4, 2, 256, 256)], ids=str)
def test_attention_equal_weights_are_divided(shape):
    """Equal keys and whole values: weights and sums are exact, so over up to
    one tile of positions the mean comes out correctly rounded (a product with
    the rounded reciprocal would not)."""
    heads, n_kv, qd, vd = shape
    q, kc, vc = inputs(1, 16, 16, heads, n_kv, qd, vd)
    kc[:] = kc[:, :1]
    vc = np.round(vc * 100)
    args = ([0] * 16, list(range(16)), heads, n_kv, qd, vd, 1.0 / math.sqrt(qd), 0)
    got = run(q, kc, vc, *args).reshape(16, heads, vd)
    total = np.cumsum(vc[0].reshape(16, n_kv, vd), 0, dtype=np.float32)
    want = (total / np.arange(1, 17, dtype=np.float32)[:, None, None]).repeat(heads // n_kv, 1)
    assert np.array_equal(got, want)


@pytest.mark.parametrize("shape", [(8, 2, 64, 64), (16, 16, 192, 128), (32, 8, 128, 128), (4, 2, 256, 256)], ids=str)
def test_attention_values_near_the_largest(shape):
    """A mean of values near f32's largest is one of their range: sums of
    weights that are not yet divided must not leave it."""
    heads, n_kv, qd, vd = shape
    rows = ROWS["mixed"] + [(1, p) for p in range(200, 299)]
    seq, pos = zip(*rows)
    q, kc, vc = inputs(4, 300, len(rows), heads, n_kv, qd, vd)
    vc = (3e38 * np.tanh(4 * vc + 2)).astype(np.float32)
    for window in (0, 40):
        args = (seq, pos, heads, n_kv, qd, vd, 3.0 / math.sqrt(qd), window)
        got, want = run(q, kc, vc, *args), attend64(q, kc, vc, *args)
        # Scores three times those of test_attention_shapes: their errors too.
        assert np.abs(got - want).max() < 3 * TOL * np.abs(want).max()

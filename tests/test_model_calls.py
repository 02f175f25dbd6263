"""The Python side of a model call on the CPU: which rows head reads and which
calls are refused, with the kernels replaced by the reads they make."""
import pytest
import torch

from moe_amd.model import Model, Spec


class Reads(Model):
    """Model's calls without a checkpoint: the norm hands on the rows it reads."""

    def __init__(self, hidden=8):
        self.spec = Spec(hidden=hidden, layers=0, heads=1, kv_heads=1, head_dim=hidden, vocab=4)
        self.device = torch.device("cpu")
        self.out_norm = torch.ones(hidden)
        self.trunks = 0

    def _rmsnorm(self, x, w, out, stream, rows=None, n=None, xs=None, os_=None):
        out.copy_(torch.as_strided(x, (rows, n), (xs, 1)))

    def _workspace(self, t):
        return None

    def lm_head(self, nx, logits, ws, stream=None):
        return nx

    def trunk(self, tokens, st, seqs=None, stream=None):
        self.trunks += 1
        return torch.zeros(sum(map(len, tokens)), self.spec.hidden), None


@pytest.mark.parametrize("rows", [[0], [5], [0, 1, 2, 3, 4, 5], [1, 3, 5], [2, 5], [5, 2], [1, 1], [0, 1, 3]], ids=str)
def test_head_reads_its_rows(rows):
    m = Reads()
    wide = torch.randn(6, 20)
    for x in (wide[:, :8].contiguous(), wide[:, 4:12], wide[:, ::2][:, :8], torch.randn(8, 6).T):
        assert torch.equal(m.head(x, rows), x[rows])


@pytest.mark.parametrize("rows", [[], [-1], [6], [-1, 0], [-1, 1], [0, 3, 6], [5, 6], [7, 1], [1, 1, 9]], ids=str)
def test_head_refuses_rows_outside(rows):
    with pytest.raises(ValueError):
        Reads().head(torch.randn(6, 8), rows)


@pytest.mark.parametrize("tokens", [[[], [3]], [[3], []], [[]]], ids=str)
def test_forward_refuses_a_sequence_without_tokens(tokens):
    """Before anything runs: the state does not advance."""
    m = Reads()
    with pytest.raises(ValueError):
        m.forward(tokens, None)
    assert m.trunks == 0


class Layer:
    """An FFN that records its calls."""

    def __init__(self):
        self.calls = []

    def workspace_size(self, t):
        return 256

    def feed_forward(self, x, out, residual=None, stream=None, workspace=None):
        self.calls.append((tuple(x.shape), tuple(out.shape), tuple(residual.shape), workspace.numel()))


class Ok:
    """A library whose functions all succeed and do nothing."""

    def __getattr__(self, name):
        return lambda *args: 0


def test_trunk_runs_the_layers_it_holds(monkeypatch):
    """Each layer's FFN runs through its own feed_forward (and that one's
    checks), also when a layer has been replaced since the last call."""
    from types import SimpleNamespace

    from moe_amd import model as M

    monkeypatch.setattr(M.L, "lib", Ok)
    monkeypatch.setattr(M, "_stream_ptr", lambda s: 0 if s is None else s)
    m = Reads()
    m.embed = SimpleNamespace(offset=0, dt=0, rows=4, cols=8)
    m.store = SimpleNamespace(region=SimpleNamespace(device_ptr=lambda: 0))
    m._attention = lambda *args: None
    m._mws = None
    m.layers = [dict(ln1=torch.ones(8), ln2=torch.ones(8), moe=Layer()),
                dict(ln1=torch.ones(8), ln2=torch.ones(8), mlp=SimpleNamespace(layer=Layer()))]
    st = SimpleNamespace(pos=[0], ctx=16)
    first = m.layers[0]["moe"]
    M.Model.trunk(m, [[1, 2, 3]], st, stream=7)
    m.layers[0]["moe"] = Layer()
    M.Model.trunk(m, [[1]], st, stream=7)
    want = lambda t: ((t, 8), (t, 8), (t, 8), 256)  # noqa: E731
    assert first.calls == [want(3)] and m.layers[0]["moe"].calls == [want(1)]
    assert m.layers[1]["mlp"].layer.calls == [want(3), want(1)] and st.pos == [4]


def test_rows_are_not_copied_inside_a_capture(monkeypatch):
    """The queued copy of the rows' ids reads a host block of this call alone:
    a capture would replay it from memory that is another call's by then."""
    from moe_amd.model import Batch

    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    with pytest.raises(RuntimeError, match="captured into a graph"):
        Batch([0], [0], 8, "cpu", [1], queued=True)
    b = Batch([0, 2], [3, 1], 8, "cpu", [1, 7])
    assert b.dst.tolist() == [3, 17] and b.ids.tolist() == [1, 7] and b.max_pos == 3

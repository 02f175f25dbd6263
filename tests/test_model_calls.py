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

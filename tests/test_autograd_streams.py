"""Which stream the launches of a differentiable apply go to, on the CPU with
a stand-in for liblfr that records its calls: every launch follows a stream
setting of its own, so that a launch goes to its caller's stream also when
another thread has used the same context since the launch before it."""
from types import SimpleNamespace

import pytest

torch = pytest.importorskip("torch")

from lfric_core_amd import api, autograd  # noqa: E402

NC, NL, NT, NF = 2, 3, 4, 6
UNDF_TO, UNDF_FROM = 20, 30


class RecordingLib:
    """Records (launch, stream); after every launch another thread sets its stream."""

    def __init__(self):
        self.stream, self.calls = None, []

    def lfr_set_stream(self, h, s):
        self.stream = s
        return 0

    def __getattr__(self, name):
        def launch(h, prec, *args):
            self.calls.append((name, self.stream, prec))
            self.stream = "another thread's"
            return 0
        return launch


@pytest.fixture
def rec(monkeypatch):
    lib = RecordingLib()
    for mod in (api, autograd):
        monkeypatch.setattr(mod, "lib", lambda: lib)
    monkeypatch.setattr(api.Context, "sync_stream", lambda self: lib.lfr_set_stream(self.h, "mine"))
    return lib


def _op(dtype, discontinuous=False):
    ctx = object.__new__(api.Context)
    ctx.h, ctx.device = None, torch.device("cpu")
    fs = SimpleNamespace(ncell_3d=NC * NL, is_discontinuous=discontinuous)

    def space(ndf, undf):
        sp = SimpleNamespace(ctx=ctx, fs=fs, ndf=ndf, undf=undf, h=None)

        def plan(colouring, kind):   # building a plan lets other threads run
            api.lib().stream = "another thread's"
            return SimpleNamespace(h=None)
        sp.plan = plan
        return sp
    m = torch.ones((NF, NT, NC * NL), dtype=dtype)
    return api.LMAOperator(m, space(NT, UNDF_TO), space(NF, UNDF_FROM), SimpleNamespace())


@pytest.mark.parametrize("discontinuous", [False, True])
@pytest.mark.parametrize("want", [(True, True), (True, False), (False, True)])
@pytest.mark.parametrize("transpose", [False, True])
def test_every_launch_sets_its_stream(rec, transpose, want, discontinuous):
    op = _op(torch.float64, discontinuous)
    M = op.matrix.clone().requires_grad_(want[0])
    x = torch.ones(UNDF_TO if transpose else UNDF_FROM, dtype=M.dtype).requires_grad_(want[1])
    y = (autograd.lma_apply_transpose if transpose else autograd.lma_apply)(M, x, op)
    assert len(rec.calls) == 1
    torch.autograd.grad(y, [t for t in (M, x) if t.requires_grad], torch.ones_like(y))
    assert len(rec.calls) == 1 + sum(want)
    assert [s for _, s, _ in rec.calls] == ["mine"] * len(rec.calls), rec.calls


@pytest.mark.parametrize("transpose", [False, True])
def test_matrix_gradient_has_the_matrix_dtype(rec, transpose):
    """A matrix of another precision than the operator's own: its gradient is
    formed in the precision of the fields that the kernel reads."""
    op = _op(torch.float64)
    M = op.matrix.float().requires_grad_()
    x = torch.ones(UNDF_TO if transpose else UNDF_FROM, dtype=M.dtype)
    y = (autograd.lma_apply_transpose if transpose else autograd.lma_apply)(M, x, op)
    g, = torch.autograd.grad(y, (M,), torch.ones_like(y))
    assert g.dtype == torch.float32
    assert [p for _, _, p in rec.calls] == [4, 4]

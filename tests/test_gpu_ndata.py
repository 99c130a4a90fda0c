"""Multidata applies (lfr_matrix_vector_ndata): every field of an
(undf, ndata) "ndata first" field equals, bit for bit, the single-field apply
of that field (which the LMA tests pin to the oracle), for matrix_vector and
transpose_matrix_vector, GH_INC and overwrite, FP32 and FP64."""

import numpy as np
import pytest

import oracle
from lfric_core_amd.function_space import build_dofmap, colour_cells
from lfric_core_amd.mesh import cubed_sphere
from lfric_core_amd.rng import Stream
from lfric_core_amd.configs import normal_lma
from test_gpu_lma import _limited_area

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _setup(ctx, nc, nl, k, spaces):
    from lfric_core_amd import api
    m = cubed_sphere(nc)
    col = colour_cells(m)
    fs = {s: build_dofmap(m, s, nl, k) for s in spaces}
    sp = {s: api.Space(ctx, f) for s, f in fs.items()}
    return m, col, fs, sp


def _t(a, ctx):
    return torch.from_numpy(np.ascontiguousarray(a)).to(ctx.device)


CASES = [
    # (nc, nl, k, to, from, ndata, transpose)
    (3, 4, 1, "W2", "W2", 16, False),   # 36 dofs per cell: plan-entry classes
    (4, 5, 0, "W2", "W2", 16, False),
    (4, 5, 0, "W2", "W2", 3, False),
    (6, 10, 0, "W0", "W0", 16, False),
    (4, 5, 0, "W3", "W2", 16, True),    # D^T onto W2
]


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("nc,nl,k,to,frm,nd,tr", CASES)
def test_ndata_equals_single_field(ctx, dtype, nc, nl, k, to, frm, nd, tr):
    from lfric_core_amd import api
    print(f"case ndata nc={nc} nl={nl} k={k} {to}<-{frm} nd={nd} transpose={tr} {dtype.__name__}",
          flush=True)
    m, col, fs, sp = _setup(ctx, nc, nl, k, {to, frm})
    st = Stream(31)
    n3 = m.ncells * nl
    M = normal_lma(st, n3, fs[to].ndf, fs[frm].ndf).astype(dtype)
    op = api.LMAOperator(_t(M, ctx), sp[to], sp[frm], col)
    lsp, xsp = (frm, to) if tr else (to, frm)
    X = _t(st.uniform(fs[xsp].undf * nd).reshape(fs[xsp].undf, nd).astype(dtype), ctx)
    Y0 = _t(st.uniform(fs[lsp].undf * nd).reshape(fs[lsp].undf, nd).astype(dtype), ctx)
    Yi = Y0.clone()
    api.matrix_vector_ndata(Yi, X, op, transpose=tr)
    Yo = torch.full_like(Y0, float("nan"))
    api.matrix_vector_ndata(Yo, X, op, overwrite=True, transpose=tr)
    single = api.transpose_matrix_vector if tr else api.matrix_vector
    for r in range(nd):
        xr = X[:, r].contiguous()
        yi = Y0[:, r].contiguous()
        single(yi, xr, op)
        yo = torch.empty_like(yi)
        single(yo, xr, op, overwrite=True)
        assert torch.equal(Yi[:, r], yi), f"field {r} (increment)"
        assert torch.equal(Yo[:, r], yo), f"field {r} (overwrite)"
    if not tr and nd == 3:   # one direct oracle check
        ref = oracle.invoke_coloured(0, col, nl, np.zeros(fs[to].undf, dtype), X[:, 1].cpu().numpy(), M,
                                     fs[to].dofmap, fs[frm].dofmap)
        np.testing.assert_array_equal(Yo[:, 1].cpu().numpy(), ref)


def test_ndata_bad_args(ctx):
    from lfric_core_amd import api
    from lfric_core_amd._ffi import LfrError
    print("case ndata errors", flush=True)
    m, col, fs, sp = _setup(ctx, 2, 3, 0, {"W2"})
    M = torch.zeros((6, 6, m.ncells * 3), dtype=torch.float64, device=ctx.device)
    op = api.LMAOperator(M, sp["W2"], sp["W2"], col)
    u = fs["W2"].undf
    with pytest.raises(LfrError):   # ndata above 64
        api.matrix_vector_ndata(torch.zeros(u, 65, dtype=torch.float64, device=ctx.device),
                                torch.zeros(u, 65, dtype=torch.float64, device=ctx.device), op)
    with pytest.raises(LfrError):   # different ndata
        api.matrix_vector_ndata(torch.zeros(u, 4, dtype=torch.float64, device=ctx.device),
                                torch.zeros(u, 3, dtype=torch.float64, device=ctx.device), op)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("space,k", [("W2", 1), ("W0", 1), ("W2", 2)])
@pytest.mark.parametrize("nl", [1, 2, 5])
def test_bundled_applies_bitexact(ctx, dtype, space, k, nl):
    """Higher-order spaces, whose columns go four dofs of one mesh entity to a
    thread (W2) or one (W0, 27 dofs a cell), against the oracle: one field,
    and 1 to 20 fields (quads of lanes at multiples of 4, 4 to 1 fields a
    thread), matrix_vector and its transpose, increment and overwrite."""
    from lfric_core_amd import api
    nc = 2 if k == 2 else 3
    m, col, fs, sp = _setup(ctx, nc, nl, k, {space})
    fs, sp = fs[space], sp[space]
    st = Stream(33)
    M = normal_lma(st, m.ncells * nl, fs.ndf, fs.ndf).astype(dtype)
    op = api.LMAOperator(_t(M, ctx), sp, sp, col)
    for nd in (1, 2, 3, 4, 8, 12, 16, 20):
        print(f"case bundles {space} k={k} C{nc} nl={nl} nd={nd} {dtype.__name__}", flush=True)
        X = st.uniform(fs.undf * nd).reshape(fs.undf, nd).astype(dtype)
        Y0 = st.uniform(fs.undf * nd).reshape(fs.undf, nd).astype(dtype)
        for kind in (0, 1):
            yi = _t(Y0, ctx)
            yo = torch.full_like(yi, float("nan"))
            api.matrix_vector_ndata(yi, _t(X, ctx), op, transpose=kind == 1)
            api.matrix_vector_ndata(yo, _t(X, ctx), op, overwrite=True, transpose=kind == 1)
            torch.cuda.synchronize()
            yi, yo = yi.cpu().numpy(), yo.cpu().numpy()
            for r in sorted({0, nd // 2, nd - 1}):
                xr, y0 = np.ascontiguousarray(X[:, r]), np.ascontiguousarray(Y0[:, r])
                ref = oracle.invoke_coloured(kind, col, nl, y0.copy(), xr, M, fs.dofmap, fs.dofmap)
                np.testing.assert_array_equal(yi[:, r], ref)
                ref = oracle.invoke_coloured(kind, col, nl, np.zeros_like(y0), xr, M, fs.dofmap, fs.dofmap)
                np.testing.assert_array_equal(yo[:, r], ref)
                if nd == 1:
                    single = api.matrix_vector if kind == 0 else api.transpose_matrix_vector
                    ys = torch.empty(fs.undf, dtype=op.matrix.dtype, device=ctx.device)
                    single(ys, _t(xr, ctx), op, overwrite=True)
                    torch.cuda.synchronize()
                    np.testing.assert_array_equal(ys.cpu().numpy(), ref)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("nl", [15, 16, 17, 33])
def test_quads_across_bundles_bitexact(ctx, dtype, nl):
    """A wavefront of quads loads 16 levels' matrix values for all its lanes:
    columns of just under, exactly and just over 16 levels (a wavefront then
    holds levels of one bundle or of two, at any offset), both kinds, against
    the oracle."""
    from lfric_core_amd import api
    m, col, fs, sp = _setup(ctx, 2, nl, 1, {"W2"})
    fs, sp = fs["W2"], sp["W2"]
    st = Stream(34)
    M = normal_lma(st, m.ncells * nl, fs.ndf, fs.ndf).astype(dtype)
    op = api.LMAOperator(_t(M, ctx), sp, sp, col)
    for nd in (4, 16, 24):
        print(f"case quads nl={nl} nd={nd} {dtype.__name__}", flush=True)
        X = st.uniform(fs.undf * nd).reshape(fs.undf, nd).astype(dtype)
        for kind in (0, 1):
            y = torch.full((fs.undf, nd), float("nan"), dtype=op.matrix.dtype, device=ctx.device)
            api.matrix_vector_ndata(y, _t(X, ctx), op, overwrite=True, transpose=kind == 1)
            torch.cuda.synchronize()
            for r in (0, nd - 1):
                ref = oracle.invoke_coloured(kind, col, nl, np.zeros(fs.undf, dtype), np.ascontiguousarray(X[:, r]), M,
                                             fs.dofmap, fs.dofmap)
                np.testing.assert_array_equal(y[:, r].cpu().numpy(), ref)


def _check_against_oracle(ctx, label, op, tr, fields, st):
    """matrix_vector (tr: transpose_matrix_vector) on 1 (None: the single-field
    call) to several fields, increment and overwrite, bit for bit."""
    from lfric_core_amd import api
    lsp, xsp = (op.from_space, op.to_space) if tr else (op.to_space, op.from_space)
    nl, dtype = lsp.fs.nlayers, np.float32 if op.matrix.dtype == torch.float32 else np.float64
    M = op.matrix.cpu().numpy()
    for nd in fields:
        print(f"case {label} transpose={tr} nl={nl} nd={nd} {dtype.__name__}", flush=True)
        n = nd or 1
        X = st.uniform(xsp.undf * n).reshape(xsp.undf, n).astype(dtype)
        Y0 = st.uniform(lsp.undf * n).reshape(lsp.undf, n).astype(dtype)
        for over in (False, True):
            y = _t(np.full_like(Y0, np.nan) if over else Y0, ctx)
            if nd is None:
                call = api.transpose_matrix_vector if tr else api.matrix_vector
                call(y.view(-1), _t(X, ctx).view(-1), op, overwrite=over)
            else:
                api.matrix_vector_ndata(y, _t(X, ctx), op, overwrite=over, transpose=tr)
            y = y.cpu().numpy()
            for r in sorted({0, n // 2, n - 1}):
                start = np.zeros(lsp.undf, dtype) if over else np.ascontiguousarray(Y0[:, r])
                ref = oracle.invoke_coloured(int(tr), op.colouring, nl, start, np.ascontiguousarray(X[:, r]), M,
                                             lsp.fs.dofmap, xsp.fs.dofmap)
                np.testing.assert_array_equal(y[:, r], ref)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("nl", [1, 2, 5])
@pytest.mark.parametrize("to,frm", [("WTHETA", "WTHETA"), ("W2V", "W2V"), ("W2", "WTHETA"), ("W2", "W3"),
                                    ("WTHETA", "W3")])
def test_few_input_dofs_bitexact(ctx, dtype, nl, to, frm):
    """One and two input dofs a cell: less than a block of the gather."""
    from lfric_core_amd import api
    m, col, fs, sp = _setup(ctx, 5, nl, 0, {to, frm})
    st = Stream(35)
    M = normal_lma(st, m.ncells * nl, fs[to].ndf, fs[frm].ndf).astype(dtype)
    op = api.LMAOperator(_t(M, ctx), sp[to], sp[frm], col)
    for tr in (False, True):
        if not sp[frm if tr else to].fs.is_discontinuous:
            _check_against_oracle(ctx, f"{to}<-{frm}", op, tr, (None, 1, 2, 3, 4, 6, 7), st)


def _vector_vertices(mesh, nl):
    """Four dofs at every vertex: W0 with each column four times over."""
    import dataclasses
    from lfric_core_amd.function_space import DofCounts
    fs = build_dofmap(mesh, "W0", nl)
    z = fs.dofmap.astype(np.int64) - 1
    column, shift = z // (nl + 1), z % (nl + 1)             # every W0 column has nl + 1 dofs
    dm = ((4 * column[:, :, None] + np.arange(4)) * (nl + 1) + shift[:, :, None] + 1).reshape(mesh.ncells, 32)
    return dataclasses.replace(fs, counts=DofCounts(vert=4, cell=32), dofmap=np.ascontiguousarray(dm, dtype=np.int32),
                               undf=4 * fs.undf, dof_shift=np.repeat(fs.dof_shift, 4),
                               dof_height=np.repeat(fs.dof_height, 4))


# name: function space on its mesh, classes of its plan with and without the
# few-column ones having joined a larger one, and whether the single-field
# apply goes through bundles as well
ABSENT = {
    # the 8 cube corners among 858 vertices: two entries a cell, one column a bundle
    "W0 C12": (lambda nl: build_dofmap(cubed_sphere(12), "W0", nl), 2, 1, False),
    # order 1: corner vertices, and corner edges, whose columns have one entry
    # a cell and nl levels (the unmasked form but for the absent entries)
    "W0 order 1 C12": (lambda nl: build_dofmap(cubed_sphere(12), "W0", nl, 1), 8, 6, True),
    # a limited area's edge faces, one entry a cell, one column a bundle
    "W2 area": (lambda nl: build_dofmap(_limited_area(40), "W2", nl), 3, 2, False),
    # the same with four columns a bundle
    "W2H order (0, 3) area": (lambda nl: build_dofmap(_limited_area(40), "W2H", nl, 0, 3), 2, 1, True),
    # two entries a cell, four columns a bundle
    "vector vertices C12": (lambda nl: _vector_vertices(cubed_sphere(12), nl), 2, 1, True),
}


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("nl", [2, 3])
@pytest.mark.parametrize("name", list(ABSENT))
def test_absent_entries_in_bundles_bitexact(ctx, dtype, name, nl):
    """Columns that joined a class of more cells a column, so that whole cells
    of theirs are absent; the number of the plan's classes says that they did."""
    from lfric_core_amd import api
    make, apart, joined, single = ABSENT[name]
    fs = make(nl)
    col, sp = colour_cells(fs.mesh), api.Space(ctx, fs)
    assert joined < apart
    for kind in (0, 1):
        assert sp.plan(col, kind).info()["nclasses"] == joined
    st = Stream(36)
    M = normal_lma(st, fs.mesh.ncells * nl, fs.ndf, fs.ndf).astype(dtype)
    op = api.LMAOperator(_t(M, ctx), sp, sp, col)
    for tr in (False, True):
        _check_against_oracle(ctx, name, op, tr, ((None,) if single else ()) + (1, 2, 3, 4, 16), st)

"""GPU tests of the stage kernels without a diagnostics launch (regular
hexagonal mesh, uniform coefficients): bit for bit against the CPU oracle at
the edges of their tiles, level chunks and term sets, and the auxiliary state
they leave against the diagnostics kernels'."""
import numpy as np
import pytest

from oracle import pyoracle as po
from omega_playground_amd import swe

from helpers import params_dict, rich_state, same_bits
from test_gpu_parity import make_pair, upload

pytestmark = pytest.mark.gpu

# PV, KE and SSH with each set of mixing terms
TERM_SETS = [7, 7 + 8, 7 + 16, 7 + 64, 7 + 8 + 32, 7 + 32 + 64, 127]


def compare(got, ref, *tag):
    for name, a, b in zip(("h", "vn", "tr"), got, ref):
        assert same_bits(a, b), (name,) + tag


# grids at, below and above the 8 x 8, 16 x 8 and 16 x 16 tiles; one level to
# several chunks of levels, odd counts (one level per lane) and even ones
@pytest.mark.parametrize("nx,ny,L,ntr", [(4, 4, 1, 1), (16, 16, 1, 2), (33, 18, 1, 5), (17, 6, 2, 3),
                                         (9, 8, 3, 1), (16, 10, 4, 2), (8, 8, 7, 1), (7, 10, 8, 4),
                                         (24, 16, 10, 1), (12, 14, 25, 2), (10, 6, 60, 3),
                                         (9, 6, 66, 1), (8, 18, 130, 2), (40, 32, 16, 3)])
def test_stage_shapes_bitwise(nx, ny, L, ntr):
    om, omodel, gm, gmodel, state = make_pair(nx, ny, L, ntr, seed=L)
    for terms in (79, 127):
        print("case", nx, ny, L, ntr, terms, flush=True)
        omodel.terms = gmodel.terms = terms
        ref = omodel.new_state()
        omodel.compute_tendency(ref, state, 0.0)
        gt = swe.ShallowWaterState(gm, ntr)
        gmodel.compute_tendency(gt, upload(gm, ntr, state), 0.0)
        compare(gt.download(), ref, terms)
        for kind, graph in (("rk4", True), ("lsrk", False), ("lsrk", True)):
            st = swe.RK4Stepper(gmodel) if kind == "rk4" else swe.LSRKStepper(gmodel, 5)
            st.set_graph(graph)
            gs, ref = upload(gm, ntr, state), tuple(a.copy() for a in state)
            st.run(0.0, 20.0, 3, gs)
            po.Stepper(omodel, kind, 5).run(0.0, 20.0, 3, ref)
            compare(gs.download(), ref, terms, kind, graph)


@pytest.mark.parametrize("terms", TERM_SETS)
@pytest.mark.parametrize("L,ntr", [(64, 2), (5, 0), (6, 3)])
def test_stage_term_sets_bitwise(terms, L, ntr):
    om, omodel, gm, gmodel, state = make_pair(18, 12, L, ntr, seed=terms)
    omodel.terms = gmodel.terms = terms
    print("case", terms, L, ntr, flush=True)
    rng = np.random.default_rng(terms)
    prev = tuple(rng.standard_normal(a.shape) for a in state)
    for inc in (False, True):
        ref = tuple(a.copy() for a in prev)
        omodel.compute_tendency(ref, state, 0.0, increment=inc)
        gt = upload(gm, ntr, prev)
        gmodel.compute_tendency(gt, upload(gm, ntr, state), 0.0,
                                add_mode=swe.ADD_INCREMENT if inc else swe.ADD_REPLACE)
        compare(gt.download(), ref, inc)
    gs, ref = upload(gm, ntr, state), tuple(a.copy() for a in state)
    swe.LSRKStepper(gmodel, 5).run(0.0, 30.0, 2, gs)
    po.Stepper(omodel, "lsrk", 5).run(0.0, 30.0, 2, ref)
    compare(gs.download(), ref, "lsrk")


@pytest.mark.parametrize("L", [6, 9, 64])
@pytest.mark.parametrize("how", ["tendency", "do_step", "run", "run_graph", "lsrk"])
def test_stage_leaves_the_auxiliary_state(L, how):
    """After a tendency or a step the auxiliary arrays and the per-field
    tendencies are those of the last stage's input, as with the kernels that
    store the diagnostics (forms 3)."""
    got = []
    for forms in (15, 3):
        om, omodel, gm, gmodel, state = make_pair(14, 10, L, 2, seed=L)
        gmodel.set_kernel_forms(forms)
        gs, gt = upload(gm, 2, state), swe.ShallowWaterState(gm, 2)
        st = swe.LSRKStepper(gmodel, 5) if how == "lsrk" else swe.RK4Stepper(gmodel)
        st.set_graph(how == "run_graph")
        if how == "tendency":
            gmodel.compute_tendency(gt, gs, 0.0)
        elif how == "do_step":
            st.do_step(0.0, 20.0, gs)
        else:
            st.run(0.0, 20.0, 3, gs)
        aux = [gmodel.aux_array(n) for n in ("rvort_vertex", "inv_thick_vertex", "ke_cell",
                                             "vel_div_cell", "tracer_del2_cell")]
        if how == "tendency":
            h, vn, tr = gs.device_ptrs()
            th, tv, tt = gt.device_ptrs()
            gmodel.compute_h_tendency_dev(th, h, vn, swe.ADD_INCREMENT)
            gmodel.compute_vn_tendency_dev(tv, h, vn, swe.ADD_INCREMENT)
            gmodel.compute_tr_tendency_dev(tt, tr, vn, swe.ADD_INCREMENT)
            aux += list(gt.download())
        got.append(aux + list(gs.download()))
    for a, b in zip(*got):
        assert same_bits(a, b)


@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf])
def test_stage_nonfinite_rows_spread_as_with_stored_diagnostics(value):
    """A NaN or an infinity in any one row reaches the same elements as
    through the kernels that store the diagnostics."""
    for field, at in ((0, 37), (0, 5), (1, 55), (1, 112), (1, 201), (2, 40)):
        out = []
        for forms in (15, 3):
            om, omodel, gm, gmodel, state = make_pair(12, 10, 8, 1, seed=1)
            gmodel.terms = 127
            gmodel.set_kernel_forms(forms)
            s = tuple(a.copy() for a in state)
            (s[2][0] if field == 2 else s[field])[at, 3] = value
            gt = swe.ShallowWaterState(gm, 1)
            gmodel.compute_tendency(gt, upload(gm, 1, s), 0.0)
            out.append(gt.download())
        for a, b in zip(*out):
            assert same_bits(a, b), (field, at)


@pytest.mark.parametrize("kind,graph", [("rk4", False), ("lsrk", True)])
def test_stage_ensemble_members_step_as_alone(kind, graph):
    """An ensemble whose members differ in grid, layer and tracer counts and
    term sets, with one member on the kernels that store diagnostics: every
    member ends with the bits of stepping alone."""
    shapes = [(16, 16, 1, 1, 79), (9, 8, 5, 0, 15), (12, 10, 25, 2, 127 - 16), (8, 6, 60, 3, 79),
              (10, 8, 64, 1, 7), (6, 4, 130, 2, 79), (10, 10, 16, 2, 127), (17, 6, 2, 1, 39)]
    batch, alone = swe.Batch(kind, 5), []
    batch.set_graph(graph)
    keep = []
    for i, (nx, ny, L, ntr, terms) in enumerate(shapes):
        om, omodel, gm, gmodel, state = make_pair(nx, ny, L, ntr, seed=i)
        gmodel.terms = terms
        s = upload(gm, ntr, state)
        batch.add(gmodel, s, 10.0 + i)
        keep.append((gm, gmodel, s))
        t = upload(gm, ntr, state)
        st = swe.RK4Stepper(gmodel) if kind == "rk4" else swe.LSRKStepper(gmodel, 5)
        alone.append((st, t, 10.0 + i))
    batch.run(3)
    for i, ((_, _, s), (st, t, dt)) in enumerate(zip(keep, alone)):
        got = s.download()
        st.run(0.0, dt, 3, t)
        compare(got, t.download(), shapes[i])


@pytest.mark.parametrize("L,ntr,terms", [(1, 1, 127), (2, 5, 127), (5, 0, 31), (33, 4, 79), (66, 9, 111),
                                         (130, 1, 255)])
def test_general_mesh_edge_means_bitwise(L, ntr, terms):
    """General meshes (pentagons; 9 and 10 edges on edge) through the stored
    edge means, at odd and even layer counts, tracer groups and level chunks,
    with bottom drag: the oracle's bits, and the auxiliary state the per-field
    tendencies read afterwards."""
    from test_gpu_general_mesh import DT, make
    om, omodel, gm, gmodel, pd, state = make(2, L, ntr, terms=terms, seed=L)
    ref = omodel.new_state()
    omodel.compute_tendency(ref, state, 0.0)
    gs, gt = upload(gm, ntr, state), swe.ShallowWaterState(gm, ntr)
    gmodel.compute_tendency(gt, gs, 0.0)
    compare(gt.download(), ref, "tendency")
    h, vn, tr = gs.device_ptrs()
    fields = gt.device_ptrs()
    gmodel.compute_h_tendency_dev(fields[0], h, vn)
    gmodel.compute_vn_tendency_dev(fields[1], h, vn)
    if ntr:
        gmodel.compute_tr_tendency_dev(fields[2], tr, vn)
    compare(gt.download(), ref, "fields")
    for kind, graph in (("rk4", True), ("lsrk", False)):
        st = swe.RK4Stepper(gmodel) if kind == "rk4" else swe.LSRKStepper(gmodel, 5)
        st.set_graph(graph)
        s, r = upload(gm, ntr, state), tuple(a.copy() for a in state)
        st.run(0.0, DT, 2, s)
        po.Stepper(omodel, kind, 5).run(0.0, DT, 2, r)
        compare(s.download(), r, kind)


@pytest.mark.parametrize("L,ntr", [(1, 1), (5, 2), (20, 1), (60, 0), (66, 3)])
@pytest.mark.parametrize("terms", [7, 15, 79, 127])
@pytest.mark.parametrize("kind", ["rk4", "lsrk"])
def test_step_adjoint_rows_written_by_the_stage_kernels(kind, terms, L, ntr):
    """Step adjoints whose stage recomputation writes the VJP's rows at any
    layer count give the bits of the VJP's own pre-pass (forms 7)."""
    print("case", kind, terms, L, ntr, flush=True)
    om, omodel, gm, gmodel, state = make_pair(12, 10, L, ntr, seed=L)
    gmodel.terms = terms
    rng = np.random.default_rng(terms)
    cot = tuple(rng.standard_normal(a.shape) for a in state)
    got = []
    for forms in (15, 7):
        gmodel.set_kernel_forms(forms)
        assert bool(gmodel.kernel_flags() & 16) == (forms == 15)
        st = swe.RK4Stepper(gmodel) if kind == "rk4" else swe.LSRKStepper(gmodel, 5)
        gc = upload(gm, ntr, cot)
        gp = swe.step_vjp(st, 0.0, 30.0, upload(gm, ntr, state), gc)
        got.append(list(gc.download()) + [gp])
    for a, b in zip(*got):
        assert same_bits(a, b)


@pytest.mark.parametrize("nx,ny,L,ntr", [(12, 10, 3, 1), (10, 8, 64, 0), (64, 64, 64, 1),
                                         (64, 66, 64, 1), (16, 8, 20, 3)])
def test_vjp_at_a_state_whose_stage_is_not_run(nx, ny, L, ntr):
    """The tendency VJP gets its diagnostics and rows from the stage kernels
    without a stage (with tracer del4 up to the sizes of one launch, with 64
    layers and one tracer 4096 cells): the bits of the diagnostics launch and
    the VJP's pre-pass (forms 7), and the same auxiliary state."""
    mesh = swe.PlanarHexagonalMesh(nx, ny, 10e3, L)
    model = swe.ShallowWaterModel(mesh, swe.ShallowWaterParams(**params_dict(10e3, ntr)))
    state = rich_state(mesh, L, ntr, 3)
    rng = np.random.default_rng(4)
    cot, out = (tuple(rng.standard_normal(a.shape) for a in state) for _ in range(2))
    for terms in (7, 15, 23, 79, 127):
        print("case", nx, ny, L, ntr, terms, flush=True)
        model.terms = terms
        got = []
        for forms in (15, 7):
            model.set_kernel_forms(forms)
            so, s = upload(mesh, ntr, out), upload(mesh, ntr, state)
            gp = swe.tendency_vjp(model, s, upload(mesh, ntr, cot), so)
            aux = [model.aux_array(n) for n in ("rvort_vertex", "inv_thick_vertex", "ke_cell",
                                                "vel_div_cell")]
            if terms & 64 and ntr:
                aux.append(model.aux_array("tracer_del2_cell"))
            got.append(list(so.download()) + [gp] + aux)
        for a, b in zip(*got):
            assert same_bits(a, b), terms


# 24 bytes a level in a cell's edge rows: the last count a 24-bit factor holds
# and the next one, which other kernels take (tests/test_host_side.py)
@pytest.mark.parametrize("L", [699050, 699051])
def test_tallest_columns_bitwise(L):
    print("case", L, flush=True)
    nx, ny, dc, few = 4, 4, 10e3, 5
    pd = params_dict(dc, 1, all_terms=False)
    om = po.Mesh(nx, ny, dc, few)
    omodel = po.Model(om, **pd)
    state = rich_state(om, few, 1, 3)
    ref = omodel.new_state()
    omodel.compute_tendency(ref, state, 0.0)
    gm = swe.PlanarHexagonalMesh(nx, ny, dc, L)
    gmodel = swe.ShallowWaterModel(gm, swe.ShallowWaterParams(**pd))

    def columns(a):  # levels do not see each other: the few, over and over
        return np.ascontiguousarray(a[..., np.arange(L) % few])

    gs, gt = upload(gm, 1, [columns(a) for a in state]), swe.ShallowWaterState(gm, 1)
    gmodel.compute_tendency(gt, gs, 0.0)
    compare(gt.download(), [columns(a) for a in ref], L)


@pytest.mark.parametrize("terms", [79, 127])
def test_block_order_does_not_change_bits(terms):
    """Large enough for launches of their own for momentum and tracers: with
    and without the XCD order, alone and as an ensemble's member."""
    nx, ny, L, ntr = 72, 70, 64, 2
    mesh = swe.PlanarHexagonalMesh(nx, ny, 10e3, L)
    model = swe.ShallowWaterModel(mesh, swe.ShallowWaterParams(**params_dict(10e3, ntr)))
    model.terms = terms
    y0, out = rich_state(mesh, L, ntr, 2), []
    for order in (1, 0):
        model.set_launch(0, 0, order)
        s, b = upload(mesh, ntr, y0), swe.Batch("rk4", 4)
        m = upload(mesh, ntr, y0)
        b.add(model, m, 20.0)
        swe.RK4Stepper(model).run(0.0, 20.0, 2, s)
        b.run(2)
        out += [s.download(), m.download()]
    for got in out[1:]:
        compare(got, out[0], terms)


@pytest.mark.parametrize("nx,L", [(12, 64), (12, 9), (72, 60)])
def test_cells_per_block_do_not_change_bits(nx, L):
    """Set or tuned cells per block where all fields share a launch (12) and
    where they do not (72), alone and as an ensemble's member."""
    ntr, out = 2, []
    mesh = swe.PlanarHexagonalMesh(nx, nx, 10e3, L)
    model = swe.ShallowWaterModel(mesh, swe.ShallowWaterParams(**params_dict(10e3, ntr)))
    model.terms = 79
    y0 = rich_state(mesh, L, ntr, 2)
    for rows in (256, 4, 2, 1):
        print("case", nx, L, rows, flush=True)
        model.set_launch(rows)
        s, m, b = upload(mesh, ntr, y0), upload(mesh, ntr, y0), swe.Batch("lsrk", 5)
        b.add(model, m, 20.0)
        swe.LSRKStepper(model, 5).run(0.0, 20.0, 2, s)
        b.run(2)
        out += [s.download(), m.download()]
    for got in out[1:]:
        compare(got, out[0])


@pytest.mark.parametrize("kind", ["rk4", "lsrk"])
@pytest.mark.parametrize("del4", [True, False])
def test_ensemble_of_any_terms_and_layers_bitwise(kind, del4):
    """Members of every set of terms, tile shape and levels per lane share
    their launches and end with the bits of their solo steps."""
    b, members = swe.Batch(kind, 5), []
    sets = [7 + x for x in (0, 8, 32, 40) + ((64, 72, 96, 104) if del4 else ())]
    for L in (1, 2, 3, 4, 10, 66):
        for i, terms in enumerate(sets):
            nx, ny, ntr = 8 + i, 10 + 2 * (L % 3), (i + L) % 4
            mesh = swe.PlanarHexagonalMesh(nx, ny, 10e3, L)
            model = swe.ShallowWaterModel(mesh, swe.ShallowWaterParams(**params_dict(10e3, ntr)))
            model.terms = terms
            y0 = rich_state(mesh, L, ntr, L + i)
            s = upload(mesh, ntr, y0)
            b.add(model, s, 15.0)
            members.append((mesh, model, ntr, y0, s))
    print("case", kind, del4, len(members), flush=True)
    b.set_graph(True)
    b.run(3)
    for mesh, model, ntr, y0, s in members:
        solo = upload(mesh, ntr, y0)
        (swe.RK4Stepper(model) if kind == "rk4" else swe.LSRKStepper(model, 5)).run(0.0, 15.0, 3, solo)
        compare(s.download(), solo.download(), mesh.nlayers, model.terms)


@pytest.mark.parametrize("kind", ["rk4", "lsrk"])
@pytest.mark.parametrize("graph", [True, False])
def test_ensemble_side_by_side_bitwise(kind, graph):
    """Members on the stage kernels beside members on the others (momentum
    del4, kernel forms), too large to share launches: several replays with
    uploads, downloads and solo steps between them."""
    b, members = swe.Batch(kind, 5), []
    for i, (nx, L, ntr, terms, forms) in enumerate(((66, 64, 1, 79, 15), (12, 8, 2, 127, 15),
                                                    (40, 5, 3, 111, 15), (12, 64, 1, 15, 3))):
        mesh = swe.PlanarHexagonalMesh(nx, nx, 10e3, L)
        model = swe.ShallowWaterModel(mesh, swe.ShallowWaterParams(**params_dict(10e3, ntr)))
        model.terms = terms
        model.set_kernel_forms(forms)
        y0 = rich_state(mesh, L, ntr, i)
        s, solo = upload(mesh, ntr, y0), upload(mesh, ntr, y0)
        b.add(model, s, 15.0)
        st = swe.RK4Stepper(model) if kind == "rk4" else swe.LSRKStepper(model, 5)
        members.append((s, solo, st))
    b.set_graph(graph)
    for again in range(4):
        print("case", kind, graph, again, flush=True)
        b.run(2)
        for i, (s, solo, st) in enumerate(members):
            st.run(0.0, 15.0, 2, solo)
            got = s.download()
            compare(got, solo.download(), again, i)
            s.upload(*got)


@pytest.mark.parametrize("terms", [79, 127])
@pytest.mark.parametrize("L", [7, 64])
def test_ensemble_of_one_model_bitwise(terms, L):
    """Members that share a model: the stage kernels (79) and, with momentum
    del4, the kernels that store the diagnostics."""
    ntr, n = 2, 5
    mesh = swe.PlanarHexagonalMesh(14, 12, 10e3, L)
    model = swe.ShallowWaterModel(mesh, swe.ShallowWaterParams(**params_dict(10e3, ntr)))
    model.terms = terms
    y0 = [rich_state(mesh, L, ntr, i) for i in range(n)]
    b, states = swe.Batch("lsrk", 5), [upload(mesh, ntr, y) for y in y0]
    for s in states:
        b.add(model, s, 15.0)
    b.run(3)
    aux = model.aux_array("ke_cell")
    for i in reversed(range(n)):
        solo = upload(mesh, ntr, y0[i])
        swe.LSRKStepper(model, 5).run(0.0, 15.0, 3, solo)
        compare(states[i].download(), solo.download(), i)
    assert same_bits(aux, model.aux_array("ke_cell"))

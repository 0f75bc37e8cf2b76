"""GPU tests of what adjoint runs keep between calls: a call on a used stepper
or batch gives the bits of a call on a new one, whatever changed in between."""
import numpy as np
import pytest

from omega_playground_amd import swe

from helpers import same_bits
from test_gpu_batch_adjoint import DC, make_batch, make_ensemble, stepper, upload

pytestmark = pytest.mark.gpu


def same(a, b):
    return a[0] == b[0] and same_bits(a[1], b[1]) and all(
        same_bits(x, y) for s, t in zip(a[2], b[2]) for x, y in zip(s, t))


@pytest.mark.parametrize("kind", ["rk4", "lsrk"])
def test_gradient_on_a_used_stepper(kind):
    mesh, pd, members = make_ensemble(M=2, L=5, kind=kind, n=4)
    model = members[0][0]
    used = stepper(model, kind)

    def run(st, m, n, snaps):
        g = swe.ShallowWaterState(mesh, 2)
        J, gp = swe.adjoint_run(st, 0.0, 40.0, n, upload(mesh, 2, members[m][1]), members[m][2], g,
                                n_snapshots=snaps)
        return J, gp, [g.download()]

    for m, n, snaps in ((0, 4, 3), (1, 4, 3), (1, 7, 2), (0, 1, 1), (0, 6, 5)):
        print("case", kind, m, n, snaps, flush=True)
        assert same(run(used, m, n, snaps), run(stepper(model, kind), m, n, snaps))


def test_ensemble_gradient_on_a_used_batch():
    mesh, pd, members = make_ensemble(M=3, L=6, n=4)
    used, states = make_batch(mesh, 2, members[:2], "rk4", 40.0)

    def run(b, count, n):
        grads = [swe.ShallowWaterState(mesh, 2) for _ in range(count)]
        J, gp = b.adjoint_run(0.0, n, [o for _, _, o in members[:count]], grads, n_snapshots=3)
        return J, gp, [g.download() for g in grads]

    def fresh(count, n):
        return run(make_batch(mesh, 2, members[:count], "rk4", 40.0)[0], count, n)

    for n in (4, 4, 6):
        assert same(run(used, 2, n), fresh(2, n)), n
    # other initial states
    rng = np.random.default_rng(5)
    for i, (model, y0, obs) in enumerate(members[:2]):
        y0 = (y0[0] + rng.standard_normal(y0[0].shape),) + y0[1:]
        members[i] = (model, y0, obs)
        states[i].upload(*y0)
    assert same(run(used, 2, 4), fresh(2, 4))
    # other terms, then a further member
    for model, _, _ in members:
        model.terms = 15
    assert same(run(used, 2, 4), fresh(2, 4))
    third = upload(mesh, 2, members[2][1])
    used.add(members[2][0], third, 40.0)
    assert same(run(used, 3, 4), fresh(3, 4))


def test_ensemble_gradient_with_more_members_than_one_copy_launch():
    mesh, pd, members = make_ensemble(M=19, nx=4, ny=4, L=1, n=2)
    b, states = make_batch(mesh, 2, members, "rk4", 40.0)
    grads = [swe.ShallowWaterState(mesh, 2) for _ in members]
    b.adjoint_run(0.0, 2, [o for _, _, o in members], grads, n_snapshots=2)
    for m in (0, 15, 16, 18):
        model, y0, obs = members[m]
        g = swe.ShallowWaterState(mesh, 2)
        swe.adjoint_run(stepper(model, "rk4"), 0.0, 40.0, 2, upload(mesh, 2, y0), obs, g,
                        tuple(x / 19 for x in (1.0, 0.0, 1.0)), n_snapshots=2)
        for x, y in zip(grads[m].download(), g.download()):
            assert same_bits(x, y), m


@pytest.mark.parametrize("L,ntr,snaps", [(1, 0, 1), (3, 1, 2), (5, 4, 3), (16, 2, 6)])
def test_window_gradient_is_the_chain_of_step_adjoints(L, ntr, snaps):
    """Stored, restored and directly read checkpoints give the bits of step
    adjoints at the states of a forward run, at odd sizes and without tracers."""
    print("case", L, ntr, snaps, flush=True)
    n, dt = 6, 30.0
    mesh, pd, ((model, y0, obs),) = make_ensemble(M=1, L=L, ntr=ntr, n=n, dt=dt)
    st = stepper(model, "rk4")
    ys = [upload(mesh, ntr, y0) for _ in range(n + 1)]
    for i, y in enumerate(ys):
        if i:
            st.run(0.0, dt, i, y)
    cot = swe.ShallowWaterState(mesh, ntr)
    J = swe.misfit(model, ys[n], obs, cot)
    for y in reversed(ys[:n]):
        swe.step_vjp(st, 0.0, dt, y, cot)
    grad = swe.ShallowWaterState(mesh, ntr)
    Jw, _ = swe.adjoint_run(st, 0.0, dt, n, upload(mesh, ntr, y0), obs, grad, n_snapshots=snaps)
    assert J == Jw and all(same_bits(a, b) for a, b in zip(grad.download(), cot.download()))


def test_ensemble_gradient_with_a_coriolis_parameter_per_vertex():
    """The stacked model has the members' own Coriolis parameter, also after
    it changed; members that differ in it are refused."""
    mesh, pd, members = make_ensemble(M=2, L=4, n=3)
    b, states = make_batch(mesh, 2, members, "rk4", 40.0)
    grads = [swe.ShallowWaterState(mesh, 2) for _ in members]
    wanted = [o for _, _, o in members]
    for seed in (0, 1):
        f = pd["f0"] * np.random.default_rng(seed).uniform(0.5, 1.5, mesh.nvertices)
        for model, _, _ in members:
            model.set_f_vertex(f)
        b.adjoint_run(0.0, 3, wanted, grads, n_snapshots=2)
        for m, (model, y0, obs) in enumerate(members):
            g = swe.ShallowWaterState(mesh, 2)
            swe.adjoint_run(stepper(model, "rk4"), 0.0, 40.0, 3, upload(mesh, 2, y0), obs, g,
                            (0.5, 0.0, 0.5), n_snapshots=2)
            for x, y in zip(grads[m].download(), g.download()):
                assert same_bits(x, y), (seed, m)
    members[1][0].set_f_vertex(2 * f)
    with pytest.raises(RuntimeError, match="Coriolis"):
        b.adjoint_run(0.0, 3, wanted, grads, n_snapshots=2)

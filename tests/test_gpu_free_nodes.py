"""Scenes without a tetrahedron (mass points under gravity): no kernel may read an incidence or a contribution, the
engine has none.  One node, a node block partly and exactly filled and one node more, and more than the 64 node
blocks up to which several workgroups share one; CG in both summation orders and PCG.  Bit for bit against
the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _spec(n, precond=0):
    rng = np.random.default_rng(n)
    s = dict(pos=rng.standard_normal((n, 3)), tets=np.zeros((0, 4), dtype=np.int32),
             fixed=np.arange(0, n - 1, 3, dtype=np.int32), E=1e5, nu=0.45, mass=("uniform", 0.7), g=(0.0, -9.81, 1.0), dt=0.01,
             rs=0.1, rm=0.1, iters=10, tol=1e-9, thr=1e-9)
    if precond:
        s["preconditioner"] = precond
    return s


@pytest.mark.parametrize("n", [1, 255, 256, 257, 16385])
@pytest.mark.parametrize("prec,order,precond", [("FP64", 0, 0), ("FP64", 1, 0), ("FP64", 0, 1), ("FP64", 0, 2),
                                                ("FP64_TILED", 1, 0)])
def test_no_elements(prec, order, precond, n):
    from specs import oracle_from_spec
    from sofa_amd import capi, workloads
    print(f"case: {n} free nodes {prec} order {order} preconditioner {precond}", flush=True)
    spec = _spec(n, precond)
    eng = capi.Engine(0, getattr(capi, prec))
    if order:
        eng.set_dot_order(True)
    sid = workloads.add_to_engine(eng, spec)
    eng.commit()
    eng.step([sid], 3)
    x, v, _ = eng.read(sid)
    eng.close()
    o = oracle_from_spec(spec, 0 if order else 1)
    o.step(spec["dt"], 3)
    assert np.array_equal(x, o.get("x")) and np.array_equal(v, o.get("v"))
    assert np.all(v[spec["fixed"]] == 0.0) and np.all(v[-1][1:] != 0.0)

"""Scenes whose CG loops end part way (threshold, tolerance, budget), stepped together for several steps: the launch
that records a stop is the one whose workgroups all have to see it.  Scenes of few and of many node blocks (and,
tiled, of more than 256 tiles, whose partial sums are added by the workgroup).  The untiled FP64 engine and
the reference order bit for bit against the oracle; the others, twice from rest, against themselves bit for bit
and their ends against each scene stepped alone."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

STEPS = 6


def _capi():
    from sofa_amd import capi
    return capi


def _run(prec, specs, seq=False, steps=STEPS, together=True):
    from sofa_amd import workloads
    capi = _capi()
    eng = capi.Engine(0, getattr(capi, prec))
    if seq:
        eng.set_dot_order(True)
    ids = [workloads.add_to_engine(eng, s) for s in specs]
    eng.commit()
    for group in ([ids] if together else [[i] for i in ids]):
        eng.step(group, steps)
    out = [eng.read(i)[:2] + (eng.stats(i),) for i in ids]
    eng.close()
    return out


def _specs(n, prec):
    """Beams that stop by threshold (p.q of the 7th iteration or below), by tolerance and by budget."""
    from sofa_amd import workloads
    base = workloads._beam_spec(n, (1.0, 1.0, 4.0), 1e5, 0.45, 0.01, 40, tol=1e-30, thr=1e-300)
    den = _run(prec, [dict(base, iters=7)], steps=1)[0][2]["den"]
    err = _run(prec, [dict(base, iters=11)], steps=1)[0][2]["err"]
    return [dict(base, thr=1.01 * den), dict(base, tol=1.01 * err), dict(base, iters=13)]


@pytest.mark.parametrize("prec,seq,n", [("FP64", False, (3, 4, 40)), ("FP64", False, (12, 12, 70)), ("FP64", False, (21, 21, 129)),
                                        ("FP64", True, (12, 12, 70)), ("FP64_TILED", True, (12, 12, 70))])
def test_stops_bitexact(prec, seq, n):
    from specs import oracle_from_spec
    print(f"case: stops {prec} {'reference order' if seq else ''} {n}", flush=True)
    specs = _specs(n, prec)
    got = _run(prec, specs, seq)
    assert {g[2]["end_reason"] for g in got} >= {0, 2}
    for s, (x, v, st) in zip(specs, got):
        o = oracle_from_spec(s, 0 if seq else 1)
        o.step(s["dt"], STEPS)
        assert np.array_equal(x, o.get("x")) and np.array_equal(v, o.get("v")), st


@pytest.mark.parametrize("n", [(3, 4, 40), (21, 21, 81)])
@pytest.mark.parametrize("prec", ["FP64_TILED", "FP32", "SPLIT"])
def test_stops_tiled(prec, n):
    print(f"case: stops {prec} {n}", flush=True)
    specs = _specs(n, prec)
    a, b, alone = _run(prec, specs), _run(prec, specs), _run(prec, specs, together=False)
    assert {g[2]["end_reason"] for g in a} >= {0, 2}
    for (x, v, st), (y, w, su), (z, u, sv) in zip(a, b, alone):
        assert np.array_equal(x, y) and np.array_equal(v, w) and st == su
        assert np.array_equal(x, z) and np.array_equal(v, u) and st == sv

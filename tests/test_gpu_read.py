"""sofa_amd_scene_read: the state of one scene through the pinned chunks (up to 2 MiB each), for scenes that
fill part of a chunk, a little more than one (a vector's entries split over two), and several; beside a
second scene, so that the scene's vectors do not start at the arrays' first entry.  Bit for bit, FP32 rounded."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(2, 2, 2), (5, 5, 21), (13, 13, 173), (16, 16, 230), (31, 31, 65)])
@pytest.mark.parametrize("prec", ["FP64", "FP32", "SPLIT"])
def test_read_back(prec, n):
    from sofa_amd import capi, workloads
    print(f"case: read back {prec} {n}", flush=True)
    eng = capi.Engine(0, getattr(capi, prec))
    workloads.add_to_engine(eng, workloads._beam_spec((3, 2, 2), (1.0, 1.0, 4.0), 1e5, 0.45, 0.01, 5))
    sid = workloads.add_to_engine(eng, workloads._beam_spec(n, (1.0, 1.0, 4.0), 1e5, 0.45, 0.01, 5))
    eng.commit()
    rng = np.random.default_rng(5)
    shape = (int(np.prod(n)), 3)
    for scale in (1.0, 1e-3):                     # the same engine again: nothing of the first read is left
        x, v = scale * rng.standard_normal(shape), scale * rng.standard_normal(shape)
        eng.write(sid, x, v)
        xr, vr, f = eng.read(sid)
        if prec == "FP32":
            x, v = x.astype(np.float32), v.astype(np.float32)
        assert np.array_equal(xr, x) and np.array_equal(vr, v) and not np.any(f)
    eng.close()

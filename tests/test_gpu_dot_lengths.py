"""vDot in the reference's order at the lengths where its rounds (4,096 terms) and pieces (64) end, every term of
the sum a node's own: scenes of exactly n nodes, the last terms not zero.  Against the same adds one after the other
on the CPU (numpy's accumulate), bit for bit: sums that grow, that wander through zero, that tie, and that
do so for a few pieces at a time (runs of pieces that take the chain, up to and over the end of a round)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [4, 5, 63, 64, 65, 127, 128, 129, 4032, 4033, 4095, 4096, 4097, 6000, 8191, 8192, 8193, 12288, 12289, 16447]


def _terms(kind, n, rng):
    t = rng.standard_normal(n)
    if kind == "squares":
        return t ** 2
    if kind == "ties":
        t = rng.integers(-3, 8, n) * 0.25
        t[0] = 2.0 ** 52 + 1
        return t
    if kind in ("runs", "single"):       # in some pieces, pairs as large as the sum that cancel
        size = 1 if kind == "single" else 4
        out = t ** 2
        for a in range(0, n, 64):
            if (a // 64) // size % 3 == 1:
                m = out[a:a + 64]
                m[::2] += 2.0 * n
                m[1::2] -= 2.0 * n
        return out
    return t


@pytest.mark.parametrize("kind", ["squares", "signed", "ties", "single", "runs"])
@pytest.mark.parametrize("prec", ["FP64", "FP32"])
def test_vdot_lengths(kind, prec):
    from sofa_amd import capi
    rng = np.random.default_rng(11)
    dt = np.float32 if prec == "FP32" else np.float64
    eng = capi.Engine(0, getattr(capi, prec))
    scenes = []
    for n in SIZES:
        p = np.zeros((n, 3))
        p[:4] = np.eye(4, 3)
        scenes.append(eng.add_scene(p, np.array([[3, 0, 1, 2]]), [1.0], [0.3], [0]))
    eng.commit()
    out = capi.DeviceArray(np.zeros(1))
    for n, s in zip(SIZES, scenes):
        t = _terms(kind, n, rng).astype(dt)
        a, b = np.zeros((n, 3), dtype=dt), np.zeros((n, 3), dtype=dt)
        a[:, 0], b[:, 0] = t, 1.0
        ad, bd = capi.DeviceArray(a), capi.DeviceArray(b)
        eng.vdot(s, ad.ptr, bd.ptr, 1, out.ptr)
        eng.sync()
        got = out.numpy()[0]
        want = np.add.accumulate(np.concatenate([[0.0], t.astype(np.float64)]))[-1]
        assert got == want, (kind, n, got, want)
        ad.close()
        bd.close()
    out.close()
    eng.close()

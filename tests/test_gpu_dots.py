"""vDot in the reference's order by exact parallel rounding, through the C ABI, against the same adds one
after the other on the CPU (numpy's accumulate), bit for bit: sizes around the kernel's pieces (64), groups
(512) and rounds (8192), and terms that cross binades, tie, cancel, absorb or leave the finite numbers."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 63, 64, 65, 511, 512, 513, 1025, 8191, 8192, 8193, 8705, 16384, 20001, 50176]


def _terms(kind, n, rng):
    if kind == "squares":            # r.r: growing sums, absorbed terms
        return rng.standard_normal(n) ** 2
    if kind == "wide":               # 40 decades
        return 10.0 ** rng.uniform(-30, 10, n) * rng.choice([-1, 1], n, p=[0.2, 0.8])
    if kind == "signed":             # partial sums wander through zero
        return rng.standard_normal(n)
    if kind == "negative":
        return -rng.random(n)
    if kind == "ties":               # few-bit terms on a sum near 2^52: half-way cases, both parities
        t = rng.integers(-3, 8, n) * 0.25
        t[0] = 2.0 ** 52 + 1
        return t
    if kind == "edges":              # sums that start exactly on a power of two and step back and forth over it
        t = rng.choice([2.0 ** -53, -2.0 ** -53, 2.0 ** -54, -2.0 ** -52, 0.0, 2.0 ** -60], n)
        t[0] = 1.0
        return t
    if kind == "zeros":              # a clamped face: leading zeros (both signs), then terms
        t = rng.random(n)
        t[: (3 * n) // 4] = 0.0
        t[1::3] *= -0.0
        return t
    if kind == "alternate":          # large terms that cancel, small ones between
        t = rng.random(n) * 1e-8
        t[::5] = 1e8
        t[3::5] = -1e8
        return t
    if kind == "subnormal":
        return rng.random(n) * 1e-310
    if kind == "huge":               # overflows part way
        return rng.random(n) * 1e304 + 1e304
    t = rng.random(n)                # an infinity or a NaN in the middle
    t[n // 2] = np.inf if kind == "inf" else np.nan
    return t


@pytest.mark.parametrize("kind", ["squares", "wide", "signed", "negative", "ties", "edges", "zeros", "alternate",
                                  "subnormal", "huge", "inf", "nan"])
def test_vdot_sequential_order(kind):
    from sofa_amd import capi
    rng = np.random.default_rng(7)
    eng = capi.Engine(0, capi.FP64)
    scenes = []
    for n in SIZES:
        p = np.zeros((n + 4, 3))
        p[:4] = np.eye(4, 3)
        scenes.append(eng.add_scene(p, np.array([[3, 0, 1, 2]]), [1.0], [0.3], [0]))
    eng.commit()
    out = capi.DeviceArray(np.zeros(1))
    for n, s in zip(SIZES, scenes):
        t = np.concatenate([_terms(kind, n, rng), np.zeros(4)])
        a = np.zeros((n + 4, 3))
        b = np.zeros((n + 4, 3))
        a[:, 0], b[:, 0] = t, 1.0
        ad, bd = capi.DeviceArray(a), capi.DeviceArray(b)
        eng.vdot(s, ad.ptr, bd.ptr, 1, out.ptr)
        eng.sync()
        got = out.numpy()[0]
        with np.errstate(all="ignore"):
            want = np.add.accumulate(np.concatenate([[0.0], t]))[-1]
        assert got == want or (np.isnan(got) and np.isnan(want)), (kind, n, got, want)
        ad.close()
        bd.close()
    out.close()
    eng.close()

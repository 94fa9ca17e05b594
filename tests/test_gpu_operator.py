"""The tiled CG operator (k_tile_apply): tiles with few elements, a full tile and a remainder, many tiles;
one material and a material per element with a consistent mass; with and without a plane.  The
engines that run it in one CG against the oracle's step (MIXED, which refines with the FP32 engine's operator,
is compared with converged solutions elsewhere).  Bars: FP64_TILED sums shared nodes tile by tile and p.q by
blocks, a few ulp (1e-16) of the vectors per operation, amplified by at most the 10 iterations of a solve
that is far from converged: 1e-10, on x and v.  The single precision elements: 2e-5 on x, the bar of every
FP32 trajectory test; their v after two steps is the small difference that the float force pass leaves of
positions of order one, which says nothing about the operator, and is not compared."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

BARS = {"FP64_TILED": 1e-10, "FP32": 2e-5, "SPLIT": 2e-5}


def _capi():
    from sofa_amd import capi
    return capi


def _spec(n, kind):
    from sofa_amd import workloads
    s = workloads._beam_spec(n, (1.0, 1.0, 4.0), 1e5, 0.45, 0.01, 10)
    if kind == "materials":
        rng = np.random.default_rng(7)
        s["E"] = rng.uniform(0.7e5, 1.4e5, len(s["tets"]))
        s["nu"] = rng.uniform(0.3, 0.45, len(s["tets"]))
        s["mass"] = ("meshmatrix", 1000.0)
    elif kind == "plane":
        s["plane"] = dict(normal=(0.0, 1.0, 0.0), d=0.05, stiffness=500.0, damping=1.0)
    return s


@pytest.mark.parametrize("kind", ["one", "materials", "plane"])
@pytest.mark.parametrize("n", [(2, 2, 2), (3, 3, 27), (2, 3, 53), (9, 8, 30)])
@pytest.mark.parametrize("prec", ["FP64_TILED", "FP32", "SPLIT"])
def test_tile_operator(prec, n, kind):
    from specs import oracle_from_spec
    from sofa_amd import workloads
    capi = _capi()
    print(f"case: tile operator {prec} {n} {kind}", flush=True)
    spec = _spec(n, kind)
    o = oracle_from_spec(spec, 0)
    o.step(spec["dt"], 2)
    for variant in (0, 2):
        eng = capi.Engine(0, getattr(capi, prec))
        sid = workloads.add_to_engine(eng, spec)
        eng.commit()
        eng.set_apply_variant(variant)
        eng.step([sid], 2)
        x, v, _ = eng.read(sid)
        eng.close()
        for a, b in ((x, o.get("x")), (v, o.get("v")))[:2 if prec == "FP64_TILED" else 1]:
            e = float(np.linalg.norm(a - b) / np.linalg.norm(b))
            assert e <= BARS[prec], (variant, e)


@pytest.mark.parametrize("prec", ["FP64_TILED", "FP32"])
def test_many_tiles(prec):
    """More than 256 tiles: the scene's partial sums are added by the block, in the operator and in the update.  Bars
    as above."""
    from specs import oracle_from_spec
    from sofa_amd import workloads
    capi = _capi()
    print(f"case: many tiles {prec}", flush=True)
    spec = _spec((21, 21, 81), "one")
    o = oracle_from_spec(spec, 0)
    o.step(spec["dt"], 1)
    eng = capi.Engine(0, getattr(capi, prec))
    sid = workloads.add_to_engine(eng, spec)
    eng.commit()
    assert eng.tiling(sid)["tiles"] > 256
    eng.step([sid], 1)
    x = eng.read(sid)[0]
    eng.close()
    assert float(np.linalg.norm(x - o.get("x")) / np.linalg.norm(o.get("x"))) <= BARS[prec]


def test_many_node_blocks():
    """The untiled FP64 engine above 512 node blocks (131,072 nodes), where a scene's partials of p.q and r.r are
    added by a kernel of its own: the oracle's blocked sums, bit for bit."""
    from specs import oracle_from_spec
    from sofa_amd import workloads
    capi = _capi()
    print("case: many node blocks", flush=True)
    spec = dict(_spec((52, 52, 49), "one"), iters=4)
    assert len(spec["pos"]) > 512 * 256
    o = oracle_from_spec(spec, 1)
    o.step(spec["dt"], 1)
    eng = capi.Engine(0, capi.FP64)
    sid = workloads.add_to_engine(eng, spec)
    eng.commit()
    eng.step([sid], 1)
    x, v, _ = eng.read(sid)
    eng.close()
    assert np.array_equal(x, o.get("x")) and np.array_equal(v, o.get("v"))


@pytest.mark.parametrize("prec,copies", [("FP64_TILED", 6), ("FP32", 14)])
def test_large_sets(prec, copies):
    """A launch set whose element records exceed 256 MB (the operator recomputes them) against the same scenes
    stepped one by one (it reads them back): the same bits, with materials per element and one material."""
    from sofa_amd import workloads
    capi = _capi()
    print(f"case: large sets {prec}", flush=True)
    specs = [_spec((33, 33, 65), "materials"), _spec((33, 33, 65), "one")]
    out = []
    for together in (True, False):
        eng = capi.Engine(0, getattr(capi, prec))
        ids = [workloads.add_to_engine(eng, specs[k % 2]) for k in range(copies)]
        eng.commit()
        per_tet = 72 if prec == "FP32" else 168
        assert sum(eng.tiling(i)["tiles"] for i in ids) * 512 * per_tet > 256 << 20
        for group in ([ids] if together else [[i] for i in ids[:2]]):
            eng.step(group, 2)
        out.append([eng.read(i)[:2] for i in ids[:2]])
        eng.close()
    for (x, v), (xs, vs) in zip(*out):
        assert np.array_equal(x, xs) and np.array_equal(v, vs)


@pytest.mark.parametrize("order", [0, 1])
@pytest.mark.parametrize("n", [(2, 2, 2), (8, 8, 4), (8, 8, 5), (4, 5, 13), (16, 16, 64), (16, 16, 65)])
def test_few_node_blocks(n, order):
    """The untiled FP64 engine's node kernel with four workgroups per node block (up to 64 blocks, 16,384 nodes) and
    above it: one node block partly and exactly filled and one node more, the last block of the rule and the
    first beyond; both summation orders; two scenes, so that the second's nodes start inside a block of the
    flattened arrays.  Bit for bit."""
    from specs import oracle_from_spec
    from sofa_amd import workloads
    capi = _capi()
    print(f"case: few node blocks {n} order {order}", flush=True)
    spec = _spec(n, "one")
    eng = capi.Engine(0, capi.FP64)
    if order:
        eng.set_dot_order(True)
    workloads.add_to_engine(eng, _spec((3, 3, 4), "one"))
    sid = workloads.add_to_engine(eng, spec)
    eng.commit()
    eng.step([0, sid], 2)
    x, v, _ = eng.read(sid)
    eng.close()
    o = oracle_from_spec(spec, 0 if order else 1)
    o.step(spec["dt"], 2)
    assert np.array_equal(x, o.get("x")) and np.array_equal(v, o.get("v"))


@pytest.mark.parametrize("prec", ["FP64_TILED", "FP32"])
def test_cg_solve_keeps_the_force_calls_rotations(prec):
    """cg_solve computes the rotations of the engine's own positions; addDForce after it still uses the last
    addForce's, so its result has the same bits before and after."""
    from sofa_amd import workloads
    capi = _capi()
    print(f"case: cg_solve between addDForce calls, {prec}", flush=True)
    dt = np.float32 if prec == "FP32" else np.float64
    spec = _spec((3, 3, 27), "one")
    eng = capi.Engine(0, getattr(capi, prec))
    sid = workloads.add_to_engine(eng, spec)
    eng.commit()
    rng = np.random.default_rng(3)
    dev = lambda a: capi.DeviceArray(np.ascontiguousarray(a, dtype=dt))
    x, dx = dev(spec["pos"] + 0.02 * rng.standard_normal(spec["pos"].shape)), dev(rng.standard_normal(spec["pos"].shape))
    f, before, after, sol = (dev(np.zeros(spec["pos"].shape)) for _ in range(4))
    eng.fem_add_force(sid, x.ptr, f.ptr)
    eng.fem_add_dforce(sid, dx.ptr, before.ptr, 1.0)
    eng.cg_solve(sid, 1.0, 0.0, -1e-3, dx.ptr, sol.ptr)
    eng.fem_add_dforce(sid, dx.ptr, after.ptr, 1.0)
    a, b = before.numpy(), after.numpy()
    eng.close()
    assert np.any(a) and np.array_equal(a, b)


@pytest.mark.parametrize("first", [0, 1])
@pytest.mark.parametrize("prec,variant", [("FP64_TILED", 0), ("FP32", 0), ("FP32", 1), ("SPLIT", 0), ("SPLIT", 3)])
def test_cg_solve_beside_force_calls(prec, variant, first):
    """cg_solve of one scene on one stream while force calls of another scene of the same engine are in flight on
    a second stream: scenes share no buffer, so each has the bits that it has alone."""
    from sofa_amd import workloads
    capi = _capi()
    print(f"case: cg_solve of scene {first} beside force calls, {prec}", flush=True)
    dt = np.float32 if prec == "FP32" else np.float64
    specs = [_spec((9, 9, 40), "one"), _spec((8, 9, 33), "materials")]
    eng = capi.Engine(0, getattr(capi, prec))
    for s in specs:
        workloads.add_to_engine(eng, s)
    eng.commit()
    eng.set_apply_variant(variant)
    a, b = first, 1 - first
    rng = np.random.default_rng(5)
    dev = lambda v: capi.DeviceArray(np.ascontiguousarray(v, dtype=dt))
    shape = [s["pos"].shape for s in specs]
    rhs, x, dx = (dev(rng.standard_normal(shape[a])), dev(specs[b]["pos"] + 0.01 * rng.standard_normal(shape[b])),
                  dev(rng.standard_normal(shape[b])))
    one, two = capi.Stream(), capi.Stream()
    got = []
    for beside in (False, True):
        sol, f = dev(np.zeros(shape[a])), dev(np.zeros(shape[b]))
        for _ in range(8):
            for _ in range(40):
                eng.fem_add_force(b, x.ptr, f.ptr, stream=two)
                eng.fem_add_dforce(b, dx.ptr, f.ptr, -0.5, stream=two)
            if not beside:
                two.synchronize()
            eng.cg_solve(a, 1.0, 0.0, -1e-3, rhs.ptr, sol.ptr, stream=one)
        two.synchronize()
        got.append((sol.numpy(), f.numpy()))
        sol.close()
        f.close()
    eng.close()
    assert np.any(got[0][0]) and np.any(got[0][1])
    assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1])


@pytest.mark.parametrize("branches", [1, 4])
@pytest.mark.parametrize("prec", ["FP32", "SPLIT", "MIXED"])
def test_record_line(prec, branches):
    """A set of scenes whose element records exceed 150 MB (SPLIT: 96) together, in one launch sequence and in branches that each
    stay below (the operator recomputes the records), against each scene alone (it reads them back): the same
    bits, scenes of one material and of a material per element, with and without a plane."""
    from sofa_amd import workloads
    capi = _capi()
    print(f"case: record line {prec} {branches} branches", flush=True)
    specs = [_spec((17, 17, 65), k) for k in ("one", "materials", "plane")]
    out = []
    for together in (True, False):
        eng = capi.Engine(0, getattr(capi, prec))
        ids = [workloads.add_to_engine(eng, specs[k % 3]) for k in range(28)]
        eng.commit()
        eng.set_graphs(True)
        eng.set_branches(branches)
        mb = [eng.tiling(i)["tiles"] * 512 * 72 / 2 ** 20 for i in ids]
        assert sum(mb) > 150 > 2 * max(mb) and (branches == 1 or sum(mb) / branches < 72)
        for group in ([ids] if together else [[i] for i in ids[:3]]):
            eng.step(group, 2)
        out.append([eng.read(i)[:2] for i in ids[:3]])
        eng.close()
    for (x, v), (xs, vs) in zip(*out):
        assert np.any(v) and np.array_equal(x, xs) and np.array_equal(v, vs)


@pytest.mark.parametrize("prec,variant,n,bar", [("FP32", 0, (9, 9, 33), 1e-4), ("FP32", 1, (9, 9, 33), 1e-4),
                                                ("FP32", 2, (33, 33, 65), 1e-4), ("FP32", 3, (33, 33, 65), 1e-4),
                                                ("SPLIT", 0, (33, 33, 65), 1e-4), ("SPLIT", 1, (9, 9, 33), 1e-4),
                                                ("FP64_TILED", 0, (9, 9, 33), 1e-10), ("FP64_TILED", 1, (41, 41, 129), 1e-10)])
def test_cg_solve_rotations(prec, variant, n, bar):
    """cg_solve on positions turned by one radian (the rotations of the last step are those of the rest positions), in
    scenes of few and many records and every operator variant, against the untiled FP64 engine.  Bars: a few ulp of the vectors per
    operation (1e-16 double, 1e-7 float), times the 10 iterations, times 100 for what CG makes of them."""
    from sofa_amd import workloads
    capi = _capi()
    print(f"case: cg_solve on turned positions {prec} {variant} {n}", flush=True)
    spec = _spec(n, "one")
    c, s = np.cos(1.0), np.sin(1.0)
    x = spec["pos"] @ np.array([[c, s, 0.0], [-s, c, 0.0], [0.0, 0.0, 1.0]])
    rhs = np.random.default_rng(3).standard_normal(x.shape)
    got = []
    for p in ("FP64", prec):
        dt = np.float32 if p == "FP32" else np.float64
        eng = capi.Engine(0, getattr(capi, p))
        sid = workloads.add_to_engine(eng, spec)
        eng.commit()
        if p != "FP64":
            eng.set_apply_variant(variant)
        eng.write(sid, x)
        dev = lambda a: capi.DeviceArray(np.ascontiguousarray(a, dtype=dt))
        xd, f, b, sol = dev(x), dev(np.zeros(x.shape)), dev(rhs), dev(np.zeros(x.shape))
        if p == "FP64":        # the untiled engine's rotations are the last force call's
            eng.fem_add_force(sid, xd.ptr, f.ptr)
        eng.cg_solve(sid, 1.0, 0.0, -1e-3, b.ptr, sol.ptr)
        got.append(sol.numpy().astype(np.float64))
        eng.close()
    assert np.linalg.norm(got[1] - got[0]) <= bar * np.linalg.norm(got[0])

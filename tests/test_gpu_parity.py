"""GPU parity: the HIP solver (through the C ABI) against the CPU oracle.

Tolerances
  compat mode (FP64, reference local update): bit-identical to the oracle's
    restatement on the same partition; against the reference golden
    (printed with 6 decimals) within 1e-6 us.
  converge mode (FP32, exact local update): max |dT| <= 1e-4 * max(T)
    against the FP64 fixed point of the oracle, the per-config bound the
    solver is specified to.
"""
import ctypes as C

import numpy as np
import pytest

import cases
import fimpy as F
import pyoracle as O
import vtkio

pytestmark = pytest.mark.gpu


def _compat_run(mesh, pack, stims, dt, n_steps, local=F.LOCAL_REF):
    s = F.Solver(pack, mode=F.MODE_COMPAT, local=local)
    fw = mesh.front_width()
    s.reset()
    for active, tstart, vtx in stims:  # update_events_gpu at cur_time 0
        if not (tstart >= 0.0 and active):
            break
        s.seed(vtx, 0.0)
    cur = 0.0
    for _ in range(n_steps):
        ps = cur
        cur += dt
        s.step(ps, cur, dt, fw)
    phi, st = s.download()
    s.close()
    return phi, st


def test_compat_ut_mesh_matches_golden_and_oracle():
    m = F.Mesh.load_vtk(f"{cases.UT}/ut_mesh.vtk")
    m.read_tags(f"{cases.UT}/ut_mesh.tags")
    p = F.Pack(m, F.PART_TAGS)
    stims = cases.ut_plan_stimuli()
    phi, st = _compat_run(m, p, stims, 150e3, 3)
    g = vtkio.read_vtk(f"{cases.UT}/cuda_fim_res.vtk")
    gp, gs = g["point_data"]["phi"], g["point_data"]["states"]
    assert np.array_equal(st, gs.astype(np.int32))
    ours = np.where(phi < 1e50, phi, -1.0)
    assert np.max(np.abs(ours - gp)) <= 1e-6
    xyz, e2n, _ = m.arrays()
    om = O.Mesh(xyz, e2n, atags=np.loadtxt(f"{cases.UT}/ut_mesh.tags", dtype=np.int32))
    ophi, ost, _ = O.compat_solve(om, stims, 150e3, 3)
    assert np.array_equal(st, ost)
    assert np.array_equal(phi, ophi)  # bit-identical FP64


@pytest.mark.parametrize("steps", [1, 2, 4])
def test_compat_ut_mesh_windows(steps):
    m = F.Mesh.load_vtk(f"{cases.UT}/ut_mesh.vtk")
    m.read_tags(f"{cases.UT}/ut_mesh_p.tags")
    p = F.Pack(m, F.PART_TAGS)
    stims = cases.ut_plan_stimuli()
    phi, st = _compat_run(m, p, stims, 150e3, steps)
    xyz, e2n, _ = m.arrays()
    om = O.Mesh(xyz, e2n, atags=np.loadtxt(f"{cases.UT}/ut_mesh_p.tags", dtype=np.int32))
    ophi, ost, _ = O.compat_solve(om, stims, 150e3, steps)
    assert np.array_equal(st, ost)
    assert np.array_equal(phi, ophi)


def test_compat_box_rcb_partition():
    """reference semantics on a generated mesh with the own partitioner"""
    cfg = cases.scaled(cases.CUBE, 2)
    m, om = cases.box(cfg, seed=3)
    p = F.Pack(m, F.PART_RCB, max_nn=128, seed=3)
    e2s, _ = p.partition()
    om = O.Mesh(om.xyz, om.e2n, fib=om.fib, vel=om.vel, atags=e2s.astype(np.int32))
    stims = [(1, 0.0, [0])]
    fw = m.front_width()
    n_steps = int(np.ceil(1.8 * 10000 / 0.6 / 1000.0)) + 2
    phi, st = _compat_run(m, p, stims, 1000.0, n_steps)
    ophi, ost, _ = O.compat_solve(om, stims, 1000.0, n_steps, front_width=fw)
    assert np.array_equal(st, ost)
    assert np.array_equal(phi, ophi)


@pytest.mark.parametrize("block,max_nn", [(64, 64), (128, 96), (256, 128), (256, 256), (512, 300),
                                          (64, 128), (256, 700)])
def test_compat_submesh_kernels_bit_identical(block, max_nn):
    """the thread-per-copy pass (copies <= block; geometry in LDS or not; one
    wave, so a slot's candidate is not split over two) and the general pass
    (copies > block), through re-entry (tail, far) and with shared vertices
    lowered from outside: bit-identical to the oracle"""
    cfg = dict(cases.SLAB, nx=17, ny=13, nz=5, lx=17e3, ly=13e3, lz=5e3)
    m, om = cases.box(cfg, seed=5)
    p = F.Pack(m, F.PART_RCB, max_nn=max_nn, seed=3)
    e2s, _ = p.partition()
    om = O.Mesh(om.xyz, om.e2n, fib=om.fib, vel=om.vel, atags=e2s.astype(np.int32))
    dt, apd, steps = 2e3, 20e3, 45
    stims = [(1, 0.0, [0, 700]), (1, 61e3, [5])]
    s = F.Solver(p, mode=F.MODE_COMPAT, local=F.LOCAL_REF, apd=apd, block=block)
    fw = m.front_width()
    for _ in range(2):  # the second time through fim_reset in the middle of the state
        s.reset()
        cur = 0.0
        for _ in range(steps):
            ps = cur
            cur += dt
            for active, tstart, vtx in stims:
                if active and ps <= tstart < cur:
                    s.seed(vtx, tstart)
            left = s.step(ps, cur, dt, fw)
    phi, st = s.download()
    s.close()
    ophi, ost, _ = O.compat_solve(om, stims, dt, steps, apd=apd, front_width=fw, timed=True)
    assert np.array_equal(st, ost)
    assert np.array_equal(phi, ophi)
    assert left >= np.sum((st == F.NARROW) | (st == F.NEXT))  # copies against vertices


@pytest.mark.parametrize("block,max_nn", [(64, 64), (256, 256), (64, 128)])
def test_compat_submesh_kernels_exact_candidates(block, max_nn):
    """the same passes with the exact local update, against the oracle's
    windows with that update (the windows are not a fixed-point solve; its
    FP64 arithmetic differs from the device's by contraction only; bound 1e-4
    of the latest time)"""
    cfg = dict(cases.SLAB, nx=17, ny=13, nz=5, lx=17e3, ly=13e3, lz=5e3)
    m, om = cases.box(cfg, seed=5)
    p = F.Pack(m, F.PART_RCB, max_nn=max_nn, seed=3)
    e2s, _ = p.partition()
    om = O.Mesh(om.xyz, om.e2n, fib=om.fib, vel=om.vel, atags=e2s.astype(np.int32))
    s = F.Solver(p, mode=F.MODE_COMPAT, local=F.LOCAL_EXACT, block=block)
    fw = 1e9  # every earlier time may act: no upwind cut
    s.reset()
    s.seed([0], 0.0)
    cur = 0.0
    for _ in range(60):
        s.step(cur, cur + 2e3, 2e3, fw)
        cur += 2e3
    phi, _ = s.download()
    s.close()
    ref, _, _ = O.compat_solve(om, [(1, 0.0, [0])], 2e3, 60, front_width=fw, variant=O.LOCAL_EXACT)
    assert ref.max() < 1e50
    assert np.max(np.abs(phi - ref)) <= 1e-4 * ref.max()


def _converge(m, pack, sources, **kw):
    s = F.Solver(pack, **kw)
    s.seed(sources, 0.0)
    it = s.run()
    phi, st = s.download()
    res = s.residual()
    stats = s.stats()
    s.close()
    return phi, st, it, res, stats


def _check_fp32(phi, ref):
    fin = ref < 1e50
    assert np.array_equal(fin, phi < 1e50)
    err = np.max(np.abs(phi[fin] - ref[fin]))
    tol = 1e-4 * ref[fin].max()
    assert err <= tol, (err, tol)
    return err


def test_converge_cube_48k_vs_fp64_oracle():
    m, om = cases.box(cases.CUBE, seed=1)
    p = F.Pack(m, F.PART_RCB, max_nn=512, seed=1)
    phi, st, it, res, stats = _converge(m, p, [0])
    ref, _ = O.fim_solve(om, [0], variant=O.LOCAL_EXACT)
    _check_fp32(phi, ref)
    assert res < 1e-5
    assert np.all(st == F.FROZEN)


def test_converge_anisotropic_slab_vs_fp64_oracle():
    cfg = cases.scaled(cases.SLAB, 4)
    m, om = cases.box(cfg, seed=2)
    p = F.Pack(m, F.PART_RCB, max_nn=512, seed=2)
    src = cases.pacing_sites(cfg, 5, seed=2)
    phi, st, it, res, stats = _converge(m, p, src)
    ref, _ = O.fim_solve(om, src, variant=O.LOCAL_EXACT)
    _check_fp32(phi, ref)


@pytest.mark.parametrize("staged", [False, True])
@pytest.mark.parametrize("block", [64, 128, 256, 512])
def test_converge_workgroup_shapes_agree(block, staged):
    cfg = cases.scaled(cases.SLAB, 8)
    m, om = cases.box(cfg, seed=5)
    p = F.Pack(m, F.PART_RCB, max_nn=256, seed=5)
    src = cases.pacing_sites(cfg, 3, seed=5)
    phi, *_ = _converge(m, p, src, block=block, staged=staged)
    ref, _ = O.fim_solve(om, src, variant=O.LOCAL_EXACT)
    _check_fp32(phi, ref)


def test_converge_long_element_lists_and_pair_path_agree():
    # 2048-copy submeshes seeded on their whole bottom faces: sweeps mark more
    # elements than one element-list pass holds, so they run in several
    # passes.  Workgroups of 256 and 512 evaluate (element, target) pairs, of
    # 128 one element per lane: the same sweeps, so bit-identical maps, all
    # within tolerance of the FP64 oracle.
    cfg = cases.scaled(cases.SLAB, 4)
    m, om = cases.box(cfg, seed=17)
    p = F.Pack(m, F.PART_RCB, max_nn=2048, seed=17)
    assert p.info["ne_max"] < (1 << 14)  # the pair path is taken at 256
    xyz, _, _ = m.arrays()
    src = np.nonzero(xyz[:, 2] < xyz[:, 2].min() + 0.2 * cfg["lz"] / cfg["nz"])[0]
    assert len(src) > 1000  # a bottom layer of ~2,400 tets per submesh is marked at once
    maps = {}
    for block in (128, 256, 512):
        s = F.Solver(p, block=block, window=0.0, local_iters=4)
        s.seed(src, 0.0)
        s.run()
        maps[block] = s.download()[0]
        s.close()
    assert np.array_equal(maps[128], maps[256]) and np.array_equal(maps[128], maps[512])
    ref, _ = O.fim_solve(om, src, variant=O.LOCAL_EXACT)
    _check_fp32(maps[256], ref)


@pytest.mark.parametrize("max_nn", [256, 1280])
def test_converge_register_variants_agree(max_nn):
    # the compute kernel built for 5..8 waves per SIMD: same arithmetic, so the
    # same fixed point bit for bit, single and batched, and the FP64 oracle's
    cfg = cases.scaled(cases.SLAB, 8)
    m, om = cases.box(cfg, seed=11)
    p = F.Pack(m, F.PART_RCB, max_nn=max_nn, seed=11)
    srcs = [cases.pacing_sites(cfg, k + 1, seed=40 + k) for k in range(3)]
    ref, _ = O.fim_solve(om, srcs[0], variant=O.LOCAL_EXACT)
    base = None
    for waves in (0, 5, 6, 7, 8):
        s = F.Solver(p, n_instances=3, window=50.0, local_iters=4, waves=waves, block=256)
        for i, src in enumerate(srcs):
            s.seed(src, 0.0, inst=i)
        s.run()
        maps = [s.download(inst=i)[0] for i in range(3)]
        s.close()
        _check_fp32(maps[0], ref)
        if base is None:
            base = maps
        for a_, b_ in zip(base, maps):
            assert np.array_equal(a_, b_), waves


def test_seed_batch_equals_per_instance_seeds():
    cfg = cases.scaled(cases.SLAB, 8)
    m, _ = cases.box(cfg, seed=13)
    p = F.Pack(m, F.PART_RCB, max_nn=256, seed=13)
    sets = [cases.pacing_sites(cfg, k % 3 + 1, seed=60 + k) for k in range(4)]
    a = F.Solver(p, n_instances=5, window=50.0)
    b = F.Solver(p, n_instances=5, window=50.0)
    for i, src in enumerate(sets):
        a.seed(src, 0.0, inst=i + 1)
    b.seed_batch(sets + [np.zeros(0, np.int64)], 0.0, insts=[1, 2, 3, 4, 0])
    a.run()
    b.run()
    for i in range(5):
        pa, sa = a.download(inst=i)
        pb, sb = b.download(inst=i)
        assert np.array_equal(pa, pb) and np.array_equal(sa, sb), i
    assert np.all(a.download(inst=0)[0] > 1e50)  # instance 0 was never seeded
    with pytest.raises(F.FimError):
        b.seed_batch([sets[0]], 0.0, insts=[5])  # instance out of range
    with pytest.raises(F.FimError):
        b.seed_batch([np.array([m.nn], np.int64)], 0.0)  # vertex out of range
    a.close()
    b.close()


def test_stream_maps_equal_lockstep_maps():
    # continuous batching: 10 solves through 3 instances, recycled as they
    # converge; every map equals the same solve run on its own, bit for bit
    from fimpy.stream import stream_solve
    cfg = cases.scaled(cases.SLAB, 8)
    m, om = cases.box(cfg, seed=19)
    p = F.Pack(m, F.PART_RCB, max_nn=256, seed=19)
    sets = [cases.pacing_sites(cfg, k % 3 + 1, seed=70 + k) for k in range(10)]
    got = {}
    s = F.Solver(p, n_instances=3, window=200.0, local_iters=4)

    def keep(j, inst):
        got[j] = s.download(inst=inst)[0]

    stream_solve(s, sets, on_map=keep)
    s.close()
    assert sorted(got) == list(range(10))
    for j in (0, 4, 9):
        one = F.Solver(p, n_instances=1, window=200.0, local_iters=4)
        one.seed(sets[j], 0.0)
        one.run()
        ref = one.download()[0]
        one.close()
        assert np.array_equal(got[j], ref), j
    ref, _ = O.fim_solve(om, sets[9], variant=O.LOCAL_EXACT)
    _check_fp32(got[9], ref)
    # an instance with queued work cannot be recycled
    s = F.Solver(p, n_instances=2, window=200.0)
    s.seed(sets[0], 0.0, inst=0)
    with pytest.raises(F.FimError):
        s.recycle([0])
    s.close()


def test_converge_deterministic_and_batched():
    cfg = cases.scaled(cases.SLAB, 8)
    m, om = cases.box(cfg, seed=7)
    p = F.Pack(m, F.PART_RCB, max_nn=256, seed=7)
    srcs = [cases.pacing_sites(cfg, k + 1, seed=100 + k) for k in range(4)]
    singles = [_converge(m, p, s)[0] for s in srcs]
    again = _converge(m, p, srcs[0])[0]
    assert np.array_equal(singles[0], again)  # run-to-run bitwise
    b = F.Solver(p, n_instances=4)
    for i, s in enumerate(srcs):
        b.seed(s, 0.0, inst=i)
    b.run()
    for i in range(4):
        phi, _ = b.download(inst=i)
        assert np.array_equal(phi, singles[i])  # batching changes nothing
    b.close()


@pytest.mark.parametrize("unit", [1, 3, 16])
@pytest.mark.parametrize("grid", [0, 8, 13])
def test_converge_work_units_and_grid_change_nothing(unit, grid):
    """work units of 1..16 instances, dealt to grids of 8, 13 or all
    workgroups, give bitwise the same maps (12 instances, uneven buckets)"""
    cfg = cases.scaled(cases.SLAB, 8)
    m, _ = cases.box(cfg, seed=9)
    p = F.Pack(m, F.PART_RCB, max_nn=256, seed=9)
    srcs = [cases.pacing_sites(cfg, 1 + k % 3, seed=200 + k) for k in range(12)]

    def solve(**kw):
        s = F.Solver(p, n_instances=12, window=500.0, **kw)
        for i, src in enumerate(srcs):
            s.seed(src, 0.0, inst=i)
        s.run()
        out = [s.download(inst=i)[0] for i in range(12)]
        s.close()
        return out

    base = solve(unit=4)
    for a, b in zip(base, solve(unit=unit, grid=grid)):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("block,max_nn", [(256, 300), (512, 300), (512, 1500)])
def test_few_submesh_variant_agrees(block, max_nn):
    """a list of at most one unit per submesh runs the variant that works on
    two rounds of pairs at a time; waves=8 asks for the other: bitwise the same
    maps"""
    cfg = cases.scaled(cases.SLAB, 5)
    m, _ = cases.box(cfg, seed=4)
    p = F.Pack(m, F.PART_RCB, max_nn=max_nn, seed=4)
    src = cases.pacing_sites(cfg, 3, seed=41)
    maps = [_converge(m, p, src, block=block, waves=w, window=1500.0)[0] for w in (0, 8)]
    assert np.array_equal(maps[0], maps[1])


@pytest.mark.parametrize("n", [14, 20, 60, 240])
def test_vertices_of_many_elements(n):
    """a fan of tets around one vertex, and each of them split once: 24, 36,
    116 and 476 elements at the centre (below and above the 32 ids that a copy
    keeps in a row), against the FP64 oracle"""
    from scipy.spatial import ConvexHull
    rng = np.random.default_rng(n)
    x = rng.normal(size=(n, 3))
    x *= 5000.0 / np.linalg.norm(x, axis=1, keepdims=True)
    tri = ConvexHull(x).simplices
    out = 2.0 * x
    xyz = np.concatenate([[[0.0, 0.0, 0.0]], x, out])
    e2n = [[0, 1 + a, 1 + b, 1 + c] for a, b, c in tri]
    for t in tri:  # the prism outside each face, split along ascending ids
        a, b, c = sorted(int(v) for v in t)
        A, B, C = 1 + n + a, 1 + n + b, 1 + n + c
        e2n += [[1 + a, 1 + b, 1 + c, C], [1 + a, 1 + b, B, C], [1 + a, A, B, C]]
    e2n = np.array(e2n)
    m = F.Mesh.from_arrays(xyz, e2n)
    xyz, e2n, _ = m.arrays()
    fib, vel = m.material()
    om = O.Mesh(xyz, e2n, fib=fib, vel=vel)
    for src in ([n + 1], [0]):
        phi, _, _, _, _ = _converge(m, F.Pack(m, F.PART_RCB, max_nn=4096, seed=1), src)
        ref, _ = O.fim_solve(om, src, variant=O.LOCAL_EXACT)
        _check_fp32(phi, ref)


@pytest.mark.parametrize("n_inst,unit", [(1, 0), (3, 4), (5, 2)])
def test_interrupted_runs_change_nothing(n_inst, unit):
    """a run stopped after a few iterations, with pushes on their way to the
    copies of other submeshes, then looked at (residual, support), resumed,
    reset or given a new field: bitwise the maps of uninterrupted solves (one
    work unit per bucket, and several)"""
    cfg = cases.scaled(cases.SLAB, 8)
    m, _ = cases.box(cfg, seed=9)
    p = F.Pack(m, F.PART_RCB, max_nn=200, seed=9)
    srcs = [cases.pacing_sites(cfg, 1 + k % 3, seed=500 + k) for k in range(n_inst)]
    s = F.Solver(p, n_instances=n_inst, window=500.0, unit=unit, graph_iters=3)

    def seed():
        s.reset()
        s.seed_batch(srcs, 0.0)

    def maps():
        return [s.download(inst=i)[0] for i in range(n_inst)]

    seed()
    s.run()
    base = maps()
    seed()
    left = 1
    for k in range(1000):
        left = s.advance(3, reset_stats=k == 0)
        if k % 2:
            assert s.residual(inst=k % n_inst) >= 0.0 and s.support(inst=0) >= 0.0
        if left == 0:
            break
    assert left == 0
    for a, b in zip(base, maps()):
        assert np.array_equal(a, b)
    assert all(s.residual(inst=i) <= 1e-5 for i in range(n_inst))
    # reset in the middle of a run leaves nothing behind
    seed()
    assert s.advance(6, reset_stats=True) > 0
    seed()
    s.run()
    for a, b in zip(base, maps()):
        assert np.array_equal(a, b)
    # a field given in the middle of a run is what is solved from (its window
    # is further on then: the fixed point, not the last bits)
    up = (base[0] + 3000.0).astype(np.float32)
    up[srcs[0]] = 0.0
    s.reset()
    s.init_field(up, inst=0)
    s.run()
    warm = s.download(inst=0)[0]
    seed()
    assert s.advance(6, reset_stats=True) > 0
    s.init_field(up, inst=0)
    s.run()
    assert np.max(np.abs(s.download(inst=0)[0] - warm)) <= 1e-4 * warm.max()
    for a, b in zip(base[1:], maps()[1:]):
        assert np.array_equal(a, b)
    s.close()


def test_run_multi_contexts_change_nothing():
    """12 instances at their own windows, solved by one context and by three
    contexts of 5 + 4 + 3 instances run together (fim_run_multi, one host
    thread feeding three streams): bitwise the same maps, so the oracle pins
    of the single context carry over"""
    cfg = cases.scaled(cases.SLAB, 8)
    m, _ = cases.box(cfg, seed=9)
    p = F.Pack(m, F.PART_RCB, max_nn=256, seed=9)
    srcs = [cases.pacing_sites(cfg, 1 + k % 3, seed=300 + k) for k in range(12)]
    wins = [250.0 + 75.0 * k for k in range(12)]
    one = F.Solver(p, n_instances=12, window=500.0)
    for i, src in enumerate(srcs):
        one.set_window(wins[i], inst=i)
        one.seed(src, 0.0, inst=i)
    one.run()
    base = [one.download(inst=i)[0] for i in range(12)]
    iters_one = one.stats()["global_iters"]
    one.close()
    g = F.SolverGroup([F.Solver(p, n_instances=n, window=500.0) for n in (5, 4, 3)])
    for ctx, a, b in g.parts(12):
        for i in range(a, b):
            ctx.set_window(wins[i], inst=i - a)
            ctx.seed(srcs[i], 0.0, inst=i - a)
    its = F.run_many(g.solvers)
    assert len(its) == 3 and max(its) <= iters_one and all(k > 0 for k in its)
    for i in range(12):
        assert np.array_equal(g.download(inst=i)[0], base[i])
    # a second run of the same group after a reset gives the same maps again
    for ctx, a, b in g.parts(12):
        ctx.reset()
        for i in range(a, b):
            ctx.seed(srcs[i], 0.0, inst=i - a)
    g.run()
    for i in range(12):
        assert np.array_equal(g.download(inst=i)[0], base[i])
    g.close()
    # profile mode (direct launches, every compute launch event-timed)
    g = F.SolverGroup([F.Solver(p, n_instances=n, window=500.0, profile=True) for n in (6, 6)])
    for ctx, a, b in g.parts(12):
        for i in range(a, b):
            ctx.set_window(wins[i], inst=i - a)
            ctx.seed(srcs[i], 0.0, inst=i - a)
    g.run()
    st = g.stats()
    assert st["compute_launches"] > 0 and st["compute_ms"] > 0.0
    for i in range(12):
        assert np.array_equal(g.download(inst=i)[0], base[i])
    g.close()


def test_run_multi_rejects_bad_context_lists():
    cfg = cases.scaled(cases.SLAB, 8)
    m, _ = cases.box(cfg, seed=9)
    p = F.Pack(m, F.PART_RCB, max_nn=256, seed=9)
    a = F.Solver(p, n_instances=1)
    c = F.Solver(p, mode=F.MODE_COMPAT)
    with pytest.raises(F.FimError, match="listed twice"):
        F.run_many([a, a])
    with pytest.raises(F.FimError, match="converge mode"):
        F.run_many([a, c])
    with pytest.raises(F.FimError, match="max_iters"):
        F.run_many([a], max_iters=0)
    # an iteration cap below what the solve needs ends every context's run
    # and reports FIM_ENOCONV; a later run finishes the maps
    b = F.Solver(p, n_instances=1, window=500.0)
    b.seed(cases.pacing_sites(cfg, 1, seed=301), 0.0)
    with pytest.raises(F.FimError, match="iteration cap"):
        F.run_many([b], max_iters=1)
    assert b.stats()["global_iters"] >= 1
    F.run_many([b])
    b.close()
    a.close()
    c.close()


@pytest.mark.parametrize("staged", [False, True])
@pytest.mark.parametrize("window", [300.0, 1000.0, 4000.0])
def test_converge_time_window_same_fixed_point(window, staged):
    """the per-iteration time window changes the processing order only"""
    cfg = cases.scaled(cases.SLAB, 4)
    m, om = cases.box(cfg, seed=2)
    p = F.Pack(m, F.PART_RCB, max_nn=512, seed=2)
    src = cases.pacing_sites(cfg, 5, seed=2)
    phi, st, it, res, stats = _converge(m, p, src, window=window, staged=staged)
    ref, _ = O.fim_solve(om, src, variant=O.LOCAL_EXACT)
    _check_fp32(phi, ref)
    assert res < 1e-5


def test_per_instance_windows_same_fixed_point():
    """fim_set_window: four instances of one batch with windows 0 (plain FIM
    order), 0.5, 1 and 4 ms reach the oracle's fixed point, and each equals
    the same solve run alone with that window as the context's, bit for bit"""
    cfg = cases.scaled(cases.SLAB, 4)
    m, om = cases.box(cfg, seed=2)
    p = F.Pack(m, F.PART_RCB, max_nn=512, seed=2)
    src = cases.pacing_sites(cfg, 5, seed=2)
    wins = (0.0, 500.0, 1000.0, 4000.0)
    s = F.Solver(p, n_instances=len(wins), window=1000.0)
    for i, w in enumerate(wins):
        s.set_window(w, inst=i)
        s.seed(src, 0.0, inst=i)
    s.run()
    maps = [s.download(inst=i)[0] for i in range(len(wins))]
    with pytest.raises(F.FimError):
        s.set_window(-1.0, inst=0)
    s.close()
    ref, _ = O.fim_solve(om, src, variant=O.LOCAL_EXACT)
    for i, w in enumerate(wins):
        _check_fp32(maps[i], ref)
        one, *_ = _converge(m, p, src, window=w)
        assert np.array_equal(one, maps[i]), w


def test_warm_start_from_upper_bound_reaches_same_fixed_point():
    """init_field with every vertex active: an upper bound (oracle + 5 %)
    converges to the cold-start fixed point"""
    cfg = cases.scaled(cases.SLAB, 8)
    m, om = cases.box(cfg, seed=9)
    p = F.Pack(m, F.PART_RCB, max_nn=256, seed=9)
    src = cases.pacing_sites(cfg, 2, seed=9)
    cold, *_ = _converge(m, p, src)
    ref, _ = O.fim_solve(om, src, variant=O.LOCAL_EXACT)
    s = F.Solver(p)
    s.seed(src, 0.0)
    s.init_field((ref * 1.05 + 100.0).astype(np.float32))
    s.seed(src, 0.0)
    s.run()
    warm, _ = s.download()
    s.close()
    _check_fp32(warm, ref)
    assert np.max(np.abs(warm - cold)) <= 1e-4 * ref.max()


def test_regional_scaling_equals_scaled_mesh():
    """one instance with all four regional factors s equals the mesh with
    both speeds multiplied by s (times divide by s)"""
    cfg = cases.scaled(cases.CUBE, 4)
    m, om = cases.box(cfg, seed=4)
    p = F.Pack(m, F.PART_RCB, max_nn=128, seed=4)
    s = F.Solver(p, n_instances=2)
    s.seed([0], 0.0, inst=0)
    s.seed([0], 0.0, inst=1)
    s.set_scaling(np.full(4, 1.25, np.float32), inst=1)
    s.run()
    a, _ = s.download(inst=0)
    b, _ = s.download(inst=1)
    s.close()
    fin = a < 1e50
    assert np.allclose(b[fin] * 1.25, a[fin], rtol=2e-6, atol=1e-3)


def test_multi_mesh_batch_with_regional_scalings():
    """one batch over a union of four meshes (cube + three slabs, reduced),
    each instance paced on one component with four quadrant speed factors;
    each map equals the oracle's fixed point on the union mesh with every
    element's speeds multiplied by its region's factor"""
    from fimpy import workloads as W
    parts = [(n, cases.scaled(c, 3)) for n, c in W.MULTI]
    m, offs, cfgs = W.multi_mesh(parts, 7)
    solves = W.multi_solves(cfgs, offs, 8, 11)
    p = F.Pack(m, F.PART_RCB, max_nn=512, seed=7)
    s = F.Solver(p, n_instances=len(solves), window=1000.0)
    for i, sv in enumerate(solves):
        s.seed(sv["sites"], 0.0, inst=i)
        s.set_scaling(sv["scale"], inst=i)
    s.run()
    xyz, e2n, _ = m.arrays()
    fib, vel = m.material()
    reg = np.concatenate([W.quadrant_regions(F.Mesh.gen_box(seed=7 + k, **c))
                          for k, (_, c) in enumerate(parts)])
    bounds = offs + [m.nn]
    for i, sv in enumerate(solves):
        phi, _ = s.download(inst=i)
        om = O.Mesh(xyz, e2n, fib=fib, vel=vel * sv["scale"].astype(np.float64)[reg][:, None])
        ref, _ = O.fim_solve(om, sv["sites"], variant=O.LOCAL_EXACT)
        _check_fp32(phi, ref)
        k = sv["part"]
        reached = np.flatnonzero(ref < 1e50)
        assert reached.min() >= bounds[k] and reached.max() < bounds[k + 1]
    s.close()


def test_scarred_shell_vs_fp64_oracle():
    """prolate shell with twelve slow scars at the 1M-tet resolution the
    large workload is checked at, three pacing sites on the inner surface"""
    from fimpy import workloads as W
    m = W.shell(1, h=850.0)
    xyz, e2n, _ = m.arrays()
    fib, vel = m.material()
    om = O.Mesh(xyz, e2n, fib=fib, vel=vel)
    p = F.Pack(m, F.PART_RCB, max_nn=1024, seed=1)
    sites = W.inner_surface_sites(m, 3, 5)
    phi, st, it, res, stats = _converge(m, p, sites, window=2000.0)
    ref, _ = O.fim_solve(om, sites, variant=O.LOCAL_EXACT)
    _check_fp32(phi, ref)


def test_compat_timed_events_two_beats_bit_identical():
    """multi-beat pacing with events fired in the window holding their start
    time (re-entry through tail -> far): GPU compat mode equals the oracle's
    timed restatement bit for bit"""
    cfg = cases.scaled(cases.CUBE, 2)
    m, om = cases.box(cfg, seed=3)
    p = F.Pack(m, F.PART_RCB, max_nn=128, seed=3)
    e2s, _ = p.partition()
    om = O.Mesh(om.xyz, om.e2n, fib=om.fib, vel=om.vel, atags=e2s.astype(np.int32))
    dt, apd, steps = 10e3, 50e3, 18
    stims = [(1, 0.0, [0]), (1, 120e3, [0]), (1, 125e3, [1330])]
    s = F.Solver(p, mode=F.MODE_COMPAT, local=F.LOCAL_REF, apd=apd)
    fw = m.front_width()
    s.reset()
    cur = 0.0
    for _ in range(steps):
        ps = cur
        cur += dt
        for active, tstart, vtx in stims:
            if active and ps <= tstart < cur:
                s.seed(vtx, tstart)
        s.step(ps, cur, dt, fw)
    phi, st = s.download()
    s.close()
    ophi, ost, _ = O.compat_solve(om, stims, dt, steps, apd=apd, front_width=fw, timed=True)
    assert np.array_equal(st, ost)
    assert np.array_equal(phi, ophi)


def test_converge_edge_cases():
    """a seed time shifts the map; an unreached component stays unreached;
    an iteration cap reports FIM_ENOCONV and a further run finishes the
    same map"""
    from fimpy import workloads as W
    cfg = cases.scaled(cases.SLAB, 8)
    a = F.Mesh.gen_box(seed=1, **cfg)
    b = F.Mesh.gen_box(seed=2, **cases.scaled(cases.CUBE, 4))
    u = F.Mesh.concat([a, b])
    p = F.Pack(u, F.PART_RCB, max_nn=256, seed=1)
    src = cases.pacing_sites(cfg, 2, seed=3)
    s = F.Solver(p, n_instances=3, window=1000.0)
    s.seed(src, 0.0, inst=0)
    s.seed(src, 5000.0, inst=1)
    s.run()
    p0, _ = s.download(inst=0)
    p1, _ = s.download(inst=1)
    p2, st2 = s.download(inst=2)  # never seeded
    fin = p0 < 1e50
    assert np.array_equal(np.flatnonzero(fin), np.arange(a.nn))  # only the first component
    assert np.allclose(p1[fin], p0[fin] + 5000.0, rtol=0, atol=1e-4 * p0[fin].max())
    assert np.all(p2 >= 1e50) and np.all(st2 == F.FAR)
    # iteration cap, then completion
    s.reset()
    s.seed(src, 0.0, inst=0)
    with pytest.raises(F.FimError, match="FIM_ENOCONV"):
        s.run(max_iters=3)
    s.run()
    again, _ = s.download(inst=0)
    assert np.array_equal(again, p0)
    s.close()


@pytest.mark.parametrize("n", [1, 2, 5, 9])
@pytest.mark.parametrize("n_inst", [1, 3])
def test_reset_leaves_nothing(n, n_inst):
    """a reset after a run, at array lengths of every remainder by the 16-byte
    fills: every vertex FAR, the counters of a run start at zero, the factors
    set in between take effect, and the next run gives the maps of a context
    that had none before"""
    cfg = dict(cases.CUBE, nx=n, ny=n, nz=n + 1)
    m = F.Mesh.gen_box(seed=3, **cfg)
    p = F.Pack(m, F.PART_RCB, max_nn=64, seed=3)
    far = np.finfo(np.float64).max

    def run(s):
        for i in range(n_inst):
            s.set_scaling([1.0 + 0.25 * i] * 4, inst=i)
            s.seed([i % m.nn], 0.0, inst=i)
        s.run()
        return [s.download(inst=i)[0] for i in range(n_inst)], s.stats()["activations"]

    s = F.Solver(p, n_instances=n_inst, window=0.0)
    want, acts = run(s)
    for i in range(n_inst):
        s.set_scaling([3.0] * 4, inst=i)
        s.seed([m.nn - 1], 0.0, inst=i)
    s.run()
    s.reset()
    for i in range(n_inst):
        phi, st = s.download(inst=i)
        assert (phi == far).all() and (st == 0).all()
    got, again = run(s)
    assert again == acts and all(np.array_equal(a, b) for a, b in zip(got, want))
    s.close()
    c = F.Solver(p, mode=F.MODE_COMPAT)
    steps = []
    for _ in range(2):
        c.seed([0], 0.0)
        steps.append([c.step(0.0, 2000.0, 2000.0, 1e6), *c.download()])
        c.reset()
        phi, st = c.download()
        assert (phi == far).all() and (st == 0).all()
    assert steps[0][0] == steps[1][0] and all(np.array_equal(a, b) for a, b in zip(steps[0][1:], steps[1][1:]))
    c.close()


ITER_END = 2 ** 30 - 2  # iteration numbers stay below (csrc/solver.hip, kIterEnd)


@pytest.mark.parametrize("n_inst,unit", [(1, 0), (5, 2)])
@pytest.mark.parametrize("before", [4, 5, 10, 31])
def test_iteration_numbers_start_over(n_inst, unit, before):
    """a context whose iteration numbers run out `before` iterations later (it
    has never been reset): runs with work queued and pushes on their way, a
    recycled instance and later runs give bitwise the maps and activations of
    a context that counts from 0"""
    cfg = cases.scaled(cases.SLAB, 8)
    m, _ = cases.box(cfg, seed=9)
    p = F.Pack(m, F.PART_RCB, max_nn=200, seed=9)
    srcs = [cases.pacing_sites(cfg, 1 + k % 3, seed=500 + k) for k in range(n_inst)]

    def solves(number):
        s = F.Solver(p, n_instances=n_inst, window=500.0, unit=unit, graph_iters=3)
        if number is not None:
            assert F.lib().fim_ctx_renumber(s.h, number) == 0
        out, counts = [], []
        s.seed_batch(srcs, 0.0)
        for k in range(1000):
            if s.advance(3, reset_stats=k == 0) == 0:
                break
        out += [s.download(inst=i)[0] for i in range(n_inst)]
        counts.append(s.stats()["activations"])
        assert not np.any(s.active())
        for beat in range(2):
            s.recycle([0])
            s.seed(srcs[0][:1], 0.0)
            s.run()
            out.append(s.download()[0])
            counts.append(s.stats()["activations"])
        s.close()
        return out, counts

    want, n = solves(None)
    got, k = solves(ITER_END - before)
    for a, b in zip(want, got):
        assert np.all(b < 1e30)
        assert np.array_equal(a, b)
    assert n == k


@pytest.mark.parametrize("max_nn", [128, 700])
@pytest.mark.parametrize("before", [1, 2, 3, 7, 12])
def test_window_numbers_start_over(max_nn, before):
    """a context that has worked through 2^32 windows but `before`, in the
    middle of a map (submeshes listed, shared vertices to be merged): bitwise
    the times and states, and the pending copies after every window, of a
    context that counts from 0"""
    cfg = dict(cases.SLAB, nx=17, ny=13, nz=5, lx=17e3, ly=13e3, lz=5e3)
    m, _ = cases.box(cfg, seed=5)
    p = F.Pack(m, F.PART_RCB, max_nn=max_nn, seed=3)
    fw, dt = m.front_width(), 2e3

    def windows(number):
        s = F.Solver(p, mode=F.MODE_COMPAT, local=F.LOCAL_REF, apd=20e3)
        s.seed([0, 700], 0.0)
        left = [s.step(0.0, dt, dt, fw)]
        if number is not None:
            assert F.lib().fim_ctx_renumber(s.h, C.c_uint32(number)) == 0
        left += [s.step(k * dt, (k + 1) * dt, dt, fw) for k in range(1, 20)]
        phi, st = s.download()
        s.close()
        return phi, st, left

    want, got = windows(None), windows(2 ** 32 - before)
    assert max(want[2][8:]) > 0
    assert want[2] == got[2]
    assert np.array_equal(want[0], got[0]) and np.array_equal(want[1], got[1])


@pytest.mark.parametrize("block", [64, 128, 256, 512])
def test_algorithmic_bytes_of_a_large_submesh(block):
    """one submesh of 63,888 elements, all of them evaluated: 32 B each and
    10 B a copy, whatever the workgroup's size (with 64 threads a lane adds up
    to 1,024 of the evaluated elements' bits, with 128 up to 512)"""
    m = F.Mesh.gen_box(seed=4, **dict(cases.CUBE, nx=22, ny=22, nz=22))
    p = F.Pack(m, F.PART_RCB, max_nn=16000, max_ne=65535, seed=4)
    assert p.info["nsub"] == 1 and p.info["ne_global"] == 63888
    s = F.Solver(p, block=block)
    s.seed([0], 0.0)
    s.run()
    st = s.stats()
    s.close()
    assert st["alg_bytes"] == st["activations"] * (32 * 63888 + 10 * p.info["nn_global"])


def test_contexts_made_at_once_share_a_pack():
    """the element bounds that contexts of a pack share are worked out by
    the first of them: four threads making contexts of a fresh pack at once
    get the maps of one made alone"""
    import threading
    cfg = cases.scaled(cases.SLAB, 8)
    m, _ = cases.box(cfg, seed=9)
    src = cases.pacing_sites(cfg, 2, seed=9)
    want = _converge(m, F.Pack(m, F.PART_RCB, max_nn=300, seed=9), src)[0]
    p = F.Pack(m, F.PART_RCB, max_nn=300, seed=9)
    got, gate = [None] * 4, threading.Barrier(4)

    def work(i):
        gate.wait()
        got[i] = _converge(m, p, src)[0]

    ts = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    for g in got:
        assert g is not None and np.array_equal(g, want)


def test_contexts_come_and_go_while_others_run():
    """distinct contexts are independent: threads that create a context, build
    its graph in the first run and destroy it, again and again, beside each
    other get the maps of one context alone"""
    import threading
    cfg = cases.scaled(cases.SLAB, 8)
    m, _ = cases.box(cfg, seed=9)
    src = cases.pacing_sites(cfg, 2, seed=9)
    p = F.Pack(m, F.PART_RCB, max_nn=300, seed=9)
    want = _converge(m, p, src)[0]
    bad, gate = [], threading.Barrier(6)

    def work(i):
        gate.wait()
        try:
            for k in range(12):
                n = 1 + (i + k) % 4  # with and without a plan kernel
                if not np.array_equal(_converge(m, p, src, n_instances=n)[0], want):
                    bad.append((i, k, n))
        except F.FimError as e:
            bad.append((i, str(e)))

    ts = [threading.Thread(target=work, args=(i,)) for i in range(6)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad, bad


def test_device_memory_of_a_context_is_what_its_kernels_read():
    """an unstaged context keeps 81 B an element (node ids 8, region 1,
    geometry 24, record 48), 89 B a copy (ids 12, time 4, flag 1, adjacency 68,
    vertex offsets at most 4), 60 B and twice 4 an interface copy: no heights,
    which only the staged kernel reads.  8 MB for rounding and the rest, half
    of what the heights of this mesh's 1.57 M elements take."""
    def free():  # of the HIP runtime that the library is linked with
        f, total = C.c_size_t(), C.c_size_t()
        assert F.lib().hipMemGetInfo(C.byref(f), C.byref(total)) == 0
        return f.value

    m = F.Mesh.gen_box(seed=1, **dict(cases.CUBE, nx=64, ny=64, nz=64))
    p = F.Pack(m, F.PART_RCB, max_nn=2816, seed=1)
    F.Solver(p).close()  # what the first context of a process brings
    before = free()
    s = F.Solver(p)
    used = before - free()
    s.close()
    i = p.info
    need = 81 * i["ne_global"] + 89 * i["ncopy"] + 68 * i["n_iface_copies"]
    assert used <= need + (8 << 20), (used, need)


@pytest.mark.parametrize("block,max_nn", [(256, 150), (256, 450), (512, 40), (512, 320), (512, 900), (512, 1300)])
def test_lists_of_few_waves_change_nothing(block, max_nn):
    """sweeps listed by few waves (a grid that the units fill, small submeshes)
    and by all waves (a grid that they do not): bitwise the same maps, on
    submeshes below, between and above the two sizes per wave, at one and at
    several instances a unit, and within the oracle's tolerance"""
    cfg = cases.scaled(cases.SLAB, 4)
    m, om = cases.box(cfg, seed=6)
    p = F.Pack(m, F.PART_RCB, max_nn=max_nn, seed=6)
    n_inst = 7
    srcs = [cases.pacing_sites(cfg, 1 + k % 3, seed=40 + k) for k in range(n_inst)]
    maps = []
    for grid, unit in ((16, 1), (16, 3), (65536, 1), (0, 2)):
        s = F.Solver(p, n_instances=n_inst, block=block, grid=grid, unit=unit, window=2000.0, local_iters=3)
        s.seed_batch(srcs, 0.0)
        s.run()
        maps.append([s.download(inst=i)[0] for i in range(n_inst)])
        s.close()
    for got in maps[1:]:
        for a, b in zip(maps[0], got):
            assert np.array_equal(a, b)
    ref, _ = O.fim_solve(om, srcs[0], variant=O.LOCAL_EXACT)
    _check_fp32(maps[0][0], ref)

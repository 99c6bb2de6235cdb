"""Test harness: parity cases run against the CPU-emulated build of libsmokesim
(tests/emu/Makefile) under AddressSanitizer, compared bit for bit with the
FP32 oracle.  Run as a child process with the ASan runtime preloaded:

    python emu_cases.py <path to libsmokesim_emu.so> [case ...]

Every kernel access is checked against its allocation, so an out-of-bounds
index shows up here, on the CPU, with a stack trace.  Prints "ok <case>" per
case and exits non-zero on the first failure."""
import os
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(os.path.dirname(HERE))
sys.path[:0] = [os.path.join(ROOT, "smoke-simulation_amd"), os.path.join(ROOT, "tests"),
                os.path.join(ROOT, "oracle"), ROOT]

import numpy as np  # noqa: E402

import smokesim  # noqa: E402
from helpers import assert_bitwise_equal, gpu_for, oracle_for  # noqa: E402
from smokesim import scenes  # noqa: E402


def same_bits(a, b, what):
    assert np.array_equal(np.ascontiguousarray(a).view(np.uint32),
                          np.ascontiguousarray(b, dtype=np.float32).view(np.uint32)), what


def case_single():
    for proj, its, dims, seed in [(0, 6, (15, 13, 11), 1), (1, 5, (12, 16, 9), 2),
                                  (2, 9, (17, 11, 13), 3)]:
        sc = scenes.test_scene(dims, seed=seed, projection=proj, iterations=its)
        g, o = gpu_for(sc), oracle_for(sc, 32)
        for _ in range(2):
            g.step(sc["dt"], readback=False)
        o.step(sc["dt"], 2)
        assert_bitwise_equal(g.state(), o.state(), f"single p{proj}")
        g.close()


def case_plans():
    sc = scenes.test_scene((19, 14, 12), seed=4, projection=2, iterations=7)
    o = oracle_for(sc, 32)
    o.step(sc["dt"], 1)
    for t, tile, zc in [(3, 1, 7), (6, 0, 4), (2, 1, 64), (6, 2, 5), (4, 3, 9), (5, 2, 64)]:
        g = gpu_for(sc)
        g.set_jacobi_plan(sweeps_per_launch=t, tile=tile, zc=zc)
        g.step(sc["dt"], readback=False)
        assert_bitwise_equal(g.state(), o.state(), f"plan {(t, tile, zc)}")
        g.close()


def case_batch():
    dims = [(13, 11, 9), (9, 15, 12), (16, 8, 10)]
    scs = []
    for k, d in enumerate(dims):
        sc = scenes.test_scene(d, seed=20 + k, projection=2, iterations=6, n_sources=1 + k % 2,
                               n_obstacles=k % 2)
        sc["dt"] = 0.03 + 0.01 * k
        scs.append(sc)
    for plan in (None, (5, 2, 4), (3, 3, 64)):
        sims = [gpu_for(sc) for sc in scs]
        with smokesim.Batch(sims, [sc["dt"] for sc in scs]) as b:
            if plan:
                b.set_jacobi_plan(sweeps_per_launch=plan[0], tile=plan[1], zc=plan[2])
            b.step(use_graph=False)
            for _ in range(2):
                b.step(use_graph=True)
            b.synchronize()
            states = [s.state() for s in sims]
        for sc, st in zip(scs, states):
            o = oracle_for(sc, 32)
            o.step(sc["dt"], 3)
            assert_bitwise_equal(st, o.state(), f"batch {sc['name']} plan {plan}")
        for s in sims:
            s.close()


def _req(dims, seed, dt, its=6):
    sc = scenes.test_scene(dims, seed=seed, projection=2, iterations=its, n_sources=2,
                           n_obstacles=1)
    sc["dt"] = dt
    return sc


def _drain(srv):
    for _ in range(200):
        a, q = srv.tick()
        if a == 0 and q == 0:
            return
    raise AssertionError("server did not drain")


def case_server():
    a = _req((14, 12, 10), 60, 0.05)
    others = [(_req((16, 10, 13), 61, 0.03), 5), (_req((9, 15, 8), 62, 0.07), 2),
              (_req((12, 12, 12), 63, 0.04), 3)]
    alone = smokesim.Server(1 << 30, 6)
    ia = alone.submit(a, 4)
    _drain(alone)
    _, d_alone, _, _ = alone.result(ia)
    alone.close()
    mix = smokesim.Server(1 << 30, 6)
    ids = [mix.submit(others[0][0], others[0][1]), mix.submit(others[1][0], others[1][1])]
    mix.tick()
    ia2 = mix.submit(a, 4)           # arrives while others run
    mix.tick()
    ids.append(mix.submit(others[2][0], others[2][1]))
    _drain(mix)
    _, d_mix, _, _ = mix.result(ia2)
    same_bits(d_mix, d_alone, "server: alone vs mix")
    o = oracle_for(a, 32)
    o.step(a["dt"], 4)
    same_bits(d_mix, o.output_density(), "server: mix vs oracle")
    for rid, (sc, steps) in zip(ids, others):
        _, d, _, _ = mix.result(rid)
        o = oracle_for(sc, 32)
        o.step(sc["dt"], steps)
        same_bits(d, o.output_density(), f"server: {sc['name']}")
    s = mix.stats()
    assert s["completed"] == 4 and s["hbm_used"] == 0, s
    ms, nreq = mix.tick_ms()
    assert len(ms) == s["ticks"] and nreq.max() == 3, (len(ms), s["ticks"], nreq)
    mix.close()
    # admission under a budget that holds two requests
    fp = smokesim.footprint_bytes(12, 12, 12)
    srv = smokesim.Server(int(2.5 * fp), 6)
    scs = [_req((12, 12, 12), 70 + k, 0.05) for k in range(4)]
    rids = [srv.submit(sc, 2) for sc in scs]
    assert srv.tick() == (2, 2)
    _drain(srv)
    st = srv.stats()
    assert st["completed"] == 4 and st["hbm_peak"] <= st["hbm_budget"], st
    for rid, sc in zip(rids, scs):
        _, d, _, _ = srv.result(rid)
        o = oracle_for(sc, 32)
        o.step(sc["dt"], 2)
        same_bits(d, o.output_density(), f"budgeted {sc['name']}")
    srv.close()


def case_step_graph():
    # Steps replayed from a captured graph give the eager bits, through
    # changes that force a new capture (moved objects, parameters, dt).
    for proj, its, plan in ((0, 3, None), (2, 5, (2, 0, 64))):
        sc = scenes.test_scene((14, 12, 10), seed=34, projection=proj, iterations=its,
                               n_sources=1, n_obstacles=1)
        sims = [gpu_for(sc), gpu_for(sc)]
        sims[1].set_step_graph(True)
        if plan:
            for g in sims:
                g.set_jacobi_plan(sweeps_per_launch=plan[0], tile=plan[1], zc=plan[2])
        dt = sc["dt"]
        for k in range(4):
            if k == 1:
                for g in sims:
                    g.move_object(0, 7.0, 5.0, 4.0)
                    g.move_object(1, 6.0, 3.0, 5.0)
            if k == 2:
                for g in sims:
                    g.set_params(iterations=its + 2)
                dt = sc["dt"] * 0.5
            outs = [g.step(dt) for g in sims]
            same_bits(outs[1], outs[0], f"graph step {k} projection {proj}")
        assert_bitwise_equal(sims[1].state(), sims[0].state(), f"graph projection {proj}")
        for g in sims:
            g.close()


def case_readback():
    sc = scenes.test_scene((13, 12, 11), seed=5, projection=2, iterations=5)
    g = gpu_for(sc)
    for k in range(3):
        g.step_async(sc["dt"])
        g.readback_begin(smokesim.READBACK_F32)
        host, step = g.readback_wait()
        assert step == k + 1
        same_bits(host, g.read_density(), "readback f32")
    g.close()


def _rel_l2(a, b):
    a = np.asarray(a, dtype=np.float64)
    b = np.asarray(b, dtype=np.float64)
    n = np.linalg.norm(b)
    return float(np.linalg.norm(a - b) / n) if n > 0 else float(np.linalg.norm(a))


def case_precision():
    # REFINED (FP32 and BF16 fields) against FP64 Jacobi with the same number
    # of sweeps, BF16 conversions, and the tolerance-driven loop.
    sc = scenes.test_scene((18, 14, 12), seed=7, projection=2, iterations=12)
    o = oracle_for(sc, 64)
    o.step(sc["dt"], 2)
    ref = o.state()
    for storage in (smokesim.STORAGE_FP32, smokesim.STORAGE_BF16, smokesim.STORAGE_FP16,
                    smokesim.STORAGE_FP16_VELOCITY):
        g = gpu_for(sc, storage=storage)
        g.set_params(projection=smokesim.PROJ_REFINED, inner_sweeps=6, iterations=12)
        for _ in range(2):
            g.step(sc["dt"], readback=False)
        st = g.state()
        rel, nref = g.solve_info()
        assert nref == 2 and 0.0 < rel < 1.0, (rel, nref)
        assert np.array_equal(st["flags"], ref["flags"])
        for k in ("rho0", "rho1", "u0", "u1", "v0", "v1", "w0", "w1"):
            e = _rel_l2(st[k], ref[k])
            assert e < 3e-2, (storage, k, e)
        e = _rel_l2(g.get_pressure(), o.get_pressure())
        assert e < 3e-2, (storage, "pressure", e)
        g.close()
    # BF16 round trip: stored values are the round-to-nearest-even BF16 of the input
    g = smokesim.Simulation(9, 7, 5, storage=smokesim.STORAGE_BF16)
    x = np.random.default_rng(1).standard_normal((5, 7, 9)).astype(np.float32)
    g.set_density(0, x)
    b = x.view(np.uint32).astype(np.uint64)
    rne = ((b + 0x7FFF + ((b >> 16) & 1)) >> 16 << 16).astype(np.uint32).view(np.float32)
    same_bits(g.get_density(0), rne, "bf16 store rounding")
    g.close()
    # FP16 round trip: binary16 round to nearest even (numpy's conversion)
    g = smokesim.Simulation(9, 7, 5, storage=smokesim.STORAGE_FP16)
    g.set_density(0, x)
    same_bits(g.get_density(0), x.astype(np.float16).astype(np.float32), "fp16 store rounding")
    g.close()
    # tolerance-driven refinement on a small grid
    sc = scenes.test_scene((8, 7, 6), seed=8, projection=2, iterations=10, box_fraction=0.0,
                           n_obstacles=0)
    g = gpu_for(sc)
    g.set_params(projection=smokesim.PROJ_REFINED, inner_sweeps=10, iterations=2000,
                 tolerance=1e-5)
    g.step(sc["dt"], readback=False)
    rel, nref = g.solve_info()
    assert rel <= 1e-5 and 1 <= nref < 1000, (rel, nref)
    g.close()


def case_refine_groups():
    # The refined solve's FP16 sweeps give the same bits however they are
    # grouped into fused launches (plans T = 2, 4, 6 split 10 inner sweeps as
    # 2+2+2+2+2, 4+4+2 or 6+4) and whatever the tile (one or two rows per
    # thread).
    sc = scenes.test_scene((21, 13, 11), seed=9, projection=2, iterations=20)
    states = []
    for t, tile in ((2, 0), (4, 0), (6, 0), (4, 2), (6, 3)):
        g = gpu_for(sc, storage=smokesim.STORAGE_BF16_VELOCITY)
        g.set_jacobi_plan(sweeps_per_launch=t, tile=tile, zc=5)
        g.set_params(projection=smokesim.PROJ_REFINED, inner_sweeps=10, iterations=20)
        for _ in range(2):
            g.step(sc["dt"], readback=False)
        states.append((t, g.state(), g.get_pressure()))
        g.close()
    for t, st, pr in states[1:]:
        assert_bitwise_equal(st, states[0][1], f"refined, plan T={t}")
        same_bits(pr, states[0][2], f"refined pressure, plan T={t}")


def case_proxy():
    # Proxy-plane geometry: one and two chunks of the 1024-lane workgroup,
    # through the host entry point (pinned workspace, completion mark).
    import oracle as orc
    rng = np.random.default_rng(5)
    for steps in (1, 100, 1025):
        dims = rng.integers(16, 160, 3).astype(np.float32)
        view = (np.zeros(3, np.float32), dims, rng.uniform(-300, 300, 3).astype(np.float32),
                rng.normal(size=3).astype(np.float32))
        gv, gi, gp = smokesim.proxy_geometry(*view, steps)
        ov, oi, op = orc.proxy_geometry(*view, steps)
        assert np.array_equal(gi, oi) and np.array_equal(gp, op), steps
        nan = np.isnan(ov)
        assert np.array_equal(np.isnan(gv), nan), steps
        assert np.array_equal(gv[~nan].view(np.uint32), ov[~nan].view(np.uint32)), steps


def case_vorticity():
    # Vorticity confinement after the force stage, under each projection.
    for proj, its, dims, seed in [(0, 4, (14, 12, 11), 30), (1, 4, (11, 15, 9), 31),
                                  (2, 6, (16, 10, 12), 32)]:
        sc = scenes.test_scene(dims, seed=seed, projection=proj, iterations=its, noise=0.5)
        sc["params"]["vorticity"] = 1.5
        g, o = gpu_for(sc), oracle_for(sc, 32)
        for _ in range(2):
            g.step(sc["dt"], readback=False)
        o.step(sc["dt"], 2)
        assert_bitwise_equal(g.state(), o.state(), f"vorticity p{proj}")
        g.close()


def case_advection():
    # Velocity advection tiles: grids wider than one 64-cell tile row with
    # partial tiles, and back-traces longer than the tile halo (large noise
    # and dt) next to short ones.
    for dims, seed, noise, dt in [((70, 11, 10), 40, 0.5, 0.05), ((67, 18, 9), 41, 40.0, 0.1),
                                  ((130, 9, 6), 42, 8.0, 0.3)]:
        sc = scenes.test_scene(dims, seed=seed, projection=2, iterations=4, noise=noise)
        sc["dt"] = dt
        g, o = gpu_for(sc), oracle_for(sc, 32)
        for _ in range(2):
            g.step(sc["dt"], readback=False)
        o.step(sc["dt"], 2)
        assert_bitwise_equal(g.state(), o.state(), f"advection {dims}")
        g.close()


def case_norms():
    # Step norms (two-pass fixed-order reduction with lane exchanges) against
    # the oracle's restatement on the simulation's own fields.
    import oracle as orc
    sc = scenes.test_scene((70, 9, 11), seed=12, projection=2, iterations=5, noise=0.3)
    g = gpu_for(sc)
    g.norms_enable(True)
    for _ in range(2):
        g.step(sc["dt"], readback=False)
    n = g.step_norms()
    ref = orc.step_norms(g, sc["dt"])
    for k in ("max_u", "max_v", "max_w", "max_density", "nonfinite"):
        assert n[k] == ref[k], (k, n[k], ref[k])
    for k in ("div_l2", "density_sum", "cfl"):
        assert abs(n[k] - ref[k]) <= 1e-12 * abs(ref[k]), (k, n[k], ref[k])
    assert n["rhs_l2"] > n["div_l2"]
    g.close()


class EmuDevice:
    """Device memory of the emulator, as a caller of the C ABI holds it."""

    def __init__(self, nbytes):
        import ctypes
        self.lib = smokesim.load()
        self.lib.emu_copies_into.restype = ctypes.c_longlong
        self.lib.emu_copies_into.argtypes = [ctypes.c_void_p]
        self.lib.hipFree.argtypes = [ctypes.c_void_p]
        p = ctypes.c_void_p()
        assert self.lib.hipMalloc(ctypes.byref(p), ctypes.c_size_t(nbytes)) == 0
        self.p = p
        self.floats = np.ctypeslib.as_array(ctypes.cast(p, ctypes.POINTER(ctypes.c_float)), (nbytes // 4,))

    def copies(self):
        return self.lib.emu_copies_into(self.p)

    def free(self):
        del self.floats
        assert self.lib.hipFree(self.p) == 0


def case_read_targets():
    # A blocking read into device memory is one copy by the runtime, whatever
    # its size and whatever reads into host memory came before; only plain host
    # memory is written by the CPU.
    import ctypes
    rng = np.random.default_rng(11)
    for dims in ((20, 17, 13), (40, 33, 30), (120, 100, 91)):  # 17 KB, 155 KB, 4.2 MB
        x = rng.standard_normal(dims[::-1]).astype(np.float32)
        g = smokesim.Simulation(*dims, density=x)
        for _ in range(6):
            same_bits(g.get_density(0), x, f"{dims} into host memory")
        dev = EmuDevice(x.nbytes)
        smokesim._check(g.lib.smoke_get_density(g.h, 0, ctypes.cast(dev.p, ctypes.POINTER(ctypes.c_float))))
        assert dev.copies() == 1, (dims, dev.copies())
        same_bits(dev.floats, x.ravel(), f"{dims} into device memory")
        dev.free()
        g.close()


def _emu(name, *args):
    import ctypes
    f = getattr(smokesim.load(), name)
    f.restype = ctypes.c_longlong
    return f(*[ctypes.c_size_t(a) for a in args])


def case_small_reads():
    # Reads that come to less than the pinned slots' size are the runtime's
    # copies; from then on a small read is one copy into the slots.
    rng = np.random.default_rng(12)
    for dims, n in (((40, 33, 30), 20), ((101, 100, 99), 3)):  # 155 KB, 3.8 MB
        x = rng.standard_normal(dims[::-1]).astype(np.float32)
        with smokesim.Simulation(*dims, density=x) as g:
            for _ in range(n):
                same_bits(g.get_density(0), x, f"{dims}")
    assert _emu("emu_pinned_calls") == 0
    with smokesim.Simulation(101, 100, 99, density=x) as g:
        for _ in range(6):
            same_bits(g.get_density(0), x, "with slots")
        assert _emu("emu_pinned_calls") == 1 == _emu("emu_pinned_held")
        for dims in ((20, 17, 13), (40, 33, 30), (64, 64, 33)):
            y = rng.standard_normal(dims[::-1]).astype(np.float32)
            with smokesim.Simulation(*dims, density=y) as h:
                same_bits(h.get_density(0), y, f"with slots {dims}")
    assert _emu("emu_pinned_held") == 0


def case_read_slots():
    # The pinned slots of the blocking reads: built once the reads add up to
    # their size, one set per device, kept while a simulation of the device
    # lives, and refused without harm.
    lib = smokesim.load()
    dims = (120, 100, 91)  # 4.2 MB
    x = np.random.default_rng(13).standard_normal(dims[::-1]).astype(np.float32)

    def read(g, n, what):
        for _ in range(n):
            same_bits(g.get_density(0), x, what)

    for k in range(5):  # too little is read in any one life
        with smokesim.Simulation(*dims, density=x) as g:
            read(g, 2, f"life {k}")
    assert _emu("emu_pinned_calls") == 0
    sims = []
    for d in (0, 1):
        assert lib.hipSetDevice(d) == 0
        sims.append(smokesim.Simulation(*dims, density=x))
    for k in range(8):
        for d, g in enumerate(sims):
            assert lib.hipSetDevice(d) == 0
            read(g, 1, f"device {d} read {k}")
    assert _emu("emu_pinned_calls") == 2 and _emu("emu_pinned_held") == 2
    sims[0].close()
    assert _emu("emu_pinned_held") == 1
    sims[1].close()
    assert _emu("emu_pinned_held") == 0
    assert lib.hipSetDevice(0) == 0
    with smokesim.Simulation(*dims, density=x) as g:
        _emu("emu_refuse_above", 4 << 20)
        read(g, 9, "refused")
        assert _emu("emu_pinned_calls") == 4 and _emu("emu_pinned_held") == 0
        _emu("emu_refuse_above", 2 ** 63)
        read(g, 5, "later")
        assert _emu("emu_pinned_held") == 1
    assert _emu("emu_pinned_held") == 0


def _sweep_launches(g, dt):
    """Launches of the projection's sweeps in one step."""
    g.timing_enable(True)
    g.timing_reset()
    g.step(dt, readback=False)
    n = g.timing_sweeps()[1]
    g.timing_enable(False)
    return n


def case_batch_autotune():
    # Every candidate takes the same time here: the plan in force, fitted or
    # given, stays.
    scs = [scenes.test_scene(d, seed=50 + k, projection=2, iterations=1, n_obstacles=0)
           for k, d in enumerate([(12, 10, 9), (9, 12, 20)])]
    for given in (None, dict(sweeps_per_launch=3, tile=1, zc=5)):
        sims = [gpu_for(sc) for sc in scs]
        b = smokesim.Batch(sims, [0.05, 0.05])
        if given:
            b.set_jacobi_plan(**given)
        plan, _ = b.autotune()
        assert plan == (given or dict(sweeps_per_launch=5, tile=0, zc=plan["zc"])), plan
        assert plan["zc"] < 32 and b.get_jacobi_plan() == plan, plan
        b.step(use_graph=False)
        b.synchronize()
        for sc, g in zip(scs, sims):
            o = oracle_for(sc, 32)
            o.step(0.05, 1)
            assert_bitwise_equal(g.state(), o.state(), f"{sc['name']} {plan}")
        b.close()
        for g in sims:
            g.close()


def _same_state(g, o, what):
    assert_bitwise_equal(g.state(), o.state(), what)
    same_bits(g.get_pressure(), o.get_pressure(), what + " pressure")


def case_reference_memory():
    # The reference form holds no more than the footprint: its half-sweeps use
    # the pressure form's fields, which are zero again for everything that reads
    # them.
    dims, its = (14, 12, 10), 4
    fp = smokesim.footprint_bytes(*dims)

    def both(seed, **kw):
        sc = scenes.test_scene(dims, seed=seed, projection=0, iterations=its, **kw)
        return sc, gpu_for(sc), oracle_for(sc, 32)

    def step(sc, g, o, n=1):
        for _ in range(n):
            g.step(sc["dt"], readback=False)
        o.step(sc["dt"], n)

    def change(g, o, **kw):
        for s in (g, o):
            s.set_params(**kw)

    for graph in (False, True):
        sc, g, o = both(60)
        assert _emu("emu_device_bytes") == fp
        g.set_step_graph(graph)
        assert _sweep_launches(g, sc["dt"]) < 2 * its
        o.step(sc["dt"], 1)
        step(sc, g, o, 3)
        assert _emu("emu_device_bytes") == fp
        _same_state(g, o, f"graph {graph}")           # the pressure is still zero
        step(sc, g, o, 2)                             # (a replay after it was cleared)
        blob = g.snapshot()
        step(sc, g, o)
        r = gpu_for(sc)
        r.restore(blob)
        r.step(sc["dt"], readback=False)
        _same_state(r, o, f"restored, graph {graph}")
        r.close()
        for proj, warm in ((2, 0), (1, 1), (2, 1), (0, 0), (1, 1)):
            change(g, o, projection=proj, warm_start=warm)
            step(sc, g, o, 2)
            _same_state(g, o, f"then projection {proj}, graph {graph}")
        g.close()
    # Warm from the zero pressure; norms, whose right-hand side is kept; a batch.
    sc, g, o = both(61, noise=0.4)
    step(sc, g, o)
    change(g, o, projection=1, warm_start=1)
    step(sc, g, o)
    _same_state(g, o, "warm after reference")
    g.close()
    import oracle as orc
    sc, g, o = both(62, noise=0.4)
    step(sc, g, o)
    g.norms_enable(True)
    step(sc, g, o)
    n, m = g.step_norms(), orc.step_norms(g, sc["dt"])
    assert n["rhs_l2"] > n["div_l2"] and abs(n["div_l2"] - m["div_l2"]) <= 1e-12 * m["div_l2"]
    g.norms_enable(False)
    step(sc, g, o, 2)
    _same_state(g, o, "norms")
    change(g, o, projection=2)
    b = smokesim.Batch([g], [sc["dt"]])
    for _ in range(2):
        b.step(use_graph=False)
    b.close()
    o.step(sc["dt"], 2)
    _same_state(g, o, "batch")
    change(g, o, projection=0)
    step(sc, g, o, 2)
    _same_state(g, o, "after the batch")
    g.close()


def case_sweep_tail():
    # A fitted plan leaves no launch for a last sweep alone; a plan that was set
    # runs as it was set.
    import ctypes
    lib = smokesim.load()
    lib.emu_launches.restype = ctypes.c_longlong
    for its, given, single in [(6, None, 0), (11, None, 0), (1, None, 1),
                               (6, dict(sweeps_per_launch=5, tile=0, zc=8), 1)]:
        sc = scenes.test_scene((14, 12, 10), seed=65, projection=2, iterations=its)
        g, o = gpu_for(sc), oracle_for(sc, 32)
        if given:
            g.set_jacobi_plan(**given)
        before = lib.emu_launches(b"k_jacobi")
        assert _sweep_launches(g, sc["dt"]) == -(-its // 5)
        assert lib.emu_launches(b"k_jacobi") - before == single, (its, given)
        o.step(sc["dt"], 1)
        _same_state(g, o, f"{its} sweeps {given}")
        g.close()


def case_refused_set():
    # Without memory for the reference form's own velocity set (after a pressure
    # form) its steps run in place with the same bits; setting the parameters
    # again asks again.
    sc = scenes.test_scene((14, 12, 10), seed=64, projection=2, iterations=4)
    g, o = gpu_for(sc), oracle_for(sc, 32)

    def step(**kw):
        for s in (g, o):
            s.set_params(**kw)
        o.step(sc["dt"], 1)
        return _sweep_launches(g, sc["dt"])

    step()
    _emu("emu_refuse_above", 1000)
    assert step(projection=0) == 8
    o.step(sc["dt"], 1)
    assert _sweep_launches(g, sc["dt"]) == 8
    _same_state(g, o, "refused")
    _emu("emu_refuse_above", 2 ** 63)
    assert step(iterations=5) < 10
    blob = g.snapshot()
    _same_state(g, o, "allocated")
    r = gpu_for(sc)
    _emu("emu_refuse_above", 1000)
    r.restore(blob)
    assert _sweep_launches(r, sc["dt"]) == 10
    _emu("emu_refuse_above", 2 ** 63)
    r.restore(blob)
    assert _sweep_launches(r, sc["dt"]) < 10
    o.step(sc["dt"], 1)
    _same_state(r, o, "restored")
    r.close()
    g.close()


def case_thin_reference():
    # Grids whose columns would be mostly empty run one half-sweep per launch,
    # others several, with the same bits; a change of the iteration count may
    # change the route.
    for dims, its, several in [((3, 4, 2570), 3, False), ((14, 12, 10), 3, True),
                               ((14, 12, 10), 1, False)]:
        sc = scenes.test_scene(dims, seed=38, projection=0, iterations=its, box_fraction=0.0,
                               n_obstacles=0)
        g, o = gpu_for(sc), oracle_for(sc, 32)
        n = _sweep_launches(g, sc["dt"])
        assert (n < 2 * its) == several, (dims, its, n)
        o.step(sc["dt"], 1)
        assert_bitwise_equal(g.state(), o.state(), f"thin {dims} x{its}")
        g.close()


def case_thin_pressure():
    # The same for the pressure form, cold and warm; the pressure changes
    # buffers or not by the route.
    for dims, its, warm, several in [((60, 3, 400), 20, 1, False), ((60, 3, 400), 20, 0, False),
                                     ((14, 12, 10), 3, 1, True)]:
        sc = scenes.test_scene(dims, seed=39, projection=1, iterations=its, box_fraction=0.0,
                               n_obstacles=0)
        sc["params"]["warm_start"] = warm
        g, o = gpu_for(sc), oracle_for(sc, 32)
        n = _sweep_launches(g, sc["dt"])
        assert (n < 2 * its) == several, (dims, its, n)
        g.step(sc["dt"], readback=False)
        o.step(sc["dt"], 2)
        assert_bitwise_equal(g.state(), o.state(), f"thin {dims} x{its} warm {warm}")
        same_bits(g.get_pressure(), o.get_pressure(), f"thin {dims} x{its} warm {warm}")
        g.close()


def case_foreign_capture():
    # A first step of the reference form while another stream is captured in
    # the global mode: the capture goes on, and this and later steps run
    # several half-sweeps per launch.
    import ctypes
    sc = scenes.test_scene((14, 12, 10), seed=36, projection=0, iterations=6)
    g, o = gpu_for(sc), oracle_for(sc, 32)
    hip = smokesim.load()

    def captured_step():
        st, graph = ctypes.c_void_p(), ctypes.c_void_p()
        assert hip.hipStreamCreateWithFlags(ctypes.byref(st), 1) == 0
        assert hip.hipStreamBeginCapture(st, 0) == 0
        g.step(sc["dt"], readback=False)
        assert hip.hipStreamEndCapture(st, ctypes.byref(graph)) == 0
        assert hip.hipGraphDestroy(graph) == 0 and hip.hipStreamDestroy(st) == 0

    captured_step()
    assert _sweep_launches(g, sc["dt"]) < 2 * 6
    o.step(sc["dt"], 2)
    for s in (g, o):
        s.set_params(projection=2)  # after it the reference form has a set of its own
    g.step(sc["dt"], readback=False)
    o.step(sc["dt"], 1)
    for s in (g, o):
        s.set_params(projection=0)
    captured_step()
    assert _sweep_launches(g, sc["dt"]) < 2 * 6
    o.step(sc["dt"], 2)
    assert_bitwise_equal(g.state(), o.state(), "foreign capture")
    g.close()


CASES = {"sweep_tail": case_sweep_tail, "refused_set": case_refused_set, "reference_memory": case_reference_memory, "batch_autotune": case_batch_autotune, "thin_pressure": case_thin_pressure, "thin_reference": case_thin_reference, "read_slots": case_read_slots, "small_reads": case_small_reads, "foreign_capture": case_foreign_capture, "read_targets": case_read_targets, "step_graph": case_step_graph, "proxy": case_proxy, "refine_groups": case_refine_groups, "single": case_single, "norms": case_norms, "plans": case_plans, "batch": case_batch,
         "server": case_server, "readback": case_readback, "precision": case_precision,
         "vorticity": case_vorticity, "advection": case_advection}


def main():
    smokesim.LIB_PATH = sys.argv[1]
    names = sys.argv[2:] or list(CASES)
    for n in names:
        CASES[n]()
        print("ok", n, flush=True)


if __name__ == "__main__":
    main()

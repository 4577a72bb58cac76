"""Launch and kernel variants chosen by size: each against the oracle or the general path."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def ctx1(nyx, n, lo=(0, 0, 0), hi=(1, 1, 1), **kw):
    return nyx.PMContext(nyx.BoxGeom(tuple(int(v) for v in n), tuple(lo), tuple(hi)), **kw)


def mean_free(n, seed):
    f = np.random.default_rng(seed).standard_normal((n[2], n[1], n[0]))
    return f - f.mean()


@pytest.mark.parametrize("n", [(32, 32, 32), (66, 18, 10), (130, 34, 6), (40, 24, 18), (15, 16, 14),
                               (144, 112, 144)])
def test_residual_chunks_bitwise(nyx, orc, n):
    # the level-0 residual by pairs of cells (small boxes of even nx, blocks past the
    # last pair), and by marched columns that pass its edge (odd nx, and above 2^21
    # cells): iterates and norms of two V-cycles from a
    # non-zero guess, bit for bit
    f = mean_free(n, 31)
    guess = mean_free(n, 32)
    dx = [1.0 / 32] * 3
    hi = [v / 32 for v in n]
    with ctx1(nyx, n, hi=hi) as c:
        phi, it, norms = c.solve_poisson(f, guess, fixed_iters=2)
    ref, it2, st, _ = orc.mg_solve(n, dx, f, guess, fixed_iters=2)
    assert np.array_equal(norms[:2], st[:2])
    if n[0] % 2:  # a bottom alone, solved exactly: only the first residual compares in bits
        return
    assert it == it2 == 2
    assert np.array_equal(phi, ref)
    assert norms[2] == st[2]


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("n", [
    (16, 16, 16),    # three smoothing levels over a 2^3 bottom, the whole cycle in one workgroup
    (12, 20, 16),    # two levels, 3 x 5 x 4 bottom
    (4, 16, 64),     # 2 x 8 x 32 bottom, pairs whose x-neighbours are themselves
    (10, 14, 6),     # one level, 5 x 7 x 3 bottom
    (9, 5, 7),       # a bottom alone
    (14, 12, 13),    # a bottom too large to be staged (2184 cells)
    (36, 40, 48),    # finer levels above a 9 x 10 x 12 workgroup level
    (36, 36, 36),                 # a 9^3 bottom: odd rows of one piece
    (44, 20, 12),                 # an 11 x 5 x 3 bottom: rows of two pieces
])
def test_coarse_workgroup_equals_per_level(nyx, orc, n, precision):
    # the one-workgroup coarse cycle against one launch per level and step, bit for
    # bit, from zero, and in FP64 against the oracle (a bottom alone: to rounding,
    # the library's and the oracle's Green's functions come from two compilers)
    f = mean_free(n, 33)
    hi = [v / 32 for v in n]
    out = []
    for coarse in ("workgroup", "per_level"):
        with ctx1(nyx, n, hi=hi, precision=precision, coarse=coarse) as c:
            out.append(c.solve_poisson(f, fixed_iters=3)[0])
    assert np.array_equal(out[0], out[1])
    if precision == "fp64":
        ref, _, _, _ = orc.mg_solve(n, [1.0 / 32] * 3, f, fixed_iters=3)
        if any(v % 2 for v in n):
            assert np.abs(out[0] - ref).max() <= 1e-12 * np.abs(ref).max()
        else:
            assert np.array_equal(out[0], ref)


def test_coarse_workgroup_keeps_the_correction(nyx):
    # grouped FP32 cycles continue from the previous correction also where the
    # whole V-cycle runs in the workgroup (a converged mixed solve, no fixed count)
    n = (16, 16, 16)
    f = mean_free(n, 34)
    out = []
    for coarse in ("workgroup", "per_level"):
        with ctx1(nyx, n, precision="mixed", coarse=coarse) as c:
            out.append(c.solve_poisson(f)[:2])
    assert out[0][1] == out[1][1]
    assert np.array_equal(out[0][0], out[1][0])


@pytest.mark.parametrize("npart", [1, 300, 2 ** 18, 2 ** 18 + 77])
@pytest.mark.parametrize("slack", [0.0, -1.0])
def test_device_download_equals_host_download(nyx, npart, slack):
    # downloads into device arrays (directly, or through records above 2^18
    # particles where the idle buffer holds them) against the host path, for the
    # second box of a batch, whole and with components left out, also between a
    # kick-drift and its re-sort (moves waiting in the idle buffer), whose list must
    # survive
    import torch
    r = np.random.default_rng(41)
    geoms = [nyx.BoxGeom((16, 16, 16)), nyx.BoxGeom((48, 32, 32), (0, 0, 0), (1.5, 1, 1))]
    with nyx.PMContext(geoms, resort_slack=slack) as c, nyx.PMContext(geoms, resort_slack=slack) as c2:
        pos = [r.random(npart) * (1.5 if d == 0 else 1.0) for d in range(3)]
        vel = [r.standard_normal(npart) for _ in range(3)]
        small = [r.random(500) for _ in range(3)]
        for q in (c, c2):
            q.upload(0, small, [np.zeros(500)] * 3, m=r.random(500))
            q.upload(1, pos, vel, m_const=1.0 / npart)
            q.pm_init()
        out = torch.full((6, npart), -7.0, dtype=torch.float64, device="cuda")
        addr = [out[k].data_ptr() for k in range(6)]

        def check(use):
            out.fill_(-7.0)
            torch.cuda.synchronize()
            c.download_device([a if k in use else None for k, a in enumerate(addr)], box=1)
            p, v = c.download(1)
            got = out.cpu().numpy()
            for k, ref in enumerate(list(p) + list(v)):
                assert np.array_equal(got[k], ref if k in use else np.full(npart, -7.0))

        check(range(6))
        c.assign_density(want=False)
        check(range(6))
        for q in (c, c2):
            q.move_kick_drift(1e-3)
        check((1, 3, 4))
        check(range(6))
        assert np.array_equal(c.assign_density(1), c2.assign_density(1))
        check((0, 5))


@pytest.mark.parametrize("slack", [0.0, -1.0])
@pytest.mark.parametrize("use", [(0, 1), (3, 5), (0, 1, 2), (0, 2, 3, 5), (1, 2, 3, 4, 5), (0, 1, 2, 3, 4, 5)])
def test_device_download_of_some_components(nyx, use, slack):
    # records of two, four and eight doubles, and the launch per component where they find
    # no room (no slack: the idle buffer is too small for eight) or a list of moves waits
    import torch
    npart = 2 ** 18 + 77
    r = np.random.default_rng(43)
    pos = [r.random(npart) for _ in range(3)]
    vel = [r.standard_normal(npart) for _ in range(3)]
    with ctx1(nyx, (32, 32, 32), resort_slack=slack) as c:
        c.upload(0, pos, vel, m_const=1.0 / npart)
        c.pm_init()
        for moving in (False, True):
            if moving:
                c.move_kick_drift(1e-3)
            out = torch.full((6, npart + 1), -7.0, dtype=torch.float64, device="cuda")
            torch.cuda.synchronize()
            # (8-byte aligned destinations)
            c.download_device([out[k, 1:].data_ptr() if k in use else None for k in range(6)])
            p, v = c.download()
            got = out.cpu().numpy()
            assert (got[:, 0] == -7.0).all()
            for k, ref in enumerate(list(p) + list(v)):
                assert np.array_equal(got[k, 1:], ref if k in use else np.full(npart, -7.0))


@pytest.mark.parametrize("sweep2", [0, 9])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("boxes", [
    [(64, 64, 64)],
    [(8, 12, 64)],                # narrower than a leg's region
    [(72, 40, 24)],               # columns that overlap their neighbours in x and y
    [(36, 20, 16)],               # a narrow column shape, one level above the workgroup
    [(16, 8, 40)],                # the smallest shape
    [(5, 5, 5), (100, 36, 28)],   # a batch whose first box has no smoothing level
    [(144, 80, 48), (48, 64, 40)],
    [(160, 80, 96)],              # restrictions by narrow marched tiles
])
def test_paired_smoothing_equals_half_sweeps(nyx, boxes, precision, sweep2):
    # whole cycle legs in one launch (sweep2 = 0, these sizes) and smoothing pairs as
    # one pass (sweep2 = 9: uneven z-chunks of 9) in both precisions, against separate
    # half sweeps, bit for bit: the solves of two steps (the correction kept between
    # grouped FP32 cycles, phi updated by the last pass)
    r = np.random.default_rng(51)
    parts = []
    for n in boxes:
        npart = 3000
        parts.append(([r.random(npart) * (v / 32) for v in n], [0.1 * r.standard_normal(npart) for _ in range(3)]))
    out = []
    for sm in ("fused", "half"):
        geoms = [nyx.BoxGeom(n, (0, 0, 0), tuple(v / 32 for v in n)) for n in boxes]
        with nyx.PMContext(geoms, precision=precision, smoother=sm, sweep2=sweep2) as c:
            for b, (pos, vel) in enumerate(parts):
                c.upload(b, pos, vel, m_const=1e-3)
            c.pm_init()
            it = c.pm_steps(2, 1e-3)
            out.append([it] + [c.get_phi(b) for b in range(len(boxes))] + [x for b in range(len(boxes))
                                                                             for x in sum(map(list, c.download(b)), [])])
    for a, b in zip(*out):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("npart", [4096, 4097, 30011])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_split_tile_deposit(nyx, orc, npart, precision):
    # a clump inside one tile: one block up to 4096 slots, above that parts whose
    # fixed-point sums meet in global memory.  AssignDensity (FP64 weights) against
    # the oracle, repeated (the accumulators are zero again) and through other tile
    # shapes; the step's deposit (FP32 weights in mixed precision, the interpolation
    # error of a weight is below 4 roundings of 2^-24) through the right-hand side
    r = np.random.default_rng(61)
    n = (32, 32, 32)
    pos = [(9.0 + 5.0 * r.random(npart)) / 32 for _ in range(3)]
    pos = [np.concatenate([p, r.random(2000)]) for p in pos]
    m = 0.5 + r.random(npart + 2000)
    ref = orc.deposit(n, (0, 0, 0), (1, 1, 1), *pos, m=m)
    with ctx1(nyx, n, precision=precision) as c, ctx1(nyx, n, tile=(32, 8, 4), precision=precision) as c2:
        for q in (c, c2):
            q.upload(0, pos, [np.zeros_like(m)] * 3, m=m)
        rho = c.assign_density()
        assert np.abs(rho - ref).max() <= 1e-13 * ref.max()
        assert np.array_equal(c.assign_density(), rho)
        assert np.abs(c2.assign_density() - ref).max() <= 1e-13 * ref.max()
        c.pm_init()
        rhs = -(ref - ref.mean())
        tol = 1e-13 if precision == "fp64" else 4 * 2.0 ** -24
        assert np.abs(c.get_rhs() - rhs).max() <= tol * ref.max()
        assert np.array_equal(c.assign_density(), rho)


@pytest.mark.parametrize("clump", [0, 6001])
def test_density_and_vels_second_box_of_a_batch(nyx, orc, clump):
    # the momentum deposits (three components in one launch, a clump's tile in parts)
    # and the one-pass fold, for a box with partial tiles behind another one: the
    # density is AssignDensity's, the velocities the oracle's to the rounding of a sum
    # of its contributions (cells with mass), and a second call gives the same bits
    r = np.random.default_rng(71)
    n, hi = (36, 20, 24), (1.8, 1.0, 1.2)
    npart = 5000
    pos = [r.random(npart) * h for h in hi]
    pos = [np.concatenate([p, 0.41 + 0.02 * r.random(clump)]) for p in pos]
    vel = [r.standard_normal(npart + clump) * (d + 1) for d in range(3)]
    m = 0.5 + r.random(npart + clump)
    geoms = [nyx.BoxGeom((16, 16, 16)), nyx.BoxGeom(n, (0, 0, 0), hi)]
    with nyx.PMContext(geoms) as c:
        small = [r.random(100) for _ in range(3)]
        c.upload(0, small, small, m=0.1 + r.random(100))
        c.upload(1, pos, vel, m=m)
        rho = c.assign_density(1)
        out = c.assign_density_and_vels(1)
        assert np.array_equal(c.assign_density_and_vels(1), out)
        assert np.array_equal(c.assign_density(1), rho)
        # the solver's pools held the momentum sums: a solve after it is unaffected
        c.solve_for_phi(use_guess=False)
        phi = c.get_phi(1)
    with nyx.PMContext(geoms) as c:
        c.upload(0, small, small, m=0.1 + r.random(100))
        c.upload(1, pos, vel, m=m)
        c.assign_density(want=False)
        c.solve_for_phi(use_guess=False)
        assert np.array_equal(c.get_phi(1), phi)
    assert np.array_equal(out[0], rho)
    ref = orc.deposit_vels(n, (0, 0, 0), hi, pos, vel, m=m)
    big = ref[0] > 1e-3 * ref[0].max()
    for d in range(3):
        assert np.abs(out[d + 1] - ref[d + 1])[big].max() <= 1e-11 * (d + 1)
        assert np.array_equal(out[d + 1] == 0, out[0] == 0)


@pytest.mark.parametrize("per_tile,clump", [(40, 0), (3400, 0), (3400, 30001)])
def test_density_and_vels_scratch(nyx, orc, per_tile, clump):
    # the momentum deposits' halo slots in the idle buffer (60 B a slot) or their own where
    # those are more, and the accumulators of split tiles, which only this call allocates:
    # what the context holds after it, the oracle's fields, and the steps go on as without
    n = (64, 32, 40)
    hi = (1.6, 0.8, 1.0)
    tiles = 4 * 4 * 5
    npart = per_tile * tiles
    r = np.random.default_rng(73)
    pos = [np.concatenate([r.random(npart) * h, 0.41 + 0.02 * r.random(clump)]) for h in hi]
    vel = [r.standard_normal(npart + clump) for _ in range(3)]
    m = (0.5 + r.random(npart + clump)) / npart
    halo = 3 * tiles * (17 * 9 * 9 - 16 * 8 * 8) * 8
    res = []
    for call in (False, True):
        with ctx1(nyx, n, hi=hi) as c:
            c.upload(0, pos, vel, m=m)
            c.pm_init()
            c.pm_steps(2, 1e-4)
            c.assign_density(want=False)
            if call:
                ref = orc.deposit_vels(n, (0, 0, 0), hi, *c.download(), m=m)
                held = c.device_bytes()
                out = c.assign_density_and_vels()
                more = c.device_bytes() - held
                assert np.array_equal(c.assign_density_and_vels(), out)
                assert c.device_bytes() - held == more
                slots = npart + clump + ((npart + clump) * 256 + 1023 >> 10) + 16 * tiles
                split = 8 * (slots // 4096 * 3 * 2 * 17 * 9 * 9 + (slots // 4096 * 3 + 1) // 2)
                assert more == split + (halo if slots * 60 < halo else 0)
                assert np.abs(out[0] - ref[0]).max() <= 1e-13 * ref[0].max()
                big = ref[0] > 1e-3 * ref[0].max()
                for d in range(3):
                    assert np.abs(out[d + 1] - ref[d + 1])[big].max() <= 1e-11
            c.pm_steps(2, 1e-4)
            p, v = c.download()
            res.append(list(p) + list(v) + [c.get_phi()])
    for a, b in zip(*res):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("npart", [3000, 2 ** 18 + 5])
def test_tiled_gather_equals_thread_per_particle(nyx, npart, precision):
    # the staged gather (written directly, and as records above 2^18 particles) against
    # the thread-per-particle kernel, which a context that has not binned its particles
    # takes: after the deposit, after a kick-drift whose moves still wait (particles
    # outside their tile and outside the box) and after its periodic shift
    r = np.random.default_rng(81)
    n, hi = (40, 24, 36), (2.0, 1.2, 1.8)
    pos = [r.random(npart) * h for h in hi]
    vel = [r.standard_normal(npart) for _ in range(3)]
    phi = r.standard_normal((n[2], n[1], n[0]))
    with ctx1(nyx, n, hi=hi, precision=precision) as c:
        c.upload(0, pos, vel, m_const=1.0)
        c.set_phi(phi)

        def unbinned():
            p, v = c.download()
            with ctx1(nyx, n, hi=hi, precision=precision) as c2:
                c2.upload(0, p, v, m_const=1.0)
                c2.set_phi(phi)
                return c2.gather_accel()

        assert np.array_equal(c.gather_accel(), unbinned())
        c.assign_density(want=False)
        assert np.array_equal(c.gather_accel(), unbinned())
        c.move_kick_drift(0.05)
        assert np.array_equal(c.gather_accel(), unbinned())
        c.assign_density(want=False)
        assert np.array_equal(c.gather_accel(), unbinned())
        c.redistribute()
        assert np.array_equal(c.gather_accel(), unbinned())
        if npart <= 2 ** 20:
            assert np.array_equal(c.gather_accel_noalloc(), unbinned())


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("per_tile", [71, 72, 114, 115])
def test_gather_of_sparse_tiles(nyx, per_tile, precision):
    # either side of the particles per tile from which the gather stages g per tile (115
    # of 16x8x8 cells in FP64, 72 in mixed precision): the values of the
    # thread-per-particle kernel of a context that has not binned them, bit for bit
    n = (352, 160, 192)
    npart = per_tile * (n[0] // 16) * (n[1] // 8) * (n[2] // 8)
    hi = [v / 352 for v in n]
    r = np.random.default_rng(83)
    pos = [r.random(npart) * h for h in hi]
    zero = np.zeros(npart)
    phi = r.standard_normal((n[2], n[1], n[0]))
    res = []
    for binned in (False, True):
        with ctx1(nyx, n, hi=hi, precision=precision) as c:
            c.upload(0, pos, [zero] * 3, m_const=1.0)
            if binned:
                c.assign_density(want=False)
            c.set_phi(phi)
            res.append(c.gather_accel())
    assert np.array_equal(*res)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("slack,speed", [(0.25, 0.02), (0.002, 1.0), (0.5, 6.0)])
def test_captured_resort_equals_eager(nyx, precision, slack, speed):
    # captured steps re-sort incrementally and decide on the device about the full sort
    # (few particles moving; tiles that run out of slack; emptied slots past their
    # limit), over several replays and calls with eager steps between them, against
    # eager steps bit for bit, with per-particle masses, and with what the host counts
    r = np.random.default_rng(91)
    sizes, npart = [(32, 32, 32), (24, 24, 24)], 20000
    parts = [([r.random(npart) for _ in range(3)], [speed * 0.3 * r.standard_normal(npart) for _ in range(3)],
              0.5 / npart + r.random(npart) / npart) for _ in sizes]
    res = []
    for graph in (False, True):
        with nyx.PMContext([nyx.BoxGeom(n) for n in sizes], precision=precision, resort_slack=slack) as c:
            for b, (pos, vel, m) in enumerate(parts):
                c.upload(b, pos, vel, m=m)
            c.pm_init()
            states = []
            for nsteps in (8, 5, 10):
                c.pm_steps(nsteps, 1e-3, use_graph=graph)
                for b in range(2):
                    p, v = c.download(b)
                    states += list(p) + list(v) + [c.get_phi(b)]
            st = c.sort_stats()
            res.append(states)
            print("sorts", graph, st, flush=True)
            if speed < 0.1:
                assert st["full"] == 1 and st["incremental"] == 23 and st["moved"] > 0
            else:
                assert st["full"] > 3
                assert speed > 2 or st["incremental"] > 3
    for a, b in zip(*res):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("kind", ["pair", "separate", "faithful"])
def test_captured_full_sorts_of_many_moves(nyx, kind):
    # from 2^22 particles, captured steps record plain full sorts while more than 6/1024 of
    # the particles change tile per step (0.02 cells: not; 0.1: they do; 2: tiles overflow),
    # over calls that change between these, against eager steps bit for bit
    n, npart = (64, 64, 64), 2 ** 22 + 3
    r = np.random.default_rng(97)
    pos = [r.random(npart) for _ in range(3)]
    vel = [r.standard_normal(npart) for _ in range(3)]
    m = (0.5 + r.random(npart)) / npart
    res = []
    for graph in (False, True):
        with ctx1(nyx, n, precision="mixed", pair_kicks=kind != "separate") as c:
            c.upload(0, pos, vel, m=m)
            c.pm_init(four_pi_G=1e-3)
            states = []
            for cells, nsteps in ((0.02, 6), (0.1, 8), (0.1, 7), (2.0, 7), (0.02, 6)):
                st0 = c.sort_stats()
                c.pm_steps(nsteps, cells / 64, four_pi_G=1e-3, use_graph=graph, nyx_faithful=kind == "faithful")
                st = {k: v - st0[k] for k, v in c.sort_stats().items()}
                print(kind, graph, cells, nsteps, st, flush=True)
                assert st["full"] + st["incremental"] >= nsteps
                if graph and cells > 0.05:  # all but the first, which looks
                    assert st["incremental"] <= 1
                p, v = c.download()
                states += list(p) + list(v) + [c.get_phi()]
            res.append(states)
    for a, b in zip(*res):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_cycles_issued_ahead(nyx, precision):
    # V-cycles issued before the host looks at a check (one fewer than the last solve
    # took): solves that need fewer, none, more or a fixed number of cycles than the one
    # before give the bits, counts and norms of a context that has solved nothing else
    n = (40, 24, 32)
    f = mean_free(n, 91)
    hard = dict(rel_tol=1e-12)
    def runs(c, phi):
        return [lambda: c.solve_poisson(f, **hard), lambda: c.solve_poisson(f, rel_tol=1e-3),
                lambda: c.solve_poisson(f, phi, rel_tol=1e-6), lambda: c.solve_poisson(f, **hard),
                lambda: c.solve_poisson(f, fixed_iters=3), lambda: c.solve_poisson(0 * f),
                lambda: c.solve_poisson(f, phi, **hard)]
    with ctx1(nyx, n, precision=precision) as c:
        phi = c.solve_poisson(f, **hard)[0]
        together = [g() for g in runs(c, phi)]
    for i, (p, it, norms) in enumerate(together):
        with ctx1(nyx, n, precision=precision) as c:
            p1, it1, norms1 = runs(c, phi)[i]()
        assert it == it1 and np.array_equal(norms, norms1) and np.array_equal(p, p1)
    assert together[2][1] == together[5][1] == 0 and together[4][1] == 3


def test_cycles_issued_ahead_up_to_the_limit(nyx):
    # ... and a solve that runs into max_iter raises with its count, whatever was issued
    n = (32, 32, 32)
    f = mean_free(n, 92)
    with ctx1(nyx, n, max_iter=4) as c:
        assert c.solve_poisson(f, rel_tol=1e-2)[1] <= 4
        for _ in range(2):
            with pytest.raises(nyx.NyxPMError, match="after 4 cycles"):
                c.solve_poisson(f, rel_tol=1e-14)
        assert c.solve_poisson(f, rel_tol=1e-2)[1] <= 4


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_cycles_issued_ahead_fit_the_solve(nyx, precision):
    # a solve that needs few cycles launches no more than it needs (one level-0 residual
    # each, and the first) after one that failed, one from zero, one of another
    # tolerance; alternating hard and easy guesses, at most one
    n = (32, 32, 32)
    f = mean_free(n, 93)
    first = 5 if precision == "mixed" else 1

    def residuals(c, solve):
        c.timing_reset()
        c.timing_enable(True)
        try:
            it = solve()
        finally:
            c.timing_enable(False)
            got = c.timing("residual")[0]
        need = 1 if it == 0 else 2 if it <= first else 2 + it - first
        return got - need

    with ctx1(nyx, n, precision=precision, max_iter=60) as c:
        phi = c.solve_poisson(f, rel_tol=1e-13)[0]
        with pytest.raises(nyx.NyxPMError):
            c.solve_poisson(f, abs_tol=1e-300, rel_tol=0.0)
        for rel in (0.0, 1e-9):
            with pytest.raises(nyx.NyxPMError):
                c.solve_poisson(f, rel_tol=rel / 1e300, abs_tol=0.0)
            assert residuals(c, lambda: c.solve_poisson(0 * f, 0 * f, rel_tol=rel / 1e300)[1]) == 0
        easy = lambda: c.solve_poisson(f, phi, rel_tol=1e-9)[1]
        hard = lambda: c.solve_poisson(f, rel_tol=1e-9)[1]
        assert easy() == 0
        hard()
        assert residuals(c, easy) <= 1
        hard()
        assert residuals(c, easy) <= 1
    pos, vel, m = nyx.ics.lattice_gaussian(32, nyx.ics.SEED_BASE, sigma_cells=1.0)
    with ctx1(nyx, n, precision=precision) as c:
        c.upload(0, pos, vel, m_const=m)
        c.assign_density(want=False)
        solve = lambda guess, rel=1e-10: int(c.solve_for_phi(rel_tol=rel, use_guess=guess)[0][0])
        for _ in range(3):
            assert solve(False) > 3
            assert residuals(c, lambda: solve(True, 1e-9)) == 0
        for _ in range(2):
            solve(False)
        assert residuals(c, lambda: solve(False, 1e-2)) == 0
        assert residuals(c, lambda: solve(False)) == 0


def test_autotune_times_what_the_rule_chose(nyx):
    # a level that only the narrowest column of the smoothing pair fits: it is timed, kept,
    # and the solves keep their bits
    geoms = [nyx.BoxGeom((64, 8, 512), (0, 0, 0), (2.0, 0.25, 16.0))] * 3
    r = np.random.default_rng(95)
    rho = [r.random((512, 8, 64)) for _ in geoms]
    res = []
    for precision in ("fp64", "mixed"):
        with nyx.PMContext(geoms, precision=precision) as c:
            for tune in (False, True):
                if tune:
                    rep = c.autotune()
                    for key in ("sweep2.d0", "sweep2.fp64.d0"):
                        assert rep[key]["shape"] == [16, 8] and 0 < rep[key]["us"] < 1e6 and rep[key]["on"]
                for b in range(3):
                    c.set_density(rho[b], b)
                its = c.solve_for_phi(rel_tol=1e-8, use_guess=False)[0]
                res.append((list(its), [c.get_phi(b) for b in range(3)]))
    for a, b in (res[:2], res[2:]):
        assert a[0] == b[0] and all(np.array_equal(p, q) for p, q in zip(a[1], b[1]))


def test_uploads_across_the_particle_buffers_kinds(nyx):
    # particle buffers of an allocation per array (below 2^18 slots) and of one for all, with
    # and without masses, replaced by each other in one context: as in a context of its own
    n = (32, 32, 32)

    def steps(c, npart, mass, seed):
        r = np.random.default_rng(seed)
        pos = [r.random(npart) for _ in range(3)]
        vel = [r.standard_normal(npart) for _ in range(3)]
        m = (0.5 + r.random(npart)) / npart if mass else None
        c.upload(0, pos, vel, m=m, m_const=1.0 / npart)
        c.pm_init()
        c.pm_steps(2, 1e-3)
        p, v = c.download()
        return list(p) + list(v) + [c.get_phi()]

    runs = [(5000, False), (300000, False), (5000, True), (300000, True), (209000, True), (7000, True)]
    with ctx1(nyx, n) as c:
        together = [steps(c, npart, mass, 100 + i) for i, (npart, mass) in enumerate(runs)]
    for i, (npart, mass) in enumerate(runs):
        with ctx1(nyx, n) as c:
            alone = steps(c, npart, mass, 100 + i)
        for a, b in zip(together[i], alone):
            assert np.array_equal(a, b)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("share", [0.3, 1.0])
def test_items_of_a_clump_by_a_wave(nyx, precision, share):
    # tiles of more items and deposit parts than one thread writes, next to tiles of few:
    # steps with the default kick items and with items of 256 particles, against the
    # thread-per-particle kick
    r = np.random.default_rng(103)
    n, npart = (48, 32, 32), 60000
    clump = int(share * npart)
    pos = [r.random(npart) * 1.5 if d == 0 else r.random(npart) for d in range(3)]
    for d in range(3):
        pos[d][:clump] = (0.4, 0.61, 0.27)[d] + r.random(clump) / 64
    vel = [0.1 * r.standard_normal(npart) for _ in range(3)]
    res = []
    for kw in (dict(kick="global"), {}, dict(kick_chunk=256)):
        with ctx1(nyx, n, hi=(1.5, 1, 1), precision=precision, **kw) as c:
            c.upload(0, pos, vel, m_const=1.0 / npart)
            c.pm_init(four_pi_G=1e-3)
            c.pm_steps(3, 1e-3, four_pi_G=1e-3)
            p, v = c.download()
            res.append(list(p) + list(v) + [c.get_phi(), c.assign_density()])
    for other in res[1:]:
        for a, b in zip(res[0], other):
            assert np.array_equal(a, b)

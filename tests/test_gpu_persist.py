"""The persistent kernel for small single systems (persist.hip): every step of
a run in one launch, the workgroups meeting at a grid barrier each step, the
lane rows built inside the kernel.

Checked against the FP64 oracle (positions, velocities, temperatures,
energies) for NVE velocity Verlet, NVE leapfrog and leapfrog Berendsen, for
each lanes-per-atom shape; against the tile path; over several calls in a row
and a hand-back to the tile path; through a row overflow (the run replayed
with longer rows); and for the 10,000-step NVE energy drift."""
import dataclasses
import sys

import numpy as np
import pytest

from md_gpu_amd import systems as S
from conftest import rel_rms

pytestmark = pytest.mark.gpu


def say(*a):
    print("[case]", *a, file=sys.stderr, flush=True)


@pytest.fixture(scope="module")
def E():
    from md_gpu_amd import engine
    return engine


def perturbed(sys_, amp, seed=11):
    s = sys_.copy()
    rng = np.random.default_rng(seed)
    p = s.pos.astype(np.float64) + rng.normal(0.0, amp, s.pos.shape)
    s.pos = S.wrap_centered(p, s.box.astype(np.float64)).astype(np.float32)
    return s


def arxe_one(n=2000, seed=21):
    """One Ar-Xe mixture (two atom types), NVT leapfrog Berendsen."""
    return S.arxe_replicas(nrep=1, seed=seed, nmin=n, nmax=n)[0]


CASES = [
    ("argon_vv_nve", lambda: perturbed(S.argon(), 0.1), 100),
    ("argon_lf_nve", lambda: dataclasses.replace(perturbed(S.argon(), 0.1), integrator="leapfrog",
                                                 thermostat="none"), 100),
    ("arxe2000_lf_berendsen", lambda: arxe_one(), 100),
]


def persist_engine(E, s, lanes):
    e = E.Engine.from_system(s)
    e.set_launch(persist=1, lanes=lanes)
    return e


def check_vs_oracle(st, pos, vel, r, box, pos_tol=2e-4):
    d = pos.astype(np.float64) - r["pos"]
    d -= box * np.rint(d / box)
    say("  max |dx|", np.abs(d).max(), "T", st["temp"][-1, 0], r["temp"][-1])
    assert np.abs(d).max() < pos_tol
    assert rel_rms(vel, r["vel"]) < 1e-4
    assert np.allclose(st["temp"][:, 0], r["temp"], rtol=1e-4)
    assert np.allclose(st["ke"][:, 0], r["ke"], rtol=1e-4)
    assert np.allclose(st["pe_lj"][:, 0], r["pe"], rtol=1e-4, atol=1e-4 * np.abs(r["pe"]).max())


@pytest.mark.parametrize("lanes", [4, 8, 16])
@pytest.mark.parametrize("name,mk,nsteps", CASES)
def test_persist_matches_oracle(E, orc, name, mk, nsteps, lanes):
    s = mk()
    say("persist", name, s.n, "lanes", lanes, "steps", nsteps)
    e = persist_engine(E, s, lanes)
    pos0, vel0, _ = e.download()
    so = s.copy()
    so.pos, so.vel = pos0, vel0
    st = e.run(nsteps, energy_every=1)
    info = e.persist_info()
    assert info["runs"] == 1 and info["replays"] == 0, info
    pos, vel, _ = e.download()
    r = orc.md_run(so, nsteps)
    check_vs_oracle(st, pos, vel, r, s.box)
    assert e.info()["steps"] == nsteps
    e.close()


def test_persist_matches_tile_path(E):
    s = perturbed(S.argon(), 0.1)
    say("persist vs tile path argon", s.n)
    out = []
    for persist in (0, 1):
        e = E.Engine.from_system(s)
        e.set_launch(persist=persist, lanes=16)
        st = e.run(100, energy_every=1)
        assert e.persist_info()["runs"] == persist
        pos, vel, force = e.download()
        out.append((st, pos, vel, force))
        e.close()
    (st0, p0, v0, f0), (st1, p1, v1, f1) = out
    d = p1.astype(np.float64) - p0
    d -= s.box * np.rint(d / s.box)
    say("  max |dx|", np.abs(d).max(), "force rel rms", rel_rms(f1, f0))
    assert np.abs(d).max() < 1e-4
    assert rel_rms(f1, f0) < 1e-4
    assert np.allclose(st1["conserved"][:, 0], st0["conserved"][:, 0], rtol=1e-5)


def test_persist_consecutive_runs_and_hand_back(E, orc):
    """Three persistent runs (40, 1, 39 steps), then 40 steps on the tile path:
    the 120-step trajectory of one engine against the oracle's."""
    s = dataclasses.replace(perturbed(S.argon(), 0.1), integrator="leapfrog", thermostat="berendsen", tau=100.0,
                            T0=120.0)
    say("persist consecutive runs + tile path", s.n)
    e = persist_engine(E, s, 8)
    pos0, vel0, _ = e.download()
    so = s.copy()
    so.pos, so.vel = pos0, vel0
    temps = []
    for n in (40, 1, 39):
        temps.append(e.run(n, energy_every=1)["temp"][:, 0])
    assert e.persist_info()["runs"] == 3
    e.set_launch(persist=0)
    temps.append(e.run(40, energy_every=1)["temp"][:, 0])
    assert e.persist_info()["runs"] == 3
    assert all(v == 0 for v in e.check_lists().values())
    pos, vel, _ = e.download()
    r = orc.md_run(so, 120)
    d = pos.astype(np.float64) - r["pos"]
    d -= s.box * np.rint(d / s.box)
    say("  max |dx|", np.abs(d).max())
    assert np.abs(d).max() < 2e-4
    assert np.allclose(np.concatenate(temps), r["temp"], rtol=1e-4)
    assert e.info()["steps"] == 120
    e.close()


def test_persist_row_overflow_replays(E, orc):
    """A list capacity of 16 entries per atom (about 80 neighbors lie within
    r_list) makes the lane rows too short: the run is replayed from its start with
    rows twice as long until they fit, and ends on the oracle's trajectory."""
    s = perturbed(S.argon(), 0.1)
    say("persist row overflow argon", s.n)
    e = persist_engine(E, s, 16)
    e.set_list_capacity(16)
    row0 = e.persist_info()["row_len"]
    pos0, vel0, _ = e.download()
    so = s.copy()
    so.pos, so.vel = pos0, vel0
    st = e.run(60, energy_every=1)
    info = e.persist_info()
    say("  rows per lane", row0, "->", info["row_len"], "replays", info["replays"])
    assert info["replays"] >= 1 and info["row_len"] > row0 and info["runs"] == 1
    pos, vel, _ = e.download()
    r = orc.md_run(so, 60)
    check_vs_oracle(st, pos, vel, r, s.box)
    e.close()


def test_persist_ineligible_system_runs_tiles(E, orc):
    """A charged system is not the persistent kernel's: persist = 1 runs the tile path."""
    s = dataclasses.replace(perturbed(S.nacl(nsites=12), 0.1), thermostat="none")
    say("persist ineligible nacl", s.n)
    e = persist_engine(E, s, 8)
    st = e.run(10, energy_every=1)
    assert e.persist_info()["runs"] == 0
    r = orc.md_run(s, 10)
    assert np.allclose(st["temp"][:, 0], r["temp"], rtol=1e-4)
    e.close()


def _slope_and_error(H, nblock=10):
    t = np.arange(H.size, dtype=np.float64)
    slope = np.polyfit(t, H, 1)[0]
    m = H.size // nblock
    bs = np.array([np.polyfit(t[:m], H[b * m:(b + 1) * m], 1)[0] for b in range(nblock)])
    return slope, bs.std(ddof=1) / np.sqrt(nblock)


def test_persist_nve_drift_10000_steps(E, orc):
    """Argon 864, NVE velocity Verlet dt 2 fs, 10,000 steps in one persistent
    launch: |drift| of the conserved energy <= the oracle's + 2 sigma (block
    standard errors of the two slopes)."""
    n = 10000
    s = S.argon()
    say("persist nve drift argon 10000")
    e = persist_engine(E, s, 16)
    st = e.run(n, energy_every=1)
    assert e.persist_info()["runs"] == 1
    H = st["conserved"][:, 0].astype(np.float64)
    e.close()
    r = orc.md_run(s, n)
    Ho = r["conserved"]
    sg, eg = _slope_and_error(H)
    so, eo = _slope_and_error(Ho)
    sigma = np.hypot(eg, eo)
    say("  drift per 1000 steps gpu", sg * 1e3, "+-", eg * 1e3, "oracle", so * 1e3, "+-", eo * 1e3)
    assert abs(H[0] - Ho[0]) <= 1e-4 * abs(Ho[0])
    assert abs(sg) <= abs(so) + 2.0 * sigma


# the workgroups' edges: two atoms, part of a workgroup, 32 workgroups of 512 threads (they fit
# one XCD) and 33 (then 1024 threads), the most atoms, more workgroups than an XCD has CUs
@pytest.mark.parametrize("n,lanes", [(2, 4), (33, 16), (1024, 16), (1025, 16), (2048, 8), (2049, 8), (4096, 4),
                                     (2049, 16), (4096, 16)])
@pytest.mark.parametrize("thermostat", ["none", "berendsen"])
def test_persist_workgroup_edges(E, orc, n, lanes, thermostat):
    """Forces of the last step equal the oracle's at the positions that came with them, and the
    recorded kinetic energy is that of the velocities, whatever the split into workgroups."""
    say("persist edges", n, lanes, thermostat)
    rng = np.random.default_rng(n)
    s = S.argon(ncell=4).copy()
    m = max(9, int(np.ceil(n ** (1 / 3))))
    g = rng.permutation(m ** 3)[:n]
    L = 4.0 * m
    x = (np.stack([g // m // m, g // m % m, g % m], 1) + 0.5) * 4.0 - L / 2 + rng.uniform(-0.3, 0.3, (n, 3))
    s.box, s.pos = np.full(3, L, np.float32), x.astype(np.float32)
    s.vel = rng.normal(0.0, 2e-3, (n, 3)).astype(np.float32)
    s.type, s.charge = np.zeros(n, np.int32), np.zeros(n, np.float32)
    s.integrator, s.thermostat = ("vverlet", "none") if thermostat == "none" else ("leapfrog", "berendsen")
    e = E.Engine.from_system(s)
    e.set_launch(lanes=lanes, persist=1)
    x0 = e.download()[0]
    st = e.run(5)
    assert e.persist_info()["runs"] == 1
    p, v, f = e.download()
    so = s.copy()
    # velocity Verlet returns forces and positions of one time, leapfrog forces of the step before
    so.pos = p if thermostat == "none" else S.wrap_centered(p.astype(np.float64) - s.dt * v.astype(np.float64),
                                                            s.box.astype(np.float64)).astype(np.float32)
    Fo = orc.forces(so)[0]
    # leapfrog: the position is rounded once more (2^-23 L), against a curvature of some 1e3 kJ/mol/A^2
    assert np.abs(f - Fo).max() <= (1e-5 if thermostat == "none" else 1e-3) * max(np.abs(Fo).max(), 1.0)
    ke = 0.5 * (1e4 * s.ff.masses[0] * v.astype(np.float64) ** 2).sum()
    assert abs(st["ke"][-1, 0] - ke) <= 1e-6 * ke
    assert not np.array_equal(p, x0)
    e.close()


def test_persist_engines_side_by_side(E):
    """Several engines' persistent runs at once, a thread each, give the bits of one alone."""
    import threading
    s = perturbed(S.argon(), 0.1)

    def work(out, k):
        e = persist_engine(E, s, 16)
        for _ in range(10):
            e.run(100, stats=False)
        out[k] = e.download()
        e.close()

    alone, beside = {}, {}
    work(alone, 0)
    threads = [threading.Thread(target=work, args=(beside, k)) for k in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert len(beside) == 3
    for k in beside:
        for a, b in zip(alone[0], beside[k]):
            assert np.isfinite(a).all() and np.array_equal(a, b)


@pytest.mark.parametrize("thermostat", ["none", "berendsen"])
@pytest.mark.parametrize("stats", [False, True])
def test_persist_one_step_runs(E, thermostat, stats):
    """Leapfrog runs of a single step (without sums nothing is exchanged between the workgroups),
    from even and odd steps, between two longer ones: the tile path's trajectory.  Ten steps
    differ by the rounding of FP32 force sums (some 1e-6 of a force) and of the positions
    (1e-6 A each)."""
    s = dataclasses.replace(perturbed(S.argon(), 0.1), integrator="leapfrog", thermostat=thermostat, tau=100.0, T0=120.0)
    say("persist one-step runs", s.n, thermostat, "stats", stats)
    out = []
    for persist in (0, 1):
        e = E.Engine.from_system(s)
        e.set_launch(persist=persist, lanes=16)
        frames = []
        for n in (1, 1, 1, 2, 1, 1, 3):
            e.run(n, stats=stats)
            frames.append(e.download())
        assert e.info()["steps"] == 10 and e.persist_info()["runs"] == 7 * persist
        out.append(frames)
        e.close()
    for (p0, v0, f0), (p1, v1, f1) in zip(*out):
        d = p1.astype(np.float64) - p0
        d -= s.box * np.rint(d / s.box)
        assert np.abs(d).max() < 2e-5
        assert rel_rms(v1, v0) < 1e-5 and rel_rms(f1, f0) < 1e-5


def sampled(s):
    """The bits of a few runs of an engine: statistics and the frame they end in."""
    def bits(e, runs):
        out = [e.run(n, energy_every=3) for n in runs]
        return [x.tobytes() for x in out] + [x.tobytes() for x in e.download()]
    return bits


@pytest.mark.parametrize("integrator,thermostat", [("vverlet", "none"), ("leapfrog", "berendsen")])
def test_persist_falls_back_when_its_xcd_is_taken(E, integrator, thermostat):
    """A placed run that misses a workgroup ends by its bounded wait and is replayed on any CU with
    the same bits (frames, kinetic energies, temperatures); the XCD is tried again after 16 runs,
    after 32 when it is found taken once more, and at once after a placed run or set_launch."""
    s = dataclasses.replace(perturbed(S.argon(), 0.1), integrator=integrator, thermostat=thermostat, tau=100.0, T0=120.0)
    say("persist fallback", s.n, integrator, thermostat)
    bits = sampled(s)
    runs = [20, 1, 30]
    e = persist_engine(E, s, 16)
    want = bits(e, runs)
    assert e.persist_placement() == dict(fallbacks=0, hold=0)
    e.close()
    e = persist_engine(E, s, 16)
    e.test_control(E.TEST_LATE_WORKGROUP, 1)
    assert bits(e, runs) == want
    assert e.persist_placement() == dict(fallbacks=1, hold=13)
    assert e.persist_info()["runs"] == 3 and e.persist_info()["replays"] == 0
    for _ in range(13):
        e.run(1, stats=False)
    e.test_control(E.TEST_LATE_WORKGROUP, 1)
    e.run(2, stats=False)
    assert e.persist_placement() == dict(fallbacks=2, hold=31)
    e.set_launch(persist=1)
    assert e.persist_placement()["hold"] == 0
    e.run(2, stats=False)
    assert e.persist_placement() == dict(fallbacks=2, hold=0)
    e.close()


def test_persist_engines_side_by_side_record_the_same(E):
    """Engines side by side record the statistics of one alone, whatever their placement."""
    import threading
    s = dataclasses.replace(perturbed(S.argon(), 0.1), integrator="leapfrog", thermostat="berendsen", tau=100.0, T0=120.0)
    say("persist side by side, berendsen")
    bits = sampled(s)

    def work(out, k):
        e = persist_engine(E, s, 16)
        if k % 2:
            e.test_control(E.TEST_LATE_WORKGROUP, 1)
        out[k] = bits(e, [50] * 6)
        e.close()

    out = {}
    work(out, 0)
    threads = [threading.Thread(target=work, args=(out, k)) for k in range(1, 5)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert len(out) == 5
    for k in out:
        assert out[k] == out[0], k


def test_persist_long_run_does_not_hold_back_others(E):
    """Short runs of other engines end while an engine with as many workgroups as an XCD has CUs is
    in the middle of a long run (three engines, since two streams may share a hardware queue)."""
    import threading
    import time
    s = S.argon(ncell=7).copy()   # 1,024 of its 1,372 atoms: 32 workgroups of 512 threads with 16 lanes
    s.pos, s.vel, s.type, s.charge = s.pos[:1024], s.vel[:1024], s.type[:1024], s.charge[:1024]
    say("persist long run beside short ones")
    big = persist_engine(E, s, 16)
    small = [persist_engine(E, perturbed(S.argon(ncell=4), 0.1), 16) for _ in range(3)]
    for e in [big] + small:
        e.run(10, stats=False)
    ended = {}

    def work(k, e, n):
        e.run(n, stats=False)
        ended[k] = time.perf_counter()

    threads = [threading.Thread(target=work, args=("big", big, 40000))]
    threads[0].start()
    time.sleep(0.02)
    assert "big" not in ended
    for k, e in enumerate(small):
        threads.append(threading.Thread(target=work, args=(k, e, 100)))
        threads[-1].start()
    for t in threads:
        t.join()
    assert min(ended[k] for k in range(3)) < ended["big"] - 0.02
    for e in [big] + small:
        e.close()

"""Force matching on the GPU at the benchmark's size: NaCl 4,096 ions x 64
frames (frames sampled from a GPU trajectory, targets = forces of the model
with eps, sigma and the charge scale perturbed by up to 5 %).

- loss and gradient of all 64 frames against the FP64 oracle;
- the GPU gradient against central finite differences (h = 1e-4 relative) of
  the GPU loss itself;
- one Adam step through the torch wrapper (fm_loss / FMLoss).
"""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def say(*a):
    print("[case]", *a, file=sys.stderr, flush=True)


@pytest.fixture(scope="module")
def problem():
    from md_gpu_amd import engine as E
    from md_gpu_amd.fit import nacl_problem
    say("fm problem nacl 4096 x 64 frames")
    e, fm, base, frames, tgt, theta_t = nacl_problem(E.Engine, nframes=64)
    yield e, fm, base, frames, tgt, theta_t
    e.close()


def test_all_64_frames_match_oracle(problem, orc):
    e, fm, base, frames, tgt, _ = problem
    say("fm 64 frames vs oracle")
    loss, g1, g2, gq = e.fm_loss_grad(base.ff.lj1, base.ff.lj2, 1.0)
    lo, o1, o2, oq = orc.fm_loss_grad(frames, base.type, base.charge, base.box, base.ff, 1.0, tgt)
    say("  loss", loss, lo, "gq", gq, oq)
    assert abs(loss - lo) <= 1e-5 * lo
    assert abs(gq - oq) <= 1e-5 * abs(oq)
    np.testing.assert_allclose(g1, o1, rtol=1e-5, atol=1e-5 * np.abs(o1).max())
    np.testing.assert_allclose(g2, o2, rtol=1e-5, atol=1e-5 * np.abs(o2).max())


def _central(fm, th, k, h):
    tp, tm = th.copy(), th.copy()
    tp[k] += h
    tm[k] -= h
    return (fm.loss_grad(tp)[0] - fm.loss_grad(tm)[0]) / (2 * h)


def test_gradient_matches_gpu_central_differences(problem):
    """d loss / d theta (adjoint kernel + chain rule) vs (L(theta + h e_k) -
    L(theta - h e_k)) / 2h of the GPU loss itself.

    Two error sources bound what finite differences of an FP32 force field
    can show.  Rounding: each force is an FP32 sum of ~400 pair terms, so a
    relative step of 1e-4 moves it by only ~10x its rounding error, and the
    loss difference over 786k components keeps ~1e-4 of that noise, hence the
    1e-3 bar at h = 1e-4 theta_k.  Truncation: O(h^2) terms of relative size
    ~220 (h / sigma)^2 for sigma^12.  The five-point stencil at h = 3e-3
    theta_k has thirty times less rounding noise and truncation terms below
    1e-6 of the largest component (measured on the FP64 oracle for the same
    model), so that check holds to 5e-5."""
    _, fm, *_ = problem
    th = fm.theta0() * (1.0 + 0.02 * np.cos(np.arange(7)))   # away from the base and the target
    loss, g = fm.loss_grad(th)
    gmax = np.abs(g).max()
    say("fm central FD, loss", loss)
    for k in range(fm.nparam):
        fd4 = _central(fm, th, k, 1e-4 * abs(th[k]))
        h = 3e-3 * abs(th[k])
        fdr = (4.0 * _central(fm, th, k, h) - _central(fm, th, k, 2 * h)) / 3.0   # five-point stencil
        say("  k", k, "adjoint", g[k], "fd h=1e-4", fd4, "five-point h=3e-3", fdr)
        assert abs(g[k] - fd4) <= 1e-3 * gmax, (k, g[k], fd4)
        assert abs(g[k] - fdr) <= 5e-5 * gmax, (k, g[k], fdr)


def test_loss_small_at_target_parameters(problem):
    _, fm, _, _, _, theta_t = problem
    l0, _ = fm.loss_grad(fm.theta0())
    lt, gt = fm.loss_grad(theta_t)
    say("fm loss at base / target", l0, lt)
    assert lt < 1e-8 * l0


def test_adam_step_through_torch_wrapper(problem):
    import torch
    from md_gpu_amd.fit import FMLoss, fit
    _, fm, *_ = problem
    th = torch.tensor(fm.theta0(), dtype=torch.float64, requires_grad=True)
    loss = FMLoss.apply(th, fm)
    loss.backward()
    ref_loss, ref_g = fm.loss_grad(fm.theta0())
    say("fm torch", loss.item(), ref_loss)
    assert loss.item() == ref_loss                 # the GPU evaluation is deterministic
    np.testing.assert_array_equal(th.grad.numpy(), ref_g)
    theta, losses = fit(fm, steps=3, lr=5e-3)
    say("fm adam losses", losses)
    assert losses[-1] < losses[0]
    assert np.all(np.isfinite(theta))



@pytest.mark.parametrize("lanes", [4, 8, 16])
@pytest.mark.parametrize("ntype", [1, 2, 3])
@pytest.mark.parametrize("coulomb", ["rf", "wolf", "damped"])
def test_one_pass_small_matches_oracle(orc, lanes, ntype, coulomb):
    """The single pass with every table size (1, 2 and 4 types), lane count and Coulomb kind, on
    frames with a partial last tile, at the bars of the full-size problem."""
    import dataclasses
    from md_gpu_amd import engine as E, systems as S
    from md_gpu_amd.fit import ForceMatch
    say("fm small", lanes, ntype, coulomb)
    s = S.nacl(nsites=10)
    k = [0, 1, 1][:ntype]
    ff = dataclasses.replace(s.ff, names=["Na", "Cl", "Br"][:ntype], masses=s.ff.masses[k], rc=8.0,
                             lj1=s.ff.lj1[np.ix_(k, k)], lj2=s.ff.lj2[np.ix_(k, k)],
                             coulomb={"rf": S.COUL_RF, "wolf": S.COUL_WOLF, "damped": S.COUL_DAMPED}[coulomb])
    typ = np.zeros_like(s.type) if ntype == 1 else s.type.copy()
    if ntype == 3:
        typ[::3] = np.where(typ[::3] == 1, 2, typ[::3])
    base = dataclasses.replace(s, ff=ff, type=typ)
    rng = np.random.default_rng(4)
    frames = S.wrap_centered(base.pos + np.clip(rng.normal(0.0, 0.2, (3, base.n, 3)), -0.5, 0.5),
                             base.box.astype(np.float64)).astype(np.float32)
    targets = rng.normal(0.0, 50.0, frames.shape).astype(np.float32)
    e = E.Engine.from_system(base)
    e.set_launch(lanes=lanes)
    ForceMatch(e, base, frames, targets)
    loss, g1, g2, gq = e.fm_loss_grad(ff.lj1, ff.lj2, 1.0)
    e.close()
    lo, o1, o2, oq = orc.fm_loss_grad(frames, base.type, base.charge, base.box, ff, 1.0, targets)
    assert abs(loss - lo) <= 1e-5 * lo
    assert abs(gq - oq) <= 1e-5 * abs(oq)
    np.testing.assert_allclose(g1, o1, rtol=1e-5, atol=1e-5 * np.abs(o1).max())
    np.testing.assert_allclose(g2, o2, rtol=1e-5, atol=1e-5 * np.abs(o2).max())


def _without_lj(ff, t):
    """ff with every Lennard-Jones entry of type t zero."""
    import dataclasses
    lj1, lj2 = ff.lj1.copy(), ff.lj2.copy()
    lj1[t, :] = lj1[:, t] = lj2[t, :] = lj2[:, t] = 0.0
    return dataclasses.replace(ff, lj1=lj1, lj2=lj2)


@pytest.mark.parametrize("lanes", [4, 8, 16])
@pytest.mark.parametrize("free", [0, 1])
def test_two_passes_follow_the_trial_table(orc, lanes, free):
    """The base force field has no Lennard-Jones interactions on one type, the trial table has:
    two passes and one pass both equal the oracle, at the bars of the full-size problem; so
    they do for the base's own table."""
    import dataclasses
    from md_gpu_amd import engine as E, systems as S
    from md_gpu_amd.fit import ForceMatch
    say("fm type without LJ in the base", lanes, free)
    s = S.nacl(nsites=10, ff=S.nacl_ff(rc=8.0))
    base = dataclasses.replace(s, ff=_without_lj(s.ff, free))
    rng = np.random.default_rng(6)
    frames = S.wrap_centered(base.pos + np.clip(rng.normal(0.0, 0.2, (3, base.n, 3)), -0.5, 0.5),
                             base.box.astype(np.float64)).astype(np.float32)
    targets = rng.normal(0.0, 50.0, frames.shape).astype(np.float32)
    e = E.Engine.from_system(base)
    ForceMatch(e, base, frames, targets)
    for ff in (s.ff, base.ff):
        lo, o1, o2, oq = orc.fm_loss_grad(frames, base.type, base.charge, base.box, ff, 1.0, targets)
        for fused in (0, 1):
            e.set_launch(lanes=lanes, fm_fused=fused)
            loss, g1, g2, gq = e.fm_loss_grad(ff.lj1, ff.lj2, 1.0)
            say("  fused", fused, "loss", loss, lo)
            assert abs(loss - lo) <= 1e-5 * lo
            assert abs(gq - oq) <= 1e-5 * abs(oq)
            np.testing.assert_allclose(g1, o1, rtol=1e-5, atol=1e-5 * np.abs(o1).max())
            np.testing.assert_allclose(g2, o2, rtol=1e-5, atol=1e-5 * np.abs(o2).max())
    e.close()


def test_bonded_loss_follows_the_trial_table(orc):
    """Flexible water, Lennard-Jones on the oxygens only, and a trial table with hydrogen terms
    (bonded systems always take two passes): the loss is the oracle's."""
    import ctypes as C
    import dataclasses
    from md_gpu_amd import engine as E, systems as S
    say("fm flexible water, trial table with hydrogen terms")
    base = S.water(nmol=343)
    base = dataclasses.replace(base, ff=dataclasses.replace(base.ff, rc=8.0))
    assert (base.ff.lj1[1] == 0).all()
    eps, sig = np.array([[0.65, 0.2], [0.2, 0.1]]), np.array([[3.166, 1.5], [1.5, 1.0]])
    trial = dataclasses.replace(base.ff, lj1=48.0 * eps * sig ** 12, lj2=24.0 * eps * sig ** 6)
    rng = np.random.default_rng(7)
    frame = S.wrap_centered(base.pos + np.clip(rng.normal(0.0, 0.05, (base.n, 3)), -0.1, 0.1),
                            base.box.astype(np.float64)).astype(np.float32)
    target = rng.normal(0.0, 50.0, (1, base.n, 3)).astype(np.float32)
    e = E.Engine.from_system(base)
    e.fm_set_frames(frame[None], target)
    bonds, angles = (np.ascontiguousarray(x, np.int32) for x in (base.bonds, base.angles))
    E._check(E.lib().md_set_topology(e._h, len(bonds), bonds.ctypes.data_as(C.c_void_p), len(angles),
                                     angles.ctypes.data_as(C.c_void_p)))
    for ff in (trial, base.ff):
        so = dataclasses.replace(base.copy(), ff=ff, pos=frame)
        lo = ((orc.forces(so)[0] - target[0]) ** 2).mean()
        loss = e.fm_loss_grad(ff.lj1, ff.lj2, 1.0)[0]
        say("  loss", loss, lo)
        assert abs(loss - lo) <= 1e-5 * lo
    e.close()

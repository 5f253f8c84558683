"""The moment form of the row-band iteration (csrc/strip_moment.hip) against
the CPU oracle, at the edges of what it takes: band and grid remainders, runs
clipped by the image, lines whose column is clamped, steep events, anisotropic
pixels, the smallest lists and the smallest sigma.

Tolerances, derived: a kernel value's polynomial factor is within 7.8e-7 and
its 8-term FP32 evaluation within 8 x 6e-8 x e^2 = 3.5e-6 of exact (the terms'
magnitudes sum to at most e^2 times the value); with the row terms' own FP32
rounding (under 5e-6 between the row-band kernels and the oracle) a forward
projection is within 1e-5.  Support counts are integers: exact.  Images: the
graded bar, rel-L2 1e-4.
"""
import numpy as np
import pytest

from conftest import print_case

pytestmark = pytest.mark.gpu

# n_z, n_y, pixel width, height, sigma_z, sigma_dl, R, L, phantom half sizes,
# events.  All of them take the moment form (asserted): where bins hold few pairs,
# wide lines and many bins stay on the lists.
CASES = {
    "command line defaults, sigma 1.5 px": (
        100, 100, 0.01, 0.01, 0.015, 0.06, 0.5, 1.0, 0.3, 0.3, 20_011),
    "object beyond every edge": (
        61, 37, 5.0, 5.0, 10.0, 42.0, 250.0, 700.0, 220.0, 150.0, 6_000),
    "one row past a band, flat pixels": (
        128, 33, 2.0, 1.5, 10.0, 42.0, 120.0, 500.0, 100.0, 20.0, 5_000),
    "fifteen rows, tall pixels": (
        90, 15, 2.0, 4.0, 10.0, 42.0, 120.0, 500.0, 70.0, 25.0, 3_000),
    "narrower than a run": (
        12, 200, 2.0, 2.0, 12.0, 42.0, 300.0, 500.0, 20.0, 150.0, 4_000),
    "steep events": (
        200, 64, 2.0, 2.0, 10.0, 30.0, 70.0, 1200.0, 150.0, 40.0, 5_000),
    "one event": (128, 80, 4.0, 4.0, 10.0, 42.0, 350.0, 500.0, 80.0, 60.0, 1),
    "seventeen events": (
        128, 80, 4.0, 4.0, 10.0, 42.0, 350.0, 500.0, 80.0, 60.0, 17),
    "wide line, dense bins": (
        300, 200, 1.0, 1.0, 10.0, 42.0, 250.0, 500.0, 40.0, 30.0, 30_000),
    # 21000 bins of five pairs on short lines: merged back-projection tasks,
    # clipped by the image
    "many small bins": (
        150, 70, 4.0, 4.0, 10.0, 42.0, 200.0, 500.0, 330.0, 150.0, 40_000),
    # more than 400 pairs per bin: six terms
    "full bins": (
        60, 32, 2.0, 2.0, 30.0, 42.0, 200.0, 200.0, 50.0, 25.0, 300_000),
}


def _case(pystrip_mod, phantom_mod, oracle_mod, name, seed=5):
    n_z, n_y, w, h, sz, sdl, R, L, a, b, n = CASES[name]
    ev = phantom_mod.generate_events(
        [phantom_mod.Ellipse(0.3 * a, -0.2 * b, 0.2 * a, 0.3 * b, 20, 3),
         phantom_mod.Ellipse(0, 0, a, b, 0, 1)], R, L, sz, sdl, n, seed=seed,
        batch=1 << 16)
    g = pystrip_mod.Geometry.make(R, L, n_z, n_y, w, sz, sdl, pixel_height=h)
    og = oracle_mod.geometry(R, L, n_z, n_y, w, h, sz, sdl, 0.0, 0.0)
    return ev, g, og


@pytest.mark.parametrize("name", list(CASES))
def test_moment_form_against_oracle(pystrip_mod, phantom_mod, oracle_mod,
                                    name):
    print_case("moment form:", name)
    ev, g, og = _case(pystrip_mod, phantom_mod, oracle_mod, name)
    rec = pystrip_mod.Reconstruction(g)
    rec.set_events(ev)
    assert rec.plan_forms() == (1, 0)
    _, ne = oracle_mod.support_counts(og, ev)
    assert rec.kernel_evaluations() == int(ne.sum())
    rho = np.random.default_rng(3).uniform(0.5, 2.0, rec.shape).astype(
        np.float32)
    rec.rho = rho
    d = rec.forward().astype(np.float64)
    ref = oracle_mod.forward(og, ev, rho).astype(np.float64)
    assert np.array_equal(d > 0, ref > 0)
    nz = ref > 0
    err = np.max(np.abs(d[nz] - ref[nz]) / ref[nz]) if nz.any() else 0.0
    print("events with support", int(nz.sum()), "of", len(ev), "max rel D",
          err)
    assert err < 1e-5
    rec.iterate(3)
    e = oracle_mod.rel_l2(rec.rho, oracle_mod.mlem(og, ev, rho0=rho,
                                                   iterations=3))
    print("rel-L2", e)
    assert e <= 1e-4


def test_moment_form_non_finite_pixels(pystrip_mod, phantom_mod, oracle_mod):
    # a pixel that is not finite reaches the events whose support holds it
    # and no others: as the pixel-by-pixel kernels give it
    ev, g, og = _case(pystrip_mod, phantom_mod, oracle_mod,
                      "object beyond every edge")
    for value in (np.inf, np.nan):
        print_case("moment form, pixel =", value)
        rho = np.ones((g.n_y_pixels, g.n_z_pixels), np.float32)
        rho[20, 30] = value
        rho[5, 1] = value
        out = []
        for algorithm in (1, 0):
            rec = pystrip_mod.Reconstruction(g)
            rec.set_algorithm(algorithm)
            rec.set_events(ev)
            assert rec.plan_forms() == (1 - algorithm, 0)
            rec.rho = rho
            out.append(rec.forward())
        fine = np.isfinite(out[0])
        assert 0 < fine.sum() < len(ev)
        assert np.array_equal(fine, np.isfinite(out[1]))
        assert np.array_equal(np.isnan(out[0]), np.isnan(out[1]))
        nz = fine & (out[0] > 0)
        assert np.max(np.abs(out[1][nz] - out[0][nz]) / out[0][nz]) < 1e-5


# n_z, n_y, pixel, body half sizes, R, L, events, whether the moment form is the
# faster one (an iteration over the lists and in the moment form, us); all of
# them far from where the two are alike
CHOICES = {
    "few events, long lines": (512, 512, 1.0, 200.0, 200.0, 350.0, 700.0, 300,
                               False),  # 20, 35
    "spread events, long lines": (512, 512, 1.0, 200.0, 200.0, 350.0, 700.0,
                                  10_000, False),  # 67, 202
    "dense events, long lines": (512, 512, 1.0, 200.0, 200.0, 350.0, 700.0,
                                 300_000, True),  # 808, 445
    "short lines": (256, 160, 2.0, 80.0, 60.0, 350.0, 500.0, 3_000,
                    True),  # 105, 34
    "the shortest lines, one event": (61, 37, 5.0, 100.0, 60.0, 250.0, 700.0,
                                      1, True),  # 12, 12; the shorter plan
}


@pytest.mark.parametrize("name", list(CHOICES))
def test_choice_of_the_faster_form(pystrip_mod, phantom_mod, name):
    print_case("choice of the form:", name)
    n_z, n_y, w, a, b, R, L, n, moments = CHOICES[name]
    ev = phantom_mod.generate_events([phantom_mod.Ellipse(0, 0, a, b, 0, 1)],
                                     R, L, 10.0, 42.0, n, seed=7,
                                     batch=1 << 16)
    rec = pystrip_mod.Reconstruction(
        pystrip_mod.Geometry.make(R, L, n_z, n_y, w, 10.0, 42.0))
    rec.set_events(ev)
    assert rec.plan_forms() == ((1, 0) if moments else (0, 1))


def test_moment_form_knobs(pystrip_mod, phantom_mod, oracle_mod):
    # leaving a knob's default takes the lists, returning to it the moment
    # form again: the same reconstruction within rounding
    print_case("moment form and tiling knobs")
    ev, g, og = _case(pystrip_mod, phantom_mod, oracle_mod,
                      "command line defaults, sigma 1.5 px")
    ref = oracle_mod.mlem(og, ev, iterations=2)
    rec = pystrip_mod.Reconstruction(g)
    rec.set_events(ev)
    tiling = rec.band_tiling()
    assert tiling[:2] == (32, 16) and rec.band_groups() == (2, 4)
    assert rec.span_table()
    for change, forms in ((lambda: None, (1, 0)),
                          (lambda: rec.set_exp_mode(0), (0, 1)),
                          (lambda: rec.set_exp_mode(1), (1, 0)),
                          (lambda: rec.set_span_table(False), (0, 1)),
                          (lambda: rec.set_span_table(True), (1, 0)),
                          (lambda: rec.set_algorithm(2), (0, 1)),
                          (lambda: rec.set_algorithm(0), (1, 0))):
        change()
        assert rec.plan_forms() == forms
        rec.rho = np.ones(rec.shape, np.float32)
        rec.iterate(2)
        assert oracle_mod.rel_l2(rec.rho, ref) <= 1e-4
        assert rec.band_tiling()[:2] == tiling[:2]


@pytest.mark.parametrize("name", list(CASES))
def test_moment_form_gradient_against_oracle(pystrip_mod, phantom_mod,
                                             oracle_mod, name):
    # the log-likelihood and its derivatives in FP64.  An event's log D is
    # within 1e-5 (above), its share of d ln sigma, of a size of one, within
    # 2e-5; images as everywhere against FP64: 1e-4.
    print_case("moment form, gradient:", name)
    ev, g, og = _case(pystrip_mod, phantom_mod, oracle_mod, name)
    rec = pystrip_mod.Reconstruction(g)
    rec.set_events(ev)
    assert rec.plan_forms() == (1, 0)
    rho = np.random.default_rng(8).uniform(0.5, 2.0, rec.shape).astype(
        np.float32)
    value, grad, gs = rec.loglik_gradient(rho)
    rv, rg, rs = oracle_mod.loglik_grad(og, ev.astype(np.float64),
                                        rho.astype(np.float64))
    print("value", value, rv, "image", oracle_mod.rel_l2(grad, rg), "sigma",
          gs, rs)
    assert abs(value - rv) <= 1e-5 * len(ev) + 2e-6 * abs(rv)
    assert oracle_mod.rel_l2(grad, rg) <= 1e-4
    sigma = np.array([g.sigma_z, g.sigma_dl])
    assert np.all(np.abs(gs - rs) <= 1e-3 * np.abs(rs) + 2e-5 * len(ev) / sigma)


def test_moment_form_gradient_non_finite_pixels(pystrip_mod, phantom_mod,
                                                oracle_mod):
    # as the lists give it: the events whose support holds the pixel drop out
    # of the image derivative, and no others
    ev, g, og = _case(pystrip_mod, phantom_mod, oracle_mod,
                      "object beyond every edge")
    for value in (np.inf, np.nan):
        print_case("moment form, gradient, pixel =", value)
        rho = np.ones((g.n_y_pixels, g.n_z_pixels), np.float32)
        rho[20, 30] = value
        rho[5, 1] = value
        out = []
        for algorithm in (2, 0):
            rec = pystrip_mod.Reconstruction(g)
            rec.set_algorithm(algorithm)
            rec.set_events(ev)
            assert rec.plan_forms() == ((0, 1) if algorithm else (1, 0))
            out.append(rec.loglik_gradient(rho))
        for a, b in zip(*out):
            a, b = np.asarray(a), np.asarray(b)
            assert np.array_equal(np.isnan(a), np.isnan(b))
            assert np.array_equal(np.isinf(a), np.isinf(b))
        assert np.all(np.isfinite(out[0][1]))
        assert oracle_mod.rel_l2(out[1][1], out[0][1]) <= 1e-5


# members of a batch in the moment form, which has to be a seventh faster than the
# lists there: as CASES
DENSE = {
    # 90 pairs to a bin: one wavefront to a forward task
    "eight terms, one wavefront": (300, 200, 1.0, 1.0, 10.0, 42.0, 250.0,
                                   500.0, 40.0, 30.0, 60_000),
    # 180: four
    "eight terms, four wavefronts": (300, 200, 1.0, 1.0, 10.0, 42.0, 250.0,
                                     500.0, 40.0, 30.0, 120_000),
    # more than 400 pairs to every bin, in two sizes of LDS
    "six terms": (60, 32, 2.0, 2.0, 30.0, 42.0, 200.0, 200.0, 50.0, 25.0,
                  300_000),
    "six terms, shorter lines": (60, 32, 2.5, 2.5, 30.0, 42.0, 200.0, 200.0,
                                 50.0, 25.0, 300_000),
}


@pytest.mark.parametrize("names", [
    ["six terms", "eight terms, one wavefront", "many small bins",
     "wide line, dense bins", "eight terms, four wavefronts",
     "six terms, shorter lines", "one event"],
    # no member over lists, the same kind twice
    ["six terms, shorter lines", "six terms"],
    ["eight terms, one wavefront"]])
def test_moment_form_in_a_batch(pystrip_mod, phantom_mod, oracle_mod, names,
                                monkeypatch):
    # members of every kind of task, several to a launch, among members over
    # lists, iterated together, eagerly and replayed
    # ("many small bins": merged tasks, by the member's own choice)
    print_case("moment form in a batch:", names)
    own = {"many small bins"}
    monkeypatch.setattr("test_gpu_moment.CASES", {**CASES, **DENSE})
    cases = [_case(pystrip_mod, phantom_mod, oracle_mod, n) for n in names]
    refs = [oracle_mod.mlem(og, ev, iterations=5) for ev, _, og in cases]
    for graph in (False, True):
        b = pystrip_mod.Batch()
        b.set_graph(graph)
        for ev, g, _ in cases:
            b.add(g, ev)
        for i, name in enumerate(names):
            if name in own:
                b.member(i).set_algorithm(0)
        b.iterate(2)
        b.iterate(3)
        for i, name in enumerate(names):
            e = oracle_mod.rel_l2(b.rho(i), refs[i])
            print(name, b.member(i).plan_forms(), e)
            moments = name in DENSE or name in own
            assert b.member(i).plan_forms() == ((1, 0) if moments else (0, 1))
            assert e <= 1e-4

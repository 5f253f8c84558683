"""The moment form's image derivatives against FP64, beside those of the
pixel-by-pixel lists: the moment form may not round more.  Every pixel is the
sum of hundreds of contributions less one, so that the rounding of running sums
shows; the events are ones whose pixels in FP32 and in FP64 are nearly the same
(what differs there is common to both forms and would hide the rounding).

The errors differ by 2 % from run to run (the order of the additions): the
moment form may have 1.05 times the lists'.  With all tasks adding to one image
it has 1.17 to 1.75 times the lists'.
"""
import numpy as np
import pytest

from conftest import print_case

pytestmark = pytest.mark.gpu

# n_z, n_y, pixel, sigma_z, sigma_dl, R, L, half sizes of the body, events, seed
CASES = {
    "few rows": (203, 56, 2.5, 10.0, 42.0, 200.0, 640.0, 150.0, 40.0, 96_151,
                 2),
    "long lines": (476, 197, 1.5, 12.0, 42.0, 250.0, 850.0, 200.0, 80.0,
                   150_000, 3),
    "short lines": (194, 136, 2.5, 10.0, 30.0, 260.0, 600.0, 150.0, 100.0,
                    137_443, 1),
    # 17348 bins of 15.5 pairs: back-projection tasks of several bins
    "merged tasks": (194, 136, 2.5, 10.0, 30.0, 260.0, 600.0, 150.0, 100.0,
                     90_000, 1),
}


@pytest.mark.parametrize("name", list(CASES))
def test_image_derivative_rounds_no_more_than_lists(pystrip_mod, phantom_mod,
                                                    oracle_mod, name):
    print_case("image derivative, moments and lists:", name)
    n_z, n_y, w, sz, sdl, R, L, a, b, n, seed = CASES[name]
    ev = phantom_mod.generate_events([phantom_mod.Ellipse(0, 0, a, b, 0, 1)],
                                     R, L, sz, sdl, n, seed=seed, batch=1 << 16)
    g = pystrip_mod.Geometry.make(R, L, n_z, n_y, w, sz, sdl)
    og = oracle_mod.geometry(R, L, n_z, n_y, w, w, sz, sdl, 0.0, 0.0)
    rec = pystrip_mod.Reconstruction(g)
    rec.set_events(ev)
    rho = np.random.default_rng(6).uniform(0.5, 1.5, rec.shape).astype(
        np.float32)
    error = {}
    _, ref, _ = oracle_mod.loglik_grad(og, ev.astype(np.float64),
                                       rho.astype(np.float64))
    for form, algorithm in (("moments", 0), ("lists", 2)):
        rec.set_algorithm(algorithm)
        assert rec.plan_forms() == ((1, 0) if algorithm == 0 else (0, 1))
        _, grad, _ = rec.loglik_gradient(rho)
        error[form] = oracle_mod.rel_l2(grad, ref)
    print("rel-L2 against FP64", error)
    assert error["moments"] <= 1.05 * error["lists"]

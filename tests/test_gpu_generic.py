"""The generic event pass against the CPU oracle: kernel values kept in LDS
(analytic kernel, small boxes, workgroups of 256) and evaluated twice, one image
and four to add to, boxes below, around and far beyond the 2048 pixels that are
kept, fewer workgroups than images, and one context whose event count takes it
from one image to four and back.

Tolerance: the graded bar, rel-L2 1e-4.
"""
import numpy as np
import pytest

from conftest import print_case

pytestmark = pytest.mark.gpu

# n_z, n_y, pixel, sigma_z, sigma_dl, events
SIZES = {
    "small boxes, five events": (64, 48, 4.0, 10.0, 42.0, 5),
    "boxes around 2048 pixels": (256, 160, 2.0, 12.0, 50.0, 3_000),
    "boxes beyond, odd grid": (203, 171, 1.0, 14.0, 60.0, 1_500),
}


@pytest.mark.parametrize("mode", [(1, 1, 1, 0), (0, 0, 0, 0), (0, 1, 0, 1)])
@pytest.mark.parametrize("name", list(SIZES))
def test_generic_pass_against_oracle(pystrip_mod, phantom_mod, oracle_mod,
                                     name, mode):
    print_case("generic event pass:", name, mode)
    n_z, n_y, w, sz, sdl, n = SIZES[name]
    R, L = n_y * w / 2 + 60.0, n_z * w + 100.0
    ev = phantom_mod.generate_events(
        [phantom_mod.Ellipse(0, 0, n_z * w * 0.3, n_y * w * 0.3, 0, 1)], R, L,
        sz, sdl, n, seed=4, batch=1 << 14)
    g = pystrip_mod.Geometry.make(R, L, n_z, n_y, w, sz, sdl)
    og = oracle_mod.geometry(R, L, n_z, n_y, w, w, sz, sdl, 0.0, 0.0)
    rec = pystrip_mod.Reconstruction(g, mode)
    rec.set_algorithm(1)
    rec.set_events(ev)
    rec.iterate(2)
    ref = oracle_mod.mlem(og, ev, iterations=2, mode=mode)
    fine = np.isfinite(ref)
    assert np.array_equal(fine, np.isfinite(rec.rho))
    e = oracle_mod.rel_l2(np.where(fine, rec.rho, 0), np.where(fine, ref, 0))
    print("rel-L2", e)
    assert e <= 1e-4


@pytest.mark.parametrize("threads", [64, 128, 256])
def test_generic_pass_on_changing_event_counts(pystrip_mod, phantom_mod,
                                               oracle_mod, threads):
    # 256 x 160 pixels: four images from 320 events on
    print_case("generic event pass, event counts change, threads", threads)
    n_z, n_y, w, sz, sdl, n = SIZES["boxes around 2048 pixels"]
    R, L = n_y * w / 2 + 60.0, n_z * w + 100.0
    ev = phantom_mod.generate_events(
        [phantom_mod.Ellipse(0, 0, n_z * w * 0.3, n_y * w * 0.3, 0, 1)], R, L,
        sz, sdl, n, seed=9, batch=1 << 14)
    g = pystrip_mod.Geometry.make(R, L, n_z, n_y, w, sz, sdl)
    og = oracle_mod.geometry(R, L, n_z, n_y, w, w, sz, sdl, 0.0, 0.0)
    rec = pystrip_mod.Reconstruction(g, pystrip_mod.MODE_LEGACY_GPU)
    rec.set_launch(0, threads)
    for count in (40, n, 319, 320, 7):
        rec.set_events(ev[:count])
        rec.rho = np.ones(rec.shape, np.float32)
        rec.iterate(2)
        ref = oracle_mod.mlem(og, ev[:count], iterations=2,
                              mode=pystrip_mod.MODE_LEGACY_GPU)
        fine = np.isfinite(ref)
        assert np.array_equal(fine, np.isfinite(rec.rho))
        e = oracle_mod.rel_l2(np.where(fine, rec.rho, 0),
                              np.where(fine, ref, 0))
        print(count, "rel-L2", e)
        assert e <= 1e-4

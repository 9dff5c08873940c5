"""The batched lens analysis on the GPU against the fp64 oracle.

* per ray: the same Fibonacci-lattice rays traced through the same lenses by the float32 kernel
  (roots polished in float64) and the fp64 oracle agree in acceptance, point (1e-8 m), direction
  (1e-6) and weight (1e-6), except rays within float rounding of an aperture edge;
* per lens: the spot (arrived rays, best focus, RMS radius, centroid) from the kernel's summed
  moments agrees with the oracle's over every ray of the lens at every wavelength;
* the irradiance grid holds the transmitted flux that lands on it, and is identical run to run and
  under every launch shape (integer bins);
* the reference's doublet focuses all rays and its paraxial numbers equal the oracle's.
"""
from __future__ import annotations

import math

import numpy as np
import pytest

from owe_hip import lens as L
from pyoracle import LensOracle

pytestmark = pytest.mark.gpu

LENSES = [L.DOUBLET, L.SINGLET] + L.seeded_achromats(6, seed=11, rays_max=200_000)


@pytest.fixture(scope="module")
def batch(cuda):
    b = L.LensBatch(LENSES)
    b.run()
    yield b
    b.close()


@pytest.mark.parametrize("li", range(len(LENSES)))
def test_rays_match_oracle_ray_by_ray(batch, oracle, li):
    lo = LensOracle(oracle, LENSES)
    n = min(LENSES[li].rays, 8192)
    idx = np.arange(n, dtype=np.uint64)
    for w in (0, 4, 6):
        g = batch.trace(li, w, idx)
        c = lo.trace(li, L.FRAUNHOFER7[w], idx)
        okg, okc = g[:, 6] > 0, c[:, 6] > 0
        both = okg & okc
        flips = int((okg != okc).sum())
        dp = np.abs(g[both, :3] - c[both, :3]).max(initial=0)
        dd = np.abs(g[both, 3:6] - c[both, 3:6]).max(initial=0)
        dT = np.abs(g[both, 6] - c[both, 6]).max(initial=0)
        print(f"lens {li} λ{w}: {both.sum()} both arrive, {flips} flips, |Δp| {dp:.2e} |Δd| {dd:.2e} |ΔT| {dT:.2e}",
              flush=True)
        assert flips <= max(2, n // 2000)
        assert dp < 1e-8 and dd < 1e-6 and dT < 1e-6


@pytest.mark.parametrize("li", range(len(LENSES)))
def test_spot_matches_oracle(batch, oracle, li):
    per, mom, _ = batch.results()
    lo = LensOracle(oracle, LENSES)
    ms = np.array([lo.moments(li, lam)[0] for lam in L.FRAUNHOFER7])
    _, px = lo.moments(li, L.LAMBDA_D)
    lv = px["last_vertex_z"]
    s = L.spot(ms.sum(axis=0), lv + px["bfl"], lv)
    r = per[li]
    print(f"lens {li}: arrived {r['arrived']} / {s['arrived']}, rms {r['rms_best']:.6e} / {s['rms_best']:.6e}, "
          f"focus {r['best_focus_z']:.9f} / {s['best_focus_z']:.9f}", flush=True)
    assert r["efl"] == pytest.approx(px["efl"], rel=1e-12)
    assert r["bfl"] == pytest.approx(px["bfl"], rel=1e-12)
    assert r["entrance_pupil_radius"] == pytest.approx(px["entrance_pupil_radius"], rel=1e-12)
    assert abs(r["arrived"] - s["arrived"]) <= max(2, s["arrived"] // 2000)
    assert r["rms_best"] == pytest.approx(s["rms_best"], rel=2e-3)
    assert r["best_focus_z"] == pytest.approx(s["best_focus_z"], abs=2e-7)
    assert r["centroid_y"] == pytest.approx(s["centroid_y"], abs=1e-8)
    assert np.abs(mom[li, :, 0] - ms[:, 0]).max() <= max(2, s["arrived"] // 2000)


def test_ring_pupil_matches_oracle(cuda, oracle):
    # spotAt's hexapolar rings: six (the reference's analyzeLens call) and 300 (270,901 rays).
    lenses = [L.SINGLET.with_rings(6), L.DOUBLET.with_rings(6), LENSES[2].with_rings(300)]
    b = L.LensBatch(lenses)
    b.run()
    per, mom, _ = b.results()
    lo = LensOracle(oracle, lenses)
    for li, p in enumerate(lenses):
        idx = np.arange(min(p.rays, 20000), dtype=np.uint64)
        g = b.trace(li, 4, idx)
        c = lo.trace(li, L.FRAUNHOFER7[4], idx)
        okg, okc = g[:, 6] > 0, c[:, 6] > 0
        both = okg & okc
        flips = int((okg != okc).sum())
        dp = np.abs(g[both, :3] - c[both, :3]).max(initial=0)
        ms = np.array([lo.moments(li, lam)[0] for lam in L.FRAUNHOFER7])
        print(f"rings lens {li}: {p.rays} rays, {both.sum()} both arrive, {flips} flips, |Δp| {dp:.2e}, "
              f"arrived {per[li]['arrived']} / {int(ms[:, 0].sum())}", flush=True)
        assert flips <= 2 and dp < 1e-8
        assert abs(per[li]["arrived"] - ms[:, 0].sum()) <= max(2, ms[:, 0].sum() // 2000)
    b.close()


def test_doublet_focuses_every_ray_on_axis(cuda):
    # On axis every ray of the reference's achromat arrives (tests/test_instruments.cpp:333).
    b = L.LensBatch([L.DOUBLET], L.c_settings(field_deg=0.0))
    b.run()
    r = b.results()[0][0]
    b.close()
    assert r["arrived"] == r["launched"]
    assert 0.9 < r["transmitted"] < 1.0


def test_irradiance_holds_the_flux_that_lands_and_is_reproducible(cuda):
    half = 3e-3  # wide enough for the seven wavelengths' defocus
    b = L.LensBatch(LENSES[:3], L.c_settings(half_size=half))
    b.run()
    per, mom, irr = b.results(irradiance=True)
    b.set_shape(blocks_per_cu=1, rays_per_item=64)
    b.run()
    per2, mom2, irr2 = b.results(irradiance=True)
    assert np.array_equal(irr, irr2)
    assert [r["arrived"] for r in per] == [r["arrived"] for r in per2]
    for li, p in enumerate(LENSES[:3]):
        pix = 2 * half / irr.shape[-1]
        flux = irr[li].sum() * pix * pix
        beam = math.pi * (0.999 * per[li]["entrance_pupil_radius"]) ** 2 * math.cos(math.radians(0.5))
        print(f"lens {li}: flux on the grid {flux:.6e}, transmitted {per[li]['transmitted'] * beam:.6e}", flush=True)
        # All the transmitted flux lands on the grid, up to the fixed-point rounding of each ray.
        assert flux == pytest.approx(per[li]["transmitted"] * beam, rel=1e-4)
    b.close()


def test_autotune_keeps_the_results(cuda):
    b = L.LensBatch(LENSES[:4])
    b.run()
    per, _, irr = b.results(irradiance=True)
    ms = b.autotune()
    b.run()
    per2, _, irr2 = b.results(irradiance=True)
    print(f"autotune: {ms:.3f} ms", flush=True)
    assert ms > 0
    assert np.array_equal(irr, irr2)
    for a, c in zip(per, per2):
        assert a["arrived"] == c["arrived"]
        assert c["rms_best"] == pytest.approx(a["rms_best"], rel=1e-9)
    b.close()


def _oracle_grid(lo, li, lens, per, settings, planes, step, half, px):
    """The through-focus grids binned in double from the oracle's rays: every arrived ray of every
    wavelength carries T·π(0.999 r_EP)² cos θ / (rays · nλ) of flux into the bin its line crosses on
    each plane (plane k at the paraxial image + (k − (P − 1)/2)·step)."""
    r = per[li]
    idx = np.arange(lens.rays, dtype=np.uint64)
    theta = math.radians(settings.field_deg)
    nw = settings.n_wavelengths
    grid = np.zeros((planes, px, px))
    z0 = r["last_vertex_z"] + r["bfl"]
    cy = r["efl"] * math.tan(theta)
    flux = math.pi * (0.999 * r["entrance_pupil_radius"]) ** 2 * math.cos(theta) / (lens.rays * nw)
    pix = 2 * half / px
    for w in range(nw):
        t = lo.trace(li, settings.wavelengths[w], idx)
        t = t[t[:, 6] > 0]
        for k in range(planes):
            z = z0 + (k - 0.5 * (planes - 1)) * step
            s = (z - t[:, 2]) / t[:, 5]
            gx = (t[:, 0] + t[:, 3] * s) / half
            gy = (t[:, 1] + t[:, 4] * s - cy) / half
            fx, fy = (gx + 1) * 0.5 * px, (1 - gy) * 0.5 * px
            ok = (fx >= 0) & (fy >= 0) & (fx < px) & (fy < px)
            np.add.at(grid[k], (fy[ok].astype(int), fx[ok].astype(int)), t[ok, 6] * flux / (pix * pix))
    return grid


def test_through_focus_stack_matches_the_oracle_bin_by_bin(cuda, oracle):
    """Five planes 40 µm apart about the paraxial image of two lenses: every bin of every plane
    against the oracle's rays binned in double (a ray within float rounding of a bin edge may land in
    its neighbour); the middle plane equals a one-plane run bit for bit; the sharpest plane lies at, or next to, the plane nearest the best focus."""
    lenses = [LENSES[1], LENSES[2]]
    half, planes, step = 0.25e-3, 5, 40e-6
    st = L.c_settings(half_size=half, planes=planes, focus_step=step, pixels=64)
    b = L.LensBatch(lenses, st)
    b.run()
    per, _, irr = b.results(irradiance=True)
    one = L.LensBatch(lenses, L.c_settings(half_size=half, pixels=64))
    one.run()
    _, _, irr1 = one.results(irradiance=True)
    one.close()
    b.close()
    assert irr.shape == (2, planes, 64, 64)
    assert np.array_equal(irr[:, planes // 2], irr1[:, 0])
    lo = LensOracle(oracle, lenses)
    for li, p in enumerate(lenses):
        want = _oracle_grid(lo, li, p, per, st, planes, step, half, 64)
        got = irr[li].astype(np.float64)
        close = np.abs(got - want) <= 1e-5 * np.maximum(np.abs(want), np.abs(got)).max()
        flux = got.sum(axis=(1, 2))
        print(f"lens {li}: {close.mean():.5f} of bins agree; plane flux {flux / flux.max()}; peak per plane "
              f"{got.max(axis=(1, 2))}", flush=True)
        assert close.mean() > 0.995
        assert np.abs(got.sum() - want.sum()) <= 1e-4 * want.sum()


@pytest.mark.parametrize("field", [0.5, 30.0, 55.0])
def test_conic_roots_of_every_form_match_oracle(cuda, oracle, field):
    """Rows of either curvature, shallow to hemispherical, flat, ellipsoids, paraboloids and hyperboloids,
    met steeply and at the edge of their apertures: the row's first crossing, whichever root it is.
    A coordinate here is at most 0.3 m, so it rounds to 3e-8 m at most and a direction to that over the
    row's radius (1 cm and more); 99 % of the rays stay within three and ten times those, the others graze
    a row or the critical angle, where refraction magnifies without bound."""
    rng = np.random.default_rng(int(field) + 3)
    lenses = []
    for k in range(48):
        rows = []
        for j in range(1 + k % 3):
            R = rng.uniform(12, 80) * rng.choice((-1, 1)) if rng.random() < 0.9 else math.inf
            conic = rng.choice((0.0, -1.0, rng.uniform(-2, 1)))
            sd = rng.uniform(0.1, 0.95) * min(abs(R), 60.0) / math.sqrt(max(1.0, 1 + conic))
            glass = "air" if j == 2 or (j == 1 and k % 2) else ("N-BK7", "N-SF11")[j % 2]
            rows.append(L.Surface(R, rng.uniform(1.0, 30.0), glass, sd, k=conic, stop=j == 0))
        lenses.append(L.Prescription(rows, rays=2048))
    b = L.LensBatch(lenses, L.c_settings(field_deg=field))
    lo = LensOracle(oracle, lenses, field_deg=field)
    idx = np.arange(2048, dtype=np.uint64)
    total = flips = far = 0
    for li in range(len(lenses)):
        g, c = b.trace(li, 4, idx), lo.trace(li, L.FRAUNHOFER7[4], idx)
        both = (g[:, 6] > 0) & (c[:, 6] > 0)
        total += int(both.sum())
        flips += int(((g[:, 6] > 0) != (c[:, 6] > 0)).sum())
        far += int(((np.abs(g[both, :3] - c[both, :3]).max(1) > 1e-7) |
                    (np.abs(g[both, 3:6] - c[both, 3:6]).max(1) > 3e-5)).sum())
    b.close()
    print(f"field {field}: {total} rays arrive on both, {flips} flips, {far} beyond the bound", flush=True)
    assert total > 20 * 2048 and flips <= total // 1000 and far <= total // 100


@pytest.mark.parametrize("asphere", [(3e5, -4e5, 1e5, -4e5), (0.0, -4e5, 3e5, -1e5)])
@pytest.mark.parametrize("params", [0, 2])
def test_afocal_angles_on_both_sides_of_the_axis(cuda, oracle, asphere, params):
    """Two aspheric plates (afocal, magnification 1) at 60 degrees: some rays leave more than a right angle from the
    paraxial apparent direction. The sums of angles are the oracle's up to rays that only one of the two loses
    (an angle below π/2 each) and 1e-6 a ray, the direction's error in this file's other tests times the plates' steepness."""
    rows = [L.Surface(math.inf, t, g, sd, A=(a,), stop=k == 0)
            for k, (t, g, sd, a) in enumerate(zip((4.0, 2.0, 4.0, 4.0), ("N-SF11", "air", "N-SF11", "air"),
                                                  (8.0, 12.0, 14.0, 16.0), asphere))]
    p = L.Prescription(rows, rays=4096)
    b = L.LensBatch([p], L.c_settings(field_deg=60.0, pixels=0))
    if params:
        b.set_params([(0, L.PARAM_A4), (3, L.PARAM_A4)][:params])
    b.run()
    per, mom, _ = b.results()
    lo = LensOracle(oracle, [p], field_deg=60.0)
    assert per[0]["afocal"]
    strays = 0
    for w, lam in enumerate(L.FRAUNHOFER7):
        ray = lo.trace(0, lam, np.arange(p.rays, dtype=np.uint64))
        ray = ray[ray[:, 6] > 0]
        strays += int((ray[:, 4] / ray[:, 5] * math.tan(math.radians(60.0)) < -1).sum())
        want, got = lo.moments(0, lam)[0], mom[0, w]
        flips = abs(want[0] - got[0]) + max(2, p.rays // 2000)
        print(f"line {w}: {int(got[0])} rays, Σ|Δ| {np.abs(got[1:3] - want[1:3])}", flush=True)
        assert (np.abs(got[1:3] - want[1:3]) <= flips * math.pi / 2 + 1e-6 * want[0]).all()
        assert abs(got[5] - want[5]) <= flips * (math.pi / 2) ** 2 + 3e-6 * want[0]
    assert strays > 500
    if params:
        # d(angular rms)/dθ from 64-bit differences of the rays that arrive on both sides.
        idx = np.arange(p.rays, dtype=np.uint64)
        which = [(0, L.PARAM_A4), (3, L.PARAM_A4)]

        def rms(delta):
            rays = [lo.trace_perturbed(0, lam, which, delta, idx) for lam in L.FRAUNHOFER7]
            return np.concatenate([r[:, 3:7] for r in rays])

        grads = b.gradients()[0]
        for k, step in enumerate((0.1, 0.1)):
            lo_, hi = (rms([s * step if j == k else 0.0 for j in range(2)]) for s in (-1, 1))
            ok = (lo_[:, 3] > 0) & (hi[:, 3] > 0)

            def value(r):
                bxy = r[ok, :2] / r[ok, 2:3]
                return math.sqrt(((np.arctan(bxy) - np.arctan(bxy.mean(0))) ** 2).sum(1).mean())

            fd = (value(hi) - value(lo_)) / (2 * step)
            # A ray that leaves a surface at grazing has a derivative of 1 / cos θt, 10⁴ times the others', and cos²θt
            # rounds by 1.2e-7: at cos θt = 1e-3 its share of the mean is off by a tenth (the largest share
            # alone exceeds the whole of the first design's first derivative).
            share = np.abs(np.arctan(hi[ok, 1] / hi[ok, 2]) - np.arctan(lo_[ok, 1] / lo_[ok, 2])).max() / (2 * step) / ok.sum()
            print(f"parameter {k}: {grads[k]:.6e}, 64-bit difference {fd:.6e}, largest share {share:.1e}", flush=True)
            assert abs(grads[k] - fd) <= 2e-3 * abs(fd) + 0.1 * share
    b.close()


def test_rays_share_no_error_and_weights_keep_their_digits(cuda, oracle):
    """Every ray reaches the first vertex plane after the same distance of 5 to 7 cm (ulp 3.7e-9 m) at the same slope
    0.0087: correctly rounded it moves a lens's rays by up to 1.6e-11 m in y, of either sign, so the mean over 48
    lenses lies below 1e-11, and one ulp in all of them is 3.3e-11. A weight near 0.85 after three faces, T − T R at
    each, rounds by at most half an ulp (3e-8) at each, 1.7e-8 rms, and its R ≈ 0.05 by a few
    ulps of 3.7e-9, so its rms error lies below 3.5e-8 (the indices' own rounding included)."""
    lenses = L.seeded_achromats(48, seed=77, rays_min=20000, rays_max=40000)
    b = L.LensBatch(lenses, L.c_settings(pixels=0))
    lo = LensOracle(oracle, lenses)
    dy, dT = [], []
    for li, p in enumerate(lenses):
        idx = np.arange(p.rays, dtype=np.uint64)
        g, c = b.trace(li, 3, idx), lo.trace(li, L.FRAUNHOFER7[3], idx)
        both = (g[:, 6] > 0) & (c[:, 6] > 0)
        dy.append((g - c)[both, 1])
        dT.append((g - c)[both, 6])
    b.close()
    dy, dT = np.concatenate(dy), np.concatenate(dT)
    print(f"{len(dy)} rays: mean error of y {dy.mean():.2e} m, rms of the weight {np.sqrt((dT**2).mean()):.2e}", flush=True)
    assert abs(dy.mean()) < 1e-11
    assert np.sqrt((dT**2).mean()) < 3.5e-8


def test_items_of_fewer_rays_than_threads_cost_no_more(cuda):
    """A block traces an item: 64, 128, 192 and 320 rays take the time of the next multiple of 256 (within a third, the
    spread of single launches of 0.1 ms being a tenth) and give its results."""
    b = L.LensBatch(L.gregorian_variants(16, 60, 5), L.c_settings(field_deg=0.05, pixels=0))
    b.set_params([(0, L.PARAM_CURVATURE), (1, L.PARAM_CONIC)])

    def run(rays):
        b.set_shape(3, rays)
        ms = []
        for _ in range(9):
            b.run()
            ms.append(b.last_ms())
        return float(np.median(ms)), b.results()[1], b.gradients()

    for rays, whole in ((64, 256), (128, 256), (192, 256), (320, 512)):
        (t, m, g), (tw, mw, gw) = run(rays), run(whole)
        print(f"items of {rays}: {t:.3f} ms, of {whole}: {tw:.3f} ms", flush=True)
        assert np.allclose(m, mw, rtol=1e-12, atol=1e-9) and np.allclose(g, gw, rtol=1e-9, atol=1e-9 * np.abs(gw).max())
        assert t <= tw * 4 / 3
    b.close()


@pytest.mark.parametrize("lenses,rays_max", [(1, 4096), (6, 40_000), (24, 60_000)])
def test_autotune_takes_no_slower_shape_than_the_batchs_own(cuda, lenses, rays_max):
    """The batch's own shape is among those tried, so the tuned one is no slower but for the spread of a launch (a tenth)."""
    b = L.LensBatch(L.seeded_achromats(lenses, seed=3, rays_min=2048, rays_max=rays_max))

    def median():
        ms = []
        for _ in range(15):
            b.run()
            ms.append(b.last_ms())
        return float(np.median(ms))

    own, best = median(), b.autotune()
    tuned = median()
    print(f"{lenses} lenses: own {own:.4f} ms, tuned {tuned:.4f} (as timed by the tuner {best:.4f})", flush=True)
    assert tuned <= 1.1 * own
    b.close()


def test_results_take_no_memory_and_pieces_of_the_grids_join(cuda):
    """30 million bins leave the device in two pieces: the same lens gives the same grids in each place of the batch, one
    of which lies across the join, and the first results allocate nothing."""
    import torch

    lenses = [L.DOUBLET] * 5
    b = L.LensBatch(lenses, L.c_settings(planes=6, pixels=1000, half_size=3e-3))
    b.run()
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    _, mom, irr = b.results(irradiance=True)
    assert torch.cuda.mem_get_info()[0] == free
    one = L.LensBatch(lenses[:1], L.c_settings(planes=6, pixels=1000, half_size=3e-3))
    one.run()
    alone = one.results(irradiance=True)[2][0]
    assert alone.sum() > 0
    for k in range(5):
        assert np.array_equal(irr[k], alone)
    one.close()
    b.close()


@pytest.mark.parametrize("planes,pixels,step", [(16, 1024, 2e-3), (2, 4096, 50e-3)])
def test_grids_of_many_more_bins_than_the_table(cuda, planes, pixels, step):
    """Defocused light over 50,000 bins and more of a lens, where a block's table holds 4,096: every add that finds no place goes
    to memory. The bins are those of the traced rays, but for rays within float rounding of an edge (a pixel
    is 24 µm or 6, a coordinate on the plane rounds to 5 nm: below 1 in 1,000), and no launch shape changes them."""
    p = L.Prescription(L.SINGLET.surfaces, rays=150_000)
    half = 12.5e-3
    st = L.c_settings(wavelengths=(587.56,), half_size=half, pixels=pixels, planes=planes, focus_step=step)
    b = L.LensBatch([p], st)
    grids = []
    for shape in ((3, 1024), (1, 256), (2, 16384)):
        b.set_shape(*shape)
        b.run()
        per, _, irr = b.results(irradiance=True)
        grids.append(irr[0].astype(np.float64))
    assert np.array_equal(grids[0], grids[1]) and np.array_equal(grids[0], grids[2])
    r = b.trace(0, 0, np.arange(p.rays, dtype=np.uint64))
    b.close()
    r = r[r[:, 6] > 0]
    z0 = per[0]["last_vertex_z"] + per[0]["bfl"]
    y0 = per[0]["efl"] * math.tan(math.radians(st.field_deg))
    beam = math.pi * (0.999 * per[0]["entrance_pupil_radius"]) ** 2 * math.cos(math.radians(st.field_deg))
    unit = beam / (p.rays * (2 * half / pixels) ** 2)
    moved = touched = 0.0
    for k in range(planes):
        s = (z0 + (k - 0.5 * (planes - 1)) * step - r[:, 2]) / r[:, 5]
        x = ((r[:, 0] + r[:, 3] * s) / half + 1) * 0.5 * pixels
        y = (1 - (r[:, 1] + r[:, 4] * s - y0) / half) * 0.5 * pixels
        ok = (x >= 0) & (y >= 0) & (x < pixels) & (y < pixels)
        want = np.bincount((y[ok].astype(int) * pixels + x[ok].astype(int)), r[ok, 6], pixels * pixels) * unit
        touched += (want > 0).sum()
        moved += np.abs(grids[0][k].ravel() - want).sum() / want.sum() / 2
    print(f"{planes} planes of {pixels}²: {int(touched)} bins, {moved / planes:.2e} of the light in another bin", flush=True)
    assert touched > 50_000 and moved / planes < 1e-3


def test_mirrors_behind_many_rows_obstruct(cuda, oracle):
    """33 thin plates before a Gregorian: its mirrors are rows 66 and 67, beyond the first 64, and the secondary (21 mm of 54) stops
    the centre of the beam on its way to the primary, 15 % where the primary's bore alone takes 6. Point and direction as for the telescope by itself: 24 µm of
    glass and 0.9 m of travel, coordinates of 5 cm that round to 4e-9 m, angles magnified 54 times."""
    tele = L.solve_afocal(L.GREGORIAN, 587.5618)
    rows = []
    for _ in range(33):
        rows += [L.Surface(math.inf, 0.01, "N-BK7", 60.0), L.Surface(math.inf, 0.01, "air", 60.0)]
    rows[-1].t = 700.0
    p = L.Prescription(rows + tele.surfaces, rays=8192)
    b = L.LensBatch([p], L.c_settings(field_deg=0.05, pixels=0, reference=587.5618))
    lo = LensOracle(oracle, [p], field_deg=0.05, reference=587.5618)
    idx = np.arange(8192, dtype=np.uint64)
    g, c = b.trace(0, 4, idx), lo.trace(0, L.FRAUNHOFER7[4], idx)
    b.close()
    assert [k for k, s in enumerate(p.surfaces) if s.reflect] == [66, 67]
    okg, okc = g[:, 6] > 0, c[:, 6] > 0
    both = okg & okc
    dp, dd = np.abs(g[both, :3] - c[both, :3]).max(), np.abs(g[both, 3:6] - c[both, 3:6]).max()
    print(f"{both.sum()} of {len(idx)} arrive on both, {(okg != okc).sum()} flips, |Δp| {dp:.1e}, |Δd| {dd:.1e}", flush=True)
    assert 1000 < both.sum() < 8192 * 0.9 and (okg != okc).sum() <= 4
    assert dp < 1e-7 and dd < 1e-5

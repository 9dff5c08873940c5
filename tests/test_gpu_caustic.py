"""The caustic slab's forward pass and path-replay adjoint on the GPU.

* forward against the fp64 oracle on the same particles: the same irradiance up to float rounding
  of each particle's wall point; identical passes are bit-identical (integer bins);
* adjoint against central finite differences of L = mean((E − target)²) on 64 random heights, on
  the GPU itself and in fp64 on the CPU, with a step in the linear regime of the loss (the particles
  move a few thousandths of a pixel); the 1e-4 mm step is also reported — there each particle moves
  about a third of a pixel, so the difference quotient is a secant a few percent from the tangent,
  the same for both precisions;
* the torch.autograd.Function gives the same gradient, and gradient steps lower the loss;
* the adjoint costs at most three forward passes.
"""
from __future__ import annotations

import math

import numpy as np
import pytest

from owe_hip import caustic as C
from owe_hip.lens import ciddor_air
from pyoracle import CausticOracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def setup(cuda):
    import torch

    s = C.caustic_settings(particles=1 << 18)
    c = C.Caustic(s)
    H = torch.tensor(C.initial_heights(), device="cuda")
    T = torch.tensor(C.target(s), device="cuda")
    yield s, c, H, T
    c.close()


def forward(c, s, H, pass_index=0):
    import torch

    out = torch.empty((s.pixels, s.pixels), dtype=torch.float32, device="cuda")
    c.forward_into(H.contiguous(), out, pass_index)
    torch.cuda.synchronize()
    return out


def loss_of(E, T):
    return float(((E.double() - T.double()) ** 2).mean())


def adjoint(c, s, H, T, pass_index=0):
    import torch

    E = forward(c, s, H, pass_index)
    gE = (2.0 * (E.double() - T.double()) / E.numel()).float().contiguous()
    g = torch.empty_like(H)
    c.backward_into(H.contiguous(), gE, g, pass_index)
    torch.cuda.synchronize()
    return g


def test_forward_matches_oracle(setup, oracle):
    s, c, H, T = setup
    E = forward(c, s, H).cpu().numpy().astype(np.float64)
    Eo = CausticOracle(oracle, s).forward(H.cpu().numpy().astype(np.float64))
    pix = 2 * s.wall_half / s.pixels
    tot = abs(E.sum() - Eo.sum()) / Eo.sum()
    diff = np.abs(E - Eo)
    print(f"forward: flux {E.sum() * pix * pix:.6e} vs {Eo.sum() * pix * pix:.6e} (rel {tot:.2e}), "
          f"max |ΔE| {diff.max():.3e} of max E {Eo.max():.3f}", flush=True)
    assert tot < 1e-5
    assert diff.max() < 1e-3 * Eo.max()
    assert np.array_equal(E, forward(c, s, H).cpu().numpy().astype(np.float64))


def test_adjoint_matches_finite_differences(setup, oracle):
    import torch

    s, c, H, T = setup
    g = adjoint(c, s, H, T).cpu().numpy().ravel().astype(np.float64)
    nodes = np.random.default_rng(17).integers(0, s.nodes * s.nodes, 64)
    co = CausticOracle(oracle, s)
    Hn = H.cpu().numpy().astype(np.float64)
    Tn = T.cpu().numpy().astype(np.float64)
    fd_cpu = co.fd(Hn, Tn, nodes, 1e-9)
    secant_cpu = co.fd(Hn, Tn, nodes, 1e-7)

    def fd_gpu(h):
        out = []
        flat = H.clone().view(-1)
        for k in nodes:
            v = float(flat[k])
            flat[k] = v + h
            lp = loss_of(forward(c, s, flat.view(H.shape)), T)
            flat[k] = v - h
            lm = loss_of(forward(c, s, flat.view(H.shape)), T)
            flat[k] = v
            out.append((lp - lm) / (2 * h))
        return np.array(out)

    fd = fd_gpu(3e-9)
    secant = fd_gpu(1e-7)
    a = g[nodes]
    results = {}
    for name, ref in (("gpu fd", fd), ("fp64 cpu fd", fd_cpu)):
        rel = np.linalg.norm(a - ref) / np.linalg.norm(ref)
        worst = (np.abs(a - ref) / (np.abs(ref) + 0.02 * np.abs(ref).max())).max()
        results[name] = (rel, worst)
        print(f"adjoint vs {name}: relative error {rel:.2e} (norm over 64 heights), worst component {worst:.2e}",
              flush=True)
    sec = np.linalg.norm(a - secant) / np.linalg.norm(secant)
    agree = np.linalg.norm(secant - secant_cpu) / np.linalg.norm(secant_cpu)
    print(f"1e-4 mm step: adjoint vs secant {sec:.2e}; gpu secant vs fp64 secant {agree:.2e}", flush=True)
    # Within 1 % of the GPU's own finite differences over the 64 heights, each component within 5 %
    # (the float forward's rounding makes single small differences noisy); the fp64 differences are
    # free of that noise and pin the adjoint ten times tighter.
    rel, worst = results["gpu fd"]
    assert rel < 0.01 and worst < 0.05
    rel, worst = results["fp64 cpu fd"]
    assert rel < 1e-3 and worst < 5e-3
    assert agree < 0.01


def test_autograd_function_and_descent(setup):
    import torch

    s, c, H, T = setup
    g_direct = adjoint(c, s, H, T)
    Hp = H.clone().requires_grad_(True)
    E = c.irradiance(Hp)
    L = ((E.double() - T.double()) ** 2).mean()
    L.backward()
    torch.cuda.synchronize()
    assert torch.allclose(Hp.grad, g_direct, rtol=1e-5, atol=1e-6 * float(g_direct.abs().max()))
    # A few normalised gradient steps on fresh particle passes lower the loss.
    Hs = H.clone()
    losses = []
    for it in range(6):
        Hv = Hs.clone().requires_grad_(True)
        L = ((c.irradiance(Hv, it).double() - T.double()) ** 2).mean()
        L.backward()
        losses.append(float(L.detach()))
        with torch.no_grad():
            Hs = Hs - 2e-6 * Hv.grad / Hv.grad.abs().max()
    print(f"losses: {losses}", flush=True)
    assert losses[-1] < losses[0]


def test_adjoint_costs_at_most_three_forwards(cuda):
    import torch

    s = C.caustic_settings()
    c = C.Caustic(s)
    H = torch.tensor(C.initial_heights(), device="cuda")
    T = torch.tensor(C.target(s), device="cuda")
    E = torch.empty((s.pixels, s.pixels), dtype=torch.float32, device="cuda")
    gE = torch.zeros_like(E)
    g = torch.empty_like(H)
    for _ in range(2):
        c.forward_into(H, E, 0)
        c.backward_into(H, gE + 1e-3, g, 0)
    ev = [torch.cuda.Event(enable_timing=True) for _ in range(3)]
    reps = 5
    ev[0].record()
    for k in range(reps):
        c.forward_into(H, E, k)
    ev[1].record()
    gE = (2.0 * (E - T) / E.numel()).contiguous()
    for k in range(reps):
        c.backward_into(H, gE, g, k)
    ev[2].record()
    torch.cuda.synchronize()
    f, b = ev[0].elapsed_time(ev[1]) / reps, ev[1].elapsed_time(ev[2]) / reps
    print(f"forward {f:.3f} ms, adjoint {b:.3f} ms, ratio {b / f:.2f} (1,048,576 particles)", flush=True)
    assert b <= 3.0 * f
    c.close()


@pytest.mark.parametrize("particles", [1, 255, 257, 5000, 1 << 18])
def test_adjoint_of_wide_ranges_and_remainders(cuda, particles):
    """The adjoint's block sums choose their own unit: a wall whose right half's ∂L/∂E is 10⁻¹² of the
    left's (or 10⁻³⁵, where no unit suits) gives the right's nodes what the right half alone gives, and
    an infinite pixel reaches its nodes and no others. Sums of up to a few hundred float adds in another order
    differ by at most as many half ulps: 2e-5 in norm."""
    import torch

    s = C.caustic_settings(nodes=64, pixels=128, particles=particles)
    c = C.Caustic(s)
    h = torch.tensor(C.initial_heights(64, feature=16), device="cuda")
    g = torch.Generator(device="cuda").manual_seed(3)
    base = torch.randn((128, 128), device="cuda", generator=g)
    right = torch.zeros_like(base)
    right[:, 64:] = base[:, 64:]
    left = base - right

    def adjoint(ge):
        out = torch.empty_like(h)
        c.backward_into(h, ge.contiguous(), out, 0)
        torch.cuda.synchronize()
        return out

    alone = adjoint(right).double()
    assert torch.isfinite(alone).all()
    inner = alone[:, 40:]  # nodes whose particles land well inside the right half
    for scale in (1.0, 1e-12, 1e12):
        both = adjoint(left / scale + right)[:, 40:].double()
        assert (both - inner).norm() <= 2e-5 * inner.norm()
    tiny = adjoint(right * 1e-35)[:, 40:].double() * 1e35
    assert (tiny - inner).norm() <= 1e-3 * inner.norm()  # products down to 1e-38 lose digits as floats
    assert (adjoint(torch.zeros_like(base)) == 0).all()
    spoiled = right.clone()
    spoiled[64, 32] = float("inf")
    got = adjoint(spoiled)
    assert torch.isfinite(got[:, 40:]).all() and (got[:, 40:].double() - inner).norm() <= 2e-5 * inner.norm()
    if particles >= 5000:
        assert not torch.isfinite(got[:, :40]).all()
    c.close()


@pytest.mark.parametrize("n", [1.2, 1.3, 1.4, 1.7])
def test_exits_at_the_critical_angle_add_no_light(cuda, oracle, n):
    """A tilted plane whose slope is the critical one, sin θ = 1/η: the float cos²θt = 1 − η² sin²θ takes its values
    near 0, 0 among them, where the Fresnel amplitudes round past 1 and the transmittance below 0 (by up to
    2.4e-7). cos θt stays below 0.02 there (sin θ varies by 1e-5 with the heights' rounding), so a particle
    passes at most 4 cos θt < 0.13 of its weight, 0.26 of irradiance where the full weights give 1 to 2; a negative
    weight taken for a large one is a whole unit of irradiance. (The cells at the slab's edge have other slopes.)"""
    import torch

    s = C.caustic_settings(particles=1 << 20, pixels=1024, thickness=0.06, wall_distance=0.1, wall_half=0.3)
    s.medium.index_kind, s.medium.coeff_a[0] = 0, n
    c = C.Caustic(s)
    eta = n / ciddor_air(555.0)  # air's index varies by 7e-6 over the visible range
    x = np.linspace(-s.slab_half, s.slab_half, s.nodes) / math.sqrt(eta * eta - 1)
    H = np.broadcast_to(x, (s.nodes, s.nodes)).astype(np.float32)
    E = forward(c, s, torch.tensor(H.copy(), device="cuda")).cpu().numpy().astype(np.float64)
    Eo = CausticOracle(oracle, s).forward(H.astype(np.float64))
    diff = np.abs(E - Eo).max()
    print(f"index {n}: {E.sum():.3f} / {Eo.sum():.3f}, max {E.max():.3f} / {Eo.max():.3f}, max |ΔE| {diff:.3e}", flush=True)
    assert diff < 0.26 + 1e-3 * Eo.max()
    c.close()


@pytest.mark.parametrize("kelvin", [110.0, 200.0, 300.0, 440.0])
def test_adjoint_of_cool_suns(cuda, oracle, kelvin):
    """Planck's exponent exceeds float's range over part of the visible range below 450 K and over all of it below
    195 K; the weights are ratios and stay in range. The reddest particles carry the sums there."""
    import torch

    s = C.caustic_settings(nodes=64, pixels=128, particles=1 << 16, kelvin=kelvin)
    c = C.Caustic(s)
    H = torch.tensor(C.initial_heights(64, feature=16), device="cuda")
    co = CausticOracle(oracle, s)
    E, Eo = forward(c, s, H).cpu().numpy().astype(np.float64), co.forward(H.cpu().numpy().astype(np.float64))
    # The exponent c2/(λT), up to 400, rounds by 2⁻²³ of itself twice: 1e-4 of a weight.
    assert np.linalg.norm(E - Eo) <= 3e-4 * np.linalg.norm(Eo)
    T = torch.tensor(C.target(s), device="cuda")
    g = adjoint(c, s, H, T).cpu().numpy().ravel().astype(np.float64)
    assert np.isfinite(g).all()
    nodes = np.argsort(-np.abs(g))[:: 64][:16]
    fd = co.fd(H.cpu().numpy().astype(np.float64), T.cpu().numpy().astype(np.float64), nodes, 1e-9)
    rel = np.linalg.norm(g[nodes] - fd) / np.linalg.norm(fd)
    print(f"{kelvin} K: adjoint against fp64 differences {rel:.2e}", flush=True)
    assert rel < 1e-3
    c.close()

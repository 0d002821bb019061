"""The registry kernels on the ray's line (``forward_line``, ``forward_rrm``).

Against the oracle and against the kind switch (variant 0) where the line kernels can go
wrong: rays through the Sun and at the poles, pointings normal to the observer's
direction, observers off the plane and outside cut-off spheres, exponents at the ends
of the range the kernels accept (and just outside, where the general kernel runs), ray
counts around the block and lane edges. Tolerance: the framework's parity bound, 1e-10
relative per value; the node radius (5e-15) enters the values at most to its 20th power
and, through exp(-zeta^6), with the exponent (below 746) times six, so 5e-15 x 4476 =
2e-11 bounds what two evaluations may differ by.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import zodi_oracle
from oracle.zodi_oracle import OracleModel
from zodipy_amd import Model, healpix
from zodipy_amd import units as u
from zodipy_amd._lib import Launch
from zodipy_amd.fitting import LineOfSightProblem
from zodipy_amd.runtime import OUT_COMPS

pytestmark = pytest.mark.gpu

RTOL = 1e-10


def pointings(obs):
    """Map pixels plus the directions at which the geometry degenerates."""
    o = np.asarray(obs) / np.linalg.norm(obs)
    normal = np.array([-o[1], o[0], 0.0]) / np.hypot(o[0], o[1])
    special = [[0, 0, 1], [0, 0, -1], [1, 0, 0], [0, 1, 0], [0, -1, 0], -o, o, normal,
               [np.sin(1e-9), 0, np.cos(1e-9)], [-np.cos(1e-7), np.sin(1e-7), 0]]
    return np.concatenate([healpix.pix2vec(4), np.array(special, dtype=float).T], axis=1)


def same(got, want):
    assert np.array_equal(np.isnan(got), np.isnan(want))
    ok = ~np.isnan(want)
    zero = ok & (want == 0)
    assert np.all(got[zero] == 0)
    ok &= ~zero
    rel = np.abs(got[ok] - want[ok]) / np.abs(want[ok])
    assert rel.max(initial=0.0) <= RTOL, rel.max()


def both(model, v, obs):
    dm = model.device_model
    a = dm.forward(v, obs, obs, out_mode=OUT_COMPS).cpu().numpy()
    b = dm.forward(v, obs, obs, out_mode=OUT_COMPS, launch=Launch(variant=0)).cpu().numpy()
    return a, b


@pytest.mark.parametrize("x", [25 * u.micron, 1.25 * u.micron])
@pytest.mark.parametrize("obs", [(1.0, 0.0, 0.0), (0.0, 0.9, 0.0), (0.7, -0.6, 0.3),
                                 (0.0, 0.0, 1.1), (1.25, 0.1, 0.0), (3.0, 2.0, 0.1)])
def test_degenerate_directions_against_oracle(gpu, monkeypatch, x, obs):
    # within 1e-7 of the directions to and from the Sun the arc cosine of a rounded cosine
    # holds only half the digits; the oracle takes the same angle from its tangent
    def angle(R_los, R_helio, X_los, X_helio):
        cross = np.cross(X_los, X_helio, axis=0)
        return np.arctan2(np.sqrt((cross**2).sum(axis=0)), -(X_los * X_helio).sum(axis=0))

    monkeypatch.setattr(zodi_oracle, "get_scattering_angle", angle)
    obs = np.array(obs)
    v = pointings(obs if obs[0] or obs[1] else obs + [1e-3, 0, 0])
    got = Model(x).device_model.forward(v, obs, obs, out_mode=OUT_COMPS).cpu().numpy()
    same(got, OracleModel(x).evaluate_vectors(v, obs, obs))


@pytest.mark.parametrize("obs", [(1.0, 0.0, 0.0), (0.7, -0.6, 0.3), (1.25, 0.1, 0.0),
                                 (3.0, 2.0, 0.1)])
def test_rrm_against_oracle(gpu, obs):
    """Rays inside, across and along the planes (Z_0, the bands' latitude limits)."""
    obs = np.array(obs)
    x = 25 * u.micron
    phi = np.linspace(0, 2 * np.pi, 13)
    low = np.stack([np.cos(phi), np.sin(phi), np.full(13, 0.02)])
    v = np.concatenate([pointings(obs), low / np.linalg.norm(low, axis=0)], axis=1)
    model = Model(x, name="rrm-experimental")
    got = model.device_model.forward(v, obs, obs, out_mode=OUT_COMPS).cpu().numpy()
    same(got, OracleModel(x, name="rrm-experimental").evaluate_vectors(v, obs, obs))


@pytest.mark.parametrize("change", [{"fan": {"Q": 0.0}}, {"fan": {"Z_0": 5.0}},
                                    {"comet": {"Z_0": 1e-6, "P": 0.0}},
                                    {"inner_narrow_band": {"gamma": 0.0, "beta_nb": 90.0}},
                                    {"broad_band": {"sigma_bb": 0.2, "gamma": -2.0}},
                                    {"fan": {"R_outer": 0.9}}, {"fan": {"x_0": 0.01}}])
def test_rrm_parameters_against_general_kernel(gpu, change):
    """The last one, off centre, runs the general layout kernel."""
    model = Model(25 * u.micron, name="rrm-experimental")
    p = model.get_parameters()
    for comp, values in change.items():
        p["comps"][comp].update(values)
    model.update_parameters(p)
    obs = np.array([0.98, 0.17, 0.004])
    got, want = both(model, pointings(obs), obs)
    same(got, want)


# delta and alpha up to 2 and gamma in [1/2, 6] run on the line, the rest in general.
@pytest.mark.parametrize("change", [{"delta": 2.0}, {"delta": 2.01}, {"delta": 0.0},
                                    {"delta": -0.3}, {"alpha": 2.0}, {"alpha": 2.2},
                                    {"alpha": 0.0}, {"gamma": 0.5}, {"gamma": 0.49},
                                    {"gamma": 6.0}, {"gamma": 1.0}, {"beta": 60.0},
                                    {"mu": 1e-3}, {"mu": 2.0}])
def test_exponents_against_general_kernel(gpu, change):
    model = Model(25 * u.micron)
    p = model.get_parameters()
    for k, v in change.items():
        if k in p:
            p[k] = v
        else:
            p["comps"]["cloud"][k] = v
    model.update_parameters(p)
    obs = np.array([0.98, 0.17, 0.004])
    got, want = both(model, pointings(obs), obs)
    same(got, want)


@pytest.mark.parametrize("n", [1, 31, 32, 33, 63, 65, 255, 257, 1023])
@pytest.mark.parametrize("lanes", [0, 1, 2, 4, 8])
@pytest.mark.parametrize("name", ["dirbe", "rrm-experimental"])
def test_ragged_counts(gpu, n, lanes, name):
    obs = np.array([0.99, 0.1, 0.0])
    model = Model(12 * u.micron, name=name)
    v = healpix.pix2vec(16)[:, ::3][:, :n]
    got = model.device_model.forward(v, obs, obs, out_mode=OUT_COMPS,
                                     launch=Launch(variant=1, lanes_per_ray=lanes)).cpu().numpy()
    want = model.device_model.forward(torch.as_tensor(healpix.pix2vec(16)[:, ::3].copy()), obs,
                                      obs, out_mode=OUT_COMPS).cpu().numpy()[:, :n]
    assert np.array_equal(got, want)


@pytest.mark.parametrize("rays", [1, 7, 17, 3072, 12289, 20011, 49153, 150001])
@pytest.mark.parametrize("nodes", [1, 9, 50])
@pytest.mark.parametrize("name,x", [("dirbe", 1.25 * u.micron), ("planck18", 857 * u.GHz),
                                    ("rrm-experimental", 25 * u.micron)])
def test_default_split_gives_the_bits_of_one_lane(gpu, name, x, nodes, rays):
    """The lanes per ray (1 to 32) that the launch picks from the ray count, with a last
    node step that is full, partial or the only one, against one lane per ray: equal."""
    model = Model(x, name=name, gauss_quad_degree=nodes)
    rng = np.random.default_rng(rays + nodes)
    v = rng.normal(size=(3, rays))
    v /= np.linalg.norm(v, axis=0)
    obs = np.array([0.9, 0.4, 0.02])
    for mode in ({}, {"out_mode": OUT_COMPS}):
        got = model.device_model.forward(v, obs, obs, **mode)
        one = model.device_model.forward(v, obs, obs, launch=Launch(256, 1, 0, 1), **mode)
        assert torch.equal(got, one)


@pytest.mark.parametrize("name,x,rays,lanes", [
    ("dirbe", 25 * u.micron, 393_217, 0), ("dirbe", 25 * u.micron, 200_000, 4),
    ("planck18", 857 * u.GHz, 420_001, 0), ("rrm-experimental", 25 * u.micron, 800_001, 0),
    ("dirbe", 1.25 * u.micron, 2_001, 0), ("dirbe", 1.25 * u.micron, 1, 0)])
def test_block_rows_beyond_the_resident_ones(gpu, name, x, rays, lanes):
    """The passes that take more blocks than stay resident (three rounds of tiles and more;
    4 lanes a ray reach it with the smallest workspace) against the resident blocks, and
    the chi^2 pass against the recompute path, which adds the same terms in another order:
    n additions of relative error below 2^-53 each on sums of like sign."""
    model = Model(x, name=name)
    rng = np.random.default_rng(rays)
    v = rng.normal(size=(3, rays))
    v /= np.linalg.norm(v, axis=0)
    obs = np.array([0.9, 0.4, 0.02])
    prob = LineOfSightProblem(model, v, obs, obs)
    theta = prob.space.theta0
    w = torch.as_tensor(rng.uniform(0.5, 1.5, rays), device="cuda")
    data = prob.forward(theta) * torch.as_tensor(rng.uniform(0.9, 0.99, rays), device="cuda")
    per_cu = 4 if name == "rrm-experimental" else 2
    got = {}
    for key, blocks in (("more", 0), ("resident", per_cu)):
        prob.launch = Launch(0, lanes, blocks, 0)
        got[key] = [prob.vjp(theta, w), torch.cat([g.reshape(-1) for g in
                                                   prob.chi2_and_grad(theta, data)]),
                    torch.cat([g.reshape(-1) for g in prob.chi2_spectral_grad(theta, data)])]
    prob.launch = None
    prob.store_jacobian = False
    got["recompute"] = [None, torch.cat([g.reshape(-1) for g in
                                         prob.chi2_and_grad(theta, data)]), None]
    for key in ("more", "recompute"):
        for a, b in zip(got[key], got["resident"]):
            if a is not None:
                # entries that cancel are judged against the gradient's largest
                tol = 1e-10 * b.abs() + 1e-13 * b.abs().max()
                assert torch.all((a - b).abs() <= tol)


@pytest.mark.parametrize("rays", [1, 5_000, 40_001, 98_305, 131_072, 150_001])
@pytest.mark.parametrize("x", [25 * u.micron, 1.25 * u.micron])
def test_gradient_splits_against_one_lane(gpu, x, rays):
    """The lanes per ray that the gradient passes pick from the ray count against one lane
    and the recompute path: the same terms in another order (tolerance as above)."""
    rng = np.random.default_rng(rays)
    v = rng.normal(size=(3, rays))
    v /= np.linalg.norm(v, axis=0)
    obs = np.array([0.9, 0.4, 0.02])
    prob = LineOfSightProblem(Model(x), v, obs, obs)
    theta = prob.space.theta0
    w = torch.as_tensor(rng.uniform(0.5, 1.5, rays), device="cuda")
    data = prob.forward(theta) * torch.as_tensor(rng.uniform(0.9, 0.99, rays), device="cuda")

    def both():
        c, g, model = prob.chi2_and_grad(theta, data, return_model=True)
        return torch.cat([c.reshape(1), g]), prob.vjp(theta, w), model

    got = both()
    prob.launch = Launch(0, 1, 0, 0)
    one = both()
    prob.store_jacobian = False
    again = both()
    for a, b, c in zip(got, one, again):
        for other in (a, c):
            tol = 1e-10 * b.abs() + 1e-13 * b.abs().max()
            assert torch.all((other - b).abs() <= tol)


@pytest.mark.parametrize("name", ["dirbe", "rrm-experimental"])
def test_feature_angle_next_to_the_axis(gpu, name):
    """Points whose squared distance from the z axis leaves the normal range (the feature's
    angle is then that of a scaled point) against the kind switch, which takes atan2."""
    v = np.array([[1e-170, -3e-200, 0.0, 2e-155], [2e-170, 1e-180, 1e-160, -1e-156],
                  [1.0, 1.0, 1.0, 1.0]])
    obs = np.array([0.0, 0.0, 1.1])
    same(*both(Model(25 * u.micron, name=name), v, obs))
    if name == "dirbe":
        same(*both(Model(1.25 * u.micron), v, obs))

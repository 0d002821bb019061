"""The launch tuner offers each kernel once and keeps shapes apart that run other kernels."""

from __future__ import annotations

import json

import numpy as np
import pytest
import torch

from zodipy_amd import Model, autotune
from zodipy_amd import units as u
from zodipy_amd._lib import Launch
from zodipy_amd.runtime import OUT_SUM

pytestmark = pytest.mark.gpu

OBS = np.array([0.98, 0.17, 0.004])


def model(name="dirbe", x=25 * u.micron, **cloud):
    m = Model(x, name=name)
    p = m.get_parameters()
    for comp, values in cloud.items():
        p["comps"][comp].update(values)
    m.update_parameters(p)
    return m


def test_keys_differ_where_the_kernels_do(gpu):
    """Scattering, shared cut-offs, exponents and frames select kernels; a parameter that does
    not keeps the key."""
    models = [model(), model(x=1.25 * u.micron), model(band1={"delta_r": 1.4}),
              model(cloud={"alpha": 2.5}), model(band1={"x_0": 0.01}), model(band1={"p": 3.9}),
              model(name="planck18", x=857 * u.GHz), model(name="rrm-experimental")]
    keys = [autotune.layout_key(m.device_model, 1000) for m in models]
    assert len(set(keys)) == len(keys)
    same = autotune.layout_key(model(cloud={"alpha": 1.4}).device_model, 1000)
    assert same == keys[0]
    assert autotune.layout_key(models[0].device_model, 5000) != keys[0]


@pytest.mark.parametrize("rays", [500, 40_000])
def test_line_kernels_are_timed_once(gpu, tmp_path, monkeypatch, rays):
    monkeypatch.setenv("ZODI_TUNE_CACHE", str(tmp_path / "tuning.json"))
    rng = np.random.default_rng(rays)
    v = rng.normal(size=(3, rays))
    v = torch.as_tensor(v / np.linalg.norm(v, axis=0), device="cuda")
    for m, smallest in ((model(), 256), (model(band1={"x_0": 0.01}), 64)):
        dm = m.device_model
        seg, n_seg, obs, earth, beyond, mode = dm.prepare_observers(
            OBS, OBS, np.array([0, rays]))
        launch, times = autotune.tune(dm, v, seg, n_seg, obs, earth, beyond, mode)
        shapes = [tuple(int(i) for i in k.split(",")) for k in times]
        assert min(b for b, _, _ in shapes) == smallest
        assert (256, 0, 0) in shapes  # the library's own choice, which no caller can name
        want = dm.forward(v, OBS, OBS, out_mode=OUT_SUM)
        assert torch.equal(dm.forward(v, OBS, OBS, out_mode=OUT_SUM, launch=launch), want)
        again, cached = autotune.tune(dm, v, seg, n_seg, obs, earth, beyond, mode)
        assert cached == times
        assert (again.block, again.lanes_per_ray) == (launch.block, launch.lanes_per_ray)
    kept = json.loads((tmp_path / "tuning.json").read_text())
    assert len(kept) == 2 and all(f"|r{autotune.KERNEL_REVISION}|" in k for k in kept)


def test_shapes_of_older_kernels_are_not_used(gpu, tmp_path, monkeypatch):
    """A cache written for other kernels (no revision in its keys) is left alone."""
    cache = tmp_path / "tuning.json"
    monkeypatch.setenv("ZODI_TUNE_CACHE", str(cache))
    dm = model().device_model
    key = autotune.layout_key(dm, 1000)
    old = "|".join(p for p in key.split("|") if p[0] not in "rfp" or p.startswith("AMD"))
    cache.write_text(json.dumps({old: {"best": [64, 8, 0], "times": {}}}))
    v = torch.as_tensor(np.eye(3)[:, [0, 1] * 500].copy(), device="cuda")
    seg, n_seg, obs, earth, beyond, mode = dm.prepare_observers(OBS, OBS, np.array([0, 1000]))
    launch, times = autotune.tune(dm, v, seg, n_seg, obs, earth, beyond, mode,
                                  candidates=[(256, 1, 0)])
    assert times and (launch.block, launch.lanes_per_ray) == (256, 1)
    assert isinstance(launch, Launch)

"""Which parameter sets the line kernels take (``zodi_line_domain.hpp``, built with g++).

Their power tables and exponentials hold over stated ranges; a block outside them runs the
general kernels. The header is plain C++, so its decisions are read here on packed blocks.
"""

from __future__ import annotations

import ctypes as ct
import shutil
import subprocess
from pathlib import Path

import numpy as np
import pytest

from zodipy_amd import Model
from zodipy_amd import units as u
from zodipy_amd.packing import MODEL_DTYPE

ROOT = Path(__file__).resolve().parents[1]
CSRC = ROOT / "zodipy_amd" / "csrc"

HARNESS = r"""
#include "zodi_line_domain.hpp"
extern "C" int takes(int which, const void* block) {
  const zodi_model* m = (const zodi_model*)block;
  return which == 0 ? zodi::line_match(m) : zodi::line_log_match(m);
}
"""


@pytest.fixture(scope="module")
def takes(tmp_path_factory):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("g++ not available")
    d = tmp_path_factory.mktemp("domain")
    (d / "harness.cpp").write_text(HARNESS)
    subprocess.run([cxx, "-O2", "-std=c++17", "-shared", "-fPIC", f"-I{CSRC}",
                    f"-I{ROOT / 'include'}", str(d / "harness.cpp"), "-o", str(d / "lib.so")],
                   check=True)
    lib = ct.CDLL(str(d / "lib.so"))

    def f(model):
        block = np.ascontiguousarray(model._packed.block)
        assert block.dtype == MODEL_DTYPE
        return tuple(bool(lib.takes(k, ct.c_void_p(block.ctypes.data))) for k in (0, 1))

    return f


def changed(name, values, x=25 * u.micron):
    """A model with parameters replaced: {"delta": v} or {"comp": {"field": v}}."""
    model = Model(x, name=name)
    p = model.get_parameters()
    for k, v in values.items():
        if isinstance(v, dict):
            p["comps"][k].update(v)
        else:
            p[k] = v
    with np.errstate(all="ignore"):
        model.update_parameters(p)
    return model


@pytest.mark.parametrize("name", ["dirbe", "planck13", "planck15", "planck18", "odegard",
                                  "rrm-experimental"])
def test_registry_models_take_the_line(takes, name):
    x = 25 * u.micron if name in ("dirbe", "rrm-experimental") else 857 * u.GHz
    adjoint = takes(Model(x, name=name))
    assert adjoint[1] and (adjoint[0] or name == "rrm-experimental")


# (values, forward, adjoint): g of the cloud reaches 1 + |mu|/2 and its radius the offset;
# beta g^gamma has to stay inside the exponential's range.
@pytest.mark.parametrize("cloud,forward,adjoint", [
    ({"mu": -4.0}, True, True), ({"mu": -4.01}, False, False),
    ({"mu": -4.0, "beta": 1e6, "gamma": 6.0}, False, False),
    ({"mu": -4.0, "beta": 5e3, "gamma": 6.0}, True, True),
    ({"mu": 3.0, "beta": 1e6, "gamma": 6.0}, True, True), ({"beta": 1.1e6}, False, False),
    ({"x_0": 2.0**60}, True, True), ({"z_0": -(2.0**60)}, True, True),
    ({"x_0": 2.0**60 * 1.01}, False, False), ({"y_0": -(2.0**61)}, False, False),
    ({"mu": np.float64(0)}, False, False), ({"mu": np.float64(-0.0)}, False, False),
    ({"mu": np.float64(5e-324)}, False, False), ({"mu": 1e-300}, False, False),
    ({"mu": 1e-12}, True, True), ({"mu": -1e-12}, True, True),
    ({"alpha": 2.0}, True, True), ({"alpha": 2.1}, False, True),
])
def test_cloud_ranges(takes, cloud, forward, adjoint):
    assert takes(changed("dirbe", {"cloud": cloud})) == (forward, adjoint)
    x = 857 * u.GHz
    assert takes(changed("planck18", {"cloud": cloud}, x)) == (forward, adjoint)


NOT_FINITE = [np.nan, np.inf, -np.inf, 1e18]  # (angles are packed in radians)


@pytest.mark.parametrize("value", NOT_FINITE)
@pytest.mark.parametrize("name", ["dirbe", "planck18", "rrm-experimental"])
def test_non_finite_parameters(takes, name, value):
    """Every parameter of every component, one at a time (derived constants follow them)."""
    x = 857 * u.GHz if name == "planck18" else 25 * u.micron
    model = Model(x, name=name)
    for label, comp in model.get_parameters()["comps"].items():
        for field in comp:
            if field in ("i", "Omega", "theta") and abs(value) == 1e18:
                continue  # an angle: its sine and cosine are finite
            if field in ("x_0", "y_0", "z_0") and abs(value) == 1e18:
                continue  # offsets: test_cloud_ranges
            if np.isinf(value) and field in ("i", "Omega", "theta"):
                continue  # the angle is refused before it is packed, or its sine is NaN
            got = takes(changed(name, {label: {field: np.float64(value)}}, x))
            assert got == (False, False), (label, field)


@pytest.mark.parametrize("value,ok", [(np.nan, True), (np.inf, False), (-np.inf, False),
                                      (12.1, False), (-12.1, False)])
def test_temperature_law(takes, value, ok):
    """A NaN exponent makes every temperature NaN by itself; larger ones overflow."""
    assert takes(changed("dirbe", {"delta": value})) == (ok, ok)
    assert takes(changed("planck18", {"delta": value}, 857 * u.GHz)) == (ok, ok)

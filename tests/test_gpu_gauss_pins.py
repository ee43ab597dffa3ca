"""Every kernel of the Gauss projection's steps, pinned where the size would
choose another: the streamed tiles and the site walk on lattices that take
the transports, the transports on ones that do not, against the oracle and
against each other.  That the pins take is checked without a device
(test_gauss_rules.py)."""
import numpy as np
import pytest

import lqcd
import oracle as O
import test_gpu_gauss_tiles as tiles
import test_gpu_gauss_transports as transports

pytestmark = pytest.mark.gpu

PINS = {"streamed": {"LQCD_GAUSS_TRANSPORTS": "0"}, "walk": {"LQCD_GAUSS_TILES": "0"},
        "transports": {"LQCD_GAUSS_TRANSPORTS": "1"}}


def pin(monkeypatch, name):
    for var in ("LQCD_GAUSS_TRANSPORTS", "LQCD_GAUSS_TILES"):
        monkeypatch.delenv(var, raising=False)
    for var, value in PINS[name].items():
        monkeypatch.setenv(var, value)


@pytest.mark.parametrize("name", ["streamed", "walk"])
@pytest.mark.parametrize("ext,cold", [([8, 16, 8, 4], False), ([16, 8, 8, 4], False), ([8, 8, 4, 4], True)])
def test_tiles_vs_oracle(ext, cold, name, monkeypatch):
    pin(monkeypatch, name)
    tiles.test_gauss_tiles_vs_oracle(ext, cold)


@pytest.mark.parametrize("ext", [[5, 3, 7, 4], [6, 10, 4, 8], [13, 12, 11, 10], [9, 7], [64, 2]])
@pytest.mark.parametrize("precision", [lqcd.F64, lqcd.F32])
def test_walk_vs_oracle(ext, precision, monkeypatch):
    pin(monkeypatch, "walk")
    transports.test_projection_matches_oracle(ext, precision)


# workgroups of C slices (streamed tiles): 8^4 and 16^3 x 8 C = 1, 16^3 x 64 and
# 32 x 16^2 x 32 C = 2, 64 x 16 x 32 x 16 C = 4 with one x_0 row per wavefront,
# 16^3 x 128 C = 4; no tiles: 12 x 10 x 6 x 9 and the D = 2 ones
@pytest.mark.parametrize("ext", [[8, 8, 8, 8], [16, 16, 16, 8], [16, 16, 16, 64], [32, 16, 16, 32], [64, 16, 32, 16],
                                 [16, 16, 16, 128], [12, 10, 6, 9], [70, 40], [2, 2]])
@pytest.mark.parametrize("precision", [lqcd.F64, lqcd.F32])
def test_kernels_agree(ext, precision, monkeypatch):
    d = len(ext)
    print(f"[gpu-case] gauss pins {ext} precision={precision}", flush=True)
    st = lqcd.LatticeStateDefault.new_determinist(1.0, 6.0, ext, 5, d, precision)
    ef = lqcd.LatticeStateEFSyncDefault(st)
    ef.reset_e_field(7, 0, 0.5 / 6.0)
    e0 = ef.e_field()
    got = {}
    for name in PINS:
        pin(monkeypatch, name)
        ef.set_e_field(e0)
        checks = ef.project_to_gauss(400)
        got[name] = checks, ef.e_field()
    print({name: c for name, (c, _) in got.items()}, flush=True)
    for name in ("walk", "transports"):
        assert abs(got[name][0] - got["streamed"][0]) <= 1
        # one group of steps more or less moves a site by its deviation at the
        # stop, 320 eps = 7e-14, over (1 - rate); f32 is rounded when stored
        tol = 1e-11 if precision == lqcd.F64 else 1e-7 * np.max(np.abs(e0))
        assert np.max(np.abs(got[name][1] - got["streamed"][1])) <= tol

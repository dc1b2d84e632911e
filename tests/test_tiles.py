"""The tiles the GPU's launches go by, walked on the host: in storage order
and in every strip order they visit each cell and face once, with its annulus
or pair and direction (dhx_check_orders), and a run whose kernels take their
elements from them, with the tile's group instead of a look-up, equals the run
by elements bit for bit."""
import ctypes as C
import os
import sys

import numpy as np
import pytest

from disco_amd import capi
from helpers import host_initial

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpu_engine"))
import build as cpu_build  # noqa: E402

GR = {"R_Min": 8.0, "R_Max": 20.0, "CFL": 0.2}


@pytest.mark.parametrize("merge", ["1", "0"])
@pytest.mark.parametrize("cname,over,orders", [
    # 10 layers with the ghosts: strips of 4, 8 and 10, of four kinds
    ("mhd_kep", {"Num_R": 12, "Num_Z": 6, "Max_DT": 0.02}, 12),
    # annuli of several tiles, 6 layers: strips of 4 and 6
    ("mhd_kep", {"Num_R": 6, "Num_Z": 2, "aspect": 0.15, "Max_DT": 0.002}, 8),
    ("gr_disk", {"Num_R": 8, "Num_Z": 4, "Riemann_Solver": 0, **GR}, 8),
    ("euler_yee", {"Num_R": 16, "Num_Z": 4}, None),
    ("disk_planet", {"Num_R": 12, "aspect": 0.3}, 0),
])
def test_runs_by_tiles_equal_runs_by_elements(monkeypatch, cname, over, orders, merge):
    lib = capi.load_library(cpu_build.build())
    lib.dhx_check_orders.argtypes, lib.dhx_check_orders.restype = [C.c_void_p], C.c_long
    cfg, par, a = host_initial(cname, over)
    monkeypatch.setenv("DH_CPU_MERGE", merge)
    outs = []
    for order in range(5):
        monkeypatch.setenv("DH_CPU_ORDER", str(order))
        g = capi.DiscoHip(cfg, par, a, library=lib)
        n = lib.dhx_check_orders(g.ctx)
        assert n >= 0 and (orders is None or n == orders), n
        for _ in range(3):
            g.timestep(g.getmindt())
        outs.append(g.download(a))
        g.close()
    for order, x in enumerate(outs):
        for key in ("prim", "cons", "piph", "dphi", "wiph", "phi_flux"):
            assert np.array_equal(getattr(x, key), getattr(outs[0], key)), (order, key)
    assert np.isfinite(outs[0].prim).all()
    assert not np.array_equal(outs[0].prim, a.prim)

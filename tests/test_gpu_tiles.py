"""Meshes whose annuli are long enough for the launches by tiles (at least
0.94 of the lanes of each annulus's 64-cell tiles at work), and meshes just
below that, stepped on the GPU and by the host build of the same kernels
from one state: last tiles of 1 and of 63 cells, whole tiles, and annuli of
one tile less."""
import os
import tempfile

import numpy as np
import pytest

from disco_amd import capi, configs, state_io
from disco_amd.host_lib import HostRun

pytestmark = pytest.mark.gpu


def _initial(cname, over):
    cfg = configs.get(cname)
    par = cfg.par_dict(**over)
    d = tempfile.mkdtemp(prefix="tiles_")
    run = HostRun(cname, state_io.write_par(d, dict(par, Autotune=0)))
    path = os.path.join(d, "init.dstate")
    run.write(path)
    run.close()
    return cfg, par, state_io.read_state(path)


# aspect scales the cells per annulus (Np = 2 pi r / (aspect dr))
@pytest.mark.parametrize("cname,over", [
    ("euler_yee", {"Num_R": 6, "aspect": 0.02}),       # 314 to 1884 cells
    ("euler_yee", {"Num_R": 12, "aspect": 0.0982}),    # 64 to 767: the first annulus one full tile
    ("euler_yee_n1", {"Num_R": 5, "aspect": 0.04, "Riemann_Solver": 0}),
    ("disk_planet", {"Num_R": 9, "aspect": 0.05}),
    ("mhd_kep", {"Num_R": 6, "Num_Z": 3, "aspect": 0.03}),
    ("mhd_kep", {"Num_R": 6, "Num_Z": 3, "aspect": 0.3}),  # below the rule's line
    ("gr_disk", {"Num_R": 5, "Num_Z": 3, "aspect": 0.05, "R_Min": 8.0, "R_Max": 20.0, "CFL": 0.2,
                 "Riemann_Solver": 0}),
])
def test_long_annuli_step_as_the_host_build(cname, over):
    import sys
    sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpu_engine"))
    import build as cpu_build
    from helpers import compare_states
    cfg, par, a = _initial(cname, over)
    print(f"case {cname} {over}: annuli of {a.np_.min()} to {a.np_.max()} cells", flush=True)
    gpu = capi.DiscoHip(cfg, par, a)
    cpu = capi.DiscoHip(cfg, par, a, library=capi.load_library(cpu_build.build()))
    nvar = 6
    gpu.autotune(nvar)  # every order of the tiles
    for _ in range(nvar + 1):
        dt = min(gpu.getmindt(), 1e-4)
        gpu.timestep(dt)
        cpu.timestep(dt)
    # the parity bar of the GPU against the host build (helpers.PARITY_TOL)
    print("  worst", compare_states(gpu.download(a), cpu.download(a)), flush=True)
    gpu.close()
    cpu.close()


@pytest.mark.parametrize("aspect", [0.5, 0.12, 0.06, 0.03])
def test_flips_of_strong_shear(aspect):
    """Keplerian shear of about a cell a step flips most faces: tracks of
    fewer faces than a flip batch (256) and of several batches, in whole
    steps (the lengths around a batch: test_gpu_flips).  Steps from common
    states: a trajectory of this mesh is ill-conditioned (the host build's
    own moves by 1e-10 under a one-ulp change of libm)."""
    import sys
    sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpu_engine"))
    import build as cpu_build
    from helpers import compare_states
    cfg, par, a = _initial("mhd_kep", {"Num_R": 6, "Num_Z": 3, "aspect": aspect})
    print(f"case flips aspect {aspect}: annuli of {a.np_.min()} to {a.np_.max()} cells", flush=True)
    lib = capi.load_library(cpu_build.build())
    lib.dhx_flip_count.argtypes = [__import__("ctypes").c_void_p]
    lib.dhx_flip_count.restype = __import__("ctypes").c_long
    cpu = capi.DiscoHip(cfg, par, a, library=lib)
    s = a
    for n in range(4):
        gpu = capi.DiscoHip(cfg, par, s)
        # at most about a cell of shear between neighbouring annuli
        dt = min(cpu.getmindt(), 2 * np.pi / s.np_.max())
        gpu.timestep(dt)
        cpu.timestep(dt)
        s = cpu.download(s)
        print(f"  step {n}: {lib.dhx_flip_count(cpu.ctx)} flips so far, worst",
              compare_states(gpu.download(s), s, tol=1e-9), flush=True)
        gpu.close()
    assert lib.dhx_flip_count(cpu.ctx) > a.n_real() // 10
    cpu.close()


@pytest.mark.parametrize("cells", [5, 62, 63, 64, 65, 126, 127])
def test_edge_means_at_the_tiles_ends(cells):
    """The phi edges' means are formed by tiles of 63 cells, the last cell's
    from the next tile's first or the ring's: annuli of one short tile, of
    whole ones, and of one cell more and less."""
    import sys
    sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpu_engine"))
    import build as cpu_build
    from helpers import compare_states
    # Np = floor(2 pi r / (aspect dr)), r the ring's outer radius: of eight
    # rings from 0.5 to 2 (whose ghost rings stay at r > 0) the innermost
    dr = 1.5 / 8
    aspect = 2 * np.pi * (0.5 + dr) / (dr * (cells + 0.5))
    cfg, par, a = _initial("mhd_kep", {"Num_R": 8, "Num_Z": 2, "aspect": aspect})
    print(f"case edge means: annuli of {sorted(set(a.np_.tolist()))} cells", flush=True)
    assert cells in a.np_
    gpu = capi.DiscoHip(cfg, par, a)
    cpu = capi.DiscoHip(cfg, par, a, library=capi.load_library(cpu_build.build()))
    for _ in range(3):
        dt = min(gpu.getmindt(), 1e-4)
        gpu.timestep(dt)
        cpu.timestep(dt)
    print("  worst", compare_states(gpu.download(a), cpu.download(a)), flush=True)
    gpu.close()
    cpu.close()

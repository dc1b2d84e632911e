"""The launch sequence of large meshes (every kernel its own launch, the
kernels over cells and faces in each traversal order the tuner tries: by
tiles where the annuli are long, by elements where they are short, the
relativistic fluxes under HLLD) on small ones: every step against the host
build of the same kernels from a common state.  A step of n tuned ones runs
every kernel in one of its n variants, so each variant is compared."""
import os
import sys
import tempfile

import numpy as np
import pytest

from disco_amd import capi, configs, state_io
from disco_amd.host_lib import HostRun
from helpers import field_errors, rel_l1
from test_gpu_grmhd import HLLD_STEP_TOL, STEP_TOL

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpu_engine"))
import build as cpu_build  # noqa: E402

pytestmark = pytest.mark.gpu

GR = {"R_Min": 8.0, "R_Max": 20.0, "CFL": 0.2}
CASES = [
    # 2-D: long annuli (tiles) and short ones (elements)
    ("euler_yee", {"Num_R": 6, "aspect": 0.02}, 2),
    ("euler_yee_n1", {"Num_R": 24, "Riemann_Solver": 0}, 2),
    ("disk_planet", {"Num_R": 9, "aspect": 0.05}, 2),
    # 10 layers: strips of 4, 8 and 10; last tiles of many sizes
    ("mhd_kep", {"Num_R": 6, "Num_Z": 6, "aspect": 0.03}, 5),
    ("mhd_kep", {"Num_R": 12, "Num_Z": 6}, 2),
    ("gr_disk", {"Num_R": 5, "Num_Z": 6, "aspect": 0.05, "Riemann_Solver": 0, **GR}, 5),
    # (HLLD in the gas the fixtures of HLLD_STEP_TOL hold)
    ("gr_disk", {"Num_R": 12, "Num_Z": 6, "aspect": 0.08, "Riemann_Solver": 2}, 5),
    ("gr_disk", {"Num_R": 16, "Num_Z": 6, "Riemann_Solver": 2}, 2),
    ("kerr_torus", {"Num_R": 6, "Num_Z": 6, "aspect": 0.02}, 5),
    ("kerr_torus", {"Num_R": 24, "Num_Z": 12}, 2),
]


def _large(g):
    """Makes a context take the large meshes' sequence."""
    import ctypes as C
    fn = capi.lib().dhx_merge_below
    fn.argtypes, fn.restype = [C.c_void_p, C.c_long], C.c_int
    assert fn(g.ctx, 0) == 0


def _initial(cname, over):
    cfg = configs.get(cname)
    par = cfg.par_dict(**over)
    d = tempfile.mkdtemp(prefix="large_")
    run = HostRun(cname, state_io.write_par(d, dict(par, Autotune=0)))
    path = os.path.join(d, "init.dstate")
    run.write(path)
    run.close()
    return cfg, par, state_io.read_state(path)


def _steps_as_the_host_build(g, cfg, par, a, steps):
    """Every step of context g against the host build's from g's own state."""
    tol = HLLD_STEP_TOL if cfg.hydro == "grmhd2" and par.get("Riemann_Solver") == 2 else STEP_TOL
    host = capi.load_library(cpu_build.build())
    m = a.real_mask()
    for n in range(steps):
        h = capi.DiscoHip(cfg, par, g.download(a), library=host)
        # the shear of a step stays below a cell
        dt = min(g.getmindt(), 1e-4) if cfg.hydro != "grmhd2" else g.getmindt()
        g.timestep(dt)
        h.timestep(dt)
        x, y = g.download(a), h.download(a)
        h.close()
        e = field_errors(x, y)
        k = max(e, key=e.get)
        ephi = rel_l1(x.phi_flux[:, m], y.phi_flux[:, m]) if a.nf else 0.0
        print(f"  step {n}: worst {e[k]:.2e} ({k}), Phi {ephi:.2e}", flush=True)
        assert np.isfinite(x.prim[:, m]).all()
        assert e[k] <= tol and ephi <= tol, (n, k, e[k], ephi)


@pytest.mark.parametrize("cname,over,nvar", CASES)
def test_every_order_steps_as_the_host_build(cname, over, nvar):
    cfg, par, a = _initial(cname, over)
    print(f"case {cname} {over}: annuli of {a.np_.min()} to {a.np_.max()} cells", flush=True)
    g = capi.DiscoHip(cfg, par, a)
    _large(g)
    g.autotune(nvar)
    _steps_as_the_host_build(g, cfg, par, a, nvar + 1)  # the last step in the variants kept
    variants = {name: len(row["ms_variants"]) for name, row in g.read_tuning().items()}
    print("  variants", variants, flush=True)
    assert max(variants.values()) == nvar
    for name in ("ranges_r", "faces_r", "grad_r", "update", "plm_phi"):
        assert variants[name] == nvar, (name, variants)
    for name in ("flux_phi", "flux_r"):  # by elements, in storage order
        assert variants[name] == 2
    if cfg.hydro != "euler":
        for name in ("faces_z", "grad_z", "edges_final", "update_B", "line_steps_r", "line_steps_z",
                     "edge_segments", "edge_adjust", "bfaces_c2p"):
            assert variants[name] == nvar, (name, variants)
    g.close()


@pytest.mark.parametrize("large", [False, True])
@pytest.mark.parametrize("cname,over", [
    ("euler_yee", {"Num_R": 16, "Num_Z": 4}),               # z faces, held z sides
    ("euler_yee", {"Num_R": 16, "Num_Z": 4, "PLM": 0.0}),   # cleared slopes, both directions
    ("euler_yee", {"Num_R": 16, "PLM": 0.0}),
    ("mhd_kep", {"Num_R": 8, "Num_Z": 1}),                  # transport without z faces
    ("mhd_kep", {"Num_R": 10, "Num_Z": 4, "Timestep": 1}),  # forward Euler
    # ring-averaged mesh velocity (not MHD's: HLLD branches on the contact at
    # the face's own speed there, and a step moves by 1e-8 with its rounding)
    ("euler_yee", {"Num_R": 24, "Mesh_Motion": 3, "Riemann_Solver": 0}),
    ("mhd_kep", {"Num_R": 10, "Num_Z": 4, "Mesh_Motion": 0}),
    ("gr_disk", {"Num_R": 16, "Num_Z": 1, "Riemann_Solver": 0}),
])
def test_both_sequences_step_as_the_host_build(cname, over, large):
    """Meshes and options whose launches differ: one direction alone,
    cleared slopes, mesh motions, forward Euler."""
    cfg, par, a = _initial(cname, over)
    print(f"case {cname} {over}, {'apart' if large else 'merged'}", flush=True)
    g = capi.DiscoHip(cfg, par, a)
    if large:
        _large(g)
    _steps_as_the_host_build(g, cfg, par, a, 4)
    g.close()


@pytest.mark.parametrize("cname,over", [
    ("euler_yee", {"Num_R": 24}), ("disk_planet", {"Num_R": 48}),
    ("mhd_kep", {"Num_R": 16, "Num_Z": 4}),
    ("gr_disk", {"Num_R": 16, "Num_Z": 4, "Riemann_Solver": 2, **GR}),
])
def test_merged_launches_equal_separate_ones(cname, over):
    """Bit for bit: the merged launches run the same bodies.  (Not the Kerr
    torus, whose merged kernels the compiler rounds by an ulp otherwise.)"""
    cfg, par, a = _initial(cname, over)
    print(f"case merged and apart {cname} {over}", flush=True)
    merged, apart = capi.DiscoHip(cfg, par, a), capi.DiscoHip(cfg, par, a)
    _large(apart)
    for n in range(5):
        dt = merged.getmindt()
        assert apart.getmindt() == dt, n
        merged.timestep(dt)
        apart.timestep(dt)
    x, y = merged.download(a), apart.download(a)
    for key in ("prim", "cons", "piph", "dphi", "phi_flux"):
        assert np.array_equal(getattr(x, key), getattr(y, key)), key
    names = [set(), set()]
    for i, g in enumerate((merged, apart)):
        g.enable_timers()
        g.timestep(dt)
        names[i] = {r[0] for r in g.read_timers()}
        g.close()
    assert names[0] != names[1] and len(names[0]) < len(names[1]), names

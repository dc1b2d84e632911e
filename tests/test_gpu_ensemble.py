"""Ensembles on the GPU (dh_ens_*): four disk-planet runs of different
resolution and planet mass stepped together, every kernel of their step one
launch for all four, each with its own CFL dt, planets and diagnostics.

* each member equals the same run stepped alone through dh_timestep, bit for
  bit (the grouped launch runs the same kernel bodies on the same data);
* each member matches the reference build (oracle/_ref) of its own in.par to
  the parity bar, with its Analysis sums.
"""
import os
import subprocess
import tempfile

import numpy as np
import pytest

from disco_amd import configs, state_io
from helpers import PARITY_TOL, compare_states

pytestmark = pytest.mark.gpu

MEMBERS = [(64, 1e-3), (128, 1e-5), (32, 3e-4), (96, 1e-4)]
STEPS = 12


def _par(nr, q):
    return configs.get("disk_planet").par_dict(Num_R=nr, Mass_Ratio=q, Autotune=0)


@pytest.mark.parametrize("graphs", [True, False])
def test_ensemble_members_equal_their_own_runs(graphs):
    from disco_amd.host_lib import Ensemble, HostRun
    d = tempfile.mkdtemp(prefix="ens_")
    print(f"case ensemble of {len(MEMBERS)} disk-planet runs, graphs {graphs}: {STEPS} steps",
          flush=True)
    runs = [HostRun("disk_planet", state_io.write_par(os.path.join(d, f"e{i}"), _par(nr, q)))
            for i, (nr, q) in enumerate(MEMBERS)]
    solo = [HostRun("disk_planet", state_io.write_par(os.path.join(d, f"s{i}"), _par(nr, q)))
            for i, (nr, q) in enumerate(MEMBERS)]
    ens = Ensemble(runs, graphs=graphs)
    try:
        for n in range(STEPS):
            ens.step()
            for i, r in enumerate(solo):
                dt = r.getmindt()
                assert dt == ens.dts[i], (n, i, dt, ens.dts[i])
                r.timestep(dt)
        ens.sync()
        for i, (a, b) in enumerate(zip(runs, solo)):
            pa, pb = os.path.join(d, f"a{i}.dstate"), os.path.join(d, f"b{i}.dstate")
            a.write(pa)
            b.write(pb)
            x, y = state_io.read_state(pa), state_io.read_state(pb)
            for key in ("prim", "piph", "dphi", "wiph", "planets"):
                assert np.array_equal(getattr(x, key), getattr(y, key)), (i, key)
            # conserved variables of real cells (a ghost cell's are never
            # written or read: only its primitives are boundary data)
            m = x.real_mask()
            assert np.array_equal(x.cons[:, m], y.cons[:, m]), (i, "cons")
            assert x.t == y.t
            print(f"  member {i} (Nr {MEMBERS[i][0]}): identical to its own run", flush=True)
    finally:
        ens.close()
        for r in runs + solo:
            r.close()


def test_ensemble_members_match_the_reference():
    from disco_amd.host_lib import Ensemble, HostRun
    cfg = configs.get("disk_planet")
    ref = configs.ref_binary(cfg)
    if not os.path.exists(ref):
        pytest.skip(f"{ref} not built")
    d = tempfile.mkdtemp(prefix="ensref_")
    dirs = []
    for i, (nr, q) in enumerate(MEMBERS):
        di = os.path.join(d, str(i))
        state_io.write_par(di, _par(nr, q))
        subprocess.run([ref, di, str(STEPS)], cwd=di, check=True, capture_output=True)
        dirs.append(di)
    runs = [HostRun("disk_planet", os.path.join(di, "in.par")) for di in dirs]
    ens = Ensemble(runs)
    try:
        for _ in range(STEPS):
            ens.step()
        ens.sync()
        for i, (r, di) in enumerate(zip(runs, dirs)):
            r.write(os.path.join(di, "got.dstate"))
            got = state_io.read_state(os.path.join(di, "got.dstate"))
            want = state_io.read_state(os.path.join(di, "state_final.bin"))
            worst = compare_states(got, want)
            assert abs(got.t - want.t) <= 1e-12 * want.t
            _, q_want = state_io.read_diag(os.path.join(di, "diag.bin"))
            q_got = r.diagnostics(q_want.size).reshape(q_want.shape)
            scale = np.abs(q_want).sum(axis=0)
            scale = np.maximum(scale, 1e-6 * scale.max())
            err = (np.abs(q_got - q_want).sum(axis=0) / scale).max()
            print(f"  member {i} (Nr {MEMBERS[i][0]}): worst rel L1 vs reference {worst:.2e}, "
                  f"diagnostics {err:.2e}", flush=True)
            assert worst <= PARITY_TOL and err <= PARITY_TOL
    finally:
        ens.close()
        for r in runs:
            r.close()


@pytest.mark.parametrize("graphs", [True, False])
@pytest.mark.parametrize("cname,sizes", [
    # copied ghost rings on both z sides, constrained transport with flips,
    # edge means by 63-cell tiles; annuli from under one tile to a dozen
    ("mhd_kep", [dict(Num_R=16, Num_Z=4), dict(Num_R=32, Num_Z=8),
                 dict(Num_R=10, Num_Z=6, aspect=0.1)]),
    ("gr_disk", [dict(Num_R=16, Num_Z=4, R_Min=8.0, R_Max=20.0, CFL=0.2, Riemann_Solver=2),
                 dict(Num_R=24, Num_Z=6, R_Min=8.0, R_Max=20.0, CFL=0.2, Riemann_Solver=2)]),
    # the smallest members: annuli of a few cells, polar axis
    ("euler_yee", [dict(Num_R=24), dict(Num_R=6), dict(Num_R=13)]),
])
def test_ensembles_of_every_module_equal_their_own_runs(cname, sizes, graphs):
    """The members' launches (by elements, grouped) against the same runs'
    own launches (by elements or by tiles, some merged): the same kernel
    bodies on the same data, bit for bit."""
    from disco_amd.host_lib import Ensemble, HostRun
    d = tempfile.mkdtemp(prefix="ensall_")
    print(f"case ensemble {cname} {sizes}, graphs {graphs}", flush=True)

    def open_all(tag):
        return [HostRun(cname, state_io.write_par(
            os.path.join(d, f"{tag}{i}"), configs.get(cname).par_dict(**s, Autotune=0)))
            for i, s in enumerate(sizes)]
    runs, solo = open_all("e"), open_all("s")
    ens = Ensemble(runs, graphs=graphs)
    try:
        for n in range(6):
            ens.step()
            for i, r in enumerate(solo):
                dt = r.getmindt()
                assert dt == ens.dts[i], (n, i, dt, ens.dts[i])
                r.timestep(dt)
        ens.sync()
        for i, (a, b) in enumerate(zip(runs, solo)):
            pa, pb = os.path.join(d, f"a{i}.dstate"), os.path.join(d, f"b{i}.dstate")
            a.write(pa)
            b.write(pb)
            x, y = state_io.read_state(pa), state_io.read_state(pb)
            assert np.isfinite(x.prim).all()
            for key in ("prim", "piph", "dphi", "wiph", "phi_flux"):
                assert np.array_equal(getattr(x, key), getattr(y, key)), (
                    i, key, np.abs(getattr(x, key) - getattr(y, key)).max())
            print(f"  member {i}: annuli of {x.np_.min()} to {x.np_.max()} cells, identical",
                  flush=True)
    finally:
        ens.close()
        for r in runs + solo:
            r.close()


@pytest.mark.parametrize("cname,over", [
    ("euler_yee", {"Num_R": 24}), ("disk_planet", {"Num_R": 48}),
    ("mhd_kep", {"Num_R": 12, "Num_Z": 4}),
    ("gr_disk", {"Num_R": 12, "Num_Z": 4, "R_Min": 8.0, "R_Max": 20.0, "CFL": 0.2}),
])
def test_launch_tables_are_built_once(cname, over):
    """The launches of an RK2 run have the same arguments in every step (dt,
    planets and the minima lie in device memory), so their tables are built
    in the first steps and stay: not one is freed, allocated and uploaded
    again for bytes of an argument that hold no value."""
    import ctypes as C
    from disco_amd import capi
    from disco_amd.host_lib import Ensemble, HostRun
    d = tempfile.mkdtemp(prefix="enstab_")
    print(f"case launch tables of {cname} {over}", flush=True)
    tables = capi.lib().dhx_ens_tables
    tables.argtypes, tables.restype = [C.c_void_p], C.c_long
    runs = [HostRun(cname, state_io.write_par(
        os.path.join(d, str(i)), configs.get(cname).par_dict(**over, Autotune=0))) for i in range(3)]
    ens = Ensemble(runs)
    try:
        built = []
        for _ in range(8):
            ens.step()
            built.append(tables(ens.ens))
        print("  tables built by step:", built, flush=True)
        assert built[2] > 0 and built[-1] == built[2], built
    finally:
        ens.close()
        for r in runs:
            r.close()

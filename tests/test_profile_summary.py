"""The profile summaries on the symbols the current library emits: every
kernel of a timestep has its timer name, launches by elements and by tiles of
one kernel are the same functor, and the launches of the launch tuner's sweep
are told from those after it by the timesteps."""
import os
import re
import subprocess

import pytest

from disco_amd import capi
from disco_amd.profile_summary import after_tuning, functor_of, timer_name

ELEMS = "void k_elems<dh::KGrad<8, 1> >(dh::KGrad<8, 1>, long, int)"
TILES = "void k_tiles<dh::KGrad<8, 1> >(dh::KGrad<8, 1>, dh::TileList, int)"
BOTH = ("void k_elems<dh::KBoth<dh::KGrad<8, 1>, dh::KGrad<8, 2> > >"
        "(dh::KBoth<dh::KGrad<8, 1>, dh::KGrad<8, 2> >, long, int)")
RINGS = ("void k_elems_rings<dh::KPlmPhi<5> >(dh::KPlmPhi<5>, long, unsigned int, dh::Mesh, "
         "double const*, int*)")
FLIPS = ("k_flips(dh::Mesh, dh::Faces, dh::Faces, double const*, double const*, double const*, "
         "double*, double*)")
STEP = "k_set_step(dh::StepArgs*, dh::StepArgs)"


def test_functor_of_every_launch_form():
    assert functor_of(ELEMS) == functor_of(TILES) == "dh::KGrad<8, 1>"
    assert functor_of(BOTH) == "dh::KBoth<dh::KGrad<8, 1>, dh::KGrad<8, 2> >"
    assert functor_of(RINGS) == "dh::KPlmPhi<5>"
    assert functor_of(FLIPS) == FLIPS
    assert timer_name(TILES) == "grad_r" and timer_name(BOTH) == "grad"
    assert timer_name(FLIPS) == "flips" and timer_name(RINGS) == "plm_phi_rings"


def _symbols():
    """The library's kernels as a profiler prints them (their host stubs)."""
    out = subprocess.run(["nm", "-C", capi.LIB_PATH], capture_output=True, text=True, check=True)
    syms = set()
    for ln in out.stdout.splitlines():
        m = re.match(r"[0-9a-f]+ \w (.*__device_stub__.*)$", ln)
        if m:
            syms.add(m.group(1).replace("__device_stub__", ""))
    return syms


def _sequence_names():
    path = os.path.join(os.path.dirname(capi.__file__), "csrc", "dh_pipeline.h")
    with open(path) as f:
        src = f.read()
    return set(re.findall(r'run_(?:ord|both|beside_rings)\(\s*(?:x,\s*)?"(\w+)"', src))


@pytest.mark.skipif(not os.path.exists(capi.LIB_PATH), reason="libdisco_hip.so not built")
def test_every_kernel_of_a_step_has_its_timer_name():
    syms = _symbols()
    assert len(syms) > 100
    # ensembles have no timers; the model's training and clears are no part of a step
    other = r"k_group<|k_set_steps|k_fill_u64|k_mlp_|KZeroWords|KCopyWords|KC2pHarvest|k_run<dh::KMlp"
    for s in syms:
        if not re.search(other, s):
            assert timer_name(s), s
    named = {timer_name(s) for s in syms}
    host_only = {"flip_flags_r", "flip_flags_z"}
    assert _sequence_names() - host_only <= named, _sequence_names() - host_only - named
    # the elements' and the tiles' launches of a kernel are one functor
    elems = {functor_of(s) for s in syms if s.startswith("void k_elems<")}
    tiles = {functor_of(s) for s in syms if s.startswith("void k_tiles<")}
    assert tiles & elems and not any("(" in f for f in tiles | elems)


def _run(steps, launches):
    """Rows of a run: per timestep one k_set_step and the launches."""
    rows, did = [(ELEMS, 1, 5.0)], 1
    for n in range(steps):
        for name in (STEP,) + launches:
            did += 1
            rows.append((name, did, float(n)))
    return rows


def test_after_tuning_leaves_the_sweeps_timesteps_out():
    rows = _run(6, (TILES, TILES, FLIPS))
    kept = after_tuning(rows, 4)
    assert [r[2] for r in kept if r[0] == TILES] == [4.0, 4.0, 5.0, 5.0]
    assert [r[2] for r in kept if r[0] == FLIPS] == [4.0, 5.0]
    assert not any(r[0] == ELEMS for r in kept)  # (set-up)
    # the rows' own order does not matter
    assert sorted(after_tuning(rows[::-1], 4)) == sorted(kept)


def test_after_tuning_of_a_run_that_is_all_sweep():
    with pytest.raises(ValueError, match="4 timesteps"):
        after_tuning(_run(4, (TILES,)), 4)

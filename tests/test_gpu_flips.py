"""The face flips on the GPU (flip_track: one workgroup per track, batches
of 256 faces in LDS, runs of flipped faces side by side) against the host
build's face-after-face hand-overs, bit for bit (sums of two numbers and sign
changes, in the same order for every flux): tracks of 2 and 3 faces, of a
whole batch, of one face more and less, of a batch and one and two faces (a
last batch of one face; a batch whose outer neighbours meet), of two and three
batches, under motions that flip every face, many, some and single ones."""
import os
import sys

import numpy as np
import pytest

from disco_amd import capi
import flip_mesh

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpu_engine"))
import build as cpu_build  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["reverse", "some", "many", "single"])
@pytest.mark.parametrize("seed", range(4))
def test_flips_equal_the_host_build(seed, kind):
    cfg, par, s = flip_mesh.mesh(seed)
    print(f"case flips {kind}, seed {seed}: {s.ntot} cells", flush=True)
    assert flip_mesh.LENGTHS <= ({int(v) for v in (flip_mesh.SIZES[:, 1:] + flip_mesh.SIZES[:, :-1]).ravel()}
                                 | {int(v) for v in (flip_mesh.SIZES[1:] + flip_mesh.SIZES[:-1]).ravel()})
    i = ("reverse", "some", "many", "single").index(kind)
    rng = np.random.default_rng(100 * seed + i)
    w = flip_mesh.motion(kind, s, rng)
    Phi2 = rng.standard_normal(s.phi_flux.shape)
    host = capi.load_library(cpu_build.build())
    got = flip_mesh.flips(capi.lib(), cfg, par, s, w, Phi2)
    want = flip_mesh.flips(host, cfg, par, s, w, Phi2)
    for name, x, y in zip(("Phi", "Phi2", "LR of the r faces", "LR of the z faces"), got, want):
        bad = np.flatnonzero((x != y).ravel())
        assert bad.size == 0, f"{name}: {bad.size} differ, first at {bad[:4].tolist()}"
    changed = int((want[0] != s.phi_flux).sum())
    print(f"  {changed} fluxes handed over", flush=True)
    assert changed > 0

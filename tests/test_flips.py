"""The face flips on meshes of chosen track lengths, host build: the result
of the tracks' hand-overs is what flipping face after face in order gives
(bfields.c:742-814), for every motion the GPU test uses; and those motions do
flip first and last faces of tracks of every length that the GPU kernel's
batches of 256 faces make special."""
import os
import sys

import numpy as np
import pytest

from disco_amd import capi
import flip_mesh

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpu_engine"))
import build as cpu_build  # noqa: E402


def _face_by_face(s, dim, L, R, LR, rows, phis):
    """flip_fluxes in order: face n's flux goes to face n - 1's and n + 1's
    slots, and faces n and n - 1 change owner."""
    slot = {1: (2, 1), 2: (4, 3)}[dim]
    f0 = 0
    for d, n, flag in rows:
        if d != dim:
            continue
        for i in np.flatnonzero(flag):
            f, m, p = f0 + i, f0 + (i - 1) % n, f0 + (i + 1) % n
            at = [(slot[int(LR[q] != 0)], L[q] if LR[q] == 0 else R[q]) for q in (f, m, p)]
            for Phi in phis:
                ph = Phi[at[0]]
                Phi[at[0]] = Phi[at[1]] + ph
                Phi[at[1]] = -ph
                Phi[at[2]] = Phi[at[2]] + ph
            LR[f], LR[m] = LR[f] == 0, LR[m] == 0
        f0 += n


@pytest.mark.parametrize("kind", ["reverse", "some", "many", "single"])
def test_flips_are_face_after_face(kind):
    lib = capi.load_library(cpu_build.build())
    cfg, par, s = flip_mesh.mesh(3)
    rng = np.random.default_rng(11)
    w = flip_mesh.motion(kind, s, rng)
    Phi2 = rng.standard_normal(s.phi_flux.shape)
    got = flip_mesh.flips(lib, cfg, par, s, w, Phi2)
    rows = flip_mesh.flagged(lib, cfg, par, s, w)
    assert sum(int(f.sum()) for _, _, f in rows) > (5 if kind == "single" else 100)
    want = [s.phi_flux.copy(), Phi2.copy()]
    g = capi.DiscoHip(cfg, par, s, library=lib)
    for dim in (1, 2):
        L, R, LR, _, _ = g.faces(dim)
        LR = LR.copy()
        _face_by_face(s, dim, L, R, LR, rows, want)
        assert np.array_equal(got[1 + dim], LR), dim
    g.close()
    assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])


def test_motions_flip_both_ends_of_every_special_track():
    lib = capi.load_library(cpu_build.build())
    first, last, both = set(), set(), set()
    for seed in range(4):
        cfg, par, s = flip_mesh.mesh(seed)
        for i, kind in enumerate(("reverse", "some", "many", "single")):
            w = flip_mesh.motion(kind, s, np.random.default_rng(100 * seed + i))
            for _, n, f in flip_mesh.flagged(lib, cfg, par, s, w):
                if f[0]:
                    first.add(n)
                if f[-1]:
                    last.add(n)
                if f[0] and f[-1] and not f.all():
                    both.add(n)
    # (a track of two faces between two single cells, of one owner, never flips)
    special = flip_mesh.LENGTHS - {2}
    assert special <= first & last, special - (first & last)
    assert {256, 257, 512, 514, 769} <= both

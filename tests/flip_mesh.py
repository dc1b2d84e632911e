"""A magnetised mesh of chosen annulus sizes and a set of face motions, for
the tests of the face flips."""
import ctypes as C

import numpy as np

from disco_amd import capi, configs
from disco_amd.state_io import MeshState

# Cells of annulus (j, k), k the row: neighbours in a row and in a column
# share a face track of as many faces as their cells together.
SIZES = np.array([
    [128, 128, 129, 129, 127, 128],
    [1, 1, 2, 62, 66, 190],
    [256, 256, 257, 257, 255, 256],
    [384, 385, 384, 386, 383, 384],
    [128, 129, 130, 126, 131, 5],
], dtype=np.int32)
NZ, NR = SIZES.shape
# around one, two and three flip batches (256 faces), and the shortest tracks
LENGTHS = {2, 3, 64, 128, 255, 256, 257, 258, 511, 512, 513, 514, 767, 769, 770}


def mesh(seed):
    """(config, in.par dict, state): cells of uneven width, random fluxes."""
    cfg = configs.get("mhd_kep")
    rng = np.random.default_rng(seed)
    np_ = SIZES.ravel()
    nt = int(np_.sum())
    dphi = np.concatenate([(lambda w: 2 * np.pi * w / w.sum())(rng.uniform(0.5, 1.5, n))
                           for n in np_])
    off = np.concatenate([[0], np.cumsum(np_)])
    piph = np.concatenate([(rng.uniform(0, 2 * np.pi) + np.cumsum(dphi[off[a]:off[a + 1]]))
                           % (2 * np.pi) for a in range(np_.size)])
    prim = np.zeros((cfg.nq, nt))
    prim[0] = prim[1] = 1.0
    s = MeshState(nq=cfg.nq, nf=cfg.nf, nr=NR, nz=NZ, ng=(2, 2, 2, 2), t=0.0, phi_max=2 * np.pi,
                  np_=np_.copy(), r_jph=np.linspace(0.4, 1.6, NR + 1),
                  z_kph=np.linspace(-0.3, 0.3, NZ + 1), prim=prim, cons=prim.copy(), piph=piph,
                  dphi=dphi, wiph=np.zeros(nt), phi_flux=rng.standard_normal((cfg.nf, nt)),
                  planets=np.zeros((1, capi.PLANET_STRIDE)), num_c=cfg.num_c)
    return cfg, cfg.par_dict(), s


def motion(kind, s, rng):
    """Displacements of every cell's edge: reversed order (every face
    flips), half a cell (some), two cells (many), and single cells."""
    width = 2 * np.pi / np.repeat(s.np_, s.np_)
    if kind == "reverse":
        return -2.0 * s.piph
    if kind == "some":
        return 0.5 * width * rng.standard_normal(s.ntot)
    if kind == "many":
        return 2.0 * width * rng.standard_normal(s.ntot)
    return np.where(rng.random(s.ntot) < 0.02, 3.0 * width, 0.0)  # "single"


def flips(lib, cfg, par, s, w, Phi2):
    """(Phi, Phi2, LR of the r and z faces) after the flips of faces moved
    by w, by library lib."""
    fn = lib.dhx_flips
    dp, bp = C.POINTER(C.c_double), C.POINTER(C.c_byte)
    fn.argtypes, fn.restype = [C.c_void_p, C.c_double, dp, bp, bp], C.c_int
    t = s.copy()
    t.wiph = w / 0.01
    g = capi.DiscoHip(cfg, par, t, library=lib)
    n = [len(g.faces(d)[0]) for d in (1, 2)]
    lr = [np.zeros(k, np.int8) for k in n]
    out = np.ascontiguousarray(Phi2).copy()
    rc = fn(g.ctx, 0.01, out.ctypes.data_as(dp), *[a.ctypes.data_as(bp) for a in lr])
    assert rc == 0, lib.dh_last_error()
    phi = g.download(t).phi_flux
    g.close()
    return phi, out, lr[0], lr[1]


def flagged(lib, cfg, par, s, w):
    """Per track (dim, first face, length): which faces flip, from the
    positions alone."""
    g = capi.DiscoHip(cfg, par, s, library=lib)
    rows = []
    for dim in (1, 2):
        L, R, LR, _, _ = g.faces(dim)
        o = np.where(LR == 0, L, R)
        up = s.piph[o] + (w / 0.01)[o] * 0.01
        pairs = ([(j + NR * k, j + 1 + NR * k) for k in range(NZ) for j in range(NR - 1)]
                 if dim == 1 else [(j + NR * k, j + NR * (k + 1)) for k in range(NZ - 1)
                                   for j in range(NR)])
        f = 0
        for a, b in pairs[:-1]:  # (the last track is skipped, as the reference does)
            n = int(s.np_[a] + s.np_[b])
            u = up[f:f + n]
            d = u - np.roll(u, 1)
            d -= 2 * np.pi * np.round(d / (2 * np.pi))
            rows.append((dim, n, d < 0.0))
            f += n
    g.close()
    return rows

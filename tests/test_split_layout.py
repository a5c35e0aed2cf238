"""The staging layout of bp_split_kernel, checked on the host: which bytes of a
row buffer each angle's copies write and which bytes each 4 x 4 block reads,
with the kernel's own float32 coordinates."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

TILES = ((32, 32), (32, 16), (16, 16))
MAX_SCALE = 1.17
f32 = np.float32


def layout(risa, shape, scale):
    fn = risa.load().risa_bp_split_layout
    fn.argtypes, fn.restype = [C.c_int, C.c_float, C.POINTER(C.c_int)], C.c_int
    v = (C.c_int * 7)()
    assert fn(shape, scale, v) == 0
    return dict(zip(("W", "angles", "rows", "row", "pitch", "buffer", "lds"), v))


def test_angles_do_not_share_bytes(risa):
    """Different waves copy different angles, so no byte may belong to two."""
    for shape in range(3):
        for scale in np.linspace(0.05, MAX_SCALE - 1e-4, 400):
            lay = layout(risa, shape, scale)
            end = 0
            for a in range(lay["angles"]):
                start = a * lay["pitch"]
                assert start >= end and start % 16 == 0, f"shape {shape} scale {scale}: angles {a - 1} and {a} overlap"
                end = start + lay["rows"] * lay["row"]
            assert end <= lay["buffer"] and lay["buffer"] % 16 == 0 and lay["lds"] <= 160 * 1024


def fma(a, b, c):
    return (a.astype(np.float64) * b + c).astype(f32)   # exact product, one rounding more than the hardware's


@pytest.mark.parametrize("N,D,rot", [(512, 512, 0.0), (512, 485, 0.0), (528, 500, 13.0), (512, 394, -30.0),
                                     (512, 580, 45.0), (128, 149, 7.0), (128, 98, 0.0), (128, 106, 0.0),
                                     (128, 121, -45.0), (128, 125, 0.0), (96, 41, 0.0), (70, 61, 13.0), (33, 20, 45.0)])
def test_blocks_read_their_own_rows(risa, N, D, rot):
    """Every sample with a weight lies in the rows of its angle, every read in
    the buffer."""
    P = 250
    ang = np.arange(P) * np.pi / P + rot / 180 * np.pi
    c, s = np.cos(ang).astype(f32), np.sin(ang).astype(f32)
    scale, center, cI = f32(D) / f32(N), f32((N - 1) * 0.5), int(D * 0.5)
    coord = lambda x: (np.asarray(x).astype(f32) - center) * scale
    for shape, (TX, TY) in enumerate(TILES):
        lay = layout(risa, shape, scale)
        nx, ny = -(-N // TX), -(-N // TY)
        for tx, ty in sorted({(0, 0), (nx - 1, 0), (0, ny - 1), (nx - 1, ny - 1), (nx // 2, ny // 2), (nx // 3, ny // 4)}):
            x0, y0 = tx * TX, ty * TY
            xa, xb, ya, yb = (coord(v) for v in (x0, x0 + TX - 1, y0, y0 + TY - 1))
            # angle_window
            t4 = [fma(y, s, (x * c).astype(f32)) for x in (xa, xb) for y in (ya, yb)]
            T = np.floor(np.minimum.reduce(t4))
            tm = np.minimum.reduce([fma(y, s, fma(x, c, -T)) for x in (xa, xb) for y in (ya, yb)])
            kmin = np.floor(tm).astype(int)
            odd = (T.astype(int) + cI) & 1
            first = (kmin + odd - 2) & ~1
            origin = (-T + odd).astype(f32)
            low = (f32(3) * scale * (np.minimum(c, 0) + np.minimum(s, 0)) - f32(0.01)).astype(f32)
            x, y = np.meshgrid(np.arange(TX), np.arange(TY))
            xc, yc = coord(x0 + x), coord(y0 + y)
            t = fma(yc[None], s[:, None, None], fma(xc[None], c[:, None, None], origin[:, None, None]))
            block = t[:, ::4, ::4]                                  # each block's first pixel
            kb = np.floor((block + low[:, None, None]).astype(f32)).astype(int) & ~1
            k = np.floor(t).astype(int)
            q = k - kb.repeat(4, 1).repeat(4, 2)
            assert q.min() >= 0 and q.max() <= 6
            rel = k - first[:, None, None]                          # samples rel, rel + 1 have weights
            assert rel.min() >= 0 and (rel.max() + 1) // 2 < lay["rows"]
            row = (kb - first[:, None, None]) // 2                  # rows row .. row + 3 are read
            assert row.min() >= 0
            assert (lay["angles"] - 1) * lay["pitch"] + (row.max() + 4) * lay["row"] <= lay["buffer"]

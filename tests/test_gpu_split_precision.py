"""bp_split_kernel (22-bit operands on the matrix cores) is no less exact than
bp_linear_kernel: distance to a float64 backprojection of the same filtered
sinogram, against that of the FP32 variant of the same tile."""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def sinogram(P, D, seed):
    """Parallel projections of 12 ellipses in a field of D detectors."""
    rng = np.random.default_rng(seed)
    th = np.arange(P)[:, None] * math.pi / P
    s = np.arange(D)[None, :] - D // 2
    out = np.zeros((P, D))
    for _ in range(12):
        a, b = rng.uniform(0.03, 0.2, 2) * D
        r, w, phi, mu = 0.25 * D * math.sqrt(rng.uniform()), *rng.uniform(0, 2 * math.pi, 2), rng.uniform(0.1, 1.0)
        A2 = (a * np.cos(th - phi)) ** 2 + (b * np.sin(th - phi)) ** 2
        u = s - r * np.cos(th - w)
        out += 2 * mu * a * b / A2 * np.sqrt(np.maximum(A2 - u * u, 0)) / D
    return out.astype(np.float32)


def backproject64(x, N):
    """x [S][P][D] float64 on the GPU -> images, zero outside the circle."""
    import torch

    S, P, D = x.shape
    c = torch.arange(N, device=x.device, dtype=torch.float64) - (N - 1) * 0.5
    y, xx = torch.nonzero(c[None, :] ** 2 + c[:, None] ** 2 <= N * N * 0.25, as_tuple=True)
    rows = torch.zeros((P, D + 2, S), dtype=torch.float64, device=x.device)
    rows[:, 1:D + 1] = x.permute(1, 2, 0)
    acc = torch.zeros((xx.numel(), S), dtype=torch.float64, device=x.device)
    for a in range(P):
        t = (c[xx] * math.cos(a * math.pi / P) + c[y] * math.sin(a * math.pi / P)) * (D / N)
        k = t.floor()
        f = (t - k)[:, None]
        k = k.long() + D // 2
        acc += rows[a][(k + 1).clamp(0, D + 1)] * (1 - f) + rows[a][(k + 2).clamp(0, D + 1)] * f
    img = torch.zeros((S, N, N), dtype=torch.float64, device=x.device)
    img[:, y, xx] = (acc * (math.pi / P / (D / N))).T
    return img


@pytest.mark.parametrize("N,P,D,window", [(512, 1000, 512, 0), (256, 500, 256, 1), (501, 776, 431, 3),
                                          (474, 944, 462, 4), (323, 914, 297, 0), (560, 300, 210, 2),
                                          (385, 400, 437, 0)])
def test_split_is_no_less_exact(risa, geom_c0, cuda, N, P, D, window):
    import torch
    from risa_amd import device

    lib = risa.load()
    run, size = lib.risa_bp_run_split, lib.risa_bp_split_bytes
    run.argtypes = [C.c_void_p, C.c_int, C.c_void_p, C.c_float, C.c_int, C.c_void_p, C.c_void_p, C.c_void_p]
    run.restype, size.argtypes, size.restype = C.c_int, [C.c_void_p], C.c_size_t
    g = geom_c0.replace(numberOfPixels=N, numberOfParallelProjections=P, numberOfParallelDetectors=D,
                        rotationOffset=0.0, fusedMasking=1, maskingValue=0.0, filterType=window)
    S = 2
    x = torch.from_numpy(np.stack([sinogram(P, D, N + i) for i in range(S)])).to(cuda)
    filt, bp = device.Filter(g), device.Backprojection(g)
    filt(x, S)
    want = backproject64(x.double(), N)
    packed = torch.zeros((size(bp.h),), dtype=torch.uint8, device=cuda)
    for shape in range(3):   # FP32 variants 0, 1, 2 have the split shapes' tiles
        err = []
        for split in (False, True):
            img = torch.full((S, N, N), float("nan"), dtype=torch.float32, device=cuda)
            if split:
                rc = run(bp.h, shape, x.data_ptr(), 1024.0, S, packed.data_ptr(), img.data_ptr(),
                         torch.cuda.current_stream().cuda_stream)
                assert rc == 0, lib.risa_last_error()
            else:
                bp.variant = shape
                bp.batch(x, S, img)
            err.append(float((img - want).norm() / want.norm()))
        print(f"case: N={N} P={P} D={D} shape {shape}: rel error linear {err[0]:.2e}, split {err[1]:.2e}", flush=True)
        assert err[1] <= err[0]
    filt.close()
    bp.close()

"""bp_split_kernel where its staged rows just hold the window: detector scales at
which the last row of an angle carries weights.

Tolerance: as in test_gpu_split.py, 5e-6 relative RMSE of every slice against
bp_linear_kernel (fractions of t differ by at most 2^-18 a sample pair, the
operands by 2^-21)."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from conftest import rel_rmse

pytestmark = pytest.mark.gpu

TOL = 5e-6


@pytest.mark.parametrize("N,D,P", [(512, 485, 130), (512, 394, 96), (512, 580, 96), (528, 500, 100), (128, 98, 64),
                                   (128, 106, 67), (128, 121, 64), (128, 125, 200)])
def test_split_scales(risa, geom_c0, cuda, N, D, P):
    import torch
    from risa_amd import device

    lib = risa.load()
    run, size = lib.risa_bp_run_split, lib.risa_bp_split_bytes
    run.argtypes = [C.c_void_p, C.c_int, C.c_void_p, C.c_float, C.c_int, C.c_void_p, C.c_void_p, C.c_void_p]
    run.restype, size.argtypes, size.restype = C.c_int, [C.c_void_p], C.c_size_t
    S = 32
    g = geom_c0.replace(numberOfPixels=N, numberOfParallelProjections=P, numberOfParallelDetectors=D)
    bp = device.Backprojection(g)
    x = torch.from_numpy(np.random.default_rng(N + D).standard_normal((S, P, D)).astype(np.float32)).to(cuda)
    want = torch.empty((S, N, N), dtype=torch.float32, device=cuda)
    bp.batch(x, S, want)
    want = want.cpu().numpy()
    packed = torch.zeros((size(bp.h),), dtype=torch.uint8, device=cuda)
    for shape in range(3):
        print(f"case: split N={N} D={D} P={P} shape {shape}", flush=True)
        img = [torch.full((S, N, N), float("nan"), dtype=torch.float32, device=cuda) for _ in range(2)]
        for o in img:
            rc = run(bp.h, shape, x.data_ptr(), 4096.0, S, packed.data_ptr(), o.data_ptr(),
                     torch.cuda.current_stream().cuda_stream)
            assert rc == 0, lib.risa_last_error()
        torch.cuda.synchronize()
        assert torch.equal(img[0], img[1])
        got = img[0].cpu().numpy()
        err = [rel_rmse(got[i], want[i]) for i in range(S)]
        print(f"  worst rel RMSE of a slice {max(err):.2e}", flush=True)
        assert max(err) < TOL
    bp.close()


def test_more_angles_than_a_grid_has_rows(risa, geom_c0, cuda):
    """The packing kernels launch a grid row per angle, 65535 at most; a geometry
    with more keeps the FP32 and FP16 variants."""
    from risa_amd import device

    lib = risa.load()
    sizes = [lib.risa_bp_split_bytes, lib.risa_bp_f16_pack_bytes]
    for size in sizes:
        size.argtypes, size.restype = [C.c_void_p], C.c_size_t
    square = next(v for v in range(device.bp_num_variants(True)) if device.bp_variant_shape(True, v)[:2] == (16, 16))
    for P, fits in ((65535, True), (65536, False)):
        bp = device.Backprojection(geom_c0.replace(numberOfPixels=8, numberOfParallelProjections=P,
                                                   numberOfParallelDetectors=8))
        bp.variant = square << 8
        assert [size(bp.h) > 0 for size in sizes] == [fits, fits]
        bp.close()

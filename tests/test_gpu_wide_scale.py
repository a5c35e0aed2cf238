"""Backprojection of many detectors per pixel: a tile shape whose staging cannot
hold an angle's window is refused, and never timed or taken by itself.

Tolerance: t' and k' stay below a tile's window of 44 scale entries; t' and the
staged s - k' d round by 2^-24 of that, times differences of about 1.4 of a
sample: below 2^-23 * 44 scale * 1.4, 2e-4 at 25 detectors per pixel and 5e-4 at
62.5, relative to the image's norm.  A window that is not staged whole is wrong
by the order of the image."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def exact(x, N):
    """Linear backprojection in float64: x [S][P][D] -> [S][N][N]."""
    S, P, D = x.shape
    c = (N - 1) * 0.5
    py, px = np.mgrid[0:N, 0:N] - c
    pad = np.zeros((S, P, D + 2))
    pad[:, :, 1:-1] = x
    img = np.zeros((S, N, N))
    for a in range(P):
        t = (px * np.cos(a * np.pi / P) + py * np.sin(a * np.pi / P)) * (D / N)
        k = np.floor(t).astype(int)
        f = t - k
        k += int(D * 0.5)
        img += pad[:, a, np.clip(k + 1, 0, D + 1)] * (1 - f) + pad[:, a, np.clip(k + 2, 0, D + 1)] * f
    return img * np.pi / P / (D / N)


@pytest.mark.parametrize("N,D,tol", [(20, 500, 2e-4), (16, 1000, 5e-4)])
def test_every_variant_is_right_or_refused(risa, geom_c0, cuda, N, D, tol):
    import torch
    from risa_amd import device

    P, S = 90, 5
    g = geom_c0.replace(numberOfPixels=N, numberOfParallelProjections=P, numberOfParallelDetectors=D, fusedMasking=0,
                        rotationOffset=0.0)
    bp = device.Backprojection(g)
    x = np.random.default_rng(D).standard_normal((S, P, D)).astype(np.float32)
    want = exact(x, N)
    xd = torch.from_numpy(x).to(cuda)

    def check(what):
        img = torch.full((S, N, N), float("nan"), dtype=torch.float32, device=cuda)
        bp.batch(xd, S, img)
        one = torch.full((N, N), float("nan"), dtype=torch.float32, device=cuda)
        bp(xd[0], one)
        got = img.cpu().numpy()
        err = np.linalg.norm(got - want) / np.linalg.norm(want)
        print(f"case: N={N} D={D} {what}: variant {bp.variant & 0xff}, rel error {err:.1e}", flush=True)
        assert err < tol
        assert np.array_equal(one.cpu().numpy(), got[0])

    check("as created")
    bp.autotune()
    check("tuned for one slice")
    bp.autotune_batch(S)
    check("tuned for a batch")
    ran = 0
    for v in range(device.bp_num_variants()):
        bp.variant = v
        try:
            check("set")
            ran += 1
        except risa.RisaError as e:
            assert "window" in str(e) or "LDS" in str(e)
    assert 0 < ran < device.bp_num_variants()
    bp.close()


def test_beyond_every_variant_is_refused(risa, geom_c0, cuda):
    import torch
    from risa_amd import device

    bp = device.Backprojection(geom_c0.replace(numberOfPixels=8, numberOfParallelProjections=9,
                                               numberOfParallelDetectors=520))   # 65 detectors per pixel
    x = torch.zeros((9, 520), dtype=torch.float32, device=cuda)
    with pytest.raises(risa.RisaError):
        bp(x, torch.empty((8, 8), dtype=torch.float32, device=cuda))
    bp.close()


def test_uneven_batch_is_right_or_refused(risa, cuda):
    """50 detectors per pixel (and 1): two of the persistent tile shapes stage
    such a window, a refused one leaves the batch as it was."""
    import torch
    from risa_amd import device

    rng = np.random.default_rng(5)
    jobs, want, imgs = [], [], []
    for N, P, D in ((16, 60, 800), (40, 50, 40)):
        x = rng.standard_normal((1, P, D)).astype(np.float32)
        imgs.append(torch.full((N, N), float("nan"), dtype=torch.float32, device=cuda))
        jobs.append(dict(sino=torch.from_numpy(x[0]).to(cuda), img=imgs[-1], N=N, P=P, D=D, mask=0))
        want.append(exact(x, N)[0])
    batch = device.BatchedBackprojection(jobs)

    def check(what):
        for i in imgs:
            i.fill_(float("nan"))
        batch()
        for i, w in zip(imgs, want):
            err = np.linalg.norm(i.cpu().numpy() - w) / np.linalg.norm(w)
            print(f"case: uneven batch {what}: N={w.shape[0]} rel error {err:.1e}", flush=True)
            assert err < 4e-4   # 2^-23 * 44 * 50 * 1.4

    check("as created")
    refused = 0
    for v in range(4):
        try:
            batch.set_variant(v)
        except risa.RisaError:
            refused += 1
        check(f"variant {v} asked for")
    assert refused == 2
    batch.autotune()
    check("tuned")
    batch.close()
    with pytest.raises(risa.RisaError):
        N, P, D = 8, 9, 520
        device.BatchedBackprojection([dict(sino=torch.zeros((P, D), device=cuda), img=torch.zeros((N, N), device=cuda),
                                           N=N, P=P, D=D)])

"""A filter call of more rows than one launch has threads for (256 per row pair
above a transform length of 1024): 33.6 million rows of 521 detectors."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_more_rows_than_a_launch(risa, geom_c0, cuda):
    import torch
    from risa_amd import device

    D, P, S = 521, 1000, 33_600        # padded transform of 1080 and more; 70 GB in place
    rows = P * S
    assert rows // 2 * 256 >= 1 << 32
    if torch.cuda.mem_get_info()[0] < 80 << 30:
        pytest.skip("needs 80 GB of free device memory")
    filt = device.Filter(geom_c0.replace(numberOfParallelProjections=P, numberOfParallelDetectors=D))
    x = torch.zeros((rows, D), dtype=torch.float32, device=cuda)
    # rows at both ends and around every 2^24 pairs
    at = sorted({0, 1, rows - 2, rows - 1} | {r for k in range(1, rows >> 24) for r in range((k << 24) - 2, (k << 24) + 2)}
                | {(1 << 25) - 2, (1 << 25) - 1, 1 << 25, (1 << 25) + 1})
    at = torch.tensor([r for r in at if r < rows], device=cuda)
    vals = torch.from_numpy(np.random.default_rng(1).standard_normal((len(at), D)).astype(np.float32)).to(cuda)
    x[at] = vals
    print(f"case: filter of {rows} rows of {D}", flush=True)
    filt(x, S)
    small = torch.zeros((P, D), dtype=torch.float32, device=cuda)
    pairs = sorted({int(r) // 2 for r in at})
    for i, p in enumerate(pairs):
        for k in (0, 1):
            hit = (at == 2 * p + k).nonzero()
            if len(hit):
                small[2 * i + k] = vals[hit[0, 0]]
    filt(small, 1)
    torch.cuda.synchronize()
    for i, p in enumerate(pairs):
        assert torch.equal(x[2 * p:2 * p + 2], small[2 * i:2 * i + 2]), f"rows {2 * p}, {2 * p + 1}"
    assert float(x[1000:1010].abs().max()) == 0.0
    del x
    torch.cuda.empty_cache()
    filt.close()

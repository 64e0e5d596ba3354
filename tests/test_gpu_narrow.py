"""GPU parity of the narrow-layer kernel (csrc/conv_stream.inc) against the CPU oracle: every row width and column
tiling it has, row counts round a tile and a workgroup, few and many neighbours, the fused epilogue and placed results."""
import numpy as np
import pytest
import torch

import oracle
from helpers import random_coords, rel_rms

pytestmark = pytest.mark.gpu


WIDTHS = [(8, 16), (8, 32), (16, 16), (16, 20), (32, 16), (32, 32), (32, 64), (64, 4), (64, 32)]
CLOUDS = [(1, (4, 4, 4)), (27, (3, 3, 3)), (64, (40, 40, 40)), (2049, (24, 22, 10))]
CASES = [(*w, *c) for w in WIDTHS for c in CLOUDS] + [(16, 16, 40001, (60, 60, 40)), (32, 32, 40001, (60, 60, 40))]


@pytest.mark.parametrize("cin,cout,n,box", CASES)
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_narrow_layers_match_oracle(cin, cout, n, box, dtype):
    from torchsparse_amd import backend
    rng = np.random.default_rng(n + cin + cout)
    coords = random_coords(rng, n, box)
    n = len(coords)
    omap = oracle.kmap_subm(coords, 3)
    x = torch.from_numpy(rng.standard_normal((n, cin)).astype(np.float32)).to("cuda", dtype)
    w = torch.from_numpy((rng.uniform(-1, 1, (27, cin, cout)) / np.sqrt(cin * 27)).astype(np.float32)).to("cuda", dtype)
    bias = torch.from_numpy(rng.standard_normal(cout).astype(np.float32)).to("cuda", dtype)
    res = torch.from_numpy(rng.standard_normal((n, cout)).astype(np.float32)).to("cuda", dtype)
    code = backend._dtype_code(x)
    assert backend._streams(27, cin, cout, code)
    wide = torch.zeros((n, cout + 24 - cout % 8), dtype=dtype, device="cuda")
    also = backend.ColumnSlice(wide, 8, cout) if cout % 8 == 0 else None
    f32 = lambda t: t.float().cpu().numpy()  # noqa: E731
    want = np.maximum(oracle.conv_implicit_gemm(f32(x), f32(w), omap, n) + f32(bias)[None] + f32(res), 0)
    y = backend._implicit_gemm(x, backend.pack_weights(w), 27, cin, cout, torch.from_numpy(omap).cuda(), n, bias, res, True,
                               also=also)
    tol = 1e-2 if dtype == torch.float16 else 5e-2
    assert rel_rms(f32(y), want) < tol
    if also is not None:
        assert torch.equal(wide[:, 8:8 + cout], y) and not wide[:, :8].any()

"""The projection GEMM over its whole ladder of tiles (128 x 192 down to 16 x 16, several depth groups in the small
ones): shapes at the edges of tiles, with shifted last column tiles, ragged rows, odd numbers of 32-deep steps and
depths shorter than the groups of a workgroup.  Every output against an f64 product on the device, within the bound of
tests/test_gpu_projection.py (|y - y64| <= gamma_m (sum|w x| + |b|) + 2^-21 sum|w x|, m = 2K + 2; the depth split only
shortens the chains of that bound), nothing written past the output, and a second call bit-identical (the sums of the
depth groups are added in a fixed order)."""

import pytest

from pvlc_testlib import log, pvlc

pytestmark = pytest.mark.gpu


# rows, k, n; the tile that the cost rule picks in the comment
@pytest.mark.parametrize("rows,k,n", [(5, 32, 12),        # 16 x 16: fewer columns than a tile, one half stage
                                      (16, 96, 20),       # 16 x 16: a shifted last tile would overlap: clamped rows
                                      (15, 2048, 1024),   # 16 x 16: 8 depth groups
                                      (31, 1024, 2564),   # 16 x 32: shifted last tile
                                      (64, 1056, 2560),   # 16 x 64: odd steps over 4 depth groups
                                      (128, 32, 2560),    # 32 x 64: three of four groups without a stage
                                      (211, 160, 2572),   # 64 x 64: two waves of rows, ragged rows
                                      (385, 224, 2560),   # 64 x 96: shifted last tile, one row in the last tile
                                      (1601, 224, 1020),  # 128 x 64: two groups of four waves, one row in the last tile
                                      (400, 96, 6140),    # 128 x 96: shifted last tile, odd steps
                                      (1157, 96, 2564),   # 128 x 128
                                      (2047, 160, 2556),  # 128 x 160: shifted last tile, ragged rows
                                      (2047, 352, 6136)]) # 128 x 192: shifted last tile, odd steps
def test_every_tile_writes_every_output_within_the_bound(rows, k, n):
    import torch
    log(f"case: projection tile rows={rows} k={k} n={n}")
    g = torch.Generator(device="cuda").manual_seed(rows * 7 + k + n)
    x = torch.randn(rows, k, generator=g, device="cuda") * torch.exp(torch.randn(rows, 1, generator=g, device="cuda"))
    w = (torch.randn(n, k, generator=g, device="cuda") * 0.05).half()
    b = torch.randn(n, generator=g, device="cuda")
    nbytes = pvlc.linear_projection_workspace_bytes(rows, k)
    ws = torch.empty(nbytes, dtype=torch.uint8, device="cuda")
    outs = []
    for _ in range(2):
        out = torch.full((rows * n + 64,), float("nan"), device="cuda")
        pvlc.linear_projection_f16(x, w, b, out, rows, k, n, ws, nbytes)
        torch.cuda.synchronize()
        assert bool(torch.isnan(out[rows * n:]).all()), "projection wrote past the output"
        outs.append(out[:rows * n].view(rows, n))
    got = outs[0]
    assert bool(torch.isfinite(got).all()), f"{int((~torch.isfinite(got)).sum())} outputs never written"
    assert torch.equal(got, outs[1]), "two calls differ"
    wt = w.double().t().contiguous()
    mag = x.double().abs() @ wt.abs()
    u = 2.0 ** -24
    gamma = (2 * k + 2) * u / (1 - (2 * k + 2) * u)
    allowed = gamma * (mag + b.double().abs()) + 2.0 ** -21 * mag
    ratio = float(((got.double() - (x.double() @ wt + b.double())).abs() / allowed).max())
    log(f"[parity] projection tile {rows}x{k}x{n}: max |gpu - f64| / bound = {ratio:.3f}")
    assert ratio <= 1.0

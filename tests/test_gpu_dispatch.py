"""Shapes at the edges of the launch rules: where a rule on sizes, types or alignment picks another split, tile or
kernel, the results on both sides of the line against the oracle or against independent kernels."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,L,C,N,T", [
    (1, 1024, 16, 32, 1100),     # one row group, one column block of one tile
    (1, 1500, 130, 64, 2999),    # three column blocks, the last of them two columns wide; odd period
    (1, 1977, 905, 128, 6073),   # fifteen column blocks, one per workgroup
    (3, 9000, 833, 128, 9100),   # fourteen column blocks in shares of several, the last share shorter; mirrored positions
])
def test_reconstruction_statistics_by_shares_of_column_blocks(B, L, C, N, T):
    """Every share of the column blocks against the fp32 vector kernel.  Bound: basis and scaled coefficients carry up to
    2^-11 relative rounding each, the results another 2^-11 (fp16)."""
    from fourierattention_amd import ops
    g = torch.Generator(device="cuda").manual_seed(3)
    c = torch.randn((B, 2 * N, C), generator=g, device="cuda") * (0.2 + 30 * torch.rand((1, 1, C), generator=g, device="cuda"))
    got = ops.mat_fourier_avg_std(c, L, T, torch.float16)
    ref = ops.mat_fourier_avg_std(c, L, T, torch.float16, matrix_cores=False)
    size = (ref[0].abs() + ref[1].abs()).cpu().numpy()
    for a, b in zip(got, ref):
        assert np.max((a - b).abs().cpu().numpy() / size) <= 2e-3

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


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("B,Hq,Hkv,D,n_il,L,N,k_counts,v_counts", [
    (1, 3, 1, 128, 5, 1, 5, [127], [1]),                        # one mid row; one stored K dim, one compressed V dim
    (2, 8, 1, 64, 63, 64, 16, [3], [63]),                       # one whole tile, eight heads, sixteen frequencies
    (1, 6, 2, 128, 65, 65, 100, [0, 57], [128, 0]),             # a tile and a row; a head that stores nothing and one that stores all
    (1, 10, 2, 80, 10, 191, 129, [33, 80], [80, 40]),           # head dims without the vectorised window kernel, 129 frequencies
    (2, 4, 2, 128, 130, 700, 300, [64, 64], [96, 17]),          # two rounds of frequencies per thread, several tiles per split
    (1, 7, 1, 128, 64, 300, 600, [100], [31]),                  # three rounds, seven heads
])
def test_any_shape_decode_kernels(dtype, B, Hq, Hkv, D, n_il, L, N, k_counts, v_counts):
    """The any-shape kernels on token-major and on paged mid rows against the float64 oracle.  Bound: the operands reach
    the kernels exactly and the arithmetic is single precision, 2e-4 on outputs of order one as for the other
    single-precision comparisons."""
    from fourierattention_amd import ops
    from fourierattention_amd.midstore import MidStore
    from oracle import fourier_oracle as fo
    from tests import helpers as H
    case = H.attn_case(11, B, Hq, Hkv, D, n_il, L, N, 2 * L + 7, k_counts, v_counts, dtype)
    want = fo.fourier_attn(**case)
    g = H.attn_case_gpu(case, dtype)
    lists = tuple(ops.as_i32(g[n]) for n in ("kc_list", "kc_h_list", "kn_list", "kn_h_list", "vc_list", "vc_h_list", "vn_list", "vn_h_list"))
    f = lambda t: t.float().contiguous()
    stats = [(f(g[f"avg_{t}_u"]), f(g[f"avg_{t}_d"]), f(g[f"scale_{t}"])) for t in "kv"]
    stores = []
    for t, n_h, is_v in ((g["k_mn"], lists[3], False), (g["v_mn"], lists[7], True)):
        ident = torch.arange(t.shape[2], dtype=torch.int32, device="cuda")
        st = MidStore(B, ident, n_h, n_h.tolist(), Hkv, D, L, dtype, "cuda", is_v)
        st.pack(t, 0, L)
        stores.append(st)
    for k_mn, v_mn in ((g["k_mn"], g["v_mn"]), stores):
        got = ops.decode_attn_raw(g["q"], [(g["k_il"], g["v_il"])], g["k_mc"], g["v_mc"], k_mn, v_mn, *stats, lists, Hq, Hkv, L,
                                  case["T"], force_generic=True)
        assert np.max(np.abs(got.cpu().numpy().astype(np.float64).reshape(want.shape) - want)) <= 2e-4


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D,S,q_len,G", [(128, 31, 31, 1), (128, 161, 161, 4), (64, 200, 65, 3), (128, 97, 1, 2)])
@pytest.mark.parametrize("climb", [0.0, 6.0, 40.0, -40.0])
def test_prompt_attention_with_a_moving_reference(dtype, D, S, q_len, G, climb):
    """Scores that climb (or fall) along the keys by ``climb`` per key tile, in units of log 2: the softmax reference of a
    row lags by up to 8 before it moves, so 0 never moves it after the first tile, 6 moves it every other tile, 40
    every tile.  Bound: f16 probabilities (2^-11 each, averaged) and the rounding of the result, as for the other shapes."""
    from fourierattention_amd import ops
    g = torch.Generator(device="cuda").manual_seed(7)
    q = torch.randn((1, 2 * G, q_len, D), generator=g, device="cuda")
    k = torch.randn((1, S, 2, D), generator=g, device="cuda")
    v = torch.randn((1, S, 2, D), generator=g, device="cuda")
    # one dim of every head carries the climb: q there is 8, k there is the wanted score over q and the scale
    q[..., 0] = 8.0
    k[..., 0] = (climb * torch.arange(S, device="cuda") / 32 * np.log(2) * D ** 0.5 / 8.0)[None, :, None]
    q, k, v = (t.to(dtype) for t in (q, k, v))
    got = ops.prefill_attention(q, k.reshape(1, S, 2 * D), v.reshape(1, S, 2 * D), 2).double()
    qd, kd, vd = q.double(), k.double().permute(0, 2, 1, 3).repeat_interleave(G, 1), v.double().permute(0, 2, 1, 3).repeat_interleave(G, 1)
    s = qd.matmul(kd.transpose(2, 3).contiguous()) / D ** 0.5
    seen = torch.arange(S, device="cuda")[None, :] <= torch.arange(q_len, device="cuda")[:, None] + S - q_len
    want = s.masked_fill(~seen, float("-inf")).softmax(-1).matmul(vd).transpose(1, 2)
    top = float(want.abs().max())
    ulp = 2.0 ** (np.floor(np.log2(top)) - (7 if dtype == torch.bfloat16 else 10))
    assert float((got - want).abs().max()) <= 0.5 * ulp + 1e-3

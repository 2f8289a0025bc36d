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


@pytest.mark.parametrize("B,L,C,N,T", [
    (1, 1300, 33, 1100, 2700),   # ten steps of the coefficients, the last one short; a column block of one column
    (2, 2048, 32, 1024, 2048),   # nine steps; whole blocks of positions and, with position T / 2, one of a single one
    (1, 1025, 17, 129, 1400),    # two steps, the second half full
])
def test_reconstruction_statistics_of_signals_with_a_mean(B, L, C, N, T):
    """Folded steps of the coefficients against float64, for signals whose mean outweighs their deviation.  Bound: coefficients
    and basis carry up to 2^-11 relative rounding each, independent from term to term, so a position is off by at most about
    five standard deviations (1 / sqrt(3) of the bound each, 4 in all) of 2^-11 times the 2-norm of the column's coefficients
    over N - without that of frequency 0, which is summed in single precision like the mean: 1e-5 of it.  The deviation is a
    difference of two such values.  What is not a number stays in its column."""
    from fourierattention_amd import ops
    g = torch.Generator(device="cuda").manual_seed(5)
    t = torch.arange(L, dtype=torch.float64, device="cuda")
    x = torch.randn((B, L, C), generator=g, device="cuda", dtype=torch.float64) + 40.0
    n = torch.arange(N, dtype=torch.float64, device="cuda")
    ph = 2 * np.pi / T * torch.remainder(n[:, None] * t[None], T)
    c = torch.cat([ph.cos() @ x, ph.sin() @ x], dim=1).float()
    r = (ph.cos().T @ c[:, :N].double() + ph.sin().T @ c[:, N:].double()) / N
    avg = r.mean(1)
    dev = torch.maximum(r.amax(1) - avg, avg - r.amin(1))
    got = ops.mat_fourier_avg_std(c, L, T, None)
    rest = c.double()
    rest[:, [0, N]] = 0.0
    bound = 4 * 2.0 ** -11 * rest.norm(dim=1) / N + 1e-5 * avg.abs()
    assert ((got[0].double() - avg).abs() <= bound).all()
    assert ((got[1].double() - dev).abs() <= 2 * bound).all()
    c[0, N // 2, 3], c[0, N + 1, 5], c[0, 0, 7] = float("nan"), float("inf"), float("nan")
    bad = ops.mat_fourier_avg_std(c, L, T, None)
    whole = torch.ones((B, C), dtype=torch.bool, device="cuda")
    whole[0, [3, 5, 7]] = False
    for a, b in zip(bad, got):
        assert torch.equal(a[whole], b[whole]) and not torch.isfinite(a[~whole]).any()


@pytest.mark.parametrize("N", [64, 65, 191, 192, 512])   # one step of the coefficients, one past it, two, one past those, five
def test_reconstruction_statistics_of_slow_columns(N):
    """Columns of a single low frequency, which is what a drift or a slow oscillation is made of: their extremes fall on
    positions where the basis is one, so nothing of the basis' rounding reaches the deviation (the period is a power of two and
    the whole of it is covered: the errors of the mean cancel).  Bound: a coefficient travels as two f16 terms, 2^-22 of it is
    lost, and single precision adds a few 2^-24."""
    from fourierattention_amd import ops
    T, low = 4096, 63
    g = torch.Generator(device="cuda").manual_seed(6)
    c = torch.zeros((1, 2 * N, 2 * low), device="cuda")
    n = torch.arange(1, low + 1, device="cuda")
    amp = (0.5 + torch.rand(2 * low, generator=g, device="cuda")) * 10.0 ** torch.randint(-3, 4, (2 * low,), generator=g, device="cuda")
    c[0, n, n - 1] = amp[:low]
    c[0, N + n, low + n - 1] = -amp[low:]
    avg, dev = ops.mat_fourier_avg_std(c, T, T, None)
    assert (avg[0].abs() * N <= 2.0 ** -20 * amp).all()
    assert ((dev[0] * N - amp).abs() <= 2.0 ** -20 * amp).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("B,H,S,D,first,last,spare,tokens_first", [
    (1, 1, 1, 8, 0, 1, 0, False),        # one row of one piece or two
    (2, 8, 517, 128, 4, 500, 1, False),  # the last block of rows holds six, among them the row of zeros
    (3, 2, 31, 64, 31, 0, 0, False),     # every row is a near one
    (2, 8, 300, 128, 4, 64, 1, True),    # token-major already: the rows are read in place
    (1, 5, 64, 24, 0, 0, 1, False),      # no near rows but the zeros; rows of odd widths
])
def test_rows_of_a_prompt(dtype, B, H, S, D, first, last, spare, tokens_first):
    """Copies are exact: token-major rows and near rows against the tensor operations they stand for."""
    from fourierattention_amd import ops
    g = torch.Generator(device="cuda").manual_seed(1)
    make = lambda: torch.randn((B, S, H, D) if tokens_first else (B, H, S, D), generator=g, device="cuda").to(dtype)
    k, v = ((t.transpose(1, 2) if tokens_first else t) for t in (make(), make()))
    near = tuple(torch.full((B, first + last + spare + 3, H * D), 7.0, device="cuda", dtype=dtype) for _ in range(2))
    got = ops.prompt_rows(k, v, near, first, last, spare)
    for t, rows, n in zip((k, v), got, near):
        want = t.permute(0, 2, 1, 3).reshape(B, S, H * D)
        assert torch.equal(rows, want) and (not tokens_first or rows.data_ptr() == t.data_ptr())
        assert torch.equal(n[:, :first], want[:, :first]) and torch.equal(n[:, first:first + last], want[:, S - last:])
        assert (n[:, first + last:first + last + spare] == 0).all() and (n[:, first + last + spare:] == 7).all()
    assert ops.prompt_rows(k[..., :-1], v[..., :-1]) is None                          # rows that are no multiples of 16 bytes
    assert ops.prompt_rows(k, v.transpose(2, 3).contiguous().transpose(2, 3)) is None or S == 1 or D == 1   # strides of their own


def test_prompt_of_a_window_keeps_its_tangent():
    """A prompt that fits the window comes back as tensor operations return it: with its gradient, or its tangent."""
    import torch.autograd.forward_ad as fwd
    from fourierattention_amd import DynamicCache, ExtraConfig, masks
    cache = DynamicCache(ExtraConfig(numinittokens=4, maxlocallen=40, maxmidstates=64, non_critical_dims=masks.synthetic_masks(1, 2, 128, [64] * 2, [64] * 2, seed=1),
                                     non_critical_dims_path=None, max_position_embeddings=4096, num_key_value_heads=2, max_new_tokens=8, model_type="llama"))
    k, v, dk = torch.randn((3, 1, 2, 20, 128), device="cuda").unbind(0)
    with fwd.dual_level():
        parts, _ = cache.update(fwd.make_dual(k, dk), v, 0)
        rows = fwd.unpack_dual(parts["k_local"])
        assert torch.equal(rows.primal, k.transpose(1, 2).reshape(1, 20, 256))
        assert rows.tangent is not None and torch.equal(rows.tangent, dk.transpose(1, 2).reshape(1, 20, 256))


@pytest.mark.parametrize("how", ["jvp", "make_fx", "trace", "fake"])
def test_prompt_of_a_window_where_operations_are_recorded(how):
    """A new cache and a prompt that fits its window, under a transform, a tracer and fake tensors: tensor operations throughout."""
    from torch._subclasses.fake_tensor import FakeTensorMode
    from torch.fx.experimental.proxy_tensor import make_fx
    from fourierattention_amd import DynamicCache, ExtraConfig, masks
    cfg = ExtraConfig(numinittokens=4, maxlocallen=40, maxmidstates=64, non_critical_dims=masks.synthetic_masks(1, 2, 128, [64] * 2, [64] * 2, seed=1),
                      non_critical_dims_path=None, max_position_embeddings=4096, num_key_value_heads=2, max_new_tokens=8, model_type="llama")
    rows = lambda k, v: DynamicCache(cfg).update(k, v, 0)[0]["k_local"]
    want = lambda k: k.transpose(1, 2).reshape(1, 20, 256)
    k, v, other = torch.randn((3, 1, 2, 20, 128), device="cuda").unbind(0)
    if how == "jvp":
        got, tangent = torch.func.jvp(lambda k: rows(k, v), (k,), (other,))
        assert torch.equal(got, want(k)) and torch.equal(tangent, want(other))
    elif how == "make_fx":
        assert torch.equal(make_fx(rows)(k, v)(other, v), want(other))
    elif how == "trace":
        assert torch.equal(torch.jit.trace(rows, (k, v), check_trace=False)(other, v), want(other))
    else:
        with FakeTensorMode(allow_non_fake_inputs=True) as mode:
            assert rows(mode.from_tensor(k), mode.from_tensor(v)).shape == (1, 20, 256)


def _reconstruction64(c, L, T):
    """Mean and largest deviation of the reconstruction in 64 bits, and the 2-norm of every column's coefficients over N."""
    N = c.shape[1] // 2
    ph = 2 * np.pi / T * (torch.arange(L, device="cuda")[:, None] * torch.arange(N, device="cuda")[None] % T).double()
    r = (ph.cos() @ c[:, :N].double() + ph.sin() @ c[:, N:].double()) / N
    avg = r.mean(1)
    return avg, torch.maximum(r.amax(1) - avg, avg - r.amin(1)), c.double().norm(dim=1) / N


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])    # the two kernels of the matrix cores
@pytest.mark.parametrize("B,L,C,N,T", [
    (1, 1024, 16, 32, 1100),     # one row group, one column block of one tile
    (1, 1500, 130, 64, 2999),    # three column blocks of 64, the last two columns wide; odd period; one whole step above its centre
    (1, 1977, 905, 128, 6073),   # fifteen column blocks, one per workgroup
    (3, 9000, 833, 128, 9100),   # shares of several column blocks, the last share shorter; mirrored positions
    (1, 1300, 33, 1100, 2700),   # nine steps of 128 or ten of 127, the last one short
    (2, 2048, 32, 1024, 2048),   # whole blocks of positions, and position T / 2 in one of its own
    (1, 1025, 17, 129, 1400),    # one coefficient past a step of 128
    (1, 1200, 40, 65, 1201),     # one past the first 64; every position but one mirrored
    (2, 1100, 64, 191, 1100),    # two whole steps of 127 (the first from its centre)
    (1, 2600, 100, 192, 1280),   # one past those; a sequence of two periods, nothing mirrored
    (1, 1500, 48, 318, 1499),    # three whole steps; as long as the period and one position more
])
def test_both_kernels_of_the_statistics_a_cache_keeps(dtype, B, L, C, N, T):
    """Mean and deviation as ``recon_scale`` leaves them, against float64.  Bound: coefficients and basis carry up to 2^-11
    relative rounding each, independent from term to term: a position is off by at most about five standard deviations (1 / sqrt(3) of
    the bound each, 4 in all) of 2^-11 times the 2-norm of the column's coefficients over N, a deviation by twice that;
    mean, deviation and an fp16 quotient are rounded to fp16 on top, 2^-11 each."""
    from fourierattention_amd import ops
    g = torch.Generator(device="cuda").manual_seed(L + N)
    c = torch.randn((B, 2 * N, C), generator=g, device="cuda") * (N ** 0.5 * (0.2 + 3 * torch.rand((1, 1, C), generator=g, device="cuda")))
    c[:, 0] += 2 * N * torch.randn((1, C), generator=g, device="cuda")       # means of the size of the deviation
    one = torch.ones((B, C), device="cuda")
    scale, _, _, (_, avg, _) = ops.recon_scale(c, L, T, one, one, dtype)
    avg64, dev64, norm = _reconstruction64(c, L, T)
    assert ((avg.double() - avg64).abs() <= 4 * 2.0 ** -11 * norm + 2.0 ** -11 * avg64.abs()).all()
    assert ((1 / scale.double() - dev64).abs() <= 8 * 2.0 ** -11 * norm + 2 * 2.0 ** -11 * dev64).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("B,L,C,N,T", [(2, 300, 5, 16, 400), (1, 1100, 70, 64, 1500)])   # vector kernels / matrix cores
def test_statistics_a_cache_keeps(dtype, B, L, C, N, T):
    """The same values, bit for bit, as the conversions and the division as tensor operations; in single precision on the matrix
    cores those of the kernel such a cache has for itself."""
    from fourierattention_amd import ops
    g = torch.Generator(device="cuda").manual_seed(2)
    x = (torch.randn((B, L, C), generator=g, device="cuda") * 3 + 1).to(dtype)
    c = ops.mat_fourier(x, N, T)
    u_avg, u_dev = ops.mat_avg_std(x, round_dtype=dtype)
    i_avg, i_dev = ops.mat_fourier_avg_std(c, L, T, torch.float16)
    scale = u_dev.to(dtype) / i_dev.to(torch.float16)
    got = ops.recon_scale(c, L, T, u_avg, u_dev, dtype)
    want = (scale, u_avg.to(dtype), i_avg.to(torch.float16), u_avg, i_avg, scale.float())
    have = (*got[:3], *got[3])
    assert all(a.dtype == b.dtype for a, b in zip(have, want))
    # a single-precision cache has a kernel of its own on the matrix cores: what comes of the reconstruction may round the other way
    own = dtype == torch.float32 and L > 1024
    for at in (1, 3) if own else range(6):
        assert torch.equal(have[at], want[at])
    if own:
        # (the same mean in both types, the same quotient twice, and the quotient of the deviation as fp16 holds it)
        assert torch.equal(have[2].float(), have[4]) and torch.equal(have[0], have[5])
        dev = u_dev.double() / have[0].double()
        dev16 = dev.to(torch.float16).double()
        assert ((dev - dev16).abs() <= 2.0 ** -22 * dev16).all()
        # mean and deviation against float64: at most 4 * 2^-11 of the 2-norm of a column's coefficients over N, as for the kernels
        # themselves (twice that for the deviation), and half a place of fp16
        avg64, dev64, norm = _reconstruction64(c, L, T)
        assert ((have[4].double() - avg64).abs() <= 4 * 2.0 ** -11 * norm + 2.0 ** -11 * avg64.abs()).all()
        assert ((dev16 - dev64).abs() <= 8 * 2.0 ** -11 * norm + 2.0 ** -11 * dev64).all()


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
    row moves with its maximum, so -40 never moves it after the first tile, 0 here and there, 6 and 40 on every
    tile.  Bound: f16 probabilities (2^-11 each, averaged) and the rounding of the result, as for the other shapes."""
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


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D,G", [(128, 4), (128, 3), (64, 1)])
@pytest.mark.parametrize("first,last,keys", [(16, 32, False), (5, 161, False), (5, 161, True), (37, 38, False), (1, 17, True)])
@pytest.mark.parametrize("climb", [0.0, 40.0])
def test_prompt_rows_beside_rows_that_are_not_numbers(dtype, D, G, first, last, keys, climb):
    """Query rows ``first .. last`` (and, with ``keys``, their keys) are NaN: every other row that sees no such key is what it
    is without them, and the NaN rows stay NaN.  Scores climb as above, so a vote withheld would overflow f16.  Bound: as
    above."""
    from fourierattention_amd import ops
    S = 161
    g = torch.Generator(device="cuda").manual_seed(11)
    q = torch.randn((1, 2 * G, S, D), generator=g, device="cuda")
    k = torch.randn((1, S, 2, D), generator=g, device="cuda")
    v = torch.randn((1, S, 2, D), generator=g, device="cuda")
    q[..., 0] = 8.0
    k[..., 0] = (climb * torch.arange(S, device="cuda") / 32 * np.log(2) * D ** 0.5 / 8.0)[None, :, None]
    q, k, v = (t.to(dtype) for t in (q, k, v))
    qd, kd, vd = q.double(), k.double().permute(0, 2, 1, 3).repeat_interleave(G, 1), v.double().permute(0, 2, 1, 3).repeat_interleave(G, 1)
    s = qd.matmul(kd.transpose(2, 3).contiguous()) / D ** 0.5
    rows = torch.arange(S, device="cuda")
    want = s.masked_fill(rows[None, :] > rows[:, None], float("-inf")).softmax(-1).matmul(vd).transpose(1, 2)
    q[:, :, first:last] = float("nan")
    if keys:
        k[:, first:last] = float("nan")
    got = ops.prefill_attention(q, k.reshape(1, S, 2 * D), v.reshape(1, S, 2 * D), 2).double()
    bad = (rows >= first) if keys else (rows >= first) & (rows < last)
    assert bool(got[:, bad].isnan().all())
    top = float(want.abs().max())
    ulp = 2.0 ** (np.floor(np.log2(top)) - (7 if dtype == torch.bfloat16 else 10))
    assert float((got - want)[:, ~bad].abs().max()) <= 0.5 * ulp + 1e-3


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("B,D,rows,extra,counts", [
    (1, 128, 1, 0, [128, 1]),                 # one row; a full head and a single dim
    (2, 128, 65, 3, [7, 0, 120, 33]),         # a page of one row in the second block; runs at odd columns, odd row length
    (1, 64, 2080, 0, [64, 9, 17]),            # whole pages, an odd number of them
    (3, 200, 96, 5, [200, 150]),              # heads above 128 dims
])
def test_pages_of_rows_in_order(dtype, B, D, rows, extra, counts):
    """Columns that are the stored dims already against the same pack through an index list into a zero-filled store: the
    pages bit for bit, in a store that held NaN, from rows that are slices of wider rows."""
    from fourierattention_amd.midstore import MidStore
    g = torch.Generator(device="cuda").manual_seed(rows)
    cn = sum(counts)
    src = torch.randn((B, rows, cn + extra), generator=g, device="cuda").to(dtype)[:, :, extra:]
    n_h_host = [sum(counts[:i]) for i in range(len(counts) + 1)]
    n_h = torch.tensor(n_h_host, dtype=torch.int32, device="cuda")
    ident = torch.arange(cn, dtype=torch.int32, device="cuda")
    for is_v in (False, True):
        want, got = (MidStore(B, ident, n_h, n_h_host, len(counts), D, rows, dtype, "cuda", is_v) for _ in range(2))
        want.pack(src, 0, rows)
        got.data.fill_(float("nan"))
        got.pack(src, 0, rows, in_order=True)
        assert torch.equal(got.data, want.data)
        assert torch.equal(got.dense(rows), src)


@pytest.mark.parametrize("list_dtype", [torch.int64, torch.int32])
@pytest.mark.parametrize("stat_dtype", [torch.bfloat16, torch.float16, torch.float32, torch.float64])
def test_operands_in_the_types_the_kernels_take(list_dtype, stat_dtype):
    """Lists, statistics (empty and strided ones among them) and padded offsets against the tensor operations."""
    from fourierattention_amd import _lib
    g = torch.Generator(device="cuda").manual_seed(5)
    lists = tuple(torch.randint(0, 1000, (n,), generator=g, device="cuda").to(list_dtype) for n in (0, 9, 1023, 9, 257, 9, 1, 9))
    heads = [torch.tensor([0] + [int(x) for x in torch.randint(0, 129, (8,)).cumsum(0)], device="cuda", dtype=list_dtype) for _ in range(2)]
    lists = lists[:3] + (heads[0],) + lists[4:7] + (heads[1],)
    stats = tuple(torch.randn((2, 2 * n), generator=g, device="cuda").to(stat_dtype)[:, ::s] for n, s in ((0, 1), (1, 2), (300, 1), (17, 2), (4, 1), (1023, 1)))
    l32, s32, paging = _lib.load_host().operands(lists, stats, 32, 16)
    assert all(a.dtype == torch.int32 and torch.equal(a, b.to(torch.int32)) for a, b in zip(l32, lists))
    assert all(a.dtype == torch.float32 and a.is_contiguous() and torch.equal(a, b.float()) for a, b in zip(s32, stats))
    for i, unit in enumerate((32, 16)):
        n = heads[i].cpu().diff()
        pad = torch.cat([torch.zeros(1, dtype=n.dtype), ((n + unit - 1) // unit * unit).cumsum(0)])
        assert paging[i] == heads[i].tolist() and paging[2 + i].tolist() == pad.tolist()
    assert _lib.load_host().operands(lists, stats, 0, 0)[2] is None


@pytest.mark.parametrize("L,C,N,T", [
    (512, 1, 8, 700),           # one row tile of frequencies, one column, one chunk of four steps
    (1300, 70, 136, 1301),      # a row tile past a whole workgroup, two column blocks, a ragged last step
    (33000, 1100, 24, 40000),   # more than 128 splits of the statistics; eighteen column blocks, shares at their limit
])
def test_spectral_operators_at_the_edges_of_their_tiles(L, C, N, T):
    """Coefficients and both statistics against the fp32 vector kernels.  Bounds: the basis is rounded to f16 (2^-11 per
    entry, errors of both signs over L rows: well below 5e-4 of the column's norm); statistics as above."""
    from fourierattention_amd import ops
    g = torch.Generator(device="cuda").manual_seed(L)
    a = torch.randn((2, L, C), generator=g, device="cuda").to(torch.bfloat16)
    got, ref = (ops.mat_fourier(a, N, T, matrix_cores=m) for m in (True, False))
    assert float(((got - ref).norm(dim=1) / ref.norm(dim=1)).max()) <= 5e-4
    if L >= 1024 and C >= 16 and N >= 32 or C > 1000:
        c = torch.randn((2, 2 * max(N, 32), C), generator=g, device="cuda")
        st, sr = (ops.mat_fourier_avg_std(c, L, T, torch.float16, matrix_cores=m) for m in (True, False))
        size = sr[0].abs() + sr[1].abs()
        assert all(float(((x - y).abs() / size).max()) <= 2e-3 for x, y in zip(st, sr))
    avg, dev = ops.mat_avg_std_triton(a)
    want = a.double().mean(1)
    # float32 sums of L values of order one, then one rounding to bf16: eight significant bits, so half a unit in the last
    # place is up to 2^-8 of the value
    assert float((avg.double() - want).abs().max()) <= 2.0 ** -8 * float(want.abs().max()) + 1e-5
    spread = torch.maximum(a.double().amax(1) - want, want - a.double().amin(1))
    assert float(((dev.double() - spread) / spread).abs().max()) <= 2.0 ** -8


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,K,n_out", [(1, 1024, 32), (16, 1024, 96), (5, 3072, 64), (4, 4096, 160), (2, 8192, 32), (3, 8192, 32)])
def test_projections_with_the_steps_beside_them(dtype, rows, K, n_out):
    """RMSNorm, gate and residual in the projection's launch against the launches of their own: the same bits without the
    norm (same sums, same rounding); with it the sum of squares is taken in another order, which moves the scale of a row
    by a place of float32 and with it single operands by a place of ``dtype`` (2^-8 / 2^-11 relative)."""
    from fourierattention_amd import ops
    g = torch.Generator(device="cuda").manual_seed(rows + K)
    rn = lambda *s: torch.randn(s, generator=g, device="cuda")
    pw = ops.PackedLinearWeight((rn(n_out, K) * 0.05).to(dtype))
    x, h = (rn(rows, 1, K) * 3).to(dtype), rn(rows, 1, n_out).to(dtype)
    norm = (1 + 0.1 * rn(K)).to(dtype)
    plain = ops.linear_packed(x, pw)
    kept = h.clone()
    assert ops.linear_packed_step(x, pw, residual=kept) is kept and torch.equal(kept, h + plain)
    assert torch.equal(ops.linear_packed_step(x, pw, gated=True), ops.silu_mul(*plain.chunk(2, dim=-1)))
    assert pw.normalises(x, norm) == (rows * K <= 16384) and not pw.normalises(x, torch.cat([norm, norm])[1:K + 1])
    if rows * K > 16384:
        with pytest.raises(RuntimeError):
            ops.linear_packed_step(x, pw, norm, 1e-5)
        return
    before = x.clone()
    got = ops.linear_packed_step(x, pw, norm, 1e-5)
    y = ops.add_rmsnorm(x, None, norm, 1e-5)
    want = ops.linear_packed(y, pw)
    ulp = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    bound = 2 * ulp * float(want.abs().max()) + ulp * float(y.abs().max()) * 0.2 * 4
    assert torch.equal(x, before) and float((got.float() - want.float()).abs().max()) <= bound
    gate = ops.linear_packed_step(x, pw, norm, 1e-5, gated=True)
    assert torch.equal(gate, ops.silu_mul(*got.chunk(2, dim=-1)))
    kept = h.clone()
    assert torch.equal(ops.linear_packed_step(x, pw, norm, 1e-5, residual=kept), h + got)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("K", [5120, 14336, 16384])     # two pieces of a row for some threads, the last of four for some, four for all
def test_norm_of_a_long_row_in_the_projection(dtype, K):
    """One row whose pieces share their sum of squares, against the norm as tensor operations.  Bound as above: the scale of the
    row moves by a place of float32, single operands by a place of ``dtype``."""
    from fourierattention_amd import ops
    g = torch.Generator(device="cuda").manual_seed(K)
    rn = lambda *s: torch.randn(s, generator=g, device="cuda")
    pw = ops.PackedLinearWeight((rn(64, K) * 0.05).to(dtype))
    x, norm = (rn(1, 1, K) * 3).to(dtype), (1 + 0.1 * rn(K)).to(dtype)
    f = x.float()
    y = norm * (f * torch.rsqrt(f.pow(2).mean(-1, keepdim=True) + 1e-5)).to(dtype)
    want, got = ops.linear_packed(y, pw), ops.linear_packed_step(x, pw, norm, 1e-5)
    ulp = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    assert float((got.float() - want.float()).abs().max()) <= 2 * ulp * float(want.abs().max()) + ulp * float(y.abs().max()) * 0.2 * 4
    assert torch.equal(ops.linear_packed_step(x, pw, norm, 1e-5, gated=True), ops.silu_mul(*got.chunk(2, dim=-1)))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,q_len,K,Hq,Hkv,D", [(1, 1, 1024, 1, 1, 16), (2, 1, 3072, 6, 2, 128), (3, 5, 1024, 4, 2, 64), (1, 4, 4096, 2, 1, 48)])
def test_rotary_embedding_in_the_projection(dtype, B, q_len, K, Hq, Hkv, D):
    """q, k and v of one launch against the projection on the weight in its natural order and the rotary embedding as launches
    of their own: the same bits (same sums, same rounding), with and without the norm in front."""
    from fourierattention_amd import ops
    g = torch.Generator(device="cuda").manual_seed(K + D)
    rn = lambda *s: torch.randn(s, generator=g, device="cuda")
    n_out = (Hq + 2 * Hkv) * D
    w = (rn(n_out, K) * 0.05).to(dtype)
    plain, pairs = ops.PackedLinearWeight(w), ops.PackedLinearWeight(w[ops.rotary_pairs(n_out, Hq + Hkv, D, "cuda")].contiguous())
    x, norm = (rn(B, q_len, K) * 3).to(dtype), (1 + 0.1 * rn(K)).to(dtype)
    cos, sin = rn(B, q_len, D).to(dtype), rn(B, q_len, D).to(dtype)
    for nw in (None, norm) if B * q_len * K <= 16384 else (None,):
        row = ops.linear_packed(x, plain) if nw is None else ops.linear_packed_step(x, plain, nw, 1e-5)
        q, k, v = (t.contiguous() for t in row.split((Hq * D, Hkv * D, Hkv * D), dim=-1))
        q = ops.rope_qk(q, k, cos, sin, D)
        for got, want in zip(ops.linear_packed_qkv(x, pairs, nw, 1e-5, cos, sin, Hq, Hkv, D), (q, k, v)):
            assert torch.equal(got, want.view(B, q_len, -1, D).transpose(1, 2))


@pytest.mark.parametrize("at", [1, 4])     # elements past an aligned address
def test_rotary_tables_anywhere(at):
    """Tables that start off a vector's alignment - a slice of a longer buffer - are taken as ``rope_qk`` takes them."""
    from fourierattention_amd import ops
    K, Hq, Hkv, D = 1024, 2, 1, 16
    g = torch.Generator(device="cuda").manual_seed(at)
    rn = lambda *s: torch.randn(s, generator=g, device="cuda").bfloat16()
    w = ops.PackedLinearWeight(rn((Hq + 2 * Hkv) * D, K))
    x, table = rn(1, 1, K), rn(128)
    cos, sin = (table[i + at: i + at + D].view(1, 1, D) for i in (0, 64))
    assert cos.data_ptr() % 16 and sin.data_ptr() % 16
    want = ops.linear_packed_qkv(x, w, None, 0.0, cos.clone(), sin.clone(), Hq, Hkv, D)
    for got, t in zip(ops.linear_packed_qkv(x, w, None, 0.0, cos, sin, Hq, Hkv, D), want):
        assert torch.equal(got, t)


def _launches(f):
    """Kernel launches of a call: the nodes of a graph it is captured into (which is never run)."""
    import ctypes
    from fourierattention_amd import _lib
    graph, n = torch.cuda.CUDAGraph(keep_graph=True), ctypes.c_size_t()
    with torch.cuda.graph(graph):
        f()
    get_nodes = _lib.load().hipGraphGetNodes      # (of the runtime the library runs on)
    get_nodes.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.POINTER(ctypes.c_size_t)]
    assert get_nodes(graph.raw_cuda_graph(), None, ctypes.byref(n)) == 0
    return n.value


@pytest.mark.parametrize("dtype,B,Hq,Hkv,D,states,init,W,counts,wide", [
    (torch.bfloat16, 1, 8, 2, 128, 256, 4, 100, [64, 64], False),     # matrix cores, merge in the launch, sub-splits
    (torch.bfloat16, 3, 12, 4, 128, 256, 4, 61, [128, 0, 77, 1], True),   # a head without compressed K, tokens as slices of wider rows
    (torch.float16, 2, 16, 2, 64, 512, 1, 64, [40, 13], False),       # heads of 64 dims, eight query heads
    (torch.float32, 1, 6, 2, 128, 64, 4, 33, [100, 128], False),      # single precision
    (torch.bfloat16, 2, 8, 2, 128, 64, 0, 40, [64, 100], False),      # no sink rows
    (torch.bfloat16, 1, 4, 2, 80, 64, 4, 40, [30, 50], False),        # head dims without the vectorised window kernel
    (torch.bfloat16, 7, 4, 2, 128, 1024, 4, 40, [100, 77], False),    # uneven heads, many coefficients, few sequences: apart
    (torch.bfloat16, 2, 4, 2, 128, 1024, 4, 40, [100, 92], False),    # the same where the sum is a whole number of lines
    (torch.bfloat16, 8, 4, 2, 128, 1024, 4, 40, [100, 77], False),    # eight sequences: joined
])
def test_update_in_the_attention_launch(dtype, B, Hq, Hkv, D, states, init, W, counts, wide):
    """A decode step through ``fourier_attention`` (the update in the attention's first launch, or in front of it where it
    cannot be) against ``update`` and ``decode_attention`` as calls of their own, on two caches with the same prompt:
    the same window, pages and attention arithmetic, bit for bit, over enough steps for the ring to come round."""
    from fourierattention_amd import DynamicCache, ExtraConfig, masks
    from fourierattention_amd.attention import fourier_attention
    g = torch.Generator(device="cuda").manual_seed(W)
    rn = lambda *s: torch.randn(s, generator=g, device="cuda").to(dtype)
    m = masks.synthetic_masks(1, Hkv, D, counts, counts[::-1], seed=3)
    cfg = ExtraConfig(numinittokens=init, maxlocallen=W, maxmidstates=states, non_critical_dims=m, non_critical_dims_path=None,
                      max_position_embeddings=8192, num_key_value_heads=Hkv, max_new_tokens=8, model_type="llama")
    S = init + W + states + 700
    prompt = rn(B, Hkv, S, D), rn(B, Hkv, S, D)
    one, two = DynamicCache(cfg), DynamicCache(cfg)
    one.update(*prompt, 0)
    two.update(*prompt, 0)
    for t in range(W + 5):
        q = rn(B, Hq, 1, D)
        k, v = rn(B, 1, 2 * Hkv * D).split(Hkv * D, dim=-1)
        k, v = (x.view(B, 1, Hkv, D).transpose(1, 2) if wide else x.reshape(B, Hkv, 1, D).contiguous() for x in (k, v))
        got = fourier_attention(q, k, v, one, 0, Hq, Hkv)
        two.update(k, v, 0)
        want = two.decode_attention(q, 0, Hq, Hkv, out_dtype=dtype).view(B, 1, Hq * D)
        assert torch.equal(got, want), t
    for a, b in zip((one.key_cache[0], one.value_cache[0]), (two.key_cache[0], two.value_cache[0])):
        assert all(torch.equal(a[n], b[n]) for n in a)
    assert one.get_seq_length() == two.get_seq_length() == S + W + 5
    # one launch less than the two calls, except with head dims that have no vectorised window kernel and where two are quicker
    joins = D != 80 and not (states == 1024 and B < 8)
    def both():
        two.update(k, v, 0)
        two.decode_attention(q, 0, Hq, Hkv, out_dtype=dtype)
    joined = _launches(lambda: fourier_attention(q, k, v, one, 0, Hq, Hkv))
    assert joined == _launches(both) - joins


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B,Hq,Hkv,D,rows", [(1, 2, 1, 128, 1), (2, 6, 2, 64, 64), (3, 8, 2, 80, 65), (1, 16, 2, 128, 4161), (2, 4, 4, 8, 1100),
                                             (1, 4, 1, 128, 20480), (1, 4, 1, 128, 20481)])
def test_window_only_decode(dtype, B, Hq, Hkv, D, rows):
    """A layer that keeps only a window, one tile to more tiles than the merge for it takes, against float64.  Bound: single
    precision over ``rows`` keys of order one, then the rounding of the result to ``dtype``."""
    from fourierattention_amd import ops
    g = torch.Generator(device="cuda").manual_seed(rows)
    q, k, v = (torch.randn(s, generator=g, device="cuda").to(dtype) for s in ((B, Hq, 1, D), (B, rows, Hkv * D), (B, rows, Hkv * D)))
    lists = (torch.zeros(Hkv + 1, dtype=torch.int32, device="cuda"),) * 8
    qd = q.double().view(B, Hkv, Hq // Hkv, D)
    kd, vd = (t.double().view(B, rows, Hkv, D).permute(0, 2, 1, 3).contiguous() for t in (k, v))
    p = (qd.matmul(kd.transpose(2, 3).contiguous()) / D ** 0.5).softmax(-1)
    want = p.matmul(vd).view(B, Hq, 1, D)
    for cast in (None, dtype):
        got = ops.decode_attn_raw(q, [(k, v)], None, None, None, None, None, None, lists, Hq, Hkv, 0, 1, out_dtype=cast)
        ulp = 2.0 ** -8 if got.dtype == torch.bfloat16 else 0.0
        assert got.dtype == (cast or torch.float32)
        assert bool(((got.double() - want).abs() <= 2e-5 + ulp * want.abs()).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("width,rows,slice_", [(256, 1, False), (1023, 3, False), (1024, 16, True), (7, 2, True)])
def test_append_rows(dtype, width, rows, slice_):
    """New rows behind a window, dense or slices of wider rows, aligned and not: the rows and nothing beside them."""
    from fourierattention_amd import ops
    g = torch.Generator(device="cuda").manual_seed(width)
    wide = torch.randn((2, rows, 2 * width), generator=g, device="cuda").to(dtype)
    k, v = wide.split(width, dim=-1) if slice_ else (x.contiguous() for x in wide.split(width, dim=-1))
    bufs = [torch.randn((2, 40, width), generator=g, device="cuda").to(dtype) for _ in range(2)]
    want = [b.clone() for b in bufs]
    for b, x in zip(want, (k, v)):
        b[:, 5:5 + rows] = x
    ops.append_rows(k, v, *bufs, 5)
    assert torch.equal(bufs[0], want[0]) and torch.equal(bufs[1], want[1])
    with pytest.raises(AssertionError):
        ops.append_rows(k, v, *bufs, 41 - rows)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_prompt_rows_whose_denominator_is_many_small_weights(dtype):
    """One key of weight 1 and 32767 keys of about 1.4 * 2^-24, where f16 holds multiples of 2^-24 only: together they are
    0.27% of the denominator.  The values of the many are zero, so the result is the denominator's inverse: it has to
    come from the weights in single precision.  Bound: the rounding of the result (of values just below 1), and single precision
    over 32768 weights."""
    from fourierattention_amd import ops
    S, D = 32768, 128
    q = torch.zeros((1, 4, 40, D), device="cuda", dtype=dtype)
    k = torch.zeros((1, S, D), device="cuda", dtype=dtype)
    v = torch.zeros((1, S, D), device="cuda", dtype=dtype)
    q[..., 0] = 16.0
    k[:, 0, 0] = float(np.log(2) * (24 - np.log2(1.4)) * D ** 0.5 / 16.0)
    v[:, 0] = 1.0
    score = float(k[0, 0, 0]) * 16.0 / D ** 0.5
    got = ops.prefill_attention(q, k, v, 1)[0].double()                  # row i sees keys 0 .. S - 40 + i
    seen = torch.arange(S - 40, S, device="cuda", dtype=torch.float64)
    want = (1.0 / (1.0 + seen * np.exp(-score)))[:, None, None].expand_as(got)
    assert float((got - want).abs().max()) <= 2.0 ** (-9 if dtype == torch.bfloat16 else -12) + 2e-5


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_prompt_rows_whose_largest_weight_comes_late(dtype):
    """Two keys, the second one (a tile later) ahead by up to six units of log 2, and only it has a value: its weight against
    the row's maximum is exactly one, so the result is the denominator's inverse to the rounding of the result itself (a weight
    of, say, 2^0.4 against the first key would already be rounded to f16).  Bound as above."""
    from fourierattention_amd import ops
    S, D, q_len = 64, 128, 24
    g = torch.Generator(device="cuda").manual_seed(2)
    q = torch.zeros((128, 4, q_len, D), device="cuda")
    q[..., 0] = 6 * np.log(2) * D ** 0.5 * torch.rand((128, 4, q_len), generator=g, device="cuda")
    q[..., 1] = 64.0
    k = torch.zeros((128, S, D), device="cuda")
    k[:, :, 1] = -64.0                       # every other key is out of reach
    k[:, (0, 40), 1] = 0.0
    k[:, 40, 0] = 1.0
    v = torch.zeros((128, S, D), device="cuda")
    v[:, 40] = 1.0
    q, k, v = (t.to(dtype) for t in (q, k, v))
    got = ops.prefill_attention(q, k, v, 1).double()
    want = torch.sigmoid(q[..., 0].double() / D ** 0.5).transpose(1, 2)[..., None].expand_as(got)
    assert float((got - want).abs().max()) <= 2.0 ** (-9 if dtype == torch.bfloat16 else -12) + 2e-5


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("L,k_counts,v_counts", [(70, [33, 122], [100, 121]), (1, [127, 128], [1, 127]), (130, [97, 60], [64, 128])])
def test_any_shape_decode_kernels_beside_infinities(dtype, L, k_counts, v_counts):
    """The last stored K dim of a head is -inf in some rows (their weight is zero) and the last row's first stored V dim is
    +inf (so is the result): what a kernel reads past a head's dims or past the rows must not reach a sum.  Bound as
    above."""
    from fourierattention_amd import ops
    from fourierattention_amd.midstore import MidStore
    from oracle import fourier_oracle as fo
    from tests import helpers as H
    Hq, Hkv, D = 4, 2, 128
    case = H.attn_case(13, 1, Hq, Hkv, D, 9, L, 40, 2 * L + 9, k_counts, v_counts, dtype)
    case["q"] = np.abs(case["q"]) + 0.25     # (a key of -inf scores -inf for every query head)
    case["q"] = H.to_dtype_np(case["q"], dtype)
    for h in range(Hkv):
        if case["kn_h_list"][h + 1] > case["kn_h_list"][h]:
            case["k_mn"][:, : L - 1 : 3, case["kn_h_list"][h + 1] - 1] = -np.inf
    case["v_mn"][:, L - 1, 0] = np.inf
    want = fo.fourier_attn(**case)
    g = H.attn_case_gpu(case, dtype)
    lists = tuple(ops.as_i32(g[n]) for n in ("kc_list", "kc_h_list", "kn_list", "kn_h_list", "vc_list", "vc_h_list", "vn_list", "vn_h_list"))
    f = lambda t: t.float().contiguous()
    stats = [(f(g[f"avg_{t}_u"]), f(g[f"avg_{t}_d"]), f(g[f"scale_{t}"])) for t in "kv"]
    stores = []
    for t, n_h, is_v in ((g["k_mn"], lists[3], False), (g["v_mn"], lists[7], True)):
        ident = torch.arange(t.shape[2], dtype=torch.int32, device="cuda")
        st = MidStore(1, ident, n_h, n_h.tolist(), Hkv, D, L, dtype, "cuda", is_v)
        st.pack(t, 0, L)
        stores.append(st)
    for k_mn, v_mn in ((g["k_mn"], g["v_mn"]), stores):
        got = ops.decode_attn_raw(g["q"], [(g["k_il"], g["v_il"])], g["k_mc"], g["v_mc"], k_mn, v_mn, *stats, lists, Hq, Hkv, L,
                                  case["T"], force_generic=True).cpu().numpy().astype(np.float64).reshape(want.shape)
        finite = np.isfinite(want)
        assert np.array_equal(got[~finite], want[~finite]) and (~finite).any()
        assert np.max(np.abs(got[finite] - want[finite])) <= 2e-4


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows", [1, 63, 65, 200])
def test_window_rows_with_an_infinite_value(dtype, rows):
    """The first row holds infinite values: they are the result in those dims and touch no other, however far the last
    tile reaches past the rows.  Bound: as for the window above."""
    from fourierattention_amd import ops
    B, Hq, Hkv, D = 2, 6, 2, 128
    g = torch.Generator(device="cuda").manual_seed(rows)
    q, k, v = (torch.randn(s, generator=g, device="cuda").to(dtype) for s in ((B, Hq, 1, D), (B, rows, Hkv * D), (B, rows, Hkv * D)))
    v[:, 0, 5] = float("inf")
    v[:, 0, 200] = -float("inf")
    lists = (torch.zeros(Hkv + 1, dtype=torch.int32, device="cuda"),) * 8
    kd, vd = (t.double().view(B, rows, Hkv, D).permute(0, 2, 1, 3).contiguous() for t in (k, v))
    p = (q.double().view(B, Hkv, Hq // Hkv, D).matmul(kd.transpose(2, 3).contiguous()) / D ** 0.5).softmax(-1)
    want = p.matmul(vd).view(B, Hq, 1, D)
    got = ops.decode_attn_raw(q, [(k, v)], None, None, None, None, None, None, lists, Hq, Hkv, 0, 1).double()
    inf = want.isinf()
    assert int(inf.sum()) == B * Hq and torch.equal(got[inf], want[inf])
    assert float((got - want)[~inf].abs().max()) <= 2e-5


def _two_caches(dtype, B=2, Hkv=2, D=128, W=40, states=128):
    """Two caches with the same prompt, and a source of new tokens."""
    from fourierattention_amd import DynamicCache, ExtraConfig, masks
    g = torch.Generator(device="cuda").manual_seed(21)
    rn = lambda *s: torch.randn(s, generator=g, device="cuda").to(dtype)
    m = masks.synthetic_masks(1, Hkv, D, [64, 40], [30, 64], seed=3)
    cfg = ExtraConfig(numinittokens=4, maxlocallen=W, maxmidstates=states, non_critical_dims=m, non_critical_dims_path=None,
                      max_position_embeddings=8192, num_key_value_heads=Hkv, max_new_tokens=8, model_type="llama")
    one, two = DynamicCache(cfg), DynamicCache(cfg)
    prompt = rn(B, Hkv, 4 + W + states + 300, D), rn(B, Hkv, 4 + W + states + 300, D)
    one.update(*prompt, 0)
    two.update(*prompt, 0)
    return one, two, rn


def _same_state(one, two):
    a, b = one._layers[0], two._layers[0]
    parts = zip((one.key_cache[0], one.value_cache[0]), (two.key_cache[0], two.value_cache[0]))
    return (a.n_mid, a.spare) == (b.n_mid, b.spare) and all(torch.equal(x[n], y[n]) for x, y in parts for n in x)


@pytest.mark.parametrize("refusal", ["type of q", "heads of q", "warning as an error"])
def test_a_refused_attention_leaves_the_update(refusal):
    """A decode step whose attention is refused on the way to the launch: the token is in the cache all the same, as with
    ``update`` alone, and the next step is what it is there."""
    import warnings
    from fourierattention_amd import ops
    from fourierattention_amd.attention import fourier_attention
    B, Hq, Hkv, D, dtype = 2, 8, 2, 128, torch.float16
    one, two, rn = _two_caches(dtype)
    for _ in range(2):
        q, k, v = rn(B, Hq, 1, D), rn(B, Hkv, 1, D), rn(B, Hkv, 1, D)
        two.update(k, v, 0)
        if refusal == "warning as an error":
            old = ops._REPACK_MIN_ROWS
            ops._REPACK_MIN_ROWS = 1
            ops._warned_shapes.clear()
            warn = ops._warn_if_off_the_matrix_cores
            ops._warn_if_off_the_matrix_cores = lambda *a: warnings.warn("off the matrix cores", RuntimeWarning)
            try:
                with warnings.catch_warnings(), pytest.raises(RuntimeWarning):
                    warnings.simplefilter("error")
                    fourier_attention(q, k, v, one, 0, Hq, Hkv)
            finally:
                ops._REPACK_MIN_ROWS, ops._warn_if_off_the_matrix_cores = old, warn
        else:
            with pytest.raises((AssertionError, RuntimeError)):
                fourier_attention(q.float() if refusal == "type of q" else rn(B, 9, 1, D), k, v, one, 0, Hq if refusal == "type of q" else 9, Hkv)
        assert _same_state(one, two)
        q, k, v = rn(B, Hq, 1, D), rn(B, Hkv, 1, D), rn(B, Hkv, 1, D)
        got = fourier_attention(q, k, v, one, 0, Hq, Hkv)
        two.update(k, v, 0)
        assert torch.equal(got, two.decode_attention(q, 0, Hq, Hkv, out_dtype=dtype).view(B, 1, Hq * D)) and _same_state(one, two)


def test_a_refused_update_leaves_the_layer():
    """A token of another type than the window: neither call counts a row that was never written."""
    from fourierattention_amd.attention import fourier_attention
    one, two, rn = _two_caches(torch.bfloat16)
    q, k, v = rn(2, 8, 1, 128), rn(2, 2, 1, 128), rn(2, 2, 1, 128)
    with pytest.raises(AssertionError):
        fourier_attention(q, k.float(), v.float(), one, 0, 8, 2)
    with pytest.raises(AssertionError):
        two.update(k.float(), v.float(), 0)
    a, b = one._layers[0], two._layers[0]       # (the views of the parts are of the state before, on either side)
    assert (a.n_mid, a.spare, a.version) == (b.n_mid, b.spare, b.version)
    for x, y in ((a.k, b.k), (a.v, b.v)):
        assert torch.equal(x.ring[:, :40], y.ring[:, :40]) and torch.equal(x.coef, y.coef) and torch.equal(x.mid.data, y.mid.data)


@pytest.mark.parametrize("rows,launches", [(1, 1), (3, 1), (4, 3), (16, 3)])
def test_where_the_norms_of_a_decoder_step_run(rows, launches, monkeypatch):
    """Up to three rows of 12288 elements together the two norms of a layer ride in its projections and only the final one is a
    launch; above, all three are.  The logits against the chain of tensor ops, which rounds between them: bf16 through one layer, 2^-8 of the
    largest, a few times over."""
    from fourierattention_amd import DynamicCache, ExtraConfig, masks, ops
    from fourierattention_amd.llama import LlamaConfig, random_init
    llama = LlamaConfig(hidden_size=2048, intermediate_size=2048, num_hidden_layers=1, num_attention_heads=16, num_key_value_heads=8,
                        head_dim=128, vocab_size=512)
    model = random_init(llama, torch.bfloat16, "cuda:0", seed=1)
    model.model.pack_projections()
    cfg = ExtraConfig(numinittokens=4, maxlocallen=64, maxmidstates=64, non_critical_dims=masks.synthetic_masks(1, 8, 128, [64] * 8, [64] * 8, seed=1),
                      non_critical_dims_path=None, max_position_embeddings=4096, num_key_value_heads=8, max_new_tokens=8, model_type="llama")
    ids = torch.randint(0, 512, (rows, 21), device="cuda")
    own, calls, logits = ops.add_rmsnorm, [], []
    monkeypatch.setattr(ops, "add_rmsnorm", lambda *a: (calls.append(1), own(*a))[1])
    with torch.no_grad():
        for fused in (True, False):
            model.model.fused_elementwise = fused
            cache = DynamicCache(cfg)
            model(ids[:, :20], cache)
            calls.clear()
            logits.append(model(ids[:, 20:], cache).logits)
            assert len(calls) == (launches if fused else 0)
    assert float((logits[0] - logits[1]).abs().max()) <= 4 * 2.0 ** -8 * float(logits[1].abs().max())


@pytest.mark.parametrize("rows,launches", [(4, 1), (6, 1), (7, 3)])
def test_where_the_norms_of_a_narrow_decoder_step_run(rows, launches, monkeypatch):
    """Rows of 6144 elements together ride however many they are (1024 wide: 5 rows 14.3 us a layer apart, 12.3 riding)."""
    from fourierattention_amd import DynamicCache, ExtraConfig, masks, ops
    from fourierattention_amd.llama import LlamaConfig, random_init
    llama = LlamaConfig(hidden_size=1024, intermediate_size=1024, num_hidden_layers=1, num_attention_heads=8, num_key_value_heads=8,
                        head_dim=128, vocab_size=512)
    model = random_init(llama, torch.bfloat16, "cuda:0", seed=1)
    model.model.pack_projections()
    cfg = ExtraConfig(numinittokens=4, maxlocallen=64, maxmidstates=64, non_critical_dims=masks.synthetic_masks(1, 8, 128, [64] * 8, [64] * 8, seed=1),
                      non_critical_dims_path=None, max_position_embeddings=4096, num_key_value_heads=8, max_new_tokens=8, model_type="llama")
    ids = torch.randint(0, 512, (rows, 21), device="cuda")
    own, calls, logits = ops.add_rmsnorm, [], []
    monkeypatch.setattr(ops, "add_rmsnorm", lambda *a: (calls.append(1), own(*a))[1])
    with torch.no_grad():
        for fused in (True, False):
            model.model.fused_elementwise = fused
            cache = DynamicCache(cfg)
            model(ids[:, :20], cache)
            calls.clear()
            logits.append(model(ids[:, 20:], cache).logits)
            assert len(calls) == (launches if fused else 0)
    assert float((logits[0] - logits[1]).abs().max()) <= 4 * 2.0 ** -8 * float(logits[1].abs().max())


def test_argument_forms_of_the_decode_call():
    """Lists instead of tuples, whole numbers that are not ints, timings in any mutable sequence; the sine table alone in another
    type, tables with rows to spare."""
    from collections import UserList
    from fourierattention_amd import ops
    from tests import helpers as H
    dtype = torch.float32
    case = H.attn_case(3, 1, 4, 2, 128, 9, 70, 16, 300, [64, 40], [30, 64], dtype)
    g = H.attn_case_gpu(case, dtype)
    lists = [ops.as_i32(g[n]) for n in ("kc_list", "kc_h_list", "kn_list", "kn_h_list", "vc_list", "vc_h_list", "vn_list", "vn_h_list")]
    f = lambda t: t.float().contiguous()
    stats = [[f(g[f"avg_{t}_u"]), f(g[f"avg_{t}_d"]), f(g[f"scale_{t}"])] for t in "kv"]
    args = (g["k_mc"], g["v_mc"], g["k_mn"], g["v_mn"])
    pair = [g["k_il"], g["v_il"]]
    want = ops.decode_attn_raw(g["q"], [tuple(pair)], *args, *map(tuple, stats), tuple(lists), 4, 2, 70, 300)
    got = ops.decode_attn_raw(g["q"], (pair, None), *args, *stats, lists, 4, 2, np.int64(70), 300.0, no_fuse=np.bool_(False))
    assert torch.equal(got, want)
    ms = UserList()
    assert torch.equal(ops.decode_attn_raw(g["q"], [pair], *args, *stats, lists, 4, 2, torch.tensor(70), 300, timings=ms), want)
    assert len(ms) == 4 and all(isinstance(x, float) for x in ms)
    q, k = (torch.randn((2, 3, n * 128), device="cuda").bfloat16() for n in (4, 2))
    cos, sin = torch.randn((2, 2, 3, 128), device="cuda").bfloat16().unbind(0)
    k1, k2 = k.clone(), k.clone()
    a, b = ops.rope_qk(q.clone(), k1, cos, sin, 128), ops.rope_qk(q.clone(), k2, cos, sin.float(), 128)
    assert torch.equal(a, b) and torch.equal(k1, k2)
    k1, k2 = k[:1].clone(), k[:1].clone()      # one sequence, tables with rows to spare
    a, b = ops.rope_qk(q[:1].clone(), k1, cos[:1], sin[:1], 128), ops.rope_qk(q[:1].clone(), k2, *(t.reshape(1, 6, 128) for t in (cos, sin)), 128)
    assert torch.equal(a, b) and torch.equal(k1, k2)


def test_operands_when_only_empty_lists_need_a_conversion():
    """Empty 64-bit lists beside 32-bit ones and single-precision statistics: nothing to convert, and nothing lost."""
    from fourierattention_amd import _lib
    i = lambda *v: torch.tensor(v, dtype=torch.int32, device="cuda")
    none = torch.empty(0, dtype=torch.int64, device="cuda")
    lists = (none, i(0, 0, 0), i(3, 4), i(0, 1, 2), none, i(0, 0, 0), i(7), i(0, 1, 1))
    stats = (torch.ones((1, 0), device="cuda", dtype=torch.bfloat16),) + tuple(torch.ones((1, 2), device="cuda") for _ in range(5))
    for units in ((0, 0), (32, 16)):
        l32, s32, paging = _lib.load_host().operands(lists, stats, *units)
        assert all(a.dtype == torch.int32 and a.tolist() == b.tolist() for a, b in zip(l32, lists))
        assert all(a.dtype == torch.float32 and torch.equal(a, b.float()) for a, b in zip(s32, stats))
        assert paging is None or (paging[0], paging[1], paging[2].tolist(), paging[3].tolist()) == ([0, 1, 2], [0, 1, 1], [0, 32, 64], [0, 16, 16])


@pytest.mark.parametrize("rows,C", [(1100, 33), (60, 1)])
def test_statistics_are_tensors_of_their_own(rows, C):
    """Mean and deviation share no storage (keeping or saving one keeps one) and start where an allocation does."""
    from fourierattention_amd import ops
    a = torch.randn((2, rows, C), device="cuda").bfloat16()
    c = torch.randn((2, 64, C), device="cuda")
    for pair in (ops.mat_avg_std(a), ops.mat_avg_std_triton(a), ops.mat_fourier_avg_std(c, rows, 2000), ops.mat_fourier_avg_std_triton(c, rows, 2000)):
        avg, dev = pair
        assert avg.untyped_storage().data_ptr() != dev.untyped_storage().data_ptr()
        assert all(t.storage_offset() == 0 and t.is_contiguous() and t.data_ptr() % 256 == 0 and t.shape == (2, C) for t in pair)
        assert all(t.untyped_storage().nbytes() < 2 * t.numel() * t.element_size() + 512 and t._base is None for t in pair)

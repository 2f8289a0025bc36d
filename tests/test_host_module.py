"""The native host side of the per-token calls: what it refuses before anything reaches the GPU, and the row strides it
reads off a view (on the GPU, against the same rows made dense)."""
import pytest
import torch


def test_cpu_tensors_and_wrong_types_are_refused():
    from fourierattention_amd import _lib, ops
    host = _lib.load_host()
    x = torch.zeros(2, 1, 1024)
    with pytest.raises(RuntimeError, match="GPU tensor"):
        ops.add_rmsnorm(x, None, torch.ones(1024), 1e-5)
    with pytest.raises(RuntimeError, match="GPU tensor"):
        ops.silu_mul(x, x)
    with pytest.raises(RuntimeError, match="GPU tensor"):
        ops.decode_attn_raw(x, [(x, x)], None, None, None, None, None, None, (x,) * 8, 8, 2, 0, 1)
    with pytest.raises(TypeError, match="must be a tensor"):
        host.linear_packed(None, x, 1024, 16)
    with pytest.raises(AssertionError, match="arguments"):
        host.silu_mul(x)


def test_a_library_of_another_layout_is_refused(monkeypatch):
    """The module fills argument structs for the library beside it: another version or struct size is an import error."""
    from types import SimpleNamespace
    from fourierattention_amd import _lib
    lib = _lib.load()
    own = lib.fa_abi_version(), lib.fa_decode_args_size(), lib.fa_stream_args_size()
    assert _lib.load_host().layout() == own
    for i in range(3):
        other = [v + (i == j) for j, v in enumerate(own)]
        fake = SimpleNamespace(**{n: (lambda v=v: v) for n, v in zip(("fa_abi_version", "fa_decode_args_size", "fa_stream_args_size"), other)})
        monkeypatch.setattr(_lib, "load", lambda: fake)
        monkeypatch.setattr(_lib, "_host", None)
        with pytest.raises(ImportError, match="was built for"):
            _lib.load_host()


@pytest.mark.gpu
@pytest.mark.parametrize("B,q_len", [(1, 1), (5, 1), (1, 7), (3, 4)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_row_slices_of_wider_rows(B, q_len, dtype):
    """q, k and gate, up as column slices of one projection output: the same bits as on dense copies of the slices."""
    from fourierattention_amd import ops
    g = torch.Generator(device="cuda").manual_seed(B * 10 + q_len)
    wide = torch.randn((B, q_len, 6 * 128 + 2 * 1024), generator=g, device="cuda").to(dtype)
    q, k, gate, up = wide.split((4 * 128, 2 * 128, 1024, 1024), dim=-1)
    cos, sin = (torch.randn((B, q_len, 128), generator=g, device="cuda").to(dtype) for _ in range(2))
    assert torch.equal(ops.silu_mul(gate, up), ops.silu_mul(gate.contiguous(), up.contiguous()))
    qd, kd = q.contiguous(), k.contiguous()
    want = ops.rope_qk(qd, kd, cos, sin, 128)
    got = ops.rope_qk(q, k, cos, sin, 128)
    assert torch.equal(got, want) and torch.equal(k, kd)
    if B * q_len <= 16:
        w = torch.randn((48, 1024), generator=g, device="cuda").to(dtype)
        packed = ops.PackedLinearWeight(w)
        assert torch.equal(ops.linear_packed(gate, packed), ops.linear_packed(gate.contiguous(), packed))


@pytest.mark.parametrize("how", ["instance", "class", "subclass"])
def test_a_replaced_update_is_what_the_attention_calls(how, monkeypatch):
    """``fourier_attention`` goes through ``update`` of the cache it is given, for one token as for many."""
    from fourierattention_amd import DynamicCache, ExtraConfig, masks
    from fourierattention_amd.attention import fourier_attention
    m = masks.synthetic_masks(1, 2, 16, [8, 8], [8, 8], seed=3)
    cfg = ExtraConfig(numinittokens=4, maxlocallen=16, maxmidstates=16, non_critical_dims=m, non_critical_dims_path=None,
                      max_position_embeddings=512, num_key_value_heads=2, max_new_tokens=8, model_type="llama")
    calls = []

    def update(key_states, value_states, layer_idx, cache_kwargs=None):
        calls.append(layer_idx)
        k, v = (t.transpose(1, 2).reshape(1, 1, 32) for t in (key_states, value_states))
        return ({"k_init": None, "k_compressed": None, "k_uncompressed": None, "k_local": k},
                {"v_init": None, "v_compressed": None, "v_uncompressed": None, "v_local": v})
    if how == "subclass":
        cache = type("Own", (DynamicCache,), {"update": lambda self, *a, **k: update(*a, **k)})(cfg, device="cpu")
    else:
        cache = DynamicCache(cfg, device="cpu")
        if how == "instance":
            cache.update = update
        else:
            monkeypatch.setattr(DynamicCache, "update", lambda self, *a, **k: update(*a, **k))
    q, k, v = torch.randn(1, 4, 1, 16), torch.randn(1, 2, 1, 16), torch.randn(1, 2, 1, 16)
    out = fourier_attention(q, k, v, cache, 0, 4, 2)
    assert calls == [0] and torch.allclose(out.view(1, 2, 2, 16), v.transpose(1, 2).reshape(1, 2, 1, 16).expand(1, 2, 2, 16))


@pytest.mark.gpu
def test_other_threads_run_while_a_call_waits_for_the_gpu():
    """The offsets of ``operands`` are waited for behind whatever the stream holds; another Python thread goes on meanwhile."""
    import threading
    import time
    from fourierattention_amd import _lib
    host = _lib.load_host()
    lists = tuple(torch.tensor([0, 5, 9], device="cuda") for _ in range(8))
    host.operands(lists, (), 32, 16)
    ticks, stop = [0], threading.Event()

    def tick():
        while not stop.is_set():
            ticks[0] += 1
            time.sleep(0.001)
    t = threading.Thread(target=tick)
    t.start()
    try:
        torch.cuda._sleep(int(4e8))        # a few tenths of a second
        before, t0 = ticks[0], time.perf_counter()
        paging = host.operands(lists, (), 32, 16)[2]
        waited, seen = time.perf_counter() - t0, ticks[0] - before
    finally:
        stop.set()
        t.join()
    assert paging[0] == [0, 5, 9] and waited > 0.05 and seen >= 10, (waited, seen)


@pytest.mark.gpu
def test_rows_without_elements_are_refused():
    """A width of zero is an error on the host (it divides the number of elements there)."""
    from fourierattention_amd import _lib, ops
    e = lambda *s: torch.empty(s, device="cuda", dtype=torch.bfloat16)
    with pytest.raises(AssertionError):
        ops.add_rmsnorm(e(2, 0), None, e(0), 1e-5)
    with pytest.raises(AssertionError):
        _lib.load_host().linear_packed(e(2, 0), e(0), 0, 16)
    assert ops.silu_mul(e(2, 0), e(2, 0)).shape == (2, 0) and ops.silu_mul(e(0, 8), e(0, 8)).shape == (0, 8)


def test_lists_of_a_cache_in_one_tensor():
    """Every list of the masks comes back whole, in both types, whatever its length or the type of its entries."""
    import numpy as np
    import torch
    from fourierattention_amd.cache import _device_lists
    lists = [[], [3], list(range(40)), [np.int64(5), 2 ** 31 - 1], (1, 2), [True, -4]]
    for got, want in ((_device_lists(lists, torch.device("cpu")), lists), (_device_lists([[1.5, 2]], torch.device("cpu")), [[1, 2]])):
        for tensors, dt in zip(got, (torch.int64, torch.int32)):
            assert [t.tolist() for t in tensors] == [[int(x) for x in lst] for lst in want]
            assert all(t.dtype == dt and t.is_contiguous() and t.storage_offset() % 32 == 0 for t in tensors)


def test_lists_of_a_cache_under_another_default_device():
    """A cache made where the program has set a default device (``torch.device(..)`` as a context) gets its lists on its own."""
    import torch
    from fourierattention_amd.cache import _device_lists
    with torch.device("meta"):
        got = _device_lists([[3, 1], [7]], torch.device("cpu"))
    for tensors, dt in zip(got, (torch.int64, torch.int32)):
        assert [(t.device.type, t.dtype, t.tolist()) for t in tensors] == [("cpu", dt, [3, 1]), ("cpu", dt, [7])]


def test_lists_of_a_cache_where_operations_are_recorded():
    """A cache made inside a traced or transformed function."""
    import torch
    from torch.fx.experimental.proxy_tensor import make_fx
    from fourierattention_amd.cache import _device_lists
    pick = lambda x: x[_device_lists([[3, 1], [2]], torch.device("cpu"))[0][0]]
    x, y = torch.arange(8.0).view(2, 4)
    assert make_fx(pick)(x)(y).tolist() == [7.0, 5.0]
    assert torch.jit.trace(pick, x, check_trace=False)(y).tolist() == [7.0, 5.0]
    assert torch.func.vmap(pick)(torch.stack([x, y])).tolist() == [[3.0, 1.0], [7.0, 5.0]]

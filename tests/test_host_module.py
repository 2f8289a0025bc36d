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

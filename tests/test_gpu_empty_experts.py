"""Experts without rows in the weight gradient: zeros, whatever lies between them, without an operation per expert; the entry that
clears them at its edges (a slot of one store, of exactly one and just over one workgroup, slots listed out of order and outside)."""
import pytest
import torch

from tests.test_gpu_any_k import close, deq

pytestmark = pytest.mark.gpu


def _gradient(k_blocks, M, N, dtype):
    import gcore_lowp as G
    g = torch.Generator(device="cuda").manual_seed(sum(k_blocks) + M)
    ops = [G.quant_fp8_e4m3_scale_e8m0(torch.randn(M, kb * 128, generator=g, device="cuda", dtype=torch.bfloat16), (1, 128))
           + G.quant_fp8_e4m3_scale_e8m0(torch.randn(N, kb * 128, generator=g, device="cuda", dtype=torch.bfloat16), (1, 128)) if kb else None
           for kb in k_blocks]
    flat = [torch.cat([o[i].view(torch.uint8).flatten() for o in ops if o] or [torch.empty(0, dtype=torch.uint8, device="cuda")]) for i in range(4)]
    out = torch.full((len(k_blocks), M, N), float("nan"), dtype=dtype, device="cuda")
    return ops, flat, out


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "f32"])
@pytest.mark.parametrize("k_blocks", [[0, 1, 0, 0, 3, 0, 2, 0], [0, 0, 0], [4, 0], [0, 5], [3, 1]], ids=str)
def test_gradients_of_empty_experts(k_blocks, dtype):
    import gcore_lowp as G
    ops, flat, out = _gradient(k_blocks, 256, 384, dtype)
    print("[case]", k_blocks, dtype, flush=True)
    G.gemm_fp8_rowscale_grouped(*flat, k_blocks, 256, 384, out)
    for e, o in enumerate(ops):
        if o is None:
            assert not out[e].any() and torch.isfinite(out[e]).all()
        else:
            close(out[e], deq(o[0], o[1], 1) @ deq(o[2], o[3], 1).t(), (k_blocks, e))


def test_many_empty_experts_cost_no_operation_each():
    import gcore_lowp as G
    from torch.utils._python_dispatch import TorchDispatchMode

    class Count(TorchDispatchMode):
        n = 0

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            Count.n += 1
            return func(*args, **(kwargs or {}))

    k_blocks = [1 if e % 8 == 0 else 0 for e in range(64)]
    _, flat, out = _gradient(k_blocks, 128, 128, torch.bfloat16)
    with Count():
        G.gemm_fp8_rowscale_grouped(*flat, k_blocks, 128, 128, out)
    assert Count.n <= 8, Count.n
    assert [bool(out[e].any()) for e in range(64)] == [bool(kb) for kb in k_blocks]


@pytest.mark.parametrize("slot_bytes", [16, 16384, 16400, 4096 * 5])
def test_listed_slots_are_cleared_and_no_other(slot_bytes):
    from gcore_lowp import _abi as A
    c = torch.full((7, slot_bytes), 5, dtype=torch.uint8, device="cuda")
    slots = torch.tensor([4, -1, 0, 7, 6, 2 ** 31 - 1], dtype=torch.int32, device="cuda")
    print("[case]", slot_bytes, flush=True)
    A.check(A.lib().lp_zero_slots(c.data_ptr(), slot_bytes, 6, slots.data_ptr(), 6, A.stream_ptr()))
    assert [bool((c[i] == 0).all()) for i in range(7)] == [True, False, False, False, True, False, False]
    assert bool((c[[1, 2, 3, 5, 6]] == 5).all())

"""The D = 64 backward kernels at the sizes where they can go wrong: edges of 32-row waves, 64-row tiles and 128-row
blocks, one tile and less, several tiles with a partial last one.  The D = 128 backward with a workspace that holds the
dS of some of the slices."""
import pytest
import torch

import abi
from oracle import attention_oracle as ao


@pytest.mark.gpu
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("N", [1, 31, 32, 33, 64, 65, 96, 127, 128, 129, 191, 193, 256, 257, 321, 450])
def test_backward_d64(N, causal):
    B, H, D = 2, 5, 64
    q, k, v, do = ao.make_inputs(B, N, H, D, seed=11)
    scale = D ** -0.5
    lib = abi.load()
    qg, kg, vg, dog = (t.cuda() for t in (q, k, v, do))
    out, lse = abi.forward(lib, qg, kg, vg, scale, causal)
    ref = ao.attention_backward(q, k, v, do, scale, causal)
    whole = abi.backward(lib, qg, kg, vg, out, dog, lse, scale, causal)
    split = abi.backward(lib, qg, kg, vg, out, dog, lse, scale, causal, split=True)
    for got, one_by_one, want in zip(whole[:3], split[:3], ref):
        # fp16 roundings of P, dS, delta's O and the result: the repository's bound for gradients of order 1
        assert (got.float().cpu() - want.half().float()).abs().max() <= 1e-2
        assert torch.equal(got, one_by_one)  # delta from the dQ pass or from its own kernel: the same bits
    assert torch.equal(whole[3], split[3])


@pytest.mark.gpu
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("B,H,N,room", [
    (1, 1025, 64, 512),   # three rounds of 344 slices, the last one smaller
    (2, 129, 129, 256),   # two rounds, the workspace one slice pair short of one
    (7, 57, 300, 200),    # two rounds that do not end at a batch, the full room used
    (3, 100, 300, 170),   # rounds of fewer than two blocks per compute unit: recomputes instead
])
def test_backward_in_rounds(B, H, N, room, causal):
    """Rounds give the bits of one pass over all slices; dK and dV are those bits on any path."""
    D, lib = 128, abi.load()
    q, k, v, do = (t.cuda() for t in ao.make_inputs(B, N, H, D, seed=7))
    out, lse = abi.forward(lib, q, k, v, D ** -0.5, causal)
    whole = abi.backward(lib, q, k, v, out, do, lse, D ** -0.5, causal)[:3]
    np_ = -(-N // 128) * 128
    nbytes = -(-lib.fused_mha_backward_min_workspace_bytes(B, H, N, D) // 256) * 256 + room * np_ * np_ * 2
    ws = torch.empty(nbytes, dtype=torch.uint8, device="cuda")
    got = [torch.full_like(q, float("nan")) for _ in range(3)]
    rc = lib.fused_mha_backward(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), do.data_ptr(), lse.data_ptr(),
                                ws.data_ptr(), nbytes, *(g.data_ptr() for g in got), B, H, N, N, D, D ** -0.5,
                                int(causal), torch.cuda.current_stream().cuda_stream)
    assert rc == abi.OK
    assert torch.equal(got[1], whole[1]) and torch.equal(got[2], whole[2])
    if room == 170:  # dQ of the recomputing kernel: the same products in another order, fp32 sums, fp16 results of order 1
        assert (got[0].float() - whole[0].float()).abs().max() <= 2e-3
    else:
        assert torch.equal(got[0], whole[0])


@pytest.mark.gpu
def test_backward_without_memory_for_the_spill():
    from flash_attn_v100 import flash_attn_func
    B, H, N, D = 1, 32, 4096, 128  # 1 GiB of dS
    q, k, v, do = (t.cuda() for t in ao.make_inputs(B, N, H, D, seed=3))
    grads = []
    total = torch.cuda.get_device_properties(0).total_memory
    for limit in (None, 512 << 20):
        leaves = [t.clone().requires_grad_() for t in (q, k, v)]
        out = flash_attn_func(*leaves, causal=True)
        torch.cuda.empty_cache()
        try:
            if limit:
                torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + limit) / total)
            torch.cuda.reset_peak_memory_stats()
            grads.append(torch.autograd.grad(out, leaves, do))
            assert (torch.cuda.max_memory_allocated() > 1 << 30) == (limit is None)
        finally:
            torch.cuda.set_per_process_memory_fraction(1.0)
    assert torch.equal(grads[0][1], grads[1][1]) and torch.equal(grads[0][2], grads[1][2])
    assert (grads[0][0].float() - grads[1][0].float()).abs().max() <= 2e-3

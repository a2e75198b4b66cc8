"""The D = 64 backward kernels at the sizes where they can go wrong: edges of 32-row waves, 64-row tiles and 128-row
blocks, one tile and less, several tiles with a partial last one.  The D = 128 backward with a workspace that holds the
dS of some of the slices."""
import ctypes
import os
import subprocess

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
@pytest.mark.parametrize("N", [1, 63, 64, 65, 129, 200, 321])
def test_backward_d64_strided(N, causal):
    """q, k, v and dout each with strides of their own: the bits of dense copies."""
    B, H, D = 2, 3, 64
    gen = torch.Generator(device="cuda").manual_seed(N)
    normal = lambda *shape: torch.randn(shape, device="cuda", dtype=torch.float16, generator=gen)
    q = normal(B, N, 3, H, D)[:, :, 1]          # a slice of a packed projection
    k = normal(B, H, N, D).transpose(1, 2)      # backed by (batch, heads, seqlen, head_size)
    v = normal(B, N, H, D + 8)[..., :D]         # rows longer than the head size
    do = normal(N, B, H, D).transpose(0, 1)     # sequence first
    assert len({t.stride() for t in (q, k, v, do)}) == 4
    lib, scale = abi.load(), D ** -0.5
    dense = [t.contiguous() for t in (q, k, v, do)]
    out, lse = abi.forward(lib, *dense[:3], scale, causal)
    got = abi.backward_strided(lib, q, k, v, out, do, lse, scale, causal)
    want = abi.backward(lib, *dense[:3], out, dense[3], lse, scale, causal)
    for a, b in zip(got, want):
        assert torch.equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("N", [1, 33, 64, 100, 128, 257, 500])
def test_backward_d64_has_the_bits_of_the_general_passes(N, causal):
    """Features that are zero add nothing to any sum, so D = 64 problems padded to D = 128 give the recomputing kernels of
    that size the same products to add, in the order that the D = 64 kernels have to keep: bit for bit the same."""
    B, H, D = 2, 3, 64
    q, k, v, do = (t.cuda() for t in ao.make_inputs(B, N, H, D, seed=N))
    lib, scale = abi.load(), D ** -0.5
    out, lse = abi.forward(lib, q, k, v, scale, causal)
    got = abi.backward(lib, q, k, v, out, do, lse, scale, causal)
    wide = [torch.nn.functional.pad(t, (0, D)) for t in (q, k, v, out, do)]
    want = abi.backward(lib, *wide, lse, scale, causal, min_workspace=True)
    for a, b in zip(got[:3], want[:3]):
        assert torch.equal(a, b[..., :D]) and not b[..., D:].any()
    assert torch.equal(got[3], want[3])  # delta


@pytest.mark.gpu
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("B,H,N,room", [
    (1, 1025, 64, 512),   # three rounds of 344 slices, the last one smaller: had a slice not a work group of its own
    (1, 1030, 100, 512),  # the same where it has not
    (2, 129, 129, 256),   # two rounds, the workspace one slice pair short of one
    (7, 57, 300, 200),    # two rounds that do not end at a batch, the full room used
    (3, 100, 300, 170),   # rounds of fewer than two blocks per compute unit: recomputes instead
])
def test_backward_in_rounds(B, H, N, room, causal):
    """Rounds give the bits of one pass over all slices, and so does the path that forms S and dP twice."""
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
    for a, b in zip(got, whole):
        assert torch.equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("H,N,causal", [
    (64, 2048, True),   # dQ pass: one pair of blocks of 256 queries per compute unit, persistent
    (60, 2048, True),   # nearly one pair, which does not share out evenly: handed out by the hardware
    (42, 1300, True),   # the same with the half panels of a ragged end
    (120, 512, True),   # nearly one pair of short blocks: persistent all the same
    (62, 1031, False),  # 558 blocks, 2.2 per compute unit
    (63, 1000, False),  # 252 blocks, nearly one per compute unit: persistent
])
def test_a_slice_alone_gives_the_same_gradients(H, N, causal):
    """One slice has too few blocks for any of the schedules the whole problem takes: the same bits."""
    D, lib = 128, abi.load()
    gen = torch.Generator(device="cuda").manual_seed(N + H)
    q, k, v, do = (torch.randn(1, N, H, D, device="cuda", dtype=torch.float16, generator=gen) for _ in range(4))
    out, lse = abi.forward(lib, q, k, v, D ** -0.5, causal)
    whole = abi.backward(lib, q, k, v, out, do, lse, D ** -0.5, causal)[:3]
    for h in (0, H // 2, H - 1):
        one = [t[:, :, h:h + 1].contiguous() for t in (q, k, v, out, do)]
        alone = abi.backward(lib, *one, lse[:, h:h + 1].clone(), D ** -0.5, causal)[:3]
        for a, b in zip(alone, whole):
            assert torch.equal(a, b[:, :, h:h + 1])


BY_SLICE = [(D, N, causal) for causal in (False, True) for D, Ns in (
    (128, (1, 2, 31, 32, 33, 63, 64, 65, 96, 100, 127, 128, 129, 130, 159, 160, 161, 192, 193, 223, 224, 225, 255, 256)),
    (64, (129, 159, 160, 161, 192, 193, 200, 256, 257, 287, 288, 289, 320, 383, 384, 385, 449, 480, 481, 511, 512)))
            for N in Ns if not (D == 64 and causal and 200 < N <= 256)]


def test_by_slice_cases(tmp_path):
    """The cases below have a work group for each of 256 slices on 256 compute units."""
    assert all(abi.host_rule(tmp_path, "fmha_backward_by_slice(x[0], x[1], 256, 256, x[2])", BY_SLICE))


@pytest.mark.gpu
@pytest.mark.parametrize("D,N,causal", BY_SLICE)
def test_a_work_group_for_each_slice(D, N, causal):
    """The bits of the passes one by one, delta too, also with strides and with the least workspace; every element of the
    gradients and none of the workspace but the statistics is written."""
    B, lib, scale = 2, abi.load(), D ** -0.5
    H = torch.cuda.get_device_properties(0).multi_processor_count // B
    gen = torch.Generator(device="cuda").manual_seed(N + D)
    packed = torch.randn(B, N, 4, H, D, device="cuda", dtype=torch.float16, generator=gen)
    dense = [packed[:, :, i].contiguous() for i in range(4)]
    out, lse = abi.forward(lib, *dense[:3], scale, causal)
    want = abi.backward(lib, *dense[:3], out, dense[3], lse, scale, causal, split=True)
    got = abi.backward(lib, *dense[:3], out, dense[3], lse, scale, causal, poison=True)
    least = abi.backward(lib, *dense[:3], out, dense[3], lse, scale, causal, poison=True, min_workspace=True)
    strided = abi.backward_strided(lib, *(packed[:, :, i] for i in range(3)), out, packed[:, :, 3], lse, scale, causal)
    for a, b, c in zip(got, want, least):
        assert torch.equal(a, b) and torch.equal(c, b)
    for a, b in zip(strided, want):
        assert torch.equal(a, b)
    ref = ao.attention_backward(*(t[:1, :, :2].cpu() for t in dense), scale, causal)
    for a, b in zip(got, ref):
        # fp16 roundings of P, dS, delta's O and the result: the repository's bound for gradients of order 1
        assert (a[:1, :, :2].float().cpu() - b.half().float()).abs().max() <= 1e-2
    words = 2 * B * H * N  # delta and lse * log2(e)
    ws = torch.full((words + 64,), float("nan"), device="cuda")
    grads = [torch.full_like(g, float("nan")) for g in got[:3]]
    rc = lib.fused_mha_backward(*(t.data_ptr() for t in (*dense[:3], out, dense[3], lse, ws)), 4 * ws.numel(),
                                *(g.data_ptr() for g in grads), B, H, N, N, D, scale, int(causal),
                                torch.cuda.current_stream().cuda_stream)
    assert rc == abi.OK
    assert not torch.isnan(ws[:words]).any() and torch.isnan(ws[words:]).all()
    assert torch.equal(ws[words // 2:words], (lse * torch.tensor(1.4426950408889634, device="cuda")).flatten())
    for a, b in zip(grads, want):
        assert torch.equal(a, b)


OVER_DS_AT_ONCE = [  # H, N, causal
    (520, 64, False), (515, 100, True), (517, 128, True),  # a block per slice and pass
    (261, 129, False), (200, 160, False), (200, 161, True),  # last blocks of 1, 32 and 33 rows
    (100, 384, True), (65, 512, False),
    (60, 1031, False), (37, 1056, False), (33, 1023, True),
    (18, 2047, True), (9, 4096, False),
]


def test_launches_over_ds_of_the_cases_below(tmp_path):
    """Both passes over dS go in one launch on 256 compute units, once it is not by slices."""
    blocks = "(long)((x[1] + 127) / 128) * x[0], x[1], 256, x[2]"
    assert all(abi.host_rule(tmp_path, f"fmha_ds_in_one_launch(x[0], x[1], 256, x[2]) && !fmha_passes_at_once(128, {blocks})",
                             OVER_DS_AT_ONCE))


@pytest.mark.gpu
@pytest.mark.parametrize("ticks", [5000000, 0])
@pytest.mark.parametrize("H,N,causal", OVER_DS_AT_ONCE)
def test_both_passes_over_ds_in_one_launch(H, N, causal, ticks):
    """The bits of the passes one after the other, also (ticks) where no block waits for the dS of another; what the blocks
    have counted; nothing is left over from the call before, with other inputs."""
    B, D, lib = 1, 128, abi.load()
    lib.fmha_backward_waiting.argtypes = ([ctypes.c_void_p] * 7 + [ctypes.c_size_t] + [ctypes.c_void_p] * 3 + [ctypes.c_int] * 4 +
                                          [ctypes.c_float, ctypes.c_int, ctypes.c_uint, ctypes.c_void_p])
    gen = torch.Generator(device="cuda").manual_seed(N + H)
    nbytes = lib.fused_mha_backward_workspace_bytes(B, H, N, D) + 128 * H  # room for the counts of this launch
    ws = torch.full((nbytes,), 255, dtype=torch.uint8, device="cuda")
    blocks, spread = -(-N // 128), H % 8  # of a slice; slices with blocks on several XCDs, the last ones
    for _ in range(2):
        q, k, v, do = (torch.randn(B, N, H, D, device="cuda", dtype=torch.float16, generator=gen) for _ in range(4))
        out, lse = abi.forward(lib, q, k, v, D ** -0.5, causal)
        apart = abi.backward(lib, q, k, v, out, do, lse, D ** -0.5, causal, split=True)[:3]
        got = [torch.full_like(q, float("nan")) for _ in range(3)]
        rc = lib.fmha_backward_waiting(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), do.data_ptr(), lse.data_ptr(),
                                       ws.data_ptr(), nbytes, *(g.data_ptr() for g in got), B, H, N, D, D ** -0.5, int(causal),
                                       ticks, torch.cuda.current_stream().cuda_stream)
        assert rc == abi.OK
        for a, b in zip(got, apart):
            assert torch.equal(a, b)
        counts = ws[-128 * H:].view(torch.int32).view(H, 32)
        assert (counts[:, 0] == 4 * blocks).all()  # waves that have stored dS
        assert (counts[:H - spread, 1] == 0).all() and (counts[H - spread:, 1] == blocks).all()  # dK/dV blocks that have started
        if ticks:  # dQ blocks that have formed S and dP themselves
            assert (counts[:H - spread, 2] == 0).all()
        assert (counts[:, 2] <= blocks).all() and (counts[:, 3:] == 0).all()


@pytest.mark.gpu
@pytest.mark.parametrize("H,N,causal", [(60, 1031, False), (33, 1023, True), (15, 4609, False), (22, 5889, False)])
def test_launches_over_ds_on_two_streams(H, N, causal):
    """Launches of both passes over dS at once, with slices whose blocks are on several XCDs: the bits of one alone, and no wait
    for blocks that cannot start (of the two longest, waiting blocks of either can hold all of an XCD)."""
    D, lib = 128, abi.load()
    nbytes = lib.fused_mha_backward_workspace_bytes(1, H, N, D) + 128 * H
    calls = []
    for seed in range(2):
        gen = torch.Generator(device="cuda").manual_seed(seed)
        q, k, v, do = (torch.randn(1, N, H, D, device="cuda", dtype=torch.float16, generator=gen) for _ in range(4))
        out, lse = abi.forward(lib, q, k, v, D ** -0.5, causal)
        want = abi.backward(lib, q, k, v, out, do, lse, D ** -0.5, causal)[:3]
        ws = torch.empty(nbytes, dtype=torch.uint8, device="cuda")
        calls.append(((q, k, v, out, do, lse), ws, [torch.empty_like(q) for _ in range(3)], want, torch.cuda.Stream()))
    for _ in range(5):
        for _, ws, got, _, _ in calls:
            for t in (ws.view(torch.int16), *got):
                t.fill_(-1)
        torch.cuda.synchronize()
        begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        begin.record()
        for inputs, ws, got, _, stream in calls:
            stream.wait_event(begin)
            rc = lib.fused_mha_backward(*(t.data_ptr() for t in inputs), ws.data_ptr(), nbytes, *(g.data_ptr() for g in got),
                                        1, H, N, N, D, D ** -0.5, int(causal), stream.cuda_stream)
            assert rc == abi.OK
        for *_, stream in calls:
            torch.cuda.current_stream().wait_stream(stream)
        end.record()
        torch.cuda.synchronize()
        for _, ws, got, want, _ in calls:
            assert (ws[-128 * H:].view(torch.int32).view(H, 32)[:, 0] == 4 * (-(-N // 128))).all()  # the launch with counts
            for a, b in zip(got, want):
                assert torch.equal(a, b)
        assert begin.elapsed_time(end) < 20  # ms; about 1.5 each


EITHER_MFMA = [1, 15, 16, 17, 32, 49, 64, 79, 128, 129, 200]


def _slices_of_a_busy_launch(N, causal, cus):
    blocks = cus if causal else -(-5 * cus // 8)
    return blocks // (-(-N // 128)) + 1


def test_mfmas_of_the_cases_below(tmp_path):
    """16 x 16 ones for the whole launch and 32 x 32 ones for a slice of it, on 256 compute units."""
    wide = "fmha_wide_mfmas((long)((x[0] + 127) / 128) * x[1], 256, x[2])"
    cases = [(N, _slices_of_a_busy_launch(N, causal, 256), causal) for N in EITHER_MFMA for causal in (False, True)]
    assert not any(abi.host_rule(tmp_path, wide, cases))
    assert all(abi.host_rule(tmp_path, wide, [(N, 1, causal) for N, _, causal in cases]))


@pytest.mark.gpu
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("N", EITHER_MFMA)
def test_backward_d128_with_either_mfma(N, causal):
    """A launch that has just enough blocks takes the passes with 16 x 16 MFMAs, a slice of it those with 32 x 32 ones: the
    same bits, with and without the workspace for dS.  The passes are called one by one: together, launches of this size
    go in one."""
    D, lib = 128, abi.load()
    H = _slices_of_a_busy_launch(N, causal, torch.cuda.get_device_properties(0).multi_processor_count)
    gen = torch.Generator(device="cuda").manual_seed(N)
    q, k, v, do = (torch.randn(1, N, H, D, device="cuda", dtype=torch.float16, generator=gen) for _ in range(4))
    out, lse = abi.forward(lib, q, k, v, D ** -0.5, causal)
    for least in (False, True):
        whole = abi.backward(lib, q, k, v, out, do, lse, D ** -0.5, causal, min_workspace=least, split=True)[:3]
        for h in (0, H - 1):
            one = [t[:, :, h:h + 1].contiguous() for t in (q, k, v, out, do)]
            alone = abi.backward(lib, *one, lse[:, h:h + 1].clone(), D ** -0.5, causal, min_workspace=least, split=True)[:3]
            for a, b in zip(alone, whole):
                assert torch.equal(a, b[:, :, h:h + 1])


@pytest.mark.gpu
@pytest.mark.parametrize("N", [129, 143, 159, 160, 161, 192, 193, 257, 288, 321, 385, 416])
def test_backward_d128_short_last_block_of_keys(N):
    """Up to 32 keys past a multiple of 128 are shared by all pairs of waves of a block, more are not; the last tile of queries
    is one row to a whole one.  The workspace holds NaN where nothing is written."""
    B, H, D = 1, 5, 128
    q, k, v, do = ao.make_inputs(B, N, H, D, seed=13)
    lib, scale = abi.load(), D ** -0.5
    qg, kg, vg, dog = (t.cuda() for t in (q, k, v, do))
    out, lse = abi.forward(lib, qg, kg, vg, scale, False)
    ref = ao.attention_backward(q, k, v, do, scale, False)
    least = abi.backward(lib, qg, kg, vg, out, dog, lse, scale, False, min_workspace=True)[:3]
    split = abi.backward(lib, qg, kg, vg, out, dog, lse, scale, False, split=True, poison=True)[:3]
    many = [t.repeat(1, 1, 60, 1) for t in (qg, kg, vg, out, dog)]  # enough slices for the passes over dS
    spill = abi.backward(lib, *many, lse.repeat(1, 60, 1), scale, False, poison=True)[:3]
    for i, want in enumerate(ref):
        for got in (least[i], split[i], spill[i][:, :, :H], spill[i][:, :, -H:]):
            # fp16 roundings of P, dS, delta's O and the result: the repository's bound for gradients of order 1
            assert (got.float().cpu() - want.half().float()).abs().max() <= 1e-2
            assert torch.equal(got, least[i])


LAST_ROUND = [  # H, N, D, whether fused_mha_backward goes in one launch
    (65, 1024, 64, True), (57, 1031, 64, True),      # 520 and 513 blocks on 512 places
    (65, 1024, 128, False), (57, 1031, 128, False),  # the forward alone
    (90, 1024, 64, False), (75, 1031, 64, False),    # 720 and 675
    (129, 1024, 64, False), (128, 1025, 64, False),  # 1032 blocks, and 1152, whose last ones have one row each
]


def test_launches_of_the_cases_below(tmp_path):
    """On 256 compute units, and that the passes' own launches have at most half a round behind full ones."""
    once = "fmha_passes_at_once(x[2], (long)((x[1] + 127) / 128) * x[0], x[1], 256, 0)"
    assert abi.host_rule(tmp_path, once, LAST_ROUND) == [c[3] for c in LAST_ROUND]
    for H, N, D, _ in LAST_ROUND:
        if D == 64:
            rounds, left = divmod(H * -(-N // 128), 512)
            assert 1 <= rounds < 3 and 0 < left <= 256


@pytest.mark.gpu
@pytest.mark.parametrize("H,N,D,once", LAST_ROUND)
def test_a_nearly_empty_last_round(H, N, D, once):
    """Launches in which every other wave slot goes first: the bits of a slice alone, which has no second round.  The
    passes of the D = 64 backward take them one by one, and together unless all of it goes in one launch."""
    lib = abi.load()
    gen = torch.Generator(device="cuda").manual_seed(N + H)
    q, k, v, do = (torch.randn(1, N, H, D, device="cuda", dtype=torch.float16, generator=gen) for _ in range(4))
    out, lse = abi.forward(lib, q, k, v, D ** -0.5, False)
    whole = [out] + list(abi.backward(lib, q, k, v, out, do, lse, D ** -0.5, False)[:3])
    split = [out] + list(abi.backward(lib, q, k, v, out, do, lse, D ** -0.5, False, split=True)[:3])
    for h in (0, H // 2, H - 1):
        q1, k1, v1, do1 = (t[:, :, h:h + 1].contiguous() for t in (q, k, v, do))
        out1, lse1 = abi.forward(lib, q1, k1, v1, D ** -0.5, False)
        alone = [out1] + list(abi.backward(lib, q1, k1, v1, out1, do1, lse1, D ** -0.5, False)[:3])
        assert torch.equal(lse1, lse[:, h:h + 1])
        for a, b, c in zip(alone, whole, split):
            assert torch.equal(a, b[:, :, h:h + 1]) and torch.equal(a, c[:, :, h:h + 1])


DS_IN_ONE_CALL = [(260, 300), (130, 600), (50, 300), (100, 300)]  # H, N: dS is stored, without a mask or under one


def test_dS_in_one_call(tmp_path):
    """Of the cases below on 256 compute units, and that it is by passes with 32 x 32 MFMAs too, though never under a mask."""
    at_once = "fmha_passes_at_once(128, (long)((x[1] + 127) / 128) * x[0], x[1], 256, x[2])"
    wide = "fmha_wide_mfmas((long)((x[1] + 127) / 128) * x[0], 256, x[2])"
    no_mask, causal = ([(*case, mask) for case in DS_IN_ONE_CALL] for mask in (0, 1))
    assert abi.host_rule(tmp_path, at_once, no_mask) == [False] * 4
    assert abi.host_rule(tmp_path, at_once, causal) == [False, False, True, False]
    assert abi.host_rule(tmp_path, wide, no_mask) == [False, False, True, False]
    every = [(H, N, 1) for N in (1, 20, 40, 64, 65, 128, 129, 200, 256, 257, 1031, 4096) for H in range(1, 600)]
    assert not any(abi.host_rule(tmp_path, f"!{at_once} && {wide}", every))


@pytest.mark.gpu
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("H,N", [(3, n) for n in (1, 32, 33, 64, 65, 96, 97, 128, 129, 257, 320)] + DS_IN_ONE_CALL)
def test_dq_ignores_dS_that_no_query_needs(H, N, causal):
    """The workspace holds NaN where the dK/dV pass writes nothing.  dQ is that of the recomputing path, bit for bit.  By the
    passes one by one, which store dS in every case."""
    D, lib = 128, abi.load()
    gen = torch.Generator(device="cuda").manual_seed(N)
    q, k, v, do = (torch.randn(1, N, H, D, device="cuda", dtype=torch.float16, generator=gen) for _ in range(4))
    out, lse = abi.forward(lib, q, k, v, D ** -0.5, causal)
    want = abi.backward(lib, q, k, v, out, do, lse, D ** -0.5, causal, min_workspace=True)[:3]
    for split in (True, False):  # H = 3 one by one: 32 x 32 MFMAs
        got = abi.backward(lib, q, k, v, out, do, lse, D ** -0.5, causal, split=split, poison=True)[:3]
        for a, b in zip(got, want):
            assert torch.equal(a, b)


HINT_ON_DS = [  # H, N, causal, whether the passes are called one by one, whether dS is told to be used once
    (127, 256, False, False, True), (128, 256, False, False, False),   # 15.9 and 16 MiB of dS
    (511, 127, False, True, True), (512, 127, False, True, False),
    (56, 384, False, False, True), (57, 384, False, False, False),     # 15.8 and 16.03
    (511, 50, True, True, True), (513, 50, True, False, False),        # 7.98 and 8.02 MiB
    (513, 50, True, True, False),                                      # one by one: whole, it has a work group for each slice
    (4, 1024, False, True, True), (5, 1024, False, True, False),       # 8 and 10 MiB
    (5, 1025, True, True, True), (9, 1025, True, True, False),         # 6.3 and 11.4 MiB
    (63, 1031, False, False, False), (64, 1031, False, False, True),   # 255 and 259 MiB of dS and tensors
    (71, 1031, True, False, False), (106, 1031, True, False, True),    # 197 and 294 MiB
]


def test_hint_on_ds_cases(tmp_path):
    """The cases below store dS on 256 compute units, with the hint or without as they say."""
    once = "fmha_passes_at_once(128, (long)((x[1] + 127) / 128) * x[0], x[1], 256, x[2])"
    ds = "(unsigned long)x[0] * ((x[1] + 127) / 128 * 128) * ((x[1] + 127) / 128 * 128) * 2 / (x[2] ? 2 : 1)"
    hint = f"fmha_ds_used_once({ds}, {ds} + 6ul * x[0] * x[1] * 256, x[1], x[2])"
    assert not any(abi.host_rule(tmp_path, once, [c[:3] for c in HINT_ON_DS if not c[3]]))
    assert abi.host_rule(tmp_path, hint, HINT_ON_DS) == [c[4] for c in HINT_ON_DS]


@pytest.mark.gpu
@pytest.mark.parametrize("H,N,causal,one_by_one,hint", HINT_ON_DS)
def test_hint_on_the_stores_of_ds(H, N, causal, one_by_one, hint):
    """Both sides of the lines between dS stored with and without the hint: the gradients of the recomputing path."""
    D, lib = 128, abi.load()
    gen = torch.Generator(device="cuda").manual_seed(N + H)
    q, k, v, do = (torch.randn(1, N, H, D, device="cuda", dtype=torch.float16, generator=gen) for _ in range(4))
    out, lse = abi.forward(lib, q, k, v, D ** -0.5, causal)
    want = abi.backward(lib, q, k, v, out, do, lse, D ** -0.5, causal, min_workspace=True)
    got = abi.backward(lib, q, k, v, out, do, lse, D ** -0.5, causal, split=one_by_one)
    for a, b in zip(got[:3], want[:3]):
        assert torch.equal(a, b)


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
    for a, b in zip(*grads):
        assert torch.equal(a, b)


def _workspace_and_grads(leaves, out, do):
    """Gradients and the bytes that the backward held at its height beside them."""
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    grads = torch.autograd.grad(out, leaves, do, retain_graph=True)
    return torch.cuda.max_memory_allocated() - before - sum(g.numel() * 2 for g in grads), grads


@pytest.mark.gpu
def test_backward_leaves_the_rest_of_the_memory_alone():
    """Past 16 GiB of dS (17 here) the backward takes rounds of 8 GiB where the memory is there, smaller ones where half
    of what is left does not hold those, none of it where that is not worth it, and never makes the allocator give back
    what it has cached."""
    from flash_attn_v100 import flash_attn_func
    B, H, N, D = 1, 34, 16384, 128
    gen = torch.Generator(device="cuda").manual_seed(3)
    q, k, v, do = (torch.randn(B, N, H, D, device="cuda", dtype=torch.float16, generator=gen) for _ in range(4))
    leaves = [t.requires_grad_() for t in (q, k, v)]
    out = flash_attn_func(*leaves, causal=True)
    total, results = torch.cuda.get_device_properties(0).total_memory, []
    for left, slices in ((None, 16), (7 << 30, 6), (1 << 30, 0)):
        torch.cuda.empty_cache()
        cached = [torch.empty(64 << 20, dtype=torch.uint8, device="cuda") for _ in range(4)]
        del cached
        stats = torch.cuda.memory_stats()
        try:
            if left:
                grads = 3 * q.numel() * 2
                torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + grads + left) / total)
            took, got = _workspace_and_grads(leaves, out, do)
        finally:
            torch.cuda.set_per_process_memory_fraction(1.0)
        after = torch.cuda.memory_stats()
        assert after["num_alloc_retries"] == stats["num_alloc_retries"] and after["num_ooms"] == stats["num_ooms"]
        assert after["reserved_bytes.all.current"] >= stats["reserved_bytes.all.current"]
        assert abs(took - slices * N * N * 2 - 2 * H * N * 4) <= 16 << 20  # the allocator rounds up
        results.append(got)
    for got in results[1:]:
        for a, b in zip(got, results[0]):
            assert torch.equal(a, b)


@pytest.mark.gpu
def test_backward_takes_a_cached_workspace_again():
    """What the allocator has cached is taken although nothing is left of the process's share."""
    from flash_attn_v100 import flash_attn_func
    B, H, N, D = 1, 10, 8192, 128  # 1.25 GiB of dS
    gen = torch.Generator(device="cuda").manual_seed(5)
    q, k, v, do = (torch.randn(B, N, H, D, device="cuda", dtype=torch.float16, generator=gen) for _ in range(4))
    leaves = [t.requires_grad_() for t in (q, k, v)]
    out = flash_attn_func(*leaves, causal=True)
    torch.cuda.empty_cache()
    took, grads = _workspace_and_grads(leaves, out, do)
    first = [g.cpu() for g in grads]
    del grads  # their blocks serve the second call's
    try:
        torch.cuda.set_per_process_memory_fraction(torch.cuda.memory_reserved() /
                                                   torch.cuda.get_device_properties(0).total_memory)
        took_again, grads = _workspace_and_grads(leaves, out, do)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert took == took_again > 1 << 30
    for a, b in zip(first, grads):
        assert torch.equal(a, b.cpu())


@pytest.mark.gpu
def test_capture_with_a_large_workspace():
    """A graph capture takes its memory from a pool of its own: 1 GiB of dS there, the eager result on every replay."""
    from flash_attn_v100 import flash_attn_func
    B, H, N, D = 1, 8, 8192, 128
    static = [torch.zeros(B, N, H, D, dtype=torch.float16, device="cuda") for _ in range(4)]
    leaves = [t.requires_grad_() for t in static[:3]]

    def step():
        return torch.autograd.grad(flash_attn_func(*leaves, causal=True), leaves, static[3])

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = step()
    for seed in (1, 2, 3):
        gen = torch.Generator(device="cuda").manual_seed(seed)
        with torch.no_grad():
            for t in static:
                t.copy_(torch.randn(t.shape, device="cuda", dtype=torch.float16, generator=gen))
        graph.replay()
        torch.cuda.synchronize()
        replayed = [t.clone() for t in captured]
        eager = step()
        torch.cuda.synchronize()
        for a, b in zip(replayed, eager):
            assert torch.equal(a, b)

@pytest.mark.gpu
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("B,H,N", [
    (3, 5, 1), (67, 3, 1), (9, 7, 2), (5, 1, 7), (2, 5, 15), (2, 3, 16), (3, 3, 17),  # blocks with rows of many slices and batches
    (2, 3, 31), (2, 3, 32), (3, 2, 33), (2, 4, 100), (1, 3, 1031), (2, 8, 512),
])
def test_row_statistics(B, H, N, D):
    """delta and lse * log2(e) of every row, whatever rows share a block, and nothing behind them."""
    lib = abi.load()
    gen = torch.Generator(device="cuda").manual_seed(B * H * N)
    out, do = (torch.randn(B, N, H, D, device="cuda", dtype=torch.float16, generator=gen) for _ in range(2))
    lse = torch.randn(B, H, N, device="cuda", generator=gen)
    nbytes, rows = lib.fused_mha_backward_min_workspace_bytes(B, H, N, D), B * H * N
    ws = torch.full((nbytes // 4 + 64,), float("nan"), device="cuda")
    assert lib.fused_mha_backward_delta(out.data_ptr(), do.data_ptr(), lse.data_ptr(), ws.data_ptr(), nbytes, B, H, N, D,
                                        torch.cuda.current_stream().cuda_stream) == abi.OK
    products = (out.double() * do.double()).permute(0, 2, 1, 3)
    error = (ws[:rows].view(B, H, N) - products.sum(-1)).abs()
    assert (error <= D * 2.0 ** -24 * products.abs().sum(-1)).all()  # D roundings of partial sums in fp32
    want = lse.double() / torch.log(torch.tensor(2.0, dtype=torch.float64))
    assert ((ws[rows:2 * rows].view(B, H, N) - want).abs() <= 2.0 ** -22 * want.abs()).all()  # the constant's and the product's
    assert nbytes == 8 * rows and torch.isnan(ws[2 * rows:]).all()


def test_blocks_of_two_passes_are_a_bijection(tmp_path):
    """csrc/block_map.h, compiled for the host: every block of either pass once, whole slices on one XCD, heavy blocks first or
    short ones last; and launches of both passes at once stay within the number of threads that a launch can have."""
    src = tmp_path / "check.cpp"
    src.write_text(r'''
#include <cstdio>
#include <vector>
#include "block_map.h"
int main() {
  for (int slices = 1; slices <= 300; slices += (slices < 80 ? 1 : 7))
    for (int nb : {1, 2, 3, 8, 33})
      for (int mode = 0; mode < 3; ++mode) {
        const bool heavy = mode == 0, short_last = mode == 1;
        const int total = 2 * slices * nb;
        std::vector<int> seen(total, 0), xcd(slices, -1);
        int prev = 0, drops = 0;
        for (int lin = 0; lin < total; ++lin) {
          int s = -1, b = -1;
          bool second = false;
          fmha_two_pass_block(lin, slices, nb, heavy, short_last, s, b, second);
          if (s < 0 || s >= slices || b < 0 || b >= nb || seen[2 * (s * nb + b) + second]++) {
            printf("map %d %d %d %d\n", slices, nb, mode, lin);
            return 1;
          }
          if (!short_last && s < (slices & ~7)) {
            if (xcd[s] >= 0 && xcd[s] != (lin & 7)) { printf("xcd %d %d\n", slices, nb); return 1; }
            xcd[s] = lin & 7;
          }
          if (short_last && (b == nb - 1) != (lin >= 2 * slices * (nb - 1))) { printf("short %d %d\n", slices, nb); return 1; }
          drops += heavy && b < prev;
          prev = b;
        }
        if (heavy && drops > slices / 64) { printf("order %d %d\n", slices, nb); return 1; }
      }
  for (int causal = 0; causal < 4; ++causal)
    for (int n = 1; n <= 8192; n = n < 600 ? n + 1 : n * 2)
      for (long slices = 1; slices < 1 << 23; slices += 1 + slices / 9) {
        const long blocks = slices * ((n + 127) / 128);
        if (fmha_passes_at_once(causal & 2 ? 64 : 128, blocks, n, 256, causal & 1) && 2 * blocks * 512 >= 1L << 32) { printf("threads %d\n", n); return 1; }
      }
  puts("ok");
  return 0;
}
''')
    exe = tmp_path / "check"
    inc = os.path.join(abi.ROOT, "flash-attention-v100_amd", "csrc")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-I", inc, str(src), "-o", str(exe)])
    assert subprocess.check_output([str(exe)]).decode().strip() == "ok"


def test_one_launch_only_where_it_is_worth_it(tmp_path):
    """D, N, slices, causal of launches timed both ways on 256 compute units."""
    rule = "fmha_passes_at_once(x[0], (long)((x[1] + 127) / 128) * x[2], x[1], 256, x[3])"
    apart = [
        (128, 77, 520, 0), (128, 128, 513, 0), (128, 140, 128, 0), (128, 140, 68, 0),
        (128, 200, 198, 0), (128, 257, 89, 0), (128, 1031, 20, 0), (128, 300, 90, 1), (128, 200, 218, 1), (128, 33, 520, 0),
        (64, 64, 3584, 0), (64, 80, 2560, 0), (64, 5, 5120, 0), (64, 512, 128, 0), (64, 5, 8192, 1),
    ]
    at_once = [
        (128, 33, 256, 0), (128, 64, 256, 0), (128, 64, 512, 0), (128, 110, 128, 0), (128, 100, 448, 0), (128, 77, 384, 0),
        (128, 128, 141, 0), (128, 128, 512, 0), (128, 140, 166, 0), (128, 180, 192, 0), (128, 256, 192, 0), (128, 64, 512, 1),
        (128, 40, 486, 1), (128, 200, 192, 1), (128, 1031, 28, 1), (128, 1031, 14, 0),
        (64, 48, 512, 0), (64, 64, 512, 0), (64, 80, 448, 0), (64, 120, 512, 0), (64, 128, 512, 0), (64, 24, 3800, 0),
        (64, 64, 2400, 0), (64, 128, 2048, 0), (64, 204, 256, 0), (64, 512, 96, 0), (64, 1, 4096, 1), (64, 140, 900, 1),
        (64, 1024, 64, 1),
    ]
    assert not any(abi.host_rule(tmp_path, rule, apart))
    assert all(abi.host_rule(tmp_path, rule, at_once))
    without_room = rule.replace("x[3])", "x[3], false)")  # for dS
    at_once = [(128, 300, 90, 0), (128, 512, 96, 0), (128, 1031, 42, 0), (128, 4096, 9, 0)]
    apart = [(128, 110, 520, 0), (128, 230, 256, 0), (128, 1024, 20, 0), (128, 1024, 50, 0), (128, 4096, 15, 0)]
    assert not any(abi.host_rule(tmp_path, rule, at_once))
    assert all(abi.host_rule(tmp_path, without_room, at_once))
    assert not any(abi.host_rule(tmp_path, without_room, apart))


ONE_LAUNCH = {  # B, H, N, causal by head size and by what fused_mha_backward does
    (64, "one launch, statistics made by the blocks"): [
        (1, 1, 1, False), (3, 5, 64, True), (2, 3, 65, False), (1, 3, 512, False), (2, 4, 511, True), (1, 5, 1024, True),
        (16, 40, 129, False), (1, 70, 1000, True), (1, 480, 60, False), (1, 900, 127, False), (1, 250, 193, False),
        (1, 512, 64, False), (1, 500, 65, False),
    ],
    (64, "one launch behind the kernel for the statistics"): [
        (1, 3, 513, False), (2, 2, 1025, True), (1, 5, 1031, False), (1, 3, 1536, True), (3, 20, 1031, False),
    ],
    (64, "the passes one after the other"): [
        (1, 64, 1024, False), (1, 130, 1024, True), (1, 800, 256, False), (1, 3900, 33, False), (1, 2600, 64, False),
        (1, 2600, 65, False), (1, 800, 193, False), (1, 3100, 65, True), (1, 600, 511, True), (1, 120, 1031, True),
    ],
    (128, "one launch, statistics made by the blocks"): [
        (1, 1, 1, True), (3, 5, 33, False), (2, 3, 64, True), (2, 3, 65, False), (1, 100, 128, True), (3, 100, 77, False),
        (2, 30, 255, False), (1, 70, 256, True), (1, 140, 256, False), (3, 7, 384, True), (1, 9, 321, False),
        (5, 100, 64, True), (1, 140, 250, False), (1, 400, 33, False), (1, 400, 40, True), (1, 150, 65, False),
        (1, 140, 128, False), (1, 396, 128, False), (1, 192, 160, False), (5, 100, 77, False), (1, 400, 65, False),
    ],
    (128, "one launch behind the kernel for the statistics"): [
        (1, 3, 385, False), (2, 2, 1031, True), (1, 9, 1031, False), (1, 30, 1000, True), (1, 2, 2049, False),
    ],
    (128, "the passes one after the other"): [
        (6, 100, 77, False), (1, 70, 250, False), (1, 70, 400, True), (1, 20, 1031, False), (1, 520, 33, False),
        (1, 513, 64, True), (1, 520, 40, True), (1, 520, 65, False), (1, 520, 128, False), (1, 200, 200, False),
        (1, 90, 300, False), (1, 31, 1031, False),  # one launch without room for dS
    ],
}


def test_launches_of_the_backward(tmp_path):
    """The cases below on 256 compute units."""
    shape = "x[0], (long)((x[3] + 127) / 128) * x[1] * x[2], x[3], 256, x[4]"
    for (D, what), cases in ONE_LAUNCH.items():
        cases = [(D, *case) for case in cases]
        assert abi.host_rule(tmp_path, f"fmha_passes_at_once({shape})", cases) == [what.startswith("one launch")] * len(cases)
        if what.startswith("one launch"):
            blocks = abi.host_rule(tmp_path, "fmha_blocks_make_stats(x[0], x[3], x[4])", cases)
            assert blocks == [what.endswith("by the blocks")] * len(cases)


@pytest.mark.gpu
@pytest.mark.parametrize("D,B,H,N,causal", [(D, *case) for (D, _), cases in ONE_LAUNCH.items() for case in cases])
def test_backward_in_one_launch(D, B, H, N, causal):
    """Whatever goes in one launch, gradients and delta are those of the passes one by one, bit for bit, also with strides
    and with the least workspace (at D = 128 the passes one by one store dS, the launch forms it twice)."""
    lib = abi.load()
    scale = D ** -0.5
    gen = torch.Generator(device="cuda").manual_seed(N + H)
    packed = torch.randn(B, N, 4, H, D, device="cuda", dtype=torch.float16, generator=gen)
    dense = [packed[:, :, i].contiguous() for i in range(4)]
    out, lse = abi.forward(lib, *dense[:3], scale, causal)
    want = abi.backward(lib, *dense[:3], out, dense[3], lse, scale, causal, split=True)
    got = abi.backward(lib, *dense[:3], out, dense[3], lse, scale, causal)
    strided = abi.backward_strided(lib, *(packed[:, :, i] for i in range(3)), out, packed[:, :, 3], lse, scale, causal)
    least = abi.backward(lib, *dense[:3], out, dense[3], lse, scale, causal, min_workspace=True)
    for a, b, c, d in zip(got, want, strided, least):
        assert torch.equal(a, b) and torch.equal(c, b) and torch.equal(d, b)
    assert torch.equal(got[3], want[3]) and torch.equal(least[3], want[3])

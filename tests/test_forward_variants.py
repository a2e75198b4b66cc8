"""The forward's work-group order, on the CPU, and its two kernels at the sizes where they can go wrong, on the GPU."""
import os
import subprocess

import pytest
import torch

import abi
from oracle import attention_oracle as ao


def test_scheduled_blocks_are_a_bijection(tmp_path):
    """csrc/block_map.h, compiled for the host: every (slice, block) once for any slice count, whole slices on one XCD
    up to slices % 8 of them, and (heavy_first) block indices that never fall inside a group of slices."""
    src = tmp_path / "check.cpp"
    src.write_text(r'''
#include <cstdio>
#include <vector>
#include "block_map.h"
int main() {
  for (int slices = 1; slices <= 300; slices += (slices < 150 ? 1 : 7))
    for (int bps : {1, 2, 3, 5, 8, 12, 33})
      for (int mode = 0; mode < 3; ++mode) {
        const bool heavy = mode == 0, short_last = mode == 1;
        const int total = slices * bps;
        std::vector<int> seen(total, 0), xcd(slices, -1);
        int prev = 0, drops = 0;
        for (int lin = 0; lin < total; ++lin) {
          int s = -1, b = -1;
          fmha_scheduled_block(lin, slices, bps, heavy, short_last, s, b);
          if (s < 0 || s >= slices || b < 0 || b >= bps || seen[s * bps + b]++) { printf("map %d %d %d %d\n", slices, bps, mode, lin); return 1; }
          if (heavy && s < (slices & ~7)) {
            if (xcd[s] >= 0 && xcd[s] != (lin & 7)) { printf("xcd %d %d\n", slices, bps); return 1; }
            xcd[s] = lin & 7;
          }
          if (short_last && (b == bps - 1) != (lin >= slices * (bps - 1))) { printf("short %d %d\n", slices, bps); return 1; }
          drops += heavy && b < prev;
          prev = b;
        }
        if (heavy && drops > slices / 64) { printf("order %d %d\n", slices, bps); return 1; }
      }
  puts("ok");
  return 0;
}
''')
    exe = tmp_path / "check"
    inc = os.path.join(abi.ROOT, "flash-attention-v100_amd", "csrc")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-I", inc, str(src), "-o", str(exe)])
    assert subprocess.check_output([str(exe)]).decode().strip() == "ok"


def test_paired_blocks_are_a_bijection(tmp_path):
    """csrc/block_map.h: every block once and on the same XCD for any number of blocks, and with two blocks to a CU those
    that share one weigh the same together."""
    src = tmp_path / "check.cpp"
    src.write_text(r'''
#include <cstdio>
#include <vector>
#include "block_map.h"
int main() {
  for (int total = 1; total <= 1100; ++total) {
    std::vector<int> seen(total, 0);
    for (int lin = 0; lin < total; ++lin) {
      const int at = fmha_paired_block(lin, total);
      if (at < 0 || at >= total || seen[at]++ || (at & 7) != (lin & 7)) { printf("%d of %d\n", lin, total); return 1; }
      if ((lin < kCus || lin >= 2 * kCus) && at != lin) { printf("moved %d of %d\n", lin, total); return 1; }
    }
  }
  for (int w = 0; w < kCus; ++w)
    if ((w >> 3) + (fmha_paired_block(w + kCus, 2 * kCus) >> 3) != 2 * kCus / 8 - 1) { printf("pair %d\n", w); return 1; }
  puts("ok");
  return 0;
}
''')
    exe = tmp_path / "check"
    inc = os.path.join(abi.ROOT, "flash-attention-v100_amd", "csrc")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-I", inc, str(src), "-o", str(exe)])
    assert subprocess.check_output([str(exe)]).decode().strip() == "ok"


def _persistent(tmp_path, shapes):
    """Which of the (slices, N, causal) problems the 256-query kernel takes."""
    return abi.host_rule(tmp_path, "fmha_persistent_forward_pays(x[0], x[1], 256, x[2])", shapes)


def test_rule_between_the_forward_kernels(tmp_path):
    """Causal launches with even shares: by the length alone, however many rounds they have.  Without a mask: by the last
    round."""
    pairs = [(n, 512 // (-(-n // 256)) * k) for n in (1024, 2048, 4095, 4096, 8001, 8192, 16384) for k in range(1, 9)]
    assert all(slices % 8 == 0 for _, slices in pairs)
    assert _persistent(tmp_path, [(slices, n, True) for n, slices in pairs]) == [n >= 4096 for n, _ in pairs]
    uneven = [(60, 2048), (60, 4096), (128, 4100), (64, 5120), (64, 7168), (4, 32768)]
    assert not any(_persistent(tmp_path, [(s, n, True) for s, n in uneven]))
    taken = [(64, 4096), (25, 4096), (42, 4096), (13, 8192), (30, 2048), (32, 1500), (128, 512), (256, 256)]
    left = [(24, 4096), (56, 4096), (84, 4096), (100, 4096), (28, 8192), (42, 8192), (84, 1152), (120, 1031), (224, 1024)]
    assert all(_persistent(tmp_path, [(s, n, False) for s, n in taken]))
    assert not any(_persistent(tmp_path, [(s, n, False) for s, n in left]))


def _inputs(B, N, H, D, growing):
    """growing: the score scale rises with the key index, so that nearly every 64-key tile holds a maximum that is
    more than 2^12 times (12 in the exp2 domain) above the earlier ones and the running maximum is raised in it."""
    q, k, v, _ = ao.make_inputs(B, N, H, D, seed=7)
    if growing:
        q = q.abs() * 0.25
        k = (k.abs() * 0.5 + torch.arange(N).view(1, N, 1, 1) // 64 * (60.0 / D)).half()
        q = q.half()
    return q, k, v


def _check(B, N, H, D, causal, growing, heads=None):
    q, k, v = _inputs(B, N, H, D, growing)
    out, lse = abi.forward(abi.load(), q.cuda(), k.cuda(), v.cuda(), D ** -0.5 if not growing else 1.0, causal)
    assert torch.isfinite(out).all() and torch.isfinite(lse).all()
    pick = list(range(H)) if heads is None else heads
    ref, ref_lse = ao.attention_forward(q[:, :, pick], k[:, :, pick], v[:, :, pick],
                                        D ** -0.5 if not growing else 1.0, causal)
    # the repository's bounds: fp16 probabilities and results for O of order 1, fp32 sums for the logsumexp (relative
    # to its size: a score of size s carries the fp32 rounding of D products of size s, below 2^-20 s)
    assert (out[:, :, pick].float().cpu() - ref.half().float()).abs().max() <= 2e-3 * max(1.0, ref.abs().max().item())
    assert ((lse[:, pick].cpu() - ref_lse).abs() <= 2e-3 + 1e-6 * ref_lse.abs()).all()


@pytest.mark.gpu
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("N", [1, 32, 33, 64, 65, 96, 128, 129, 192, 193, 256, 257, 320, 449])
def test_small_blocks(N, causal, D):
    for growing in (False, True):
        _check(1, N, 3, D, causal, growing)


PERSISTENT = [  # B, H, N, causal: launches of the 256-query kernel
    (5, 17, 700, False), (1, 256, 250, False),  # 255 and 256 blocks
    (1, 32, 4096, True), (1, 16, 8001, True),   # one pair of blocks per compute unit
]
FULL = [  # launches of the other kernel with as many queries
    (1, 63, 2000, True),                        # 504 blocks of 256: no even shares
    (1, 32, 3900, True), (1, 64, 2048, True),   # even ones, too short
]


def test_shapes_take_the_kernel_they_are_meant_for(tmp_path):
    """On 256 compute units."""
    several = [(2, 32, 4096, True), (1, 32, 8001, True)]
    assert all(_persistent(tmp_path, [(B * H, N, causal) for B, H, N, causal in PERSISTENT + several] +
                           [(H, N, causal) for H, N, causal in MANY_ROUNDS] +
                           [(B * H, N, causal) for B, H, N, _, causal in NOT_FINITE_PERSISTENT]))
    assert not any(_persistent(tmp_path, [(B * H, N, causal) for B, H, N, causal in FULL + [(1, 61, 4099, True)]]))


@pytest.mark.gpu
@pytest.mark.parametrize("B,H,N,causal", PERSISTENT + FULL)
def test_persistent_blocks(B, H, N, causal):
    """Launches the persistent kernel takes and such that it nearly takes."""
    for growing in (False, True):
        _check(B, N, H, 128, causal, growing, heads=[0, H // 2, H - 1])


MANY_ROUNDS = [
    (26, 2048, False), (25, 4096, False), (44, 1153, False), (37, 1500, False),  # last rounds of 208, 144, 220 and 222 blocks
    (48, 8192, True), (24, 16384, True), (96, 4096, True),                       # three pairs of rounds of work groups
]


@pytest.mark.gpu
@pytest.mark.parametrize("H,N,causal", MANY_ROUNDS)
def test_a_slice_alone_where_the_last_round_is_half_full(H, N, causal):
    """The persistent kernel without even shares and with many rounds: the bits of the 128-query kernel, which takes a slice
    alone."""
    D, lib = 128, abi.load()
    gen = torch.Generator(device="cuda").manual_seed(N + H)
    q, k, v = (torch.randn(1, N, H, D, device="cuda", dtype=torch.float16, generator=gen) for _ in range(3))
    out, lse = abi.forward(lib, q, k, v, D ** -0.5, causal)
    for h in (0, H // 2, H - 1):
        one = [t[:, :, h:h + 1].contiguous() for t in (q, k, v)]
        out1, lse1 = abi.forward(lib, *one, D ** -0.5, causal)
        assert torch.equal(out1, out[:, :, h:h + 1]) and torch.equal(lse1, lse[:, h:h + 1])


@pytest.mark.gpu
@pytest.mark.parametrize("B,H,N,causal", PERSISTENT + FULL + [
    (2, 32, 4096, True),   # two pairs of blocks per compute unit: persistent
    (1, 61, 4099, True),   # 17 blocks a slice, the last one of three queries
    (1, 32, 8001, True),   # two pairs, with a ragged end: persistent
])
def test_a_slice_alone_gives_the_same_bits(B, H, N, causal):
    """One slice has too few blocks for the persistent kernel, the whole problem takes it (or the other one: then there
    is nothing to tell apart)."""
    lib = abi.load()
    for growing in (False, True):
        q, k, v = (t.cuda() for t in _inputs(B, N, H, 128, growing))
        scale = 1.0 if growing else 128 ** -0.5
        out, lse = abi.forward(lib, q, k, v, scale, causal)
        for b, h in ((0, 0), (B - 1, H - 1), (B // 2, H // 2)):
            one = [t[b:b + 1, :, h:h + 1].contiguous() for t in (q, k, v)]
            o1, l1 = abi.forward(lib, *one, scale, causal)
            assert torch.equal(o1, out[b:b + 1, :, h:h + 1]) and torch.equal(l1, lse[b:b + 1, h:h + 1])


NOT_FINITE_PERSISTENT = [(5, 17, 700, 128, False), (1, 32, 4096, 128, True), (1, 16, 8001, 128, True)]


@pytest.mark.gpu
@pytest.mark.parametrize("B,H,N,D,causal", NOT_FINITE_PERSISTENT + [
    (1, 3, 449, 64, False), (1, 3, 449, 64, True), (1, 3, 449, 128, False), (1, 3, 449, 128, True), (1, 64, 2048, 128, True),
    (1, 200, 449, 64, False), (1, 256, 449, 64, True), (1, 130, 150, 128, False), (1, 130, 200, 128, True),  # a work group per slice
])
def test_rows_that_are_not_finite(B, H, N, D, causal):
    """Queries with a NaN or an infinity give NaN rows and make their wave raise its maximum at every tile; the finite rows
    beside them, in the forward and in dQ, stay within the usual bounds, and other heads keep their bits."""
    bad = [5, 40, 41, N - 1]
    q, k, v, do = ao.make_inputs(B, N, H, D, seed=9)
    lib, scale, h = abi.load(), D ** -0.5, 1
    clean = q.clone()
    q[:, bad[:2], h, 3] = float("nan")
    q[:, bad[2:], h, 7] = float("inf")
    qg, kg, vg, dog = (t.cuda() for t in (q, k, v, do))
    out, lse = abi.forward(lib, qg, kg, vg, scale, causal)
    dq, dk, dv = abi.backward(lib, qg, kg, vg, out, dog, lse, scale, causal)[:3]
    out0, lse0 = abi.forward(lib, clean.cuda(), kg, vg, scale, causal)
    others = [i for i in range(H) if i != h]
    assert torch.equal(out[:, :, others], out0[:, :, others]) and torch.equal(lse[:, others], lse0[:, others])
    grads0 = abi.backward(lib, clean.cuda(), kg, vg, out0, dog, lse0, scale, causal)[:3]
    for a, b in zip((dq, dk, dv), grads0):
        assert torch.equal(a[:, :, others], b[:, :, others])
    good = [i for i in range(N) if i not in bad]
    one = [t[:, :, h:h + 1] for t in (clean, k, v, do)]
    ref, ref_lse = ao.attention_forward(*one[:3], scale, causal)
    ref_dq = ao.attention_backward(*one, scale, causal)[0]
    assert torch.isnan(out[:, bad, h]).all() and torch.isnan(dq[:, bad, h]).all()
    # the repository's bounds for O, the logsumexp and gradients of order 1
    assert (out[:, good, h].float().cpu() - ref[:, good, 0].half().float()).abs().max() <= 2e-3
    assert (lse[:, h, good].cpu() - ref_lse[:, 0, good]).abs().max() <= 2e-3
    assert (dq[:, good, h].float().cpu() - ref_dq[:, good, 0].half().float()).abs().max() <= 1e-2


TAILS = [  # D, slices, N, causal, how many slices' last rows go to one block
    (64, 300, 129, 0, 2), (64, 401, 150, 0, 4), (64, 100, 257, 0, 2), (64, 110, 520, 0, 2), (64, 118, 544, 0, 4),
    (64, 59, 1031, 0, 2), (64, 61, 1537, 0, 2), (64, 62, 1550, 0, 4), (128, 300, 160, 0, 2), (128, 181, 130, 0, 4),
    (128, 90, 1025, 0, 2),  # with every other wave slot first
    (128, 203, 257, 0, 2), (128, 150, 400, 0, 4), (128, 57, 1056, 0, 2), (128, 122, 1025, 0, 4),
    (64, 300, 129, 1, 2), (64, 401, 160, 1, 4), (64, 231, 288, 1, 4), (64, 199, 416, 1, 4), (64, 173, 513, 1, 4),
    (128, 625, 288, 1, 4), (128, 301, 513, 1, 4),  # nearly as many rounds as it pays for
    (128, 150, 130, 1, 2), (128, 399, 150, 1, 4), (128, 230, 257, 1, 4), (128, 215, 385, 1, 4), (128, 170, 544, 1, 4),
]


def test_blocks_with_the_last_rows_of_slices(tmp_path):
    """The cases below on 256 compute units and others left alone; every slice's last rows once, on few XCDs."""
    rule = "fmha_tails_per_block(x[0], x[2], x[1], 256, x[3]) == x[4]"
    alone = [(64, 300, 128), (64, 300, 161), (64, 230, 129), (64, 256, 257), (64, 30, 1031), (64, 34, 900), (128, 56, 1031),
             (128, 200, 1031), (128, 34, 900), (128, 1, 129), (64, 1, 1), (128, 230, 2070)]
    causal = [(64, 256, 150), (128, 256, 129), (64, 100, 520), (64, 257, 410), (128, 264, 410), (128, 100, 520), (128, 200, 1031),
              (128, 641, 288), (128, 710, 288), (128, 481, 400), (128, 276, 416), (128, 353, 416), (128, 324, 513), (128, 385, 544)]
    alone = [(*case, 0, 0) for case in alone] + [(*case, 1, 0) for case in causal]
    assert all(abi.host_rule(tmp_path, rule, TAILS + alone))
    src, exe = tmp_path / "tails.cpp", tmp_path / "tails"
    src.write_text(r'''
#include <cstdio>
#include <vector>
#include "block_map.h"
int main() {
  for (int per = 2; per <= 4; per += 2)
    for (int slices = 1; slices <= 900; ++slices) {
      const int tails = fmha_tail_blocks(slices, per);
      std::vector<int> seen(slices, 0);
      for (int lin = 0; lin < tails; ++lin)
        for (int wave = 0; wave < per; ++wave) {
          const int s = fmha_tail_slice(lin, wave, tails, per);
          if (s < 0 || (s < slices && seen[s]++)) { printf("slice %d %d %d\n", per, slices, lin); return 1; }
        }
      for (int s = 0; s < slices; ++s)
        if (!seen[s]) { printf("none %d %d %d\n", per, slices, s); return 1; }
      if (tails % 8 || per * tails >= slices + 8 * per) { printf("many %d %d\n", per, slices); return 1; }
    }
  for (int d = 64; d <= 128; d += 64)
    for (int n = 1; n <= 1200; ++n)
      for (int slices = 1; slices <= 700; slices += 5) {
        const int per = fmha_tails_per_block(d, n, slices, 256, slices & 1);
        if (per && per != 2 && per != 4) return 1;
        if (per && fmha_tail_blocks(slices, per) >= slices) { printf("gain %d %d\n", n, slices); return 1; }
      }
  puts("ok");
}
''')
    inc = os.path.join(abi.ROOT, "flash-attention-v100_amd", "csrc")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-I", inc, str(src), "-o", str(exe)])
    assert subprocess.check_output([str(exe)]).decode().strip() == "ok"


@pytest.mark.gpu
@pytest.mark.parametrize("D,H,N,causal,per", TAILS)
def test_last_rows_of_several_slices_in_one_block(D, H, N, causal, per):
    """The bits of launches of a few slices, in which each has a block for its last rows; with maxima that are
    raised at nearly every tile, with strides and a negative scale, with rows that are not finite."""
    lib = abi.load()
    last = (N - 1) // 128 * 128
    for kind in ("plain", "growing", "strided", "not finite"):
        q, k, v = (t.cuda() for t in _inputs(1, N, H, D, kind == "growing"))
        scale = {"growing": 1.0, "strided": -(D ** -0.5)}.get(kind, D ** -0.5)
        if kind == "not finite":
            q[:, last, 1, 3], q[:, N - 1, H // 2, 5], k[:, N - 1, H - 1, 0] = float("nan"), float("inf"), float("inf")
        if kind == "strided":
            q, k, v = torch.stack((q, k, v), dim=2).unbind(2)
            out, lse = abi.forward_strided(lib, q, k, v, scale, causal)
        else:
            out, lse = abi.forward(lib, q, k, v, scale, causal)
        for h in range(0, H, 13):
            few = [t[:, :, h:h + 13].contiguous() for t in (q, k, v)]
            o, l = abi.forward(lib, *few, scale, causal)
            assert torch.equal(o.view(torch.int16), out[:, :, h:h + 13].contiguous().view(torch.int16)) or (
                kind == "not finite" and torch.equal(o.isnan(), out[:, :, h:h + 13].isnan()) and
                torch.equal(o.nan_to_num(), out[:, :, h:h + 13].nan_to_num()))
            assert torch.equal(l.nan_to_num(), lse[:, h:h + 13].nan_to_num())
            if h == 0 and kind in ("plain", "growing"):
                ref, ref_lse = ao.attention_forward(*(t[:, :, :2].cpu() for t in few), scale, bool(causal))
                # the bounds of _check
                assert (o[:, :, :2].float().cpu() - ref.half().float()).abs().max() <= 2e-3 * max(1.0, ref.abs().max().item())
                assert ((l[:, :2].cpu() - ref_lse).abs() <= 2e-3 + 1e-6 * ref_lse.abs()).all()

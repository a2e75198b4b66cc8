"""CPU tests of the host side: the C ABI library loads and exports what the
header declares, argument validation returns the documented codes before any
launch, and the extension raises RuntimeError like the reference's TORCH_CHECKs
(kernel/fused_mha_api.cpp:25-47).  No compute call is made here."""
import ctypes
import inspect
import os
import sys

import pytest
import torch

import abi


ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def lib():
    return abi.load()


def test_exports_every_declared_symbol(lib):
    names = abi.declared_symbols()
    assert names == sorted(["fused_mha_forward", "fused_mha_backward", "fused_mha_backward_workspace_bytes",
                            "fused_mha_backward_min_workspace_bytes",
                            "fused_mha_backward_noalloc", "fused_mha_backward_delta", "fused_mha_backward_dq", "fused_mha_backward_dkdv",
                            "fused_mha_forward_strided", "fused_mha_backward_strided", "fused_mha_error_string"])
    for name in names:
        assert hasattr(lib, name), name


def test_error_strings(lib):
    seen = set()
    for code in range(0, -11, -1):
        text = lib.fused_mha_error_string(code).decode()
        assert text and text not in seen
        seen.add(text)
    assert b"unknown" in lib.fused_mha_error_string(-99)


def test_workspace_bytes(lib):
    small = lib.fused_mha_backward_min_workspace_bytes
    assert small(2, 32, 4096, 128) == 2 * 2 * 32 * 4096 * 4
    assert small(1, 4, 128, 64) == 2 * 4 * 128 * 4
    assert small(1, 4, 100, 64) == 2 * 4 * 100 * 4  # any n > 0 is accepted
    assert small(1, 4, 0, 64) == 0
    assert small(1, 4, 128, 96) == 0
    # at head size 128 the preferred workspace adds room for the fp16 dS tiles: slices * np * np elements, np = n rounded
    # up to 128, behind the statistics rounded up to 256 bytes
    big = lib.fused_mha_backward_workspace_bytes
    assert big(2, 32, 4096, 128) == 2 * 2 * 32 * 4096 * 4 + 64 * 4096 * 4096 * 2
    assert big(1, 4, 100, 128) == 3328 + 4 * 128 * 128 * 2  # 3200 bytes of statistics -> 3328
    assert big(1, 4, 0, 64) == 0 and big(1, 4, 128, 96) == 0
    assert big(1, 32, 16384, 128) == small(1, 32, 16384, 128) + 32 * 16384 * 16384 * 2  # 16 GiB: all slices at once


@pytest.mark.parametrize("batch,head,n", [(1, 4, 128), (2, 3, 333), (16, 12, 512), (1, 16, 32768), (1, 64, 16384)])
def test_workspace_bytes_head_size_64(lib, batch, head, n):
    """The backward reads and writes nothing but the statistics there, so no more is asked for."""
    assert (lib.fused_mha_backward_workspace_bytes(batch, head, n, 64) ==
            lib.fused_mha_backward_min_workspace_bytes(batch, head, n, 64))


@pytest.mark.parametrize("batch,head,n,slices", [
    (1, 64, 16384, 16),   # 32 GiB of dS; 128 key blocks a slice: 8 blocks per compute unit are 16 slices
    (8, 32, 8192, 32),
    (1, 16, 32768, 8),
    (2, 16, 20000, 14),   # 157 blocks a slice: rounded up
    (1, 12, 45000, 4),    # 5 more blocks per unit would be past 16 GiB
    (1, 2, 92672, 1),     # one slice is just within 16 GiB
    (1, 2, 92673, 0),     # not even one is
    (2, 4200, 1024, 2048),  # many short slices: 4 GiB
    (512, 1024, 384, 14563),
])
def test_workspace_bytes_past_the_spill_limit(lib, batch, head, n, slices):
    """What the preferred size has room for past 16 GiB of dS: rounds of enough slices for the launches to be full."""
    least = lib.fused_mha_backward_min_workspace_bytes(batch, head, n, 128)
    np_ = -(-n // 128) * 128
    want = -(-least // 256) * 256 + slices * np_ * np_ * 2 if slices else least
    assert batch * head * np_ * np_ * 2 > 16 << 30 and slices * np_ * np_ * 2 <= 16 << 30
    assert lib.fused_mha_backward_workspace_bytes(batch, head, n, 128) == want


@pytest.mark.parametrize("batch,head,n,d,room,slices", [
    (2, 32, 4096, 128, 16 << 30, 64),          # room for all
    (2, 32, 4096, 128, (2 << 30) + (2 << 20), 64),  # just so
    (2, 32, 4096, 128, (2 << 30) + (2 << 20) - 1, 63),
    (2, 32, 4096, 128, (1 << 30) - 1, 0),      # rounds of less than 1 GiB are not worth it
    (2, 4, 1024, 128, 1 << 20, 0),
    (1, 16, 32768, 128, 9 << 30, 4),
    (1, 16, 32768, 128, 3 << 30, 0),           # one slice is one block per compute unit
    (1, 16, 32768, 128, 0, 0),
    (1, 64, 16384, 128, 64 << 30, 16),         # no more than the preferred size
    (1, 64, 16384, 64, 64 << 30, 0),
])
def test_workspace_within(lib, batch, head, n, d, room, slices):
    """The size the extension takes when it can spare `room` bytes."""
    f = lib.fmha_backward_workspace_within
    f.argtypes, f.restype = [ctypes.c_int] * 4 + [ctypes.c_size_t], ctypes.c_size_t
    least = lib.fused_mha_backward_min_workspace_bytes(batch, head, n, d)
    np_ = -(-n // 128) * 128
    assert f(batch, head, n, d, room) == (-(-least // 256) * 256 + slices * np_ * np_ * 2 if slices else least)
    assert f(batch, head, 0, d, room) == 0


@pytest.mark.parametrize("batch,head,n,d,causal,room", [
    (2, 32, 4096, 128, 1, True), (1, 8, 4096, 128, 1, False), (1, 8, 4096, 128, 0, True), (1, 4, 4096, 128, 0, False),
    (1, 600, 100, 128, 0, True), (1, 400, 100, 128, 0, False), (1, 4, 128, 64, 0, False), (1, 64, 4096, 64, 1, False),
])
def test_workspace_for(lib, batch, head, n, d, causal, room):
    """The size the extension takes for one backward: none for dS where both passes go in one launch (256 compute units)."""
    f = lib.fmha_backward_workspace_for
    f.argtypes, f.restype = [ctypes.c_int] * 5, ctypes.c_size_t
    which = lib.fused_mha_backward_workspace_bytes if room else lib.fused_mha_backward_min_workspace_bytes
    assert f(batch, head, n, d, causal) == which(batch, head, n, d)
    assert f(batch, head, 0, d, causal) == 0


def test_forward_validation_codes(lib):
    p = 0x1000  # never dereferenced: every call below is rejected before a launch
    f = lib.fused_mha_forward
    assert f(None, p, p, p, p, 1, 1, 32, 32, 64, 1.0, 0, None) == abi.ERR_NULL_POINTER
    assert f(p, p, p, p, None, 1, 1, 32, 32, 64, 1.0, 0, None) == abi.ERR_NULL_POINTER
    assert f(p, p, p, p, p, 0, 1, 32, 32, 64, 1.0, 0, None) == abi.ERR_BAD_SHAPE
    assert f(p, p, p, p, p, 1, 1, 0, 0, 64, 1.0, 0, None) == abi.ERR_BAD_SHAPE        # n == 0
    assert f(p, p, p, p, p, 1, 1, 32, 64, 64, 1.0, 0, None) == abi.ERR_BAD_SHAPE      # m != n
    assert f(p, p, p, p, p, 1, 1, 32, 32, 96, 1.0, 0, None) == abi.ERR_BAD_HEAD_DIM
    assert f(p, p, p, p, p, 1, 1, 32, 32, 64, float("nan"), 0, None) == abi.ERR_BAD_SCALE
    assert f(p, p, p, p, p, 1, 1, 32, 32, 64, float("inf"), 0, None) == abi.ERR_BAD_SCALE
    assert f(p + 2, p, p, p, p, 1, 1, 32, 32, 64, 1.0, 0, None) == abi.ERR_MISALIGNED
    # the limits of the kernels' 32-bit arithmetic and of a launch: n < 2^29, head*d < 2^24,
    # ceil(n/128)*batch*head < 2^23, batch*head*n*d/8 < 2^32
    assert f(p, p, p, p, p, 1, 1, 1 << 29, 1 << 29, 64, 1.0, 0, None) == abi.ERR_TOO_LARGE
    assert f(p, p, p, p, p, 1 << 12, 1 << 12, 1 << 14, 1 << 14, 64, 1.0, 0, None) == abi.ERR_TOO_LARGE
    assert f(p, p, p, p, p, 2048, 2048, 1 << 16, 1 << 16, 64, 1.0, 0, None) == abi.ERR_TOO_LARGE
    assert f(p, p, p, p, p, 1, 1 << 17, 128, 128, 128, 1.0, 0, None) == abi.ERR_TOO_LARGE    # head*d = 2^24
    assert f(p, p, p, p, p, 1, 1 << 18, 128, 128, 64, 1.0, 0, None) == abi.ERR_TOO_LARGE     # head*d = 2^24
    assert f(p, p, p, p, p, 1 << 11, 1 << 12, 128, 128, 64, 1.0, 0, None) == abi.ERR_TOO_LARGE  # 2^23 blocks of 128 rows
    assert f(p, p, p, p, p, 1 << 9, 1 << 12, 130, 130, 128, 1.0, 0, None) == abi.ERR_TOO_LARGE  # delta pass: 2^32 threads
    assert lib.fused_mha_backward_workspace_bytes(1, 1 << 17, 128, 128) == 0
    assert lib.fused_mha_backward_min_workspace_bytes(1, 1 << 17, 128, 128) == 0


def test_backward_validation_codes(lib):
    p = 0x1000
    b = lib.fused_mha_backward
    ws = 2 * 1 * 1 * 32 * 4
    assert b(p, p, p, p, p, p, None, ws, p, p, p, 1, 1, 32, 32, 64, 1.0, 0, None) == abi.ERR_NULL_POINTER
    assert b(p, p, p, p, p, p, p, ws, p, p, None, 1, 1, 32, 32, 64, 1.0, 0, None) == abi.ERR_NULL_POINTER
    assert b(p, p, p, p, p, p, p, ws - 1, p, p, p, 1, 1, 32, 32, 64, 1.0, 0, None) == abi.ERR_BAD_SHAPE
    assert b(p, p, p, p, p, p, p, ws, p, p, p, 1, 1, 40, 40, 64, 1.0, 0, None) == abi.ERR_BAD_SHAPE
    assert b(p, p, p, p, p, p, p, ws, p, p, p, 1, 1, 32, 32, 32, 1.0, 0, None) == abi.ERR_BAD_HEAD_DIM
    assert b(p, p, p, p, p, p, p, ws, p, p + 8, p, 1, 1, 32, 32, 64, 1.0, 0, None) == abi.ERR_MISALIGNED
    assert lib.fused_mha_backward_delta(p, None, p, p, ws, 1, 1, 32, 64, None) == abi.ERR_NULL_POINTER
    assert lib.fused_mha_backward_dq(p, p, p, p, p, p, ws, None, 1, 1, 32, 64, 1.0, 0, None) == abi.ERR_NULL_POINTER
    assert lib.fused_mha_backward_dkdv(p, p, p, p, p, p, ws, p, None, 1, 1, 32, 64, 1.0, 0, None) == abi.ERR_NULL_POINTER


def test_noalloc_validation_codes(lib):
    """Rejected before the scratch address is looked up or anything is launched."""
    p = 0x1000
    g = lib.fused_mha_backward_noalloc
    assert g(p, p, p, p, p, p, p, p, p, 1, 1, 40, 32, 64, 1.0, 0, None) == abi.ERR_BAD_SHAPE
    assert g(p, p, p, p, p, p, p, p, p, 1, 1, 32, 32, 96, 1.0, 0, None) == abi.ERR_BAD_HEAD_DIM
    rows = abi.NOALLOC_MAX_ROWS
    assert g(p, p, p, p, p, p, p, p, p, 1, 2, rows // 2 + 1, rows // 2 + 1, 64, 1.0, 0, None) == abi.ERR_SCRATCH_LIMIT
    assert g(p, p, p, p, p, p, p, p, p, 4, 64, 8192, 8192, 128, 1.0, 1, None) == abi.ERR_SCRATCH_LIMIT
    assert b"NOALLOC_MAX_ROWS" in lib.fused_mha_error_string(abi.ERR_SCRATCH_LIMIT)
    import re
    text = open(abi.HEADER).read()
    assert int(re.search(r"#define FUSED_MHA_NOALLOC_MAX_ROWS \(1 << (\d+)\)", text).group(1)) == 20


def test_strided_validation_codes(lib):
    p = 0x1000  # never dereferenced: every call below is rejected before a launch
    f = lib.fused_mha_forward_strided
    ok = abi.Strides(32 * 2 * 64, 2 * 64, 64)

    def call(qs, ks=ok, vs=ok):
        return f(p, qs, p, ks, p, vs, p, p, 1, 2, 32, 64, 1.0, 0, None)

    assert call(abi.Strides(32 * 2 * 64, 2 * 64, 68)) == abi.ERR_BAD_STRIDE      # rows off 16-byte boundaries
    assert call(ok, abi.Strides(-4096, 128, 64)) == abi.ERR_BAD_STRIDE           # negative
    assert call(ok, ok, abi.Strides(1 << 30, 1 << 24, 64)) == abi.ERR_BAD_STRIDE  # sequence stride too large
    assert f(None, ok, p, ok, p, ok, p, p, 1, 2, 32, 64, 1.0, 0, None) == abi.ERR_NULL_POINTER
    assert f(p, ok, p, ok, p, ok, p, p, 1, 2, 32, 96, 1.0, 0, None) == abi.ERR_BAD_HEAD_DIM
    g = lib.fused_mha_backward_strided
    bad = abi.Strides(4096, 130, 64)
    assert g(p, ok, p, ok, p, ok, p, p, bad, p, p, 1 << 20, p, p, p, 1, 2, 32, 64, 1.0, 0, None) == abi.ERR_BAD_STRIDE
    assert g(p, ok, p, ok, p, ok, p, p, ok, p, p, 8, p, p, p, 1, 2, 32, 64, 1.0, 0, None) == abi.ERR_BAD_SHAPE  # workspace
    assert b"stride" in lib.fused_mha_error_string(abi.ERR_BAD_STRIDE)


def test_python_api_signature():
    import flash_attn_v100
    from flash_attn_v100 import flash_attn_func
    from flash_attn_v100.flash_attn_interface import FlashAttnFunc

    assert flash_attn_v100.__version__
    params = inspect.signature(flash_attn_func).parameters
    # reference flash_attn_interface.py:101-107
    assert list(params) == ["q", "k", "v", "softmax_scale", "causal"]
    assert params["softmax_scale"].default is None and params["causal"].default is False
    assert issubclass(FlashAttnFunc, torch.autograd.Function)


def test_extension_checks_raise_runtime_error():
    import flash_attn_v100_cuda as ext

    def t(*shape, dtype=torch.float16):
        return torch.zeros(shape, dtype=dtype)

    ok = t(1, 32, 2, 64)
    cases = [
        ((t(1, 32, 2, 64, dtype=torch.float32), ok, ok), "fp16"),
        ((ok, t(1, 32, 2, 64, dtype=torch.bfloat16), ok), "same dtype"),
        ((t(32, 2, 64), ok, ok), "4 dimensions"),
        ((t(1, 32, 2, 96), t(1, 32, 2, 96), t(1, 32, 2, 96)), "head dimension"),
        ((t(1, 0, 2, 64), t(1, 0, 2, 64), t(1, 0, 2, 64)), "seqlen must be positive"),
        ((ok, t(1, 64, 2, 64), ok), "must have shape"),
        ((t(1, 32, 2, 128)[..., ::2], ok, ok), "contiguous last dimension"),
        ((ok, ok, ok), "must be on the GPU"),
    ]
    for (q, k, v), msg in cases:
        with pytest.raises(RuntimeError, match=msg):
            ext.fwd(q, k, v, None, 0.125, False)
    lse = torch.zeros(1, 2, 32)
    with pytest.raises(RuntimeError, match="must be on the GPU"):
        ext.bwd(ok, ok, ok, ok, ok, lse, None, None, None, 0.125, True)
    with pytest.raises(RuntimeError, match="lse must be fp32"):
        ext.bwd(ok, ok, ok, ok, ok, lse.half(), None, None, None, 0.125, True)
    with pytest.raises(RuntimeError, match="must have shape"):
        ext.bwd(ok, ok, ok, ok, ok, torch.zeros(1, 32, 2), None, None, None, 0.125, True)
    with pytest.raises(RuntimeError, match="4 dimensions"):
        ext.bwd(ok, ok, t(32, 2, 64), ok, ok, lse, None, None, None, 0.125, True)
    with pytest.raises(RuntimeError, match="4 dimensions"):
        ext.bwd(ok, ok, ok, t(32, 2, 64), ok, lse, None, None, None, 0.125, True)
    with pytest.raises(RuntimeError, match="4 dimensions"):
        ext.bwd(t(2, 64), ok, ok, ok, ok, lse, None, None, None, 0.125, True)


def test_python_api_rejects_cpu_tensors():
    from flash_attn_v100 import flash_attn_func

    q = torch.zeros(1, 32, 2, 64, dtype=torch.float16)
    with pytest.raises(RuntimeError, match="must be on the GPU"):
        flash_attn_func(q, q, q, None, True)


def test_block_map_is_a_bijection(tmp_path):
    """csrc/block_map.h, compiled for the host: every (slice, block) pair is produced exactly once for any slice
    count (multiples of 8 or not), and with a multiple of 8 every slice stays on one XCD (work-group id mod 8)."""
    import os
    import subprocess

    src = tmp_path / "check_block_map.cpp"
    src.write_text(r'''
#include <cstdio>
#include <vector>
#include "block_map.h"
int main() {
  for (int slices = 1; slices <= 83; ++slices)
    for (int bps = 1; bps <= 37; ++bps) {
      const int total = slices * bps;
      std::vector<int> seen(total, 0), xcd_of(slices, -1);
      int shared = 0;
      for (int lin = 0; lin < total; ++lin) {
        int s = -1, b = -1;
        fmha_slice_and_block(lin, slices, bps, s, b);
        if (s < 0 || s >= slices || b < 0 || b >= bps) { printf("range %d %d %d\n", slices, bps, lin); return 1; }
        if (seen[s * bps + b]++) { printf("twice %d %d %d\n", slices, bps, lin); return 1; }
        if (xcd_of[s] < 0) xcd_of[s] = lin & 7;
        else if (xcd_of[s] != (lin & 7) && s < (slices & ~7)) ++shared;
      }
      if (shared) { printf("slice on two XCDs %d %d\n", slices, bps); return 1; }
    }
  // heaviest first inside a slice: block indices of one slice appear in ascending order
  // (the slices beyond a multiple of 8 are cut into per-XCD runs instead)
  for (int slices : {8, 12, 64, 80}) {
    const int bps = 16;
    std::vector<int> last(slices, -1);
    for (int lin = 0; lin < slices * bps; ++lin) {
      int s, b;
      fmha_slice_and_block(lin, slices, bps, s, b);
      if (s < (slices & ~7) && b <= last[s]) { printf("order %d %d\n", slices, lin); return 1; }
      last[s] = b;
    }
  }
  puts("ok");
  return 0;
}
''')
    inc = os.path.join(abi.ROOT, "flash-attention-v100_amd", "csrc")
    exe = tmp_path / "check_block_map"
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-I", inc, str(src), "-o", str(exe)])
    assert subprocess.check_output([str(exe)]).decode().strip() == "ok"


def test_divisors_of_a_launch(tmp_path):
    """csrc/block_map.h: FmhaDivisor gives the quotients of whole numbers below 2^31, and the orders of blocks that take it are
    those that take an int."""
    import subprocess

    src = tmp_path / "check_divisors.cpp"
    src.write_text(r'''
#include <cstdio>
#include <initializer_list>
#include <vector>
#include "block_map.h"
int main() {
  const int most = 0x7fffffff;
  auto wrong = [&](int d) {
    const FmhaDivisor by(d);
    auto bad = [&](long n) { return n >= 0 && n <= most && (int)n / by != (int)n / d; };
    for (long k : {0L, 1L, 2L, 3L, (long)most / d / 2, (long)most / d - 1, (long)most / d, (long)most / d + 1})
      for (long e = -2; e <= 2; ++e)
        if (bad(k * d + e)) return true;
    for (long n = 1; n <= most; n = n * 21 / 13 + 1)
      if (bad(n) || bad(most - n)) return true;
    return bad(most);
  };
  for (int d = 1; d <= 5000; ++d)
    if (wrong(d)) { printf("divisor %d\n", d); return 1; }
  for (long d = 5001; d <= most; d = d * 9 / 8 + 7)
    if (wrong((int)d)) { printf("divisor %ld\n", d); return 1; }
  for (int bit = 12; bit < 31; ++bit)
    for (int e = -1; e <= 1; ++e)
      if (wrong((1 << bit) + e)) { printf("divisor 2^%d %+d\n", bit, e); return 1; }
  if (wrong(most) || wrong(most - 1)) { puts("largest"); return 1; }
  for (int slices : {1, 3, 7, 8, 9, 60, 64, 71, 72, 80, 127, 128, 131, 200})
    for (int blocks : {1, 2, 3, 5, 8, 9, 16, 31})
      for (bool heavy : {false, true})
        for (bool last : {false, true}) {
          const FmhaOrder one(slices, blocks, heavy, last), two(slices, blocks, heavy, last, 2), ds(slices, blocks, heavy, false);
          auto differ = [&](int lin) {
            int s = -1, b = -1, t = -1, c = -1;
            bool p = false, q = false;
            if (lin < slices * blocks) {
              fmha_scheduled_block(lin, slices, blocks, heavy, last, s, b);
              fmha_ordered_block(lin, one.slices, one.run, one.last_level, heavy, one.short_last, t, c);
              if (s != t || b != c || s < 0 || s >= slices || b < 0 || b >= blocks) return true;
              fmha_slice_and_block(lin, slices, blocks, s, b);
              fmha_slice_and_block(lin, slices, FmhaDivisor(blocks), t, c);
              if (s != t || b != c) return true;
            }
            if (lin < 2 * slices * blocks) {
              fmha_two_pass_block(lin, slices, blocks, heavy, last, s, b, p);
              fmha_two_pass_ordered_block(lin, two.slices, two.run, two.last_level, heavy, two.short_last, t, c, q);
              if (s != t || b != c || p != q || s < 0 || s >= slices || b < 0 || b >= blocks) return true;
            }
            s = t = b = c = -1;
            const bool some = fmha_ds_launch_block(lin, slices, blocks, heavy, s, b, p);
            return some != fmha_ds_launch_ordered_block(lin, ds.slices, ds.run, ds.last_level, heavy, t, c, q) || s != t || b != c ||
                   p != q;
          };
          std::vector<int> seen(3 * slices * blocks, 0);
          for (int lin = 0; lin < 2 * slices * blocks; ++lin) {
            int s, b;
            bool second = false;
            if (lin < slices * blocks) {
              fmha_scheduled_block(lin, slices, blocks, heavy, last, s, b);
              ++seen[s * blocks + b];
            }
            fmha_two_pass_block(lin, slices, blocks, heavy, last, s, b, second);
            ++seen[((second ? 2 : 1) * slices + s) * blocks + b];
          }
          for (int n : seen)
            if (n != 1) { printf("%d x %d, %d %d: a block %d times\n", blocks, slices, heavy, last, n); return 1; }
          for (int lin = 0; lin < fmha_ds_launch_blocks(slices, blocks); ++lin)
            if (differ(lin)) { printf("%d x %d, %d %d: %d\n", blocks, slices, heavy, last, lin); return 1; }
        }
  puts("ok");
  return 0;
}
''')
    inc = os.path.join(abi.ROOT, "flash-attention-v100_amd", "csrc")
    exe = tmp_path / "check_divisors"
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-I", inc, str(src), "-o", str(exe)])
    assert subprocess.check_output([str(exe)]).decode().strip() == "ok"


def test_launches_with_last_rows_in_one_block_cover_every_block_once(tmp_path):
    """csrc/block_map.h: the 128-query forward with work groups for the last rows of slices, as the kernel takes its order:
    these first, then the blocks of one index fewer, each once and on the XCD of its slice."""
    import subprocess

    src = tmp_path / "check_tails.cpp"
    src.write_text(r'''
#include <cstdio>
#include <initializer_list>
#include <vector>
#include "block_map.h"
int main() {
  for (int slices : {1, 5, 8, 31, 60, 64, 71, 80, 129, 400, 1030})
    for (int nb : {1, 2, 3, 4, 8, 9, 16})
      for (int per : {2, 4})
        for (bool causal : {false, true}) {
          const FmhaOrder order(slices, nb, causal, false);
          const int tails = fmha_tail_blocks(slices, per), grid = tails + slices * nb;
          std::vector<int> seen(slices * (nb + 1), 0);
          for (int w = 0; w < grid; ++w) {
            const int lin = causal ? fmha_paired_block(w, grid) : w;
            if (lin < 0 || lin >= grid || (lin & 7) != (w & 7)) { printf("%d of %d\n", lin, grid); return 1; }
            if (lin < tails) {
              for (int wave = 0; wave < per; ++wave) {
                const int s = fmha_tail_slice(lin, wave, tails, per);
                if (s < slices) ++seen[s * (nb + 1) + nb];
              }
            } else {
              int s = -1, b = -1, t = -1, c = -1;
              fmha_ordered_block(lin - tails, order.slices, order.run, order.last_level, causal, false, s, b);
              fmha_ordered_block(lin - tails, slices, nb, fmha_last_level(slices), causal, false, t, c);
              if (s != t || b != c || s < 0 || s >= slices || b < 0 || b >= nb) { printf("block %d of %d\n", lin, grid); return 1; }
              const int q = slices >> 3;
              if (s < 8 * q && s / q != (lin & 7)) { printf("slice %d of %d on XCD %d\n", s, slices, lin & 7); return 1; }
              ++seen[s * (nb + 1) + b];
            }
          }
          for (int n : seen)
            if (n != 1) { printf("%d blocks of %d slices, %d to a block, %d: one %d times\n", nb, slices, per, causal, n); return 1; }
        }
  puts("ok");
  return 0;
}
''')
    inc = os.path.join(abi.ROOT, "flash-attention-v100_amd", "csrc")
    exe = tmp_path / "check_tails"
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-I", inc, str(src), "-o", str(exe)])
    assert subprocess.check_output([str(exe)]).decode().strip() == "ok"


def test_persistent_schedule_covers_every_block_once_and_balances(tmp_path):
    """csrc/block_map.h, compiled for the host: the rounds of the persistent work groups visit every block exactly
    once, a work group's blocks stay on its XCD (block number mod 8), and under causal masking the static
    schedule is balanced: at the headline and the long-context shape no work group gets more than 3 % above the
    mean number of tiles."""
    import os
    import subprocess

    src = tmp_path / "check_persistent.cpp"
    src.write_text(r'''
#include <cstdio>
#include <vector>
#include <algorithm>
#include "block_map.h"
static int check(int total, int G) {
  std::vector<int> seen(total, 0);
  for (int w = 0; w < G; ++w) {
    int r = 0;
    if (fmha_persistent_block(0, w, G) >= total) { printf("first round %d %d %d\n", total, G, w); return 1; }
    int guard = 0;
    while (r >= 0) {
      const int lin = fmha_persistent_block(r, w, G);
      if (lin < 0 || lin >= total) { printf("range %d %d %d %d\n", total, G, w, r); return 1; }
      if ((lin & 7) != (w & 7) && total > G) { printf("xcd %d %d %d %d\n", total, G, w, r); return 1; }
      if (seen[lin]++) { printf("twice %d %d %d\n", total, G, lin); return 1; }
      r = fmha_persistent_next_round(r, w, G, total);
      if (++guard > total + 2) { printf("no end %d %d %d\n", total, G, w); return 1; }
    }
  }
  for (int lin = 0; lin < total; ++lin) if (!seen[lin]) { printf("missed %d %d %d\n", total, G, lin); return 1; }
  return 0;
}
// tiles per work group under causal masking: slices x bps blocks of `rows` queries, 64-key tiles
static double imbalance(int slices, int bps, int rows, int G) {
  const int total = slices * bps;
  std::vector<long> load(G, 0);
  for (int w = 0; w < G; ++w)
    for (int r = 0; r >= 0; r = fmha_persistent_next_round(r, w, G, total)) {
      int s, b;
      fmha_slice_and_block(fmha_persistent_block(r, w, G), slices, bps, s, b);
      const int mblk = bps - 1 - b;  // heavy first
      load[w] += (long)(mblk + 1) * rows / 64;
    }
  long sum = 0, mx = 0;
  for (long v : load) { sum += v; mx = std::max(mx, v); }
  return (double)mx * G / sum;
}
int main() {
  for (int G : {8, 64, 256, 304})
    for (int total = 1; total <= 5 * G + 17; total += (total < 40 ? 1 : 7)) {
      const int grid = total <= G ? total : G;  // what persistent_grid() launches
      if (check(total, grid)) return 1;
    }
  const double head_fwd = imbalance(64, 16, 256, 256), head_dq = imbalance(64, 32, 128, 256);
  const double long_fwd = imbalance(16, 64, 256, 256), long_dq = imbalance(16, 128, 128, 256);
  if (head_fwd > 1.03 || head_dq > 1.03 || long_fwd > 1.03 || long_dq > 1.03) {
    printf("imbalance %.3f %.3f %.3f %.3f\n", head_fwd, head_dq, long_fwd, long_dq);
    return 1;
  }
  puts("ok");
  return 0;
}
''')
    inc = os.path.join(abi.ROOT, "flash-attention-v100_amd", "csrc")
    exe = tmp_path / "check_persistent"
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-I", inc, str(src), "-o", str(exe)])
    assert subprocess.check_output([str(exe)]).decode().strip() == "ok"


def test_even_shares_are_even(tmp_path):
    """csrc/block_map.h, compiled for the host: where fmha_even_shares says so, no persistent work group's share of the
    tiles is above the mean under causal masking, nor above 16/15 of it without a mask; launches that just about fill
    their rounds are not called even when their shares are not."""
    import subprocess

    src = tmp_path / "check_even.cpp"
    src.write_text(r'''
#include <algorithm>
#include <cstdio>
#include <vector>
#include "block_map.h"
// largest share over the mean one, in tiles; blocks are numbered heaviest first
static double largest(int slices, int bps, int G, bool causal) {
  const int total = slices * bps, grid = total < G ? total : G;
  std::vector<long> load(grid, 0);
  long sum = 0;
  for (int w = 0; w < grid; ++w)
    for (int r = 0; r >= 0; r = fmha_persistent_next_round(r, w, grid, total)) {
      int s, b;
      fmha_slice_and_block(fmha_persistent_block(r, w, grid), slices, bps, s, b);
      load[w] += causal ? bps - b : 1;
    }
  for (long v : load) sum += v;
  return (double)*std::max_element(load.begin(), load.end()) * G / sum;
}
int main() {
  int even[2] = {0, 0};
  for (int G : {64, 256})
    for (int slices = 1; slices <= 300; ++slices)
      for (int bps = 1; bps <= 130; ++bps)
        for (int causal = 0; causal < 2; ++causal) {
          if (slices * bps > 16 * G || !fmha_even_shares(slices, bps, G, causal)) continue;
          ++even[causal];
          const double most = largest(slices, bps, G, causal);
          if (most > (causal ? 1.0001 : 16.0001 / 15)) { printf("%d %d %d %d: %.3f\n", G, slices, bps, causal, most); return 1; }
        }
  if (even[0] < 1000 || even[1] < 50) { printf("few: %d %d\n", even[0], even[1]); return 1; }
  const int uneven[][2] = {{60, 8}, {42, 12}, {120, 8}, {60, 16}, {42, 24}, {30, 32}, {4, 128}};
  for (auto& x : uneven)
    if (fmha_even_shares(x[0], x[1], 256, true) || largest(x[0], x[1], 256, true) < 1.05) { printf("uneven %d %d\n", x[0], x[1]); return 1; }
  puts("ok");
  return 0;
}
''')
    inc = os.path.join(abi.ROOT, "flash-attention-v100_amd", "csrc")
    exe = tmp_path / "check_even"
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-I", inc, str(src), "-o", str(exe)])
    assert subprocess.check_output([str(exe)]).decode().strip() == "ok"


def test_full_launches_take_the_kernels_they_are_meant_for(tmp_path):
    """On 256 compute units."""
    from test_parity_gpu import FULL_LAUNCHES

    wide = "fmha_wide_mfmas((long)((x[1] + 127) / 128) * x[0], 256, x[2])"
    shapes = [(B * H, N, causal) for B, H, N, causal in FULL_LAUNCHES]
    assert not any(abi.host_rule(tmp_path, wide, shapes))
    assert abi.host_rule(tmp_path, "fmha_persistent_forward_pays(x[0], x[1], 256, x[2])", shapes) == [True] * 3 + [False] * 2
    assert all(abi.host_rule(tmp_path, wide, [(31, 520, False), (51, 520, True), (4, 320, True)]))


def test_blocks_of_the_launch_over_ds(tmp_path):
    """csrc/block_map.h: every block of both passes once, a dQ block behind all dK/dV blocks, slices on one XCD where the order
    of either pass keeps them there."""
    import subprocess

    src = tmp_path / "check_ds.cpp"
    src.write_text(r'''
#include <cstdio>
#include <vector>
#include "block_map.h"
int main() {
  for (int slices = 1; slices <= 200; slices += slices < 40 ? 1 : 7)
    for (int nb = 1; nb <= 40; ++nb)
      for (int causal = 0; causal < 2; ++causal) {
        const int total = fmha_ds_launch_blocks(slices, nb), blocks = slices * nb;
        std::vector<int> seen(2 * blocks, -1);
        int idle = 0;
        for (int lin = 0; lin < total; ++lin) {
          int s, b;
          bool dq;
          if (!fmha_ds_launch_block(lin, slices, nb, causal, s, b, dq)) { ++idle; continue; }
          if (s < 0 || s >= slices || b < 0 || b >= nb || dq != (lin >= blocks) || seen[dq * blocks + s * nb + b] >= 0) {
            printf("%d %d %d: %d\n", slices, nb, causal, lin);
            return 1;
          }
          seen[dq * blocks + s * nb + b] = lin;
        }
        if (idle > 7 || total != 2 * blocks + idle) return 2;
        for (int at = 0; at < blocks; ++at)
          if ((seen[at] ^ seen[blocks + at]) & 7) return 3;  // the dQ block is where the dK/dV block of the same number was
      }
  puts("ok");
  return 0;
}
''')
    inc = os.path.join(abi.ROOT, "flash-attention-v100_amd", "csrc")
    exe = tmp_path / "check_ds"
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-I", inc, str(src), "-o", str(exe)])
    assert subprocess.check_output([str(exe)]).decode().strip() == "ok"


def test_launches_over_ds_at_once_do_not_hold_each_other_up(tmp_path):
    """csrc/block_map.h: launches of both passes over dS on several streams, on 8 XCDs of 32 compute units that hand out the
    blocks of a launch in order and prefer different launches.  A dQ block that waits keeps its compute unit, and the dK/dV
    blocks that it waits for may be behind such blocks of another launch, on another XCD.  The waits leave the whole no
    more than 1.4 times as long as the launches one after the other, and nobody gives up in a launch alone."""
    import subprocess

    src = tmp_path / "at_once.cpp"
    src.write_text(r'''
#include <cstdio>
#include <vector>
#include "block_map.h"
struct Block { int slice; bool dq; };
struct Cu { bool busy = false, waiting = false; int launch; Block block; double since, end; };
// us until `launches` of them are done; alone: how many dQ blocks have formed S and dP themselves
double run(int slices, int n, int launches, bool mixed, int& alone) {
  const int nb = (n + 127) / 128;
  const double block = 0.016 * n;  // us of a dK/dV block; a dQ block over dS takes half of that, one without it 1.1 times
  std::vector<Block> queue[8];
  std::vector<int> home(slices, -1);
  for (int lin = 0; lin < fmha_ds_launch_blocks(slices, nb); ++lin) {
    int s, b;
    bool dq;
    if (!fmha_ds_launch_block(lin, slices, nb, false, s, b, dq)) continue;
    queue[lin & 7].push_back({s, dq});
    if (s < (slices & ~7)) {  // the kernel counts on its dK/dV blocks having started
      if (home[s] >= 0 && home[s] != (lin & 7)) printf("%d x %d: slice %d on two XCDs\n", n, slices, s);
      home[s] = lin & 7;
    }
  }
  std::vector<std::vector<size_t>> next(launches, std::vector<size_t>(8));
  std::vector<std::vector<int>> started(launches, std::vector<int>(slices)), stored = started;
  Cu cus[8][32];
  alone = 0;
  for (double t = 0;; t += block / 16) {
    bool any = false;
    for (auto& xcd : cus)
      for (Cu& c : xcd)
        if (c.busy && !c.waiting && c.end <= t) {
          c.busy = false;
          if (!c.block.dq) ++stored[c.launch][c.block.slice];
        }
    for (int x = 0; x < 8; ++x)
      for (Cu& c : cus[x]) {
        if (c.busy && c.waiting) {
          const int s = c.block.slice;
          const bool whole = stored[c.launch][s] == nb;
          if (whole || t - c.since >= 0.01 * fmha_ds_wait_ticks(n, started[c.launch][s] == nb)) {
            c.waiting = false;
            c.end = t + (whole ? 0.5 : 1.1) * block;
            alone += !whole;
          }
        }
        for (int k = 0; k < launches && !c.busy; ++k) {
          const int l = mixed ? (x + k) % launches : k;
          if (next[l][x] == queue[x].size()) continue;
          const Block b = queue[x][next[l][x]++];
          c = {true, b.dq, l, b, t, t + block};
          if (!b.dq) ++started[l][b.slice];
        }
        any |= c.busy;
      }
    if (!any) return t;
  }
}
int main() {
  const int shapes[][2] = {{60, 1031}, {9, 4096}, {15, 4609}, {22, 5889}, {23, 5633}, {18, 8192}};
  for (auto& shape : shapes) {
    int alone;
    run(shape[0], shape[1], 1, false, alone);
    if (alone) printf("%d x %d alone: %d\n", shape[1], shape[0], alone);
    for (int launches = 2; launches <= 4; ++launches) {
      const double apart = launches * run(shape[0], shape[1], 1, false, alone), mixed = run(shape[0], shape[1], launches, true, alone);
      if (mixed > 1.4 * apart) printf("%d x %d, %d launches: %.0f us, %.0f\n", shape[1], shape[0], launches, apart, mixed);
    }
  }
  puts("ok");
}
''')
    inc = os.path.join(abi.ROOT, "flash-attention-v100_amd", "csrc")
    exe = tmp_path / "at_once"
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-I", inc, str(src), "-o", str(exe)])
    assert subprocess.check_output([str(exe)]).decode().strip() == "ok"


def test_backward_by_slice(tmp_path, lib):
    """D, N, slices, causal of backwards timed both ways on 256 compute units; and what the extension takes for them."""
    rule = "fmha_backward_by_slice(x[0], x[1], x[2], 256, x[3])"
    slices = [
        (128, 1, 129, 0), (128, 256, 129, 1), (128, 256, 256, 0), (128, 100, 257, 0), (128, 200, 320, 0), (128, 160, 320, 1),
        (128, 96, 257, 1), (128, 97, 320, 1), (128, 116, 266, 1), (128, 97, 257, 0), (128, 256, 342, 1), (128, 33, 514, 0), (128, 100, 640, 1), (128, 256, 514, 0), (128, 100, 1600, 0), (128, 64, 3000, 1),
        (64, 129, 129, 0), (64, 257, 192, 0), (64, 512, 192, 0), (64, 300, 448, 0), (64, 512, 600, 0), (64, 512, 1300, 0),
        (64, 161, 652, 0), (64, 176, 652, 0), (64, 161, 1932, 0), (64, 177, 612, 0), (64, 160, 598, 0),
        (64, 264, 608, 0), (64, 352, 840, 0), (64, 384, 1216, 0), (64, 290, 1440, 0), (64, 304, 1704, 0), (64, 320, 1264, 1),
        (64, 264, 1264, 1),
        (64, 129, 171, 1), (64, 160, 448, 1), (64, 180, 224, 1), (64, 200, 256, 1), (64, 384, 256, 1),
        (64, 512, 224, 1), (64, 512, 448, 1), (64, 512, 1030, 1),
    ]
    other = [
        (128, 97, 257, 1), (128, 97, 296, 1), (128, 105, 266, 1), (128, 112, 266, 1),
        (128, 1, 128, 0), (128, 257, 200, 0), (128, 256, 319, 0), (128, 256, 330, 1), (128, 100, 528, 0), (128, 100, 1030, 1),
        (64, 128, 256, 0), (64, 129, 128, 0), (64, 257, 176, 0), (64, 300, 384, 0), (64, 512, 590, 0), (64, 513, 256, 0),
        (64, 161, 598, 0), (64, 161, 612, 0), (64, 161, 1812, 0), (64, 176, 1812, 0),
        (64, 300, 400, 0), (64, 384, 385, 0), (64, 290, 598, 0), (64, 290, 833, 0), (64, 320, 1076, 0), (64, 290, 1352, 0),
        (64, 304, 1544, 0), (64, 320, 224, 1), (64, 384, 224, 1), (64, 384, 752, 1), (64, 320, 1014, 1),  # whole tiles of 64 rows
        (64, 129, 160, 1), (64, 201, 256, 1), (64, 200, 480, 1), (64, 300, 480, 1), (64, 512, 208, 1), (64, 512, 640, 1),
        (64, 192, 224, 1), (64, 193, 224, 1), (64, 200, 230, 1),
        (64, 300, 1030, 1), (64, 512, 96, 0), (128, 1, 1, 0), (64, 1, 1 << 23, 0),
    ]
    assert all(abi.host_rule(tmp_path, rule, slices)) and not any(abi.host_rule(tmp_path, rule, other))
    f = lib.fmha_backward_workspace_for
    f.argtypes, f.restype = [ctypes.c_int] * 5, ctypes.c_size_t
    for D, N, S, causal in slices:  # no room for dS
        assert f(1, S, N, D, causal) == lib.fused_mha_backward_min_workspace_bytes(1, S, N, D)


def test_count_bytes(lib):
    """What the extension adds behind the dS of all slices, on 256 compute units: 128 bytes a slice where one launch does both
    passes, nothing elsewhere."""
    f = lib.fmha_backward_count_bytes
    f.argtypes, f.restype = [ctypes.c_int] * 5, ctypes.c_size_t
    assert f(3, 20, 1031, 128, 0) == 60 * 128 and f(16, 12, 512, 128, 1) == 192 * 128 and f(1, 600, 100, 128, 0) == 600 * 128
    assert f(2, 32, 4096, 128, 1) == 0    # the dQ pass alone has blocks of 256 queries there
    assert f(1, 4, 1031, 128, 0) == 0     # few blocks: one launch that forms S and dP twice
    assert f(1, 600, 64, 128, 0) == 0     # a work group for each slice
    assert f(16, 12, 512, 64, 0) == 0 and f(1, 0, 512, 128, 0) == 0
    assert f(1, 33000, 512, 128, 0) == 0  # dS in rounds
    assert f(1, 239, 896, 128, 1) == 239 * 128 and f(1, 129, 1024, 128, 1) == 129 * 128
    assert f(1, 169, 900, 128, 1) == f(1, 161, 960, 128, 1) == f(1, 185, 1024, 128, 1) == 0  # the passes one by one are faster


def test_interleaved_blocks_are_a_bijection(tmp_path):
    """csrc/block_map.h: the row statistics' work groups take every block of a launch once, and few more than there are."""
    import subprocess

    src = tmp_path / "check_rows.cpp"
    src.write_text(r'''
#include <cstdio>
#include <vector>
#include "block_map.h"
int main() {
  for (unsigned blocks = 1; blocks <= 700; ++blocks)
    for (unsigned chain = 1; chain <= blocks; chain += (chain < 40 ? 1 : 13)) {
      const unsigned chains = (blocks + chain - 1) / chain;
      if (chain * chains >= blocks + chain) { printf("many %u %u\n", blocks, chain); return 1; }
      std::vector<int> seen(chain * chains, 0);
      for (unsigned lin = 0; lin < chain * chains; ++lin) {
        const unsigned at = fmha_interleaved_block(lin, chain, chains);
        if (at >= seen.size() || seen[at]++) { printf("%u %u %u\n", blocks, chain, lin); return 1; }
      }
    }
  puts("ok");
  return 0;
}
''')
    inc = os.path.join(abi.ROOT, "flash-attention-v100_amd", "csrc")
    exe = tmp_path / "check_rows"
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-I", inc, str(src), "-o", str(exe)])
    assert subprocess.check_output([str(exe)]).decode().strip() == "ok"


def test_installed_distribution_imports_without_pythonpath(tmp_path):
    """`pip install .` (the wheel `python setup.py install` / `pip wheel .` build; reference setup.py:151-172,
    README.md:21-23) puts the package, the extension and the kernel library into one place, and the package
    imports from there with no path into this tree."""
    import os
    import subprocess
    import sys

    pkg = os.path.join(abi.ROOT, "flash-attention-v100_amd")
    target = tmp_path / "site"
    subprocess.check_call([sys.executable, "-m", "pip", "install", "--no-deps", "--no-build-isolation", "--no-index",
                           "--quiet", "--target", str(target), pkg])
    assert (target / "flash_attn_v100_cuda.so").exists()
    assert (target / "flash_attn_v100" / "lib" / "libfused_mha.so").exists()
    code = ("import sys, os; sys.path.insert(0, %r); import flash_attn_v100, flash_attn_v100_cuda; "
            "assert os.path.dirname(flash_attn_v100.__file__).startswith(%r); "
            "assert flash_attn_v100_cuda.__file__.startswith(%r); "
            "print(flash_attn_v100.__version__, callable(flash_attn_v100.flash_attn_func))") % (
                str(target), str(target), str(target))
    env = {k: v for k, v in os.environ.items() if k != "PYTHONPATH"}
    out = subprocess.check_output([sys.executable, "-c", code], cwd=str(tmp_path), env=env).decode()
    assert out.split() == ["0.0.1", "True"]


def test_bench_refuses_more_than_one_gpu():
    """bench.py is a one-GPU benchmark: --gpus N with N > 1 exits with a message that says so."""
    import subprocess

    r = subprocess.run([sys.executable, os.path.join(ROOT, "bench.py"), "--gpus", "2"], capture_output=True, text=True,
                       timeout=120)
    assert r.returncode != 0
    assert "ONE GPU" in r.stderr


def test_bench_clock_sampler_helper():
    """The helper bench.py starts for the clock and power sample: parsers on recorded tool output, and the
    one-line-in, one-JSON-line-out protocol (on a machine without the tools the values are null)."""
    import json
    import subprocess

    sys.path.insert(0, ROOT)
    import bench

    text = ("GPU: 0\n    POWER:\n        SOCKET_POWER: 1315 W\n        GFX_VOLTAGE: N/A\n    CLOCK:\n"
            "        GFX_0:\n            CLK: 1885 MHz\n            MIN_CLK: 500 MHz\n            MAX_CLK: 2400 MHz\n"
            "        GFX_1:\n            CLK: 1821 MHz\n            MIN_CLK: 500 MHz\n")
    got = bench.parse_amd_smi(text)
    assert got == {"sclk_mhz": 1853, "socket_power_w": 1315, "xcd_mhz": [1885, 1821]}
    assert bench.parse_amd_smi("no such tool") == {"sclk_mhz": None, "socket_power_w": None, "xcd_mhz": None}
    assert bench.parse_rocm_smi("GPU[0]\t\t: sclk clock level: 1: (1849Mhz)\n") == 1849
    assert bench.parse_rocm_smi("") is None

    p = bench.start_clock_sampler()
    assert p is not None
    p.stdin.write("sample\n")
    p.stdin.flush()
    reply = json.loads(p.stdout.readline())
    assert set(("sclk_mhz", "socket_power_w", "xcd_mhz")) <= set(reply)
    p.stdin.close()
    assert p.wait(timeout=60) == 0


def test_flop_and_byte_counts_of_the_bench():
    sys.path.insert(0, ROOT)
    import bench

    assert bench.fwd_flops(2, 32, 4096, 128, True) == 4 * 2 * 32 * 4096 * 4096 * 128 / 2
    assert bench.fwd_flops(16, 12, 512, 64, False) == 4 * 16 * 12 * 512 * 512 * 64
    fwd_bytes, bwd_bytes = bench.min_hbm_bytes(2, 32, 4096, 128)
    tensor = 2 * 32 * 4096 * 128 * 2
    assert fwd_bytes == 4 * tensor + 2 * 32 * 4096 * 4  # q, k, v, o and lse
    assert bwd_bytes >= 8 * tensor  # q, k, v, o, dO in; dq, dk, dv out

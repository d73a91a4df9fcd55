"""The C-ABI library loads, exports every entry point include/dryft_decode.h declares, and
rejects bad arguments before launching anything (these calls never touch a GPU)."""
import ctypes
import os
import re

import pytest

import dryft_amd
from dryft_amd import _lib

HEADER = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "include",
                      "dryft_decode.h")


def header_symbols():
    text = open(HEADER).read()
    return sorted(set(re.findall(r"^\s*(?:int|size_t)\s+(dd_\w+)\s*\(", text, re.M)))


def test_header_and_binding_agree():
    assert header_symbols() == _lib.exported_symbols()


def test_library_exports_every_symbol():
    L = dryft_amd.lib()
    for name in header_symbols():
        assert hasattr(L, name), name
    assert L.dd_abi_version() == _lib.ABI_VERSION


def test_validation_rejects_without_launch():
    L = dryft_amd.lib()
    INVALID = 1
    # null pointers
    assert L.dd_capture_id(None, None) == INVALID
    assert L.dd_gemv(None, None, None, 1, 16, 64, 1, None, None, None) == INVALID
    assert L.dd_rmsnorm(None, None, None, 1, 16, 1e-6, None) == INVALID
    # shape limits checked before any pointer is used (fake, never-dereferenced addresses)
    fake = ctypes.c_void_p(0x1000)
    assert L.dd_gemv(fake, fake, fake, 17, 16, 64, 1, None, None, None) == INVALID   # M > 16
    assert L.dd_gemv(fake, fake, fake, 1, 16, 60, 1, None, None, None) == INVALID    # K % 8
    assert L.dd_gemv(ctypes.c_void_p(0x1008), fake, fake, 1, 16, 64, 1, None, None, None) == INVALID
    assert L.dd_gemv(fake, fake, fake, 1, 16, 4096, 4, None, None, None) == INVALID  # split, no ws
    assert L.dd_rmsnorm(fake, fake, fake, 1, 5000, 1e-6, None) == INVALID    # N > 4096
    assert L.dd_argmax(fake, 2, 100, fake, None, 0, None, None, None) == INVALID  # no ws
    assert L.dd_qkv_post_decode(fake, fake, fake, fake, fake, 64, fake, 0, fake, fake, fake,
                                1, 1, 32, 8, 64, 128, 1e-6, None, None) == INVALID   # HD != 128
    assert L.dd_attn_decode(fake, fake, fake, fake, 0, fake, fake, fake,
                            1, 9, 32, 8, 128, 128, 128, None) == INVALID         # W*G > 32
    assert L.dd_attn_decode(fake, fake, fake, fake, 0, fake, fake, fake,
                            1, 1, 32, 8, 128, 128, 100, None) == INVALID         # chunk % 32
    # the no-allocation attention: argument checks, then shapes past its static scratch
    # (24 MiB of split partials, 4096 counters) are refused with hipErrorOutOfMemory (2)
    assert L.dd_attn_decode_noalloc(fake, fake, fake, fake, 0, fake,
                                    1, 9, 32, 8, 128, 128, None) == INVALID          # W*G > 32
    assert L.dd_attn_decode_noalloc(None, fake, fake, fake, 0, fake,
                                    1, 1, 32, 8, 128, 128, None) == INVALID          # null q
    assert L.dd_attn_decode_noalloc(fake, fake, fake, fake, 0, fake,
                                    512, 8, 32, 8, 128, 128, None) == 2              # 68 MB ws
    assert L.dd_attn_decode_noalloc(fake, fake, fake, fake, 0, fake,
                                    513, 1, 32, 8, 128, 128, None) == 2              # B*NKV > 4096
    # prefill: HD 128 only, G <= 8 query heads per kv head, 16-byte aligned attention operands
    assert L.dd_qkv_post_prefill(fake, fake, fake, fake, fake, 64, fake, 1, 16, 0, fake, fake,
                                 fake, 32, 8, 64, 128, 1e-6, None, None) == INVALID   # HD != 128
    assert L.dd_qkv_post_prefill(None, fake, fake, fake, fake, 64, fake, 1, 16, 0, fake, fake,
                                 fake, 32, 8, 128, 128, 1e-6, None, None) == INVALID  # null qkv
    assert L.dd_qkv_post_prefill(fake, fake, fake, fake, fake, 64, fake, 0, 16, 0, fake, fake,
                                 fake, 32, 8, 128, 128, 1e-6, None, None) == INVALID  # B = 0
    assert L.dd_qkv_post_prefill(fake, fake, fake, fake, fake, 64, fake, 1, 16, 0, fake, fake,
                                 fake, 30, 8, 128, 128, 1e-6, None, None) == INVALID  # NH % NKV
    assert L.dd_attn_prefill(fake, fake, fake, fake, 1, 16, 0, fake, 72, 8, 128, 128,
                             None) == INVALID                                        # G = 9
    assert L.dd_attn_prefill(ctypes.c_void_p(0x1008), fake, fake, fake, 1, 16, 0, fake, 32, 8,
                             128, 128, None) == INVALID                              # misaligned q
    assert L.dd_attn_prefill(fake, fake, fake, None, 1, 16, 0, fake, 32, 8, 128, 128,
                             None) == INVALID                                        # no offsets
    assert L.dd_attn_prefill(fake, fake, fake, fake, 1, 0, 0, fake, 32, 8, 128, 128,
                             None) == INVALID                                        # T = 0
    # weight tiling: matrix 0..4, K a multiple of 256; aux = I > 0 for matrix 2 with N = 2 I;
    # aux = kv heads > 0 for matrix 0 with N / aux a whole number (>= 3) of 128-row heads
    assert L.dd_tile_weight(fake, fake, 64, 256, 5, 0, None) == INVALID
    assert L.dd_tile_weight(fake, fake, 64, 256, -1, 0, None) == INVALID
    assert L.dd_tile_weight(fake, fake, 768, 384, 0, 1, None) == INVALID
    assert L.dd_tile_weight(fake, fake, 64, 256, 2, 0, None) == INVALID
    assert L.dd_tile_weight(fake, fake, 64, 256, 2, 48, None) == INVALID
    assert L.dd_tile_weight(fake, fake, 64, 256, 1, 32, None) == INVALID
    assert L.dd_tile_weight(fake, fake, 768, 256, 0, 0, None) == INVALID      # no kv heads
    assert L.dd_tile_weight(fake, fake, 768, 256, 0, 5, None) == INVALID      # N % kv heads
    assert L.dd_tile_weight(fake, fake, 768, 256, 0, 3, None) == INVALID      # 256 rows per head
    assert L.dd_tile_weight(fake, fake, 512, 256, 0, 2, None) == INVALID      # < 3 heads per group
    assert L.dd_tile_weight(None, fake, 768, 256, 0, 1, None) == INVALID
    # uncached step counters: an output pointer is required; read-back needs both pointers
    assert L.dd_step_counters_alloc(None) == INVALID
    assert L.dd_step_counters_read(None, fake) == INVALID
    assert L.dd_step_counters_read(fake, None) == INVALID
    assert L.dd_tile_weight(ctypes.c_void_p(0x1008), fake, 768, 256, 0, 1, None) == INVALID


def _step_args(**kw):
    fake = ctypes.c_void_p(0x1000)
    a = dict(layer_table=fake, L=36, embed=fake, lm_tiled=fake, final_norm=fake, cos_t=fake,
             sin_t=fake, rope_rows=4096, tok=fake, out_tok=fake, pos=fake, h=fake, qkv=fake,
             attn=fake, mbuf=fake, logits=fake, ws=fake, counters=fake, err=fake, B=16, W=1,
             H=2560, NH=32, NKV=8, I=9728, V=151936, cap=3072, eps=1e-6, phase_begin=0,
             phase_end=2 + 5 * 36, stream=None)
    a.update(kw)
    return list(a.values())


@pytest.mark.parametrize("bad", [
    dict(B=17), dict(B=0), dict(W=0), dict(W=6), dict(B=16, W=6), dict(NH=64, W=5),
    dict(NH=30), dict(cap=0), dict(rope_rows=0), dict(H=2500),
    dict(I=9700), dict(H=4352), dict(V=0), dict(phase_end=3 + 5 * 36), dict(phase_begin=5, phase_end=5),
    dict(tok=None), dict(out_tok=None), dict(counters=None), dict(NKV=64, NH=64),
    dict(rope_rows=(1 << 23) + 1),
])
def test_decode_step_validation(bad):
    """dd_decode_step checks shapes and pointers before it queries the device or launches."""
    L = dryft_amd.lib()
    assert L.dd_decode_step(*_step_args(**bad)) == 1


def test_host_side_sizing():
    L = dryft_amd.lib()
    # split-K: keep >= 512 k per split, grow the grid toward 512 workgroups
    for N, K in ((151936, 2560), (6144, 2560), (2560, 4096), (2560, 9728), (19456, 2560)):
        sk = L.dd_gemv_splitk(16, N, K)
        tiles = -(-N // 16)
        assert sk >= 1 and K // sk >= 512
        # stops once the grid reaches 512 workgroups or another split would go under 512 k
        assert tiles * sk >= 512 or K // (2 * sk) < 512 or sk == 8
    assert L.dd_gemv_splitk(16, 151936, 2560) == 1
    for M, N, K in ((16, 2560, 4096), (1, 6144, 2560), (3, 64, 64)):
        sk = L.dd_gemv_splitk(M, N, K)
        assert L.dd_gemv_ws_bytes(M, N, K, sk) == (sk * M * N * 4 if sk > 1 else 0)
        # partials | hn as bf16 (rounded up to whole floats) | per-tile sums of squares
        assert L.dd_gemv_add_rmsnorm_ws_bytes(M, N, K, sk) == 4 * (sk * M * N + (M * N + 1) // 2 + -(-N // 16) * M)
        assert L.dd_gemv_counters(N) == -(-N // 16) + 1
    assert L.dd_argmax_ws_bytes(16, 151936) == 16 * 38 * 2 * 4
    assert L.dd_tiled_bytes(6144, 2560) == 6144 * 2560 * 2
    assert L.dd_step_counters() >= 1024 + 512
    # attention: chunk multiple of 128, workspace covers every split of every row
    for B, cap in ((1, 640), (16, 3072), (16, 8192)):
        c = L.dd_attn_chunk(B, 8, cap)
        assert c % 128 == 0 and c >= 128
        nsplit = -(-cap // c)
        assert L.dd_attn_ws_bytes(B, 1, 32, 8, 128, cap, c) == B * 8 * nsplit * 4 * 130 * 4


@pytest.mark.parametrize("status", [0, 1, 700])
def test_check_raises_on_nonzero(status):
    if status == 0:
        _lib.check(0, "x")
    else:
        with pytest.raises(RuntimeError):
            _lib.check(status, "x")

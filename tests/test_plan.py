"""CPU: the host-side rules that choose a kernel, through the library's
exported functions (no GPU work)."""
import pytest

import llmt
import native


def test_attention_forward_split_is_bounded_by_its_workgroups():
    """Keys are split over the waves of 32-query blocks only up to 1280
    workgroups, however few the heads, and of 16-query blocks up to 512."""
    f = native.fn(llmt.lib(), "_ZN4llmt20attn_fwd_split_tilesEiii", native.i32, *[native.i32] * 3)
    for heads in (1, 2, 3, 4, 6, 8, 12, 16, 24, 32, 64):
        for B in (b for b in (1, 2, 4) if heads % b == 0):
            for S in (1, 16, 17, 255, 256, 512, 1024, 2048, 4096, 5120, 6144, 8192, 16384, 65536):
                t = f(B, S, heads // B)
                assert t in (0, 1, 2)
                if t:
                    assert heads * -(-S // (16 * t)) <= (512 if t == 1 else 1280), (B, S, heads)
                if heads * -(-S // 16) <= 512:
                    assert t == 1, (B, S, heads)
    # both sides of the line at 8 heads, and of the heads' own
    assert [f(1, s, 8) for s in (4096, 5120, 5121, 8192)] == [2, 2, 0, 0]
    assert [f(1, s, 16) for s in (512, 513, 2048, 2049)] == [1, 2, 2, 0]
    assert [f(2, s, 16) for s in (256, 257, 512, 513)] == [1, 2, 2, 0]


def test_attention_backward_split_lines():
    """dQ blocks split their keys with up to 16 heads and 1536 workgroups: past
    320 of them, and from S = 768 at any count with at most two query heads a
    KV head (one head at S = 4096 counts exactly 320); dK/dV blocks alone up
    to 800."""
    f = native.fn(llmt.lib(), "_ZN4llmt14attn_bwd_splitEiiii", native.i32, *[native.i32] * 4)
    assert [f(1, s, 1, 1) for s in (767, 768, 4095, 4096, 4097, 19648, 19649)] == [1, 2, 2, 2, 2, 2, 0]
    assert [f(1, s, 6, 2) for s in (768, 1456, 1457, 7008, 7009)] == [1, 1, 2, 2, 0]
    assert [f(1, s, 16, 8) for s in (16, 416, 417, 2048, 2049)] == [1, 1, 2, 2, 0]
    assert [f(1, s, 32, 8) for s in (128, 768, 769)] == [1, 1, 0]

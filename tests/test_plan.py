"""CPU: the host-side rules that choose a kernel, through the library's
exported functions (no GPU work)."""
import ctypes as C

import pytest
import torch

import llmt
import native

# calls that must be refused, with addresses that are never read: only where
# a call that is not refused has no device to launch on
no_gpu = pytest.mark.skipif(torch.cuda.is_available(), reason="runs without a GPU only")


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


def _gemm(M, N, K, i8=False, split=1, A=0x10000, **kw):
    """Arguments of a GEMM of one segment (addresses that are never read)."""
    g = native.GemmArgs()
    g.A, g.lda, g.nseg, g.M, g.N, g.K, g.split = A, K, 1, M, N, K, split
    g.seg[0].ptr, g.seg[0].rows, g.seg[0].ld, g.seg[0].is_i8 = 0x20000, N, K, i8
    for i in range(1, 5):
        g.seg_start[i] = N
    g.C, g.ldc = 0x30000, N
    for k, v in kw.items():
        setattr(g, k, v)
    return g


@no_gpu
@pytest.mark.parametrize("i8", [False, True])
@pytest.mark.parametrize("M", [16, 128, 512, 1040, 4096])
def test_swiglu_gemm_refuses_a_per_k_scale(M, i8):
    """No SwiGLU epilogue applies a per-k scale, whatever tile the plan takes:
    such a GEMM is refused before any launch, not computed without the scale."""
    L = llmt.lib()
    g = _gemm(M, 12288, 2048, i8, glu=6144, glu16=0x40000, ldglu=6144, gu16=0x50000)
    g.seg[0].kscale = 0x60000
    assert native.gemm_nt(L, g) == native.HIP_ERROR_INVALID_VALUE
    assert "per-k scale" in L.llmt_last_error().decode()


@no_gpu
@pytest.mark.parametrize("M", [16, 128, 512, 4096])
@pytest.mark.parametrize("field", ["kscale", "colscale"])
def test_gemm_refuses_a_scale_on_fp16_rows(M, field):
    """The scales are int8 rows': on fp16 rows no kernel but one applied them."""
    L = llmt.lib()
    g = _gemm(M, 2048, 2048)
    setattr(g.seg[0], field, 0x60000)
    assert native.gemm_nt(L, g) == native.HIP_ERROR_INVALID_VALUE
    assert "scale" in L.llmt_last_error().decode()


@pytest.mark.parametrize("stages", ["", "0"])
def test_split_col_gemm_keeps_its_kernel(monkeypatch, stages):
    """A GEMM whose last tiles are split runs on the 256 x 256 tiles, also where
    the override takes other fp16 GEMMs of M % 128 == 0 to the register-staged
    kernel (which cannot split single tiles: the GEMM would be refused)."""
    monkeypatch.setenv("LLMT_GEMM_SKINNY_STAGES", stages)
    L = llmt.lib()
    M, N, K = 4096, 8448, 512
    col = native.gemm_split_col(L, M, N, K, False)
    assert 0 < col < N
    g = _gemm(M, N, K, split=2, split_col=col, split_stride=M * N)
    assert native.gemm_kernel_name(L, g) == "gemm_dma"


@pytest.mark.parametrize("i8", [False, True])
@pytest.mark.parametrize("M", [16, 48, 128, 144, 336, 1024, 1040, 4096])
@pytest.mark.parametrize("offset", [0, 2, 4, 8, 14])
def test_gemm_with_unaligned_rows_takes_the_register_kernel(M, offset, i8):
    """The LDS-DMA kernels move A in 16-byte pieces; rows that are not aligned to
    them go through the register-staged kernel, with or without statistics."""
    L = llmt.lib()
    g = _gemm(M, 4096, 2048, i8, A=0x10000 + offset)
    assert (native.gemm_kernel_name(L, g) == "gemm_nt") == (offset != 0)
    if not i8:
        n = native.gemm_rowstats_tiles(L, g)
        g.rowstats = 0x70000
        assert (native.gemm_kernel_name(L, g) == "gemm_nt") == (offset != 0)
        assert n == native.gemm_rowstats_tiles(L, g) and 0 < n <= 4096 // 128
    g = _gemm(M, 4096, 2048, i8, lda=2052)
    assert native.gemm_kernel_name(L, g) == "gemm_nt"


def test_standalone_products_count_their_reduction():
    """A standalone product split over K pays a second launch that sums the
    parts, so it is split only where the split saves more than that; in the step
    the sum is part of a row pass that runs anyway."""
    L = llmt.lib()
    split = lambda M, N, K, reduce: native.gemm_plan(L, M, [(N, 0)], K, reduce=reduce)[1]
    for M, N, K in ((256, 4096, 2048), (384, 4096, 2048), (512, 3072, 3072), (128, 14336, 4096)):
        assert split(M, N, K, False) > 1 and split(M, N, K, True) == 1, (M, N, K)
    for M, N, K in ((16, 2048, 6144), (128, 2048, 6144), (128, 1024, 4096), (128, 256, 151936)):
        assert split(M, N, K, True) > 1, (M, N, K)
    for M in (16, 48, 128, 512, 1024, 4096):
        for N, K in ((16, 64), (2048, 2048), (12288, 2048), (4096, 192)):
            assert split(M, N, K, True) <= split(M, N, K, False)

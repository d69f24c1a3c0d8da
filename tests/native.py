"""ctypes mirrors of the library's internal launch arguments (csrc/ops.h) and
its exported C++ entry points, for tests of one kernel or of a host-side rule
that no C entry point reaches alone."""
import ctypes as C

vp, i32, i64, f32 = C.c_void_p, C.c_int, C.c_longlong, C.c_float
HIP_ERROR_INVALID_VALUE = 1


def _struct(name, fields):
    return type(name, (C.Structure,), {"_fields_": fields})


BSeg = _struct("BSeg", [("ptr", vp), ("colscale", vp), ("kscale", vp), ("rows", i32), ("ld", i32),
                        ("is_i8", i32)])
GemmArgs = _struct("GemmArgs", [
    ("A", vp), ("lda", i32), ("seg", BSeg * 4), ("seg_start", i32 * 5), ("nseg", i32), ("C", vp),
    ("ldc", i32), ("split_stride", i64), ("M", i32), ("N", i32), ("K", i32), ("split", i32),
    ("split_col", i32), ("glu", i32), ("glu16", vp), ("ldglu", i32), ("gu16", vp),
    ("rowstats", vp)])
LoraTerm = _struct("LoraTerm", [("shr", vp), ("row0", i32), ("kp", i32), ("c0", i32), ("n", i32),
                                ("hidx", i32)])
RowIn = _struct("RowIn", [
    ("part", vp), ("split", i32), ("ss", i64), ("ldp", i32), ("split_col", i32), ("hcol", i32),
    ("nh", i32), ("nterm", i32), ("term", LoraTerm * 3), ("lscale", f32)])
NormBwdArgs = _struct("NormBwdArgs", [
    ("inp", RowIn), ("rinv_in", vp), ("gscale", f32), ("dh_out", vp), ("dh_col", i32), ("x", vp),
    ("w", vp), ("eps", f32), ("H", i32), ("dres_in", vp), ("dres_out", vp), ("dmid_out", vp),
    ("g16", vp), ("rinv_out", vp), ("g16_ks", vp), ("lora_at", vp)])


def fn(L, symbol, restype, *argtypes):
    f = getattr(L, symbol)
    f.restype, f.argtypes = restype, list(argtypes)
    return f


def norm_bwd(L, args, T, stream=None):
    """hipError_t of llmt::norm_bwd(const NormBwdArgs&, int, hipStream_t)."""
    f = fn(L, "_ZN4llmt8norm_bwdERKNS_11NormBwdArgsEiP12ihipStream_t", i32,
           C.POINTER(NormBwdArgs), i32, vp)
    return f(C.byref(args), T, stream)


def gemm_nt(L, args, stream=None):
    """hipError_t of llmt::gemm_nt(const GemmArgs&, hipStream_t)."""
    f = fn(L, "_ZN4llmt7gemm_ntERKNS_8GemmArgsEP12ihipStream_t", i32, C.POINTER(GemmArgs), vp)
    return f(C.byref(args), stream)


def gemm_kernel_name(L, args):
    """Name of the kernel gemm_nt launches for these arguments."""
    f = fn(L, "_ZN4llmt16gemm_kernel_nameERKNS_8GemmArgsE", C.c_char_p, C.POINTER(GemmArgs))
    return f(C.byref(args)).decode()


def gemm_split_col(L, M, N, K, i8):
    f = fn(L, "_ZN4llmt14gemm_split_colEiiib", i32, i32, i32, i32, C.c_bool)
    return f(M, N, K, i8)


def gemm_rowstats_tiles(L, args):
    f = fn(L, "_ZN4llmt19gemm_rowstats_tilesERKNS_8GemmArgsE", i32, C.POINTER(GemmArgs))
    return f(C.byref(args))


def gemm_plan(L, M, segs, K, glu=0, reduce=False):
    """(kernel name, split) of a GEMM of the given (rows, int8) segments, planned
    as the step plans it (reduce: as the standalone products are): the library's
    own split, or the SwiGLU epilogue.  No address is read."""
    g = GemmArgs()
    g.A, g.lda, g.M, g.K, g.nseg, g.split = 0x10000, K, M, K, len(segs), 1
    n = 0
    for i, (rows, i8) in enumerate(segs):
        g.seg[i].ptr, g.seg[i].rows, g.seg[i].ld, g.seg[i].is_i8 = 0x20000, rows, K, i8
        g.seg_start[i] = n
        n += rows
    for i in range(len(segs), 5):
        g.seg_start[i] = n
    g.N = g.ldc = n
    g.C = 0x30000
    if glu:
        g.glu = g.ldglu = glu
        g.glu16, g.gu16 = 0x40000, 0x50000
    else:
        pick = fn(L, "_ZN4llmt15gemm_pick_splitEiiiibb", i32, i32, i32, i32, i32, C.c_bool, C.c_bool)
        g.split = pick(M, n, K, 64, bool(segs[0][1]), reduce)
    return gemm_kernel_name(L, g), g.split


def layer_plan(L, d, T, i8):
    """The kernels of one layer's eight GEMMs on T tokens, by name: forward qkv,
    o, gu (gate/up), down; backward dX ddx, gudx, odx, qkvdx."""
    H, I, r = d.hidden, d.intermediate, 16
    Q, KV = d.n_heads * 128, d.n_kv_heads * 128
    NT = Q + 2 * KV
    shapes = {"qkv": ([(NT, i8), (3 * r, 0)], H, 0), "o": ([(H, i8), (r, 0)], Q, 0),
              "gu": ([(2 * I, i8)], H, I), "down": ([(H, i8)], I, 0), "ddx": ([(I, i8)], H, 0),
              "gudx": ([(H, i8)], 2 * I, 0), "odx": ([(Q, i8), (r, 0)], H, 0),
              "qkvdx": ([(H, i8), (3 * r, 0)], NT, 0)}
    return {n: gemm_plan(L, T, segs, K, glu)[0] for n, (segs, K, glu) in shapes.items()}

"""The C-ABI library loads without a GPU, exports every symbol the header
declares, and rejects bad arguments on the host before anything is launched."""
import ctypes as C
import os
import re

import pytest

from longcat_video_amd import _capi

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "bsa_mi355x.h")
FAKE = C.c_void_p(0x10000)          # never dereferenced: validation fails first


def declared_functions():
    text = re.sub(r"/\*.*?\*/", "", open(HEADER).read(), flags=re.S)
    return sorted(set(re.findall(r"\b(bsa_[a-z0-9_]+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    lib = _capi.load()
    names = declared_functions()
    assert "bsa_fwd_3d" in names and "bsa_permute_thw_to_blocks" in names and len(names) >= 12
    for n in names:
        assert hasattr(lib, n), "library lacks %s" % n
        assert n in _capi.SIGNATURES, "binding lacks %s" % n
    assert sorted(_capi.SIGNATURES) == names


def test_version_and_error_string():
    lib = _capi.load()
    assert lib.bsa_version() >= 100
    assert isinstance(_capi.last_error(), str)


@pytest.mark.parametrize("sparsity,n", [(0.875, 8), (0.9375, 1440), (0.9, 10), (0.0, 7), (1.0, 7), (0.3, 10), (0.9375, 624)])
def test_num_selected_matches_python_doubles(sparsity, n):
    assert _capi.load().bsa_num_selected(sparsity, n) == int((1 - sparsity) * n)


def test_padded_tokens():
    lib = _capi.load()
    assert lib.bsa_padded_tokens(24, 45, 80, 4, 4, 4) == 92160
    assert lib.bsa_padded_tokens(24, 30, 52, 4, 4, 4) == 39936
    assert lib.bsa_padded_tokens(4, 8, 8, 4, 4, 4) == 256
    assert lib.bsa_padded_tokens(0, 8, 8, 4, 4, 4) == -1


def test_permute_rejects_bad_arguments():
    lib = _capi.load()
    st = _capi.strides3([256 * 128, 256 * 128, 128])
    ok_tail = (1, 1, 4, 8, 8, 4, 4, 4, 128, _capi.BSA_BF16, None)
    assert lib.bsa_permute_thw_to_blocks(None, st, FAKE, None, None, *ok_tail) == _capi.BSA_ERR_BAD_ARG
    assert "null" in _capi.last_error()
    assert lib.bsa_permute_thw_to_blocks(FAKE, None, FAKE, None, None, *ok_tail) == _capi.BSA_ERR_BAD_ARG
    bad_dtype = ok_tail[:9] + (7, None)
    assert lib.bsa_permute_thw_to_blocks(FAKE, st, FAKE, None, None, *bad_dtype) == _capi.BSA_ERR_UNSUPPORTED
    odd_d = ok_tail[:8] + (100, _capi.BSA_BF16, None)     # 200-byte rows
    assert lib.bsa_permute_thw_to_blocks(FAKE, st, FAKE, None, None, *odd_d) == _capi.BSA_ERR_UNSUPPORTED
    zero = (1, 1, 0, 8, 8, 4, 4, 4, 128, _capi.BSA_BF16, None)
    assert lib.bsa_permute_thw_to_blocks(FAKE, st, FAKE, None, None, *zero) == _capi.BSA_ERR_BAD_ARG
    misaligned = C.c_void_p(0x10002)
    assert lib.bsa_permute_thw_to_blocks(misaligned, st, FAKE, None, None, *ok_tail) == _capi.BSA_ERR_BAD_ARG
    bad_stride = _capi.strides3([256 * 128, 256 * 128, 100])
    assert lib.bsa_permute_thw_to_blocks(FAKE, bad_stride, FAKE, None, None, *ok_tail) == _capi.BSA_ERR_BAD_ARG
    small_chunk = (1, 1, 4, 8, 8, 2, 2, 2, 128, _capi.BSA_BF16, None)   # 8-token chunk: no 64-slot tiles
    assert lib.bsa_permute_thw_to_blocks(FAKE, st, FAKE, None, FAKE, *small_chunk) == _capi.BSA_ERR_UNSUPPORTED


def test_topk_rejects_bad_arguments():
    lib = _capi.load()
    assert lib.bsa_topk_from_score(FAKE, FAKE, None, FAKE, 1, 1, 4, 4, 5, _capi.BSA_BF16, None) == _capi.BSA_ERR_SHAPE
    assert lib.bsa_topk_from_score(FAKE, FAKE, None, FAKE, 1, 1, 4, 5000, 5, _capi.BSA_BF16, None) == _capi.BSA_ERR_UNSUPPORTED
    assert lib.bsa_topk_from_score(FAKE, FAKE, None, FAKE, 1, 1, 4, 4096, 4097, _capi.BSA_BF16, None) == _capi.BSA_ERR_SHAPE
    assert lib.bsa_topk_from_score(None, FAKE, None, FAKE, 1, 1, 4, 4, 2, _capi.BSA_BF16, None) == _capi.BSA_ERR_BAD_ARG
    assert lib.bsa_score_topk(FAKE, FAKE, FAKE, None, FAKE, FAKE, 1, 1, 4, 4, 100, 2, _capi.BSA_BF16, None) == _capi.BSA_ERR_UNSUPPORTED
    assert lib.bsa_score_topk(FAKE, FAKE, FAKE, None, FAKE, None, 1, 1, 4, 4, 128, 2, _capi.BSA_BF16, None) == _capi.BSA_ERR_BAD_ARG
    assert lib.bsa_score_topk(FAKE, FAKE, None, None, FAKE, FAKE, 1, 1, 4, 4, 128, 2, _capi.BSA_BF16, None) == _capi.BSA_ERR_BAD_ARG


def test_fwd_rejects_bad_arguments():
    lib = _capi.load()
    ptrs = [FAKE] * 5 + [None, FAKE, None]

    def call(B=1, Hn=1, Sq=256, Sk=256, D=128, bs_q=64, bs_k=64, stride=2, scale=0.088, dtype=_capi.BSA_BF16, p=ptrs):
        return lib.bsa_fwd(*p, B, Hn, Sq, Sk, D, bs_q, bs_k, stride, scale, dtype, None)

    assert call(D=64) == _capi.BSA_ERR_UNSUPPORTED and "128" in _capi.last_error()
    assert call(bs_q=48) == _capi.BSA_ERR_UNSUPPORTED
    assert call(Sq=200) == _capi.BSA_ERR_SHAPE
    assert call(Sk=100) == _capi.BSA_ERR_SHAPE
    assert call(scale=0.0) == _capi.BSA_ERR_BAD_ARG
    assert call(scale=float("nan")) == _capi.BSA_ERR_BAD_ARG
    assert call(dtype=9) == _capi.BSA_ERR_UNSUPPORTED
    assert call(B=0) == _capi.BSA_ERR_BAD_ARG
    assert call(p=[None] + ptrs[1:]) == _capi.BSA_ERR_BAD_ARG


def test_fwd_fragment_and_bwd_shape_limits():
    """The blocked-order entry on the fragment-order kernel and the backward reject what they cannot run before any
    launch (no GPU is touched: every check comes before the first HIP call)."""
    lib = _capi.load()
    need = lib.bsa_fwd_fragment_workspace_bytes(1, 2, 640, 1280, 128, _capi.BSA_BF16)
    assert need >= 2 * 2 * 1280 * 128 * 2 and need % 256 == 0                      # K and V in fragment order, two tables
    assert lib.bsa_fwd_fragment_workspace_bytes(1, 2, 640, 1280, 128, _capi.BSA_F32) == 0
    assert lib.bsa_fwd_fragment_workspace_bytes(1, 2, 640, 1290, 128, _capi.BSA_BF16) == 0
    ptrs = [FAKE] * 5 + [None, FAKE, None]

    def call(Sq=640, Sk=1280, D=128, bs_q=64, bs_k=64, stride=3, dtype=_capi.BSA_BF16, ws=FAKE, ws_bytes=1 << 30):
        return lib.bsa_fwd_fragment(*ptrs, 1, 2, Sq, Sk, D, bs_q, bs_k, stride, 0.088, dtype, ws, ws_bytes, None)

    assert call(dtype=_capi.BSA_F32) == _capi.BSA_ERR_UNSUPPORTED
    assert call(D=64) == _capi.BSA_ERR_UNSUPPORTED
    assert call(Sq=650) == _capi.BSA_ERR_SHAPE
    assert call(stride=5000) == _capi.BSA_ERR_UNSUPPORTED and "4096" in _capi.last_error()
    assert call(ws=None) == _capi.BSA_ERR_BAD_ARG
    assert call(ws_bytes=need - 1) == _capi.BSA_ERR_WORKSPACE
    # the backward stages a KV block's query blocks in LDS: more query blocks than fit are refused, with the number
    assert lib.bsa_bwd_workspace_bytes(1, 1, 64 * 23552, 64, 128, 64, 64, 1, _capi.BSA_BF16) > 0
    assert lib.bsa_bwd_workspace_bytes(1, 1, 64 * 23553, 64, 128, 64, 64, 1, _capi.BSA_BF16) == 0
    assert "23552" in _capi.last_error()


def test_fwd_3d_plan_and_workspace():
    lib = _capi.load()
    prm = _capi.Bsa3dParams(1, 32, 128, _capi.BSA_BF16, 24, 45, 80, 24, 45, 80, 4, 4, 4, 4, 4, 4, 90, 0.0883883)
    need = lib.bsa_workspace_bytes(C.byref(prm))
    # q and o are used where they lie; k and v are rewritten once, in fragment order, at their padded size;
    # plus pooled vectors, the score matrix and the lists
    kv = 2 * 32 * 92160 * 128 * 2
    assert need > kv and need < kv + 300 * 2 ** 20
    prm32 = _capi.Bsa3dParams(1, 32, 128, _capi.BSA_F32, 24, 45, 80, 24, 45, 80, 4, 4, 4, 4, 4, 4, 90, 0.0883883)
    # fp32: no tensor is copied; pooled vectors, the score matrix and the lists, in fp32
    assert 32 * 1440 * 1440 * 4 < lib.bsa_workspace_bytes(C.byref(prm32)) < 32 * 1440 * 1440 * 4 + 200 * 2 ** 20
    st = _capi.strides3([32 * 86400 * 128, 86400 * 128, 128])
    args = (FAKE, st, FAKE, st, FAKE, st, FAKE, st)
    ws = C.c_void_p(0x100000)
    assert lib.bsa_fwd_3d(C.byref(prm), *args, ws, need - 1, None, None, None, None) == _capi.BSA_ERR_WORKSPACE
    assert lib.bsa_fwd_3d(C.byref(prm), *args, C.c_void_p(0x100010), need, None, None, None, None) == _capi.BSA_ERR_BAD_ARG
    prm.k_sel = 2000
    assert lib.bsa_workspace_bytes(C.byref(prm)) == 0
    assert lib.bsa_fwd_3d(C.byref(prm), *args, ws, need, None, None, None, None) == _capi.BSA_ERR_SHAPE
    prm.k_sel, prm.D = 90, 64
    assert lib.bsa_fwd_3d(C.byref(prm), *args, ws, need, None, None, None, None) == _capi.BSA_ERR_UNSUPPORTED
    prm.D, prm.tq = 128, 2                          # 32-token query chunks
    assert lib.bsa_fwd_3d(C.byref(prm), *args, ws, need, None, None, None, None) == _capi.BSA_ERR_UNSUPPORTED
    assert lib.bsa_fwd_3d(None, *args, ws, need, None, None, None, None) == _capi.BSA_ERR_BAD_ARG


@pytest.mark.parametrize("heads,T,H,W", [(23, 28, 28, 80), (25, 24, 48, 52), (25, 32, 36, 52), (25, 36, 32, 52)])
def test_fwd_3d_static_takes_what_its_buffer_holds(heads, T, H, W):
    """The largest problems of its 64 MiB at density 1/16: no room for an order of k's chunk means that this route does not use."""
    lib = _capi.load()
    n = T // 4 * (H // 4) * (W // 4)
    prm = _capi.Bsa3dParams(1, heads, 128, _capi.BSA_BF16, T, H, W, T, H, W, 4, 4, 4, 4, 4, 4, n // 16, 0.0883883)
    st = _capi.strides3([heads * T * H * W * 128, T * H * W * 128, 128])
    call = lambda: lib.bsa_fwd_3d_static(C.byref(prm), None, st, FAKE, st, FAKE, st, FAKE, st, None, None, None, None)      # noqa: E731
    assert call() in (_capi.BSA_ERR_HIP, _capi.BSA_ERR_BAD_ARG)      # no GPU, or the tensor that is missing: behind the test of the size
    prm.Hn = heads + 1
    assert call() == _capi.BSA_ERR_WORKSPACE


def test_which_linear_layers_work_without_a_product():
    """With a residual, a layer that the engine's GEMM serves needs the 64 MiB that every call brings; any other an fp32 product too."""
    lib = _capi.load()
    least = 64 << 20

    def alone(x=0x100000000, ldx=1024, w=0x200000000, ldw=1024, bias=0x300000000, res=0x400000000, out=0x500000000, ldo=1024, M=65536, N=1024, K=1024):
        p = lambda v: None if v is None else C.c_void_p(v)      # noqa: E731
        got = lib.bsa_linear_bf16_ld_workspace_bytes(p(x), ldx, p(w), ldw, p(bias), p(res), p(out), ldo, M, N, K)
        assert got in (least, lib.bsa_linear_bf16_workspace_bytes(M, N, 1)) and lib.bsa_linear_bf16_workspace_bytes(M, N, 1) > least
        return got == least

    assert alone() and alone(bias=None) and alone(out=0x400000000) and alone(M=16 * 256 * 4) and alone(K=64, M=3)
    assert alone(res=None)                                          # no residual: no product either
    assert not alone(M=256) and not alone(M=70 * 256)               # 4 tiles; 280: two rounds of 256, little more than half full
    assert alone(M=90 * 256 * 4)
    assert not alone(K=1000, ldx=1000) and not alone(N=1000) and not alone(ldx=1028) and not alone(ldo=1028)
    for bad in ("x", "w", "res", "out"):
        assert not alone(**{bad: 0x600000008})
    assert not alone(bias=0x300000004) and alone(bias=0x300000008)
    # results over operands that are still read: only in the residual's own place
    assert not alone(out=0x100000000) and not alone(out=0x200000000) and not alone(out=0x400000800) and not alone(out=0x300000000)
    assert not alone(out=0x100000000 + (65536 * 1024 * 2 - 16)) and alone(out=0x100000000 + 65536 * 1024 * 2)


def test_layers_behind_a_gate_or_with_a_branch_reject_bad_arguments():
    lib = _capi.load()
    p = [C.c_void_p(0x100000000 * i) for i in range(1, 9)]
    ups = (C.c_void_p * 1)(0x900000000)

    def gated(x=p[0], w=p[1], t=p[2], up=ups, res=p[3], gate=p[4], rows=4, out=p[5], M=8, N=256, K=128):
        return lib.bsa_linear_gated_bf16(x, w, None, t, 64, up, 1, 64, 1.0, 1.0, res, gate, rows, out, M, N, K, p[6], 64 << 20, None)

    for bad in ("x", "w", "up", "res", "gate", "out"):
        assert gated(**{bad: None}) == _capi.BSA_ERR_BAD_ARG
    assert gated(out=p[3]) == _capi.BSA_ERR_BAD_ARG                   # over the residual
    assert gated(M=0) == gated(N=0) == gated(K=0) == _capi.BSA_ERR_BAD_ARG
    assert gated(rows=3) == gated(rows=0) == _capi.BSA_ERR_SHAPE
    args = [p[0], p[1], None, p[2], 64, ups, 1, 64, 1.0, 1.0, p[5], 8, 256, 128, p[6], 64 << 20, None]
    for i in (0, 1, 3, 5, 10):
        assert lib.bsa_linear_lora_bf16(*args[:i], None, *args[i + 1:]) == _capi.BSA_ERR_BAD_ARG


@pytest.mark.parametrize("K,M", [(128, 8), (1000, 8), (4096, 4608)])      # served whatever the tiles; not served; served without a branch alone
def test_layers_behind_a_gate_or_with_a_branch_refuse_results_over_their_operands(K, M):
    """`out` is written while they are still read, or before: also where a few bytes meet; refused in front of any launch."""
    lib = _capi.load()
    N, r, rows = 512, 64, 4
    size = dict(x=M * K * 2, w=N * K * 2, bias=N * 2, t=((M - 1) * 72 + r) * 2, up=N * r * 2, res=M * N * 2, gate=M // rows * N * 4)
    at = {name: 0x100000000 * (i + 1) for i, name in enumerate(size)}
    ws = C.c_void_p(0xb00000000)
    p = {name: C.c_void_p(a) for name, a in at.items()}
    ups = (C.c_void_p * 1)(at["up"])

    def gated(out, t=p["t"]):
        return lib.bsa_linear_gated_bf16(p["x"], p["w"], p["bias"], t, 72, ups, 1, r, 1.0, 0.5, p["res"], p["gate"], rows, C.c_void_p(out), M, N, K, ws, 64 << 20, None)

    def lora(out):
        return lib.bsa_linear_lora_bf16(p["x"], p["w"], p["bias"], p["t"], 72, ups, 1, r, 1.0, 0.5, C.c_void_p(out), M, N, K, ws, 64 << 20, None)

    for name, a in at.items():
        for out in (a, a + size[name] // 16 * 16 - 16, a - M * N * 2 + 16):
            assert gated(out) == _capi.BSA_ERR_BAD_ARG and "own" in _capi.last_error(), name
            if name not in ("t", "up"):
                assert gated(out, None) == _capi.BSA_ERR_BAD_ARG
            if name not in ("res", "gate"):
                assert lora(out) == _capi.BSA_ERR_BAD_ARG and "own" in _capi.last_error(), name


def test_gemm_and_qkv_projection_reject_bad_arguments():
    lib = _capi.load()

    def gemm(x=FAKE, ldx=256, w=FAKE, ldw=256, bias=None, res=None, ldr=0, out=FAKE, ldo=256, M=300, N=256, K=256):
        return lib.bsa_gemm_bf16(x, ldx, w, ldw, bias, res, ldr, out, ldo, M, N, K, None)

    assert gemm(x=None) == _capi.BSA_ERR_BAD_ARG
    assert gemm(out=None) == _capi.BSA_ERR_BAD_ARG
    assert gemm(K=96, ldx=96, ldw=96) == _capi.BSA_ERR_UNSUPPORTED and "64" in _capi.last_error()
    assert gemm(N=200, ldo=200) == _capi.BSA_ERR_UNSUPPORTED and "128" in _capi.last_error()
    assert gemm(ldx=128) == _capi.BSA_ERR_BAD_ARG                   # row stride below K
    assert gemm(ldo=128) == _capi.BSA_ERR_BAD_ARG                   # row stride below N
    assert gemm(res=FAKE, ldr=100) == _capi.BSA_ERR_BAD_ARG
    assert gemm(M=0) == _capi.BSA_ERR_BAD_ARG
    assert gemm(x=C.c_void_p(0x10008)) == _capi.BSA_ERR_BAD_ARG     # 16-byte alignment
    assert gemm(ldx=1 << 23) == _capi.BSA_ERR_UNSUPPORTED

    st = _capi.strides3([4 * 256 * 128, 256 * 128, 128])

    def qkv(x=FAKE, q=FAKE, tab=FAKE, qw=FAKE, B=1, Hn=4, T=4, H=8, W=8, t0=0, table_T=4, D=128, K=512, eps=1e-6, strides=st):
        return lib.bsa_qkv_projection(x, K, FAKE, K, None, qw, FAKE, tab, q, FAKE, FAKE, strides, B, Hn, T, H, W, t0, table_T, D, K, eps, None)

    assert qkv(D=64) == _capi.BSA_ERR_UNSUPPORTED
    assert qkv(x=None) == _capi.BSA_ERR_BAD_ARG
    assert qkv(q=None) == _capi.BSA_ERR_BAD_ARG
    assert qkv(tab=None) == _capi.BSA_ERR_BAD_ARG
    assert qkv(qw=None) == _capi.BSA_ERR_BAD_ARG
    assert qkv(T=0) == _capi.BSA_ERR_BAD_ARG
    assert qkv(t0=2) == _capi.BSA_ERR_SHAPE                         # frames 2..6 of a table of 4
    assert qkv(K=100) == _capi.BSA_ERR_UNSUPPORTED
    assert qkv(eps=-1.0) == _capi.BSA_ERR_BAD_ARG
    assert qkv(strides=_capi.strides3([4 * 256 * 128, 256 * 128, 100])) == _capi.BSA_ERR_BAD_ARG


def test_fwd_3d_qknorm_rejects_bad_arguments():
    lib = _capi.load()
    prm = _capi.Bsa3dParams(1, 4, 128, _capi.BSA_BF16, 4, 8, 8, 4, 8, 8, 4, 4, 4, 4, 4, 4, 2, 0.0883883)
    need = lib.bsa_workspace_bytes(C.byref(prm))
    st = _capi.strides3([4 * 256 * 128, 256 * 128, 128])
    ws = C.c_void_p(0x100000)

    def call(p=prm, n=None, qn=FAKE, q_weight=FAKE, tab=FAKE, table_T=4, t_q=0, t_k=0, eps=1e-6):
        norm = _capi.BsaQkNorm(q_weight, FAKE, tab, table_T, t_q, t_k, eps) if n is None else n
        return lib.bsa_fwd_3d_qknorm(C.byref(p), C.byref(norm) if norm is not False else None, FAKE, st, qn, st, FAKE, st, FAKE, st,
                                     FAKE, st, ws, need, None, None, None, None)

    assert call(n=False) == _capi.BSA_ERR_BAD_ARG
    assert call(qn=None) == _capi.BSA_ERR_BAD_ARG
    assert call(q_weight=None) == _capi.BSA_ERR_BAD_ARG
    assert call(tab=None) == _capi.BSA_ERR_BAD_ARG
    assert call(table_T=3) == _capi.BSA_ERR_SHAPE
    assert call(t_k=1) == _capi.BSA_ERR_SHAPE
    assert call(eps=-1.0) == _capi.BSA_ERR_BAD_ARG
    assert call(q_weight=C.c_void_p(0x10008)) == _capi.BSA_ERR_BAD_ARG
    big = _capi.Bsa3dParams(1, 4, 128, _capi.BSA_BF16, 4, 8, 8, 4, 8, 8, 4, 4, 8, 4, 4, 8, 1, 0.0883883)      # 128-token chunks
    assert call(p=big) == _capi.BSA_ERR_UNSUPPORTED and "64-token" in _capi.last_error()
    f32 = _capi.Bsa3dParams(1, 4, 128, _capi.BSA_F32, 4, 8, 8, 4, 8, 8, 4, 4, 4, 4, 4, 4, 2, 0.0883883)
    assert call(p=f32) == _capi.BSA_ERR_UNSUPPORTED
    long_axis = _capi.Bsa3dParams(1, 4, 128, _capi.BSA_BF16, 4, 8, 16, 4, 8, 16, 1, 4, 16, 1, 4, 16, 2, 0.0883883)  # 16 positions on one axis
    assert call(p=long_axis) == _capi.BSA_ERR_UNSUPPORTED


def test_status_to_exception_mapping():
    lib = _capi.load()
    rc = lib.bsa_topk_from_score(FAKE, FAKE, None, FAKE, 1, 1, 4, 4, 5, _capi.BSA_BF16, None)
    with pytest.raises(AssertionError):
        _capi.check(rc)
    rc = lib.bsa_topk_from_score(None, FAKE, None, FAKE, 1, 1, 4, 4, 2, _capi.BSA_BF16, None)
    with pytest.raises(ValueError):
        _capi.check(rc)
    rc = lib.bsa_topk_from_score(FAKE, FAKE, None, FAKE, 1, 1, 4, 5000, 5, _capi.BSA_BF16, None)
    with pytest.raises(NotImplementedError):
        _capi.check(rc)
    _capi.check(0)


def test_header_and_library_from_a_plain_c_program(tmp_path):
    """include/bsa_mi355x.h is C, and the library needs no Python or torch around it."""
    import shutil
    import subprocess
    if shutil.which("gcc") is None:
        pytest.skip("no C compiler")
    exe = str(tmp_path / "capi_from_c")
    src = os.path.join(ROOT, "tests", "capi_from_c.c")
    subprocess.run(["gcc", "-std=c99", "-Wall", "-Werror", "-I", os.path.join(ROOT, "include"), src, "-o", exe, "-ldl"], check=True)
    _capi.load()                       # raises with the build hint if the library is missing
    out = subprocess.run([exe, _capi.LIB_PATH], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0 and out.stdout.startswith("ok"), (out.returncode, out.stdout, out.stderr)


@pytest.mark.parametrize("cus", [256, 240, 128, 32])
def test_workspace_holds_for_devices_of_any_size(cus):
    """The last, partial round of the attention kernel may be cut into parts, 33 280 bytes each, at most 16 of an item and
    two rounds of them.  How many items that round has depends on the device; the size that a caller asks for once must not.
    The lists of the CDF rule are never cut, which leaves the parts as the difference between two calls of the same sizes
    but for the CDF rule's order and queue."""
    lib = _capi.load()
    for heads, frames in ((4, 16), (7, 36), (1, 8)):                     # 256, 576, 128 query tiles a head
        size = lambda cdf: lib.bsa_workspace_bytes(C.byref(_capi.Bsa3dParams(       # noqa: E731
            1, heads, 128, _capi.BSA_BF16, frames, 32, 32, frames, 32, 32, 4, 4, 4, 4, 4, 4, 64 * frames // 4, 0.1, cdf)))
        items, round_ = heads * 64 * frames // 4, 4 * cus
        parts = size(0.0) - size(0.5) + 4 * items + 256                  # its order, its queue
        assert parts >= min(items % round_ * 16, 2 * round_) * 33280


def test_items_are_shared_where_all_teams_run_at_once():
    """Teams of wavefronts of a last round run at once (1 024 wavefronts without a device); a list by the CDF rule, which may be a
    sixteenth of its width, is not cut into parts.  By the top-k rule the estimate decides."""
    lib = _capi.load()
    out = (C.c_int32 * 4)()
    for heads in range(1, 24):
        for frames, chunk in ((4, (4, 4, 4)), (13, (4, 4, 8))):
            prm = _capi.Bsa3dParams(1, heads, 128, _capi.BSA_BF16, frames, 40, 40, frames, 40, 40, *chunk, *chunk, 0, 0.1, 0.5)
            assert lib.bsa_fwd_3d_last_round(C.byref(prm), out) == 0
            total, items, team, parts = out
            assert items == total % 1024 and parts == 1 and team in (1, 2, 4) and items * team <= 1024
            assert team > 1 if total <= 512 else team == 1
    for heads, grid, k_sel, want in ((6, (4, 40, 40), 100, (600, 600, 1, 1)), (1, (8, 64, 68), 200, (544, 544, 1, 3)),
                                     (1, (8, 64, 68), 64, (544, 544, 1, 1)), (1, (8, 64, 64), 100, (512, 512, 2, 1))):
        prm = _capi.Bsa3dParams(1, heads, 128, _capi.BSA_BF16, *grid, *grid, 4, 4, 4, 4, 4, 4, k_sel, 0.1, 0.0)
        assert lib.bsa_fwd_3d_last_round(C.byref(prm), out) == 0 and tuple(out) == want
    # keys whose last frames fill a quarter or a half of their chunks: the second wavefront of a team of two would have less to do
    for grid, chunk, k_sel, want in (((13, 26, 43), (4, 4, 8), 84, (1, 3)), ((9, 36, 57), (4, 4, 8), 172, (1, 5)), ((5, 46, 53), (4, 4, 4), 168, (1, 3)),
                                     ((16, 26, 43), (4, 4, 8), 84, (2, 1)), ((9, 50, 46), (4, 4, 4), 234, (2, 1)), ((5, 37, 15), (4, 4, 4), 64, (4, 1))):
        prm = _capi.Bsa3dParams(1, 1, 128, _capi.BSA_BF16, *grid, *grid, *chunk, *chunk, k_sel, 0.1, 0.0)
        assert lib.bsa_fwd_3d_last_round(C.byref(prm), out) == 0 and tuple(out)[2:] == want, (grid, tuple(out))
    assert lib.bsa_fwd_3d_last_round(C.byref(prm), None) == _capi.BSA_ERR_BAD_ARG
    prm.dtype = _capi.BSA_F32
    assert lib.bsa_fwd_3d_last_round(C.byref(prm), out) == _capi.BSA_ERR_UNSUPPORTED


def test_backward_workspace_holds_v_only_without_the_kept_ds():
    """With dS kept no kernel reads v in blocked order: beside bsa_bwd's workspace there are q, dO and the tables; a workspace of the
    least size has v in the place of dS, and is always smaller."""
    lib = _capi.load()
    for heads, grid, width in ((32, (24, 30, 52), 78), (1, (4, 4, 4), 1), (3, (5, 9, 13), 4), (32, (24, 45, 80), 90)):
        prm = C.byref(_capi.Bsa3dParams(1, heads, 128, _capi.BSA_BF16, *grid, *grid, 4, 4, 4, 4, 4, 4, 0, 0.1, 0.0))
        S = lib.bsa_padded_tokens(*grid, 4, 4, 4)
        total, least = lib.bsa_bwd_3d_workspace_bytes(prm, width), lib.bsa_bwd_3d_workspace_least_bytes(prm, width)
        sizes = (1, heads, S, S, 128, 64, 64, width, _capi.BSA_BF16)
        most, scratch = lib.bsa_bwd_workspace_bytes(*sizes), lib.bsa_bwd_workspace_least_bytes(*sizes)
        own = 2 * heads * S * 256 + 2 * 4 * S + S // 8 + 6 * 256
        assert scratch + heads * S * 256 <= least <= scratch + heads * S * 256 + own
        if most == scratch:                       # 24x45x80: more than is kept
            assert total == least
        else:
            assert least < total <= max(most + own, least + 256)

"""Small launches: the GEMM's 16 x 16 MFMA forms and its paired 128 x 128 tile, at the sizes
where a tile, a slab ring or a wave's share of either can go wrong.

Every tile runs the same chain of products over K for each element of C, so a
row's bits do not depend on the row count that chose the tile: each product is
compared bit for bit with the same rows of a larger one, which a 32 x 32 MFMA
tile serves (their own tests hold those to the oracle), and a part of it with
the oracle's gemm_nt at that test's bounds."""
import ctypes

import numpy as np
import pytest

import mxenc
from mxenc import from_bf16_bits, synth, to_bf16_bits
from orc import P

pytestmark = pytest.mark.gpu

NONE, POLY, ERF = mxenc.MX_EPI_NONE, mxenc.MX_EPI_GELU_POLY, mxenc.MX_EPI_GELU_ERF
GLU = 8  # the internal epilogue of the fused gated FFN (SiLU)

CASES = [
    # M, K, N, epilogue, C dtype, residual, expected kernel
    (1, 384, 1152, NONE, np.uint16, False, "lds_64x64x128_w32x32_ns3_mfma16"),  # one row
    (19, 1536, 384, NONE, np.uint16, False, "lds_64x64x128_w32x32_ns3_mfma16"),
    (65, 768, 3072, ERF, np.uint16, False, "lds_64x64x128_w32x32_ns3_mfma16"),  # a row over
    (127, 3072, 768, NONE, np.float32, True, "lds_64x64x128_w32x32_ns3_mfma16"),
    (200, 1920, 640, POLY, np.float32, True, "lds_64x64x128_w32x32_ns3_mfma16"),  # odd slabs
    (300, 768, 768, NONE, np.float32, False, "lds_64x64x128_w32x32_ns3_mfma16"),
    (1500, 1024, 1024, NONE, np.uint16, False, "lds_64x64x128_w32x32_ns2_mfma16"),
    (1473, 768, 768, POLY, np.float32, True, "lds_64x64x128_w32x32_ns2_mfma16"),
    (31, 256, 64, ERF, np.uint16, False, "lds_64x64x128_w32x32_ns2_mfma16"),  # two slabs
    (333, 448, 448, POLY, np.uint16, False, "lds_64x64x64_w32x32_ns4_mfma16"),  # K % 128 = 64
    (63, 320, 1344, NONE, np.float32, True, "lds_64x64x64_w32x32_ns4_mfma16"),
    (3000, 1280, 1280, NONE, np.float32, True, "lds_128x128x64_w64x32_ns4_mfma16"),
    (777, 512, 1000, ERF, np.uint16, False, "lds_128x128x64_w64x32_ns4_mfma16"),  # ragged M, N
    (1999, 256, 1288, ERF, np.uint16, False, "lds_128x128x64_w64x64_ns2"),  # ragged M and N
    (1500, 128, 768, NONE, np.uint16, False, "lds_128x128x64_w64x64_ns2"),  # two slabs
    (300, 192, 768, POLY, np.float32, True, "lds_128x128x64_w64x64_ns2"),
    (3940, 5120, 1280, NONE, np.float32, True, "lds_128x128x64_w64x64_ns2"),
    (3940, 5120, 1280, POLY, np.uint16, False, "lds_128x128x64_w64x64_ns2"),
    # the 64-byte 128 x 128 tile: K % 64 = 32, and an fp32 C without a residual
    (1000, 992, 1000, ERF, np.uint16, False, "lds_128x128x32_w64x64_ns4"),
    (333, 1280, 1288, POLY, np.float32, False, "lds_128x128x32_w64x64_ns4"),
]


@pytest.fixture(scope="module")
def ctx():
    c = mxenc.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("M,K,N,epi,cdt,res,plan", CASES)
def test_small_tiles(ctx, orc, M, K, N, epi, cdt, res, plan):
    print("case", M, K, N, epi, cdt, res, flush=True)
    dt = mxenc.MX_BF16 if cdt == np.uint16 else mxenc.MX_F32
    L = mxenc.lib()
    name = lambda m: L.mx_gemm_plan_for(m, N, K, dt, int(res), 0).decode()  # noqa: E731
    assert name(M).startswith(plan)
    BIG = 20000
    while "mfma16" in name(BIG):
        BIG *= 2
    rng = np.random.default_rng(M + K + N)
    A = np.zeros((BIG, K), np.uint16)
    A[:M] = to_bf16_bits(rng.standard_normal((M, K)).astype(np.float32))
    W = to_bf16_bits((rng.standard_normal((K, N)) * 0.05).astype(np.float32))
    bias = (rng.standard_normal(N) * 0.1).astype(np.float32)
    R = rng.standard_normal((BIG + 1, N)).astype(np.float32) if res else None
    dW, db = ctx.put(np.ascontiguousarray(W.T)), ctx.put(bias)

    def product(rows):
        dA = ctx.put(A[:rows])
        # one row more than C has: nothing is written past the last
        dC = ctx.put(R[:rows + 1]) if res else ctx.put(np.zeros((rows + 1, N), cdt))
        mxenc.gemm_wt(ctx, dA, rows, K, K, dW, N, db, epi, dC if res else None, dC, N)
        return dC.host()

    got, big = product(M), product(BIG)
    assert np.array_equal(got[M], R[M] if res else np.zeros(N, cdt))
    got = got[:M]
    assert np.array_equal(got.view(np.uint8), big[:M].view(np.uint8))

    rows = np.unique(np.concatenate([np.arange(min(M, 64)), np.arange(max(0, M - 64), M)]))
    want = np.empty((rows.size, N), np.float32)
    Af = np.ascontiguousarray(from_bf16_bits(A[rows]))
    Wf = np.ascontiguousarray(from_bf16_bits(W))
    orc.orc_gemm_nt(P(Af), rows.size, P(Wf), K, N, P(bias), P(want))
    if epi == POLY:
        orc.orc_gelu_poly_inplace(P(want), want.size)
    elif epi == ERF:
        orc.orc_gelu_erf_inplace(P(want), want.size)
    if res:
        want += R[rows]
    scale = np.max(np.abs(want))
    if cdt == np.uint16:
        g = from_bf16_bits(got[rows])
        assert np.max(np.abs(g - want) / (np.abs(want) + 1e-3 * scale)) < 1e-2
    else:
        assert np.max(np.abs(got[rows] - want)) / scale < 1e-5


I8_CASES = [
    # M, K, N, epilogue, C dtype, residual, expected kernel
    (1, 768, 2304, NONE, np.uint16, False, "lds_64x64x256_w32x32_ns3_mfma16"),  # one row
    (65, 1024, 4096, POLY, np.float32, False, "lds_64x64x256_w32x32_ns3_mfma16"),  # a row over
    (300, 3072, 768, NONE, np.float32, False, "lds_64x64x256_w32x32_ns3_mfma16"),
    (127, 1280, 1280, ERF, np.float32, True, "lds_64x64x256_w32x32_ns3_mfma16"),
    (300, 384, 1152, NONE, np.float32, False, "lds_128x128x128_w64x32_ns3_mfma16"),  # three slabs
    (4099, 3072, 768, NONE, np.float32, False, "lds_128x128x128_w64x32_ns3_mfma16"),
    (1000, 896, 1000, POLY, np.uint16, False, "lds_128x128x128_w64x32_ns3_mfma16"),  # ragged N
    (999, 1152, 1152, NONE, np.float32, True, "lds_128x128x128_w64x32_ns3_mfma16"),
]


@pytest.mark.parametrize("M,K,N,epi,cdt,res,plan", I8_CASES)
def test_small_tiles_i8(ctx, orc, M, K, N, epi, cdt, res, plan):
    """The int32 product is exact, so the dequantised result is the host's bit
    for bit (the exact-erf GELU and the residual's sum to one rounding)."""
    print("case", M, K, N, epi, cdt, res, flush=True)
    dt = mxenc.MX_BF16 if cdt == np.uint16 else mxenc.MX_F32
    L = mxenc.lib()
    assert L.mx_gemm_plan_for(M, N, K, dt, int(res), 1).decode().startswith(plan)
    rng = np.random.default_rng(M + K + N)
    A = rng.integers(-127, 128, (M, K)).astype(np.int8)
    W = rng.integers(-127, 128, (K, N)).astype(np.int8)
    sa = rng.uniform(1e-4, 1e-2, M).astype(np.float32)
    ws = rng.uniform(1e-4, 1e-2, N).astype(np.float32)
    b = rng.standard_normal(N).astype(np.float32)
    R = rng.standard_normal((M, N)).astype(np.float32) if res else None
    slot = mxenc.stage_weight_i8(ctx, W, ws, np.ones(K, np.float32))
    # a row more than C has: nothing is written past the last
    C = ctx.put(np.zeros((M + 1, N), cdt))
    mxenc.gemm_i8(ctx, ctx.put(A), ctx.put(sa), M, K, K, slot, ctx.put(b), epi,
                  ctx.put(R) if res else None, C, N)
    got = C.host()
    mxenc.check(L.mx_release_weight(ctx.handle, slot))
    assert not got[M].any()
    rows = np.unique(np.concatenate([np.arange(min(M, 130)), np.arange(max(0, M - 130), M)]))
    Ar, sar = np.ascontiguousarray(A[rows]), np.ascontiguousarray(sa[rows])
    c32 = np.zeros((rows.size, N), np.int32)
    orc.orc_gemm_i8(P(Ar), rows.size, K, P(W), N, P(c32))
    want = np.zeros((rows.size, N), np.float32)
    orc.orc_dequantise_c(P(c32), rows.size, N, P(sar), P(ws), P(b), P(want))
    if epi == POLY:
        orc.orc_gelu_poly_inplace(P(want), want.size)
    elif epi == ERF:
        orc.orc_gelu_erf_inplace(P(want), want.size)
    if res:
        want += R[rows]
    if cdt == np.uint16:
        assert np.array_equal(got[rows], mxenc.to_bf16_bits(want))
    elif epi == ERF:
        # the device's erf and the host's differ by a few ulp: the bound of the
        # exact-erf epilogue's own test against the host
        assert np.max(np.abs(got[rows] - want)) < 1e-4
    else:
        assert np.array_equal(got[rows], want)


class GemmArgs(ctypes.Structure):
    """mxk::GemmArgs (mx_kernels.hpp): the launch under the C ABI, which also
    takes a live row count on the device and the row count the tile is chosen
    for."""
    _fields_ = [("A", ctypes.c_void_p), ("lda", ctypes.c_int64), ("Wt", ctypes.c_void_p),
                ("M", ctypes.c_int64), ("N", ctypes.c_int64), ("K", ctypes.c_int64),
                ("bias", ctypes.c_void_p), ("epilogue", ctypes.c_int),
                ("residual", ctypes.c_void_p), ("C", ctypes.c_void_p), ("c_bf16", ctypes.c_int),
                ("ldc", ctypes.c_int64), ("rows_dev", ctypes.c_void_p),
                ("m_hint", ctypes.c_int64)]


class GemmI8Args(ctypes.Structure):
    """mxk::GemmI8Args."""
    _fields_ = [("A", ctypes.c_void_p), ("lda", ctypes.c_int64), ("Wt", ctypes.c_void_p),
                ("M", ctypes.c_int64), ("N", ctypes.c_int64), ("K", ctypes.c_int64),
                ("a_scale", ctypes.c_void_p), ("wscale", ctypes.c_void_p),
                ("bias", ctypes.c_void_p), ("epilogue", ctypes.c_int),
                ("residual", ctypes.c_void_p), ("C", ctypes.c_void_p), ("c_dtype", ctypes.c_int),
                ("ldc", ctypes.c_int64), ("rows_dev", ctypes.c_void_p),
                ("m_hint", ctypes.c_int64)]


def internal(name, args=None):
    f = mxenc.lib()[name]
    f.restype, f.argtypes = ctypes.c_int, [ctypes.POINTER(args), ctypes.c_void_p]
    return f


def plan_name(M, N, K, bf16, res, i8=False, gated=False):
    f = mxenc.lib()["_ZN3mxk14gemm_plan_nameElllbbbb"]
    f.restype, f.argtypes = ctypes.c_char_p, [ctypes.c_int64] * 3 + [ctypes.c_bool] * 4
    return f(M, N, K, bf16, res, i8, gated).decode()


def tiles_and_grid(plan, M, N):
    bm, bn = (int(x) for x in plan.split("_")[1].split("x")[:2])
    pairs = "_ns2_" in plan or plan.startswith("lds_64x64x64")
    return -(-M // bm) * -(-N // bn), 512 if pairs and bm < 256 else 256


MANY = [
    # tile for, M, K, N, epilogue, bf16 C, residual, int8, kernel
    (64, 12000, 384, 384, NONE, True, False, False, "lds_64x64x128_w32x32_ns3"),  # ring's depth
    (1000, 6000, 896, 768, POLY, False, True, False, "lds_64x64x128_w32x32_ns3"),  # odd slabs
    (64, 9000, 256, 512, ERF, True, False, False, "lds_64x64x128_w32x32_ns2"),  # ring's depth
    (64, 9000, 640, 512, NONE, False, True, False, "lds_64x64x128_w32x32_ns2"),
    (64, 9000, 320, 448, ERF, True, False, False, "lds_64x64x64_w32x32_ns4"),
    (64, 9000, 448, 448, NONE, False, True, False, "lds_64x64x64_w32x32_ns4"),
    (777, 9000, 512, 1000, ERF, True, False, False, "lds_128x128x64_w64x32_ns4"),  # ragged N
    (2000, 6000, 1216, 1152, NONE, False, True, False, "lds_128x128x64_w64x32_ns4"),  # odd slabs
    (64, 4000, 384, 1344, GLU, True, False, False, "lds_64x128x128_w32x64_ns3"),  # ragged columns
    (300, 3000, 640, 1344, GLU, True, False, False, "lds_64x128x128_w32x64_ns3"),  # odd slabs
    (20, 1500, 768, 6144, GLU, True, False, False, "lds_64x128x128_w32x64_ns3"),
    (64, 9000, 384, 1152, NONE, False, False, True, "lds_128x128x128_w64x32_ns3"),  # ring's depth
    (64, 9000, 896, 1000, POLY, True, False, True, "lds_128x128x128_w64x32_ns3"),  # ragged N
    (64, 6000, 768, 768, NONE, True, False, True, "lds_64x64x256_w32x32_ns3"),  # ring's depth
    (64, 6000, 1280, 1280, POLY, False, True, True, "lds_64x64x256_w32x32_ns3"),  # odd slabs
    (64, 3001, 2304, 2304, ERF, False, False, True, "lds_64x64x256_w32x32_ns3"),
]


@pytest.mark.parametrize("live", [False, True])
@pytest.mark.parametrize("hint,M,K,N,epi,bf16,res,i8,plan", MANY)
def test_small_tiles_walk_many(ctx, hint, M, K, N, epi, bf16, res, i8, plan, live):
    """More tiles than resident blocks, as a full batch has behind a short one:
    the slab ring, the epilogue vectors' two copies and the waits behind an
    epilogue's stores cross tile boundaries. Bit for bit the tile that the full
    row count chooses, with the row count on the host and on the device."""
    print("case", hint, M, K, N, epi, bf16, res, i8, live, flush=True)
    gated = epi == GLU
    small = plan_name(hint, N, K, bf16, res, i8, gated)
    assert small.startswith(plan) and "mfma16" in small
    assert "mfma16" not in plan_name(M, N, K, bf16, res, i8, gated)
    tiles, grid = tiles_and_grid(small, M, N)
    assert tiles > grid
    rng = np.random.default_rng(M + K + N)
    cols = N // 2 if gated else N
    rows = M - 777 if live else M
    if i8:
        A, W = (rng.integers(-127, 128, (n, K)).astype(np.int8) for n in (M, N))
    else:
        A = to_bf16_bits(rng.standard_normal((M, K)).astype(np.float32))
        W = to_bf16_bits((rng.standard_normal((N, K)) * 0.05).astype(np.float32))
    dA, dW = ctx.put(A), ctx.put(W)
    db = ctx.put((rng.standard_normal(N) * 0.1).astype(np.float32))
    sa = ctx.put(rng.uniform(1e-4, 1e-2, M).astype(np.float32))
    ws = ctx.put(rng.uniform(1e-4, 1e-2, N).astype(np.float32))
    cdt = np.uint16 if bf16 else np.float32
    start = (rng.standard_normal((M + 1, cols)).astype(np.float32) if res
             else np.full((M + 1, cols), 7, cdt))
    n_dev = ctx.put(np.array([rows], np.int32))
    stream = mxenc.lib().mx_stream_handle(ctx.stream)

    def product(m_hint):
        dC = ctx.put(start)
        common = dict(A=dA.ptr, lda=K, Wt=dW.ptr, M=M, N=N, K=K, bias=db.ptr, epilogue=epi,
                      residual=dC.ptr if res else None, C=dC.ptr, ldc=cols,
                      rows_dev=n_dev.ptr if live else None, m_hint=m_hint)
        if i8:
            a = GemmI8Args(a_scale=sa.ptr, wscale=ws.ptr, c_dtype=int(bf16), **common)
            rc = internal("_ZN3mxk7gemm_i8ERKNS_10GemmI8ArgsEP12ihipStream_t", GemmI8Args)(
                ctypes.byref(a), stream)
        else:
            a = GemmArgs(c_bf16=int(bf16), **common)
            rc = internal("_ZN3mxk4gemmERKNS_8GemmArgsEP12ihipStream_t", GemmArgs)(
                ctypes.byref(a), stream)
        assert rc == 0
        return dC.host()

    got, want = product(hint), product(0)
    assert np.array_equal(got.view(np.uint8), want.view(np.uint8))
    assert np.array_equal(got[rows:], start[rows:])  # nothing past the live rows
    assert not np.array_equal(got[:rows], start[:rows])


@pytest.mark.parametrize("name,B,S,over", [
    ("nomic", 1, 1, {}),
    ("gte", 1, 65, {}),
    ("nomic", 3, 101, {}),
    ("nomic", 2, 100, dict(hidden=384, heads=6, ffn=672)),  # the ring's depth; ragged columns
    ("gte", 3, 67, dict(hidden=640, heads=10, ffn=1312)),   # five slabs; ragged columns
])
def test_small_gated_ffn(ctx, name, B, S, over):
    """The fused gated FFN on 64 x 128 tiles: bit for bit the GEMM and the
    gated-FFN pass apart."""
    print("case", name, B, S, over, flush=True)
    m = synth.make_model(name, layers=2, ln_random=True, **over)
    assert plan_name(B * S, 2 * m["ffn"], m["hidden"], True, False, gated=True).startswith(
        "lds_64x128x128_w32x64_ns3")
    enc = mxenc.Encoder(ctx, m)
    x = np.random.default_rng(B * S).standard_normal((B * S, m["hidden"])).astype(np.float32)

    def run(fused):
        enc.set_fusion(fused)
        dx = ctx.put(x)
        enc.run(dx, None, None, B, S)
        return dx.host()

    try:
        a, b = run(True), run(False)
        assert np.isfinite(a).all()
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
    finally:
        enc.close()


@pytest.mark.parametrize("name", ["minilm", "bge_base", "nomic"])
def test_short_sequences_then_full_ones(ctx, name):
    """A single sequence, padded or not, whose tiles the sequence before it
    chose: bit for bit the padded computation."""
    print("case", name, flush=True)
    m = synth.make_model(name, layers=2, ln_random=True)
    enc = mxenc.Encoder(ctx, m)
    S = 512
    ids = np.random.default_rng(3).integers(1000, 30000, (1, S)).astype(np.int32)

    def embed(n, width, packing=True):
        am = np.zeros((1, width), np.float32)
        am[0, :n] = 1.0
        out = ctx.empty((1, m["hidden"]), np.float32)
        enc.set_packing(packing)
        enc.embed(ctx.put(ids[:, :width]), ctx.put(am), 1, width, out)
        return out.host()

    try:
        sizes = [(20, 512), (512, 512), (20, 512), (20, 20), (500, 512), (1, 512), (512, 512)]
        want = {s: embed(*s, packing=False) for s in set(sizes)}
        for s in sizes:
            assert np.array_equal(embed(*s).view(np.uint32), want[s].view(np.uint32)), s
    finally:
        enc.close()


@pytest.mark.parametrize("B,S,hd,lens,H", [
    (2, 70, 64, [1, 70], 2),
    (5, 200, 32, [200, 200, 3, 64, 129], 2),   # ties
    (64, 40, 64, None, 2),
    (65, 40, 64, None, 2),
    # ranked: more blocks than CUs, S of 128 or more
    (2, 4200, 64, [1, 4200], 4),
    (5, 1100, 32, [1100, 1100, 3, 64, 1099], 6),   # ties
    (33, 128, 32, None, 9),                     # one query block
    (64, 200, 64, None, 3),                     # the most sequences a wave ranks
    (64, 200, 32, [200] * 64, 3),               # of one length: index order
    (7, 257, 64, [0, 300, 257, 256, -5, 1, 128], 16),  # out of 1 .. S: clamped
    (65, 200, 64, None, 3),                     # one more: index order
])
def test_attention_ranks_uneven_sequences(ctx, B, S, hd, lens, H):
    """Attention over sequences of uneven length without a launch order: every
    sequence is computed once, bit for bit as when it is alone."""
    print("case", B, S, hd, lens, H, flush=True)
    d = H * hd
    rng = np.random.default_rng(B)
    lens = np.array(lens if lens else rng.integers(1, S + 1, B), np.int32)
    qkv = to_bf16_bits((rng.standard_normal((B * S, 3 * d)) * 0.5).astype(np.float32))
    mask = np.where(np.arange(S)[None, :] < lens[:, None], 0.0, -1e30).astype(np.float32)
    out = ctx.put(np.zeros((B * S, d), np.uint16))
    mxenc.attention(ctx, ctx.put(qkv), 3 * d, B, S, H, hd, 1.0, ctx.put(mask), ctx.put(lens), out,
                    d)
    got = out.host().reshape(B, S, d)
    for b in range(B):
        one = ctx.put(np.zeros((S, d), np.uint16))
        mxenc.attention(ctx, ctx.put(qkv[b * S:(b + 1) * S]), 3 * d, 1, S, H, hd, 1.0,
                        ctx.put(mask[b:b + 1]), ctx.put(lens[b:b + 1]), one, d)
        assert np.array_equal(got[b], one.host()), b

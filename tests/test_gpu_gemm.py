"""Prefill GEMM (int8 MFMA) on the GPU against the oracle: tolerance 1e-3 of the f32 reference per token row, exact
integer block sums through unit scales, the three epilogues, agreement with the GEMV on the same inputs, determinism."""
import numpy as np
import pytest

import arcinferzero_amd as az
import oracle_lib as orc
from common import (ALL_TYPES, TYPES, TYPE_NAMES, make_acts, make_weights, mixed_err, quantize_padded, rel_err_rows,
                    unit_scale_acts, unit_scale_weights)

pytestmark = pytest.mark.gpu
TOL = 1e-3
TIGHT = 2e-5


@pytest.fixture(scope="module")
def eng(rt):
    e = az.Engine(512, 5120)
    yield e
    e.close()


def run_gemm(eng, qtype, W, N, K, x, Mp, acc=0, c_init=None, ldc=None, c_off=0):
    T = x.shape[0]
    ldc = N + c_off if ldc is None else ldc
    w = eng.make_weight(qtype, N, K, W)
    xb = az.Runtime.from_numpy(x)
    eng.quantize(xb, K, K, Mp, T)
    cb = az.Runtime.alloc(Mp * ldc * 4)
    if c_init is None:
        cb.fill(0xFFFFFFFF)
    else:
        cb.write(c_init)
    eng.matmul("test", w, Mp, cb, ldc, c_off, acc)
    y = cb.read(np.float32, Mp * ldc).reshape(Mp, ldc)
    for b in (cb, xb):
        b.free()
    w.free()
    return y


@pytest.mark.parametrize("qtype", ALL_TYPES)
@pytest.mark.parametrize("T,Mp,N,K", [(16, 16, 64, 256), (100, 112, 272, 512), (128, 128, 128, 1024), (300, 384, 384, 768),
                                      (180, 192, 520, 512)])
def test_gemm_vs_oracle(eng, qtype, T, Mp, N, K):
    print(f"gemm {TYPE_NAMES[qtype]} T={T} Mp={Mp} N={N} K={K}", flush=True)
    W = make_weights(qtype, N, K, seed=31 + qtype)
    x = make_acts(T, K, seed=41 + T, outliers=True)
    y = run_gemm(eng, qtype, W, N, K, x, Mp)
    aq, asc, absum = quantize_padded(x, Mp)
    ref = orc.matmul_ref(qtype, W, N, K, aq[:T], asc)
    assert np.isfinite(y).all()
    assert not y[T:].any()                      # padding rows: zero activations give exact zeros
    err = rel_err_rows(y[:T], ref)
    form = orc.matmul_formula(qtype, 1, W, N, K, aq[:T], asc, absum)
    print(f"  rel {err.max():.2e} mixed {mixed_err(y[:T], ref):.2e} vs formula {rel_err_rows(y[:T], form).max():.2e}")
    assert err.max() <= TOL
    assert rel_err_rows(y[:T], form).max() <= TIGHT
    y2 = run_gemm(eng, qtype, W, N, K, x, Mp)
    assert np.array_equal(y.view(np.uint32), y2.view(np.uint32))   # bit-identical run to run


@pytest.mark.parametrize("qtype", ALL_TYPES)
def test_gemm_block_sums_exact(eng, qtype):
    T, N, K = 160, 160, 512
    W, wi = unit_scale_weights(qtype, N, K, seed=15)
    x = unit_scale_acts(T, K, seed=16)
    y = run_gemm(eng, qtype, W, N, K, x, 160)
    exact = x.astype(np.int64) @ wi.T
    assert np.abs(exact).max() < 2 ** 24
    assert np.array_equal(y, exact.astype(np.float32))


@pytest.mark.parametrize("qtype", ALL_TYPES)
def test_gemm_matches_gemv(eng, qtype):
    """Rows 0..7 of a 16-row GEMM against the 8-token GEMV on the same inputs: both within tolerance of the same
    reference and of each other."""
    N, K, T = 192, 1024, 16
    W = make_weights(qtype, N, K, seed=51)
    x = make_acts(T, K, seed=52)
    yg = run_gemm(eng, qtype, W, N, K, x, 16)
    w = eng.make_weight(qtype, N, K, W)
    xb = az.Runtime.from_numpy(x[:8])
    eng.quantize(xb, K, K, 16, 8)
    cb = az.Runtime.alloc(8 * N * 4)
    eng.matmul("test", w, 16, cb, N, 0, 0)
    yv = cb.read(np.float32, 8 * N).reshape(8, N)
    cb.free(); xb.free(); w.free()
    assert rel_err_rows(yg[:8], yv).max() <= TIGHT


def test_gemm_epilogues(eng):
    qtype, T, Mp, N, K = az.Q4_K, 64, 64, 128, 512
    W = make_weights(qtype, N, K, seed=61)
    x = make_acts(T, K, seed=62)
    ldc, c_off = 300, 100
    c0 = az.gen_normal(63, (Mp, ldc))
    y0 = run_gemm(eng, qtype, W, N, K, x, Mp)
    ya = run_gemm(eng, qtype, W, N, K, x, Mp, acc=1, c_init=c0, ldc=ldc, c_off=c_off)
    assert np.array_equal(ya[:, :c_off], c0[:, :c_off]) and np.array_equal(ya[:, c_off + N:], c0[:, c_off + N:])
    assert np.array_equal(ya[:, c_off:c_off + N], y0 + c0[:, c_off:c_off + N])
    ys = run_gemm(eng, qtype, W, N, K, x, Mp, acc=2, c_init=c0, ldc=ldc, c_off=c_off)
    g = c0[:, c_off:c_off + N].astype(np.float64)
    want = y0.astype(np.float64) * (g / (1.0 + np.exp(-g)))   # C = silu(C) * result (gemm.cl:562-565)
    assert np.abs(ys[:, c_off:c_off + N] - want).max() <= 1e-5 * np.abs(want).max()
    assert np.array_equal(ys[:, :c_off], c0[:, :c_off])


@pytest.mark.parametrize("qtype", [az.Q4_K, az.Q5_K])
@pytest.mark.parametrize("T,Mp,N,K", [(64, 64, 130, 4096), (40, 48, 300, 5120), (100, 112, 260, 2560), (128, 128, 128, 4096),
                                      (20, 32, 200, 4096), (17, 32, 129, 2560)])
def test_gemm_split_k(eng, qtype, T, Mp, N, K):
    """Short Q4_K / Q5_K chunks whose tiles are few: K shared out over several work-groups per tile, partial tiles added
    in a fixed order by a second kernel that also applies c_off and the accumulate mode (tiles of 32 tokens up to 32
    tokens, of 64 up to 64, of 128 above).  Parity with the oracle, the three epilogues, the same bits on every run."""
    print(f"gemm split-K {TYPE_NAMES[qtype]} T={T} Mp={Mp} N={N} K={K}", flush=True)
    W = make_weights(qtype, N, K, seed=71)
    x = make_acts(T, K, seed=72 + T, outliers=True)
    y0 = run_gemm(eng, qtype, W, N, K, x, Mp)
    aq, asc, absum = quantize_padded(x, Mp)
    ref = orc.matmul_ref(qtype, W, N, K, aq[:T], asc)
    assert rel_err_rows(y0[:T], ref).max() <= TOL and not y0[T:].any()
    assert np.array_equal(run_gemm(eng, qtype, W, N, K, x, Mp).view(np.uint32), y0.view(np.uint32))
    ldc, c_off = N + 70, 33
    c0 = az.gen_normal(73, (Mp, ldc))
    ya = run_gemm(eng, qtype, W, N, K, x, Mp, acc=1, c_init=c0, ldc=ldc, c_off=c_off)
    assert np.array_equal(ya[:, :c_off], c0[:, :c_off]) and np.array_equal(ya[:, c_off + N:], c0[:, c_off + N:])
    assert np.array_equal(ya[:, c_off:c_off + N], y0 + c0[:, c_off:c_off + N])
    ys = run_gemm(eng, qtype, W, N, K, x, Mp, acc=2, c_init=c0, ldc=ldc, c_off=c_off)
    g = c0[:, c_off:c_off + N].astype(np.float64)
    want = y0.astype(np.float64) * (g / (1.0 + np.exp(-g)))
    assert np.abs(ys[:, c_off:c_off + N] - want).max() <= 1e-5 * np.abs(want).max()
    assert np.array_equal(ys[:, :c_off], c0[:, :c_off])


@pytest.mark.parametrize("N,ldc,c_off,skip", [(1, 1, 0, 0), (255, 255, 0, 0), (257, 257, 0, 0), (1025, 1025, 0, 0), (1026, 1028, 2, 0),
                                              (1023, 1030, 7, 0), (1028, 1028, 0, 1), (1028, 1031, 3, 0), (1028, 1032, 4, 0)])
@pytest.mark.parametrize("acc", [0, 1, 2])
def test_gemm_split_k_columns(eng, N, ldc, c_off, skip, acc):
    """The reduction of the partial tiles where rows of C are whole vectors and where they are not (by N, ldc, c_off, or C
    itself `skip` floats into its buffer): integer sums, so the same bits whichever way, and nothing beside them touched."""
    T, Mp, K = 40, 48, 4096
    print(f"split-K columns N={N} ldc={ldc} c_off={c_off} skip={skip} acc={acc}", flush=True)
    W, wi = unit_scale_weights(az.Q8_0, N, K, seed=98)
    x = unit_scale_acts(T, K, seed=99)
    c0 = np.random.default_rng(100).integers(-50, 51, (Mp, ldc)).astype(np.float32)
    w = eng.make_weight(az.Q8_0, N, K, W)
    xb = az.Runtime.from_numpy(x)
    eng.quantize(xb, K, K, Mp, T)
    cb = az.Runtime.alloc((Mp * ldc + skip) * 4)
    cv = cb.view(4 * skip, Mp * ldc * 4)
    cv.write(c0)
    eng.matmul("test", w, Mp, cv, ldc, c_off, acc)
    y = cv.read(np.float32, Mp * ldc).reshape(Mp, ldc)
    for b in (cv, cb, xb, w):
        b.free()
    sums = np.zeros((Mp, N))
    sums[:T] = x.astype(np.int64) @ wi.T
    old = c0[:, c_off:c_off + N].astype(np.float64)
    want = sums if acc == 0 else sums + old if acc == 1 else sums * (old / (1.0 + np.exp(-old)))
    got = y[:, c_off:c_off + N]
    # (integers below 2^24 for a store and a sum; silu: the product of three f32 roundings and the exponential's, 2^-21)
    assert np.abs(sums).max() < 2 ** 24
    assert np.abs(got - want).max() <= (np.abs(want).max() * 2 ** -21 if acc == 2 else 0.0)
    y[:, c_off:c_off + N] = c0[:, c_off:c_off + N]
    assert np.array_equal(y, c0)


@pytest.mark.parametrize("qtype", [az.Q4_K, az.Q5_K])
@pytest.mark.parametrize("T", [64, 32])
def test_gemm_split_k_unit_scales_exact(eng, qtype, T):
    """Unit scales: the sum of the partial tiles is the exact integer sum (every partial sum below 2^24)."""
    N, K = 96, 4096
    W, wi = unit_scale_weights(qtype, N, K, seed=75)
    x = unit_scale_acts(T, K, seed=76)
    y = run_gemm(eng, qtype, W, N, K, x, T)
    assert np.array_equal(y, (x.astype(np.int64) @ wi.T).astype(np.float32))


def test_startup_self_check(rt):
    """Tuned GEMM == simple GEMM == host integer sums, bit for bit, on the reference's LCG data with unit scales
    (the start-up check in the pattern of xmx_check, zero/engine_setup.h:424-520)."""
    az.self_check()


@pytest.mark.parametrize("qtype", [az.Q4_K, az.Q6_K, az.Q8_0, az.Q4_0, az.IQ4_NL, az.MXFP4])
@pytest.mark.parametrize("T,Mp,N,K", [(1, 16, 264, 1024), (5, 16, 136, 512), (100, 112, 272, 768), (64, 64, 130, 4096)])
def test_per_256_activation_scales(eng, qtype, T, Mp, N, K):
    """act32 = 0: one activation scale per superblock (the reference's quant_store16 with act32 = 0, zero/kernels/ops.cl:
    38-72, and its non-ACT32 GEMM, gemm.cl:489-520).  The quantizer's output bit for bit against the oracle's, the
    matmul against the double-accumulated reference with that one scale on each of a superblock's eight blocks."""
    print(f"act32=0 {TYPE_NAMES[qtype]} T={T} Mp={Mp} N={N} K={K}", flush=True)
    W = make_weights(qtype, N, K, seed=91)
    x = make_acts(T, K, seed=92 + T, outliers=True)
    w = eng.make_weight(qtype, N, K, W)
    xb = az.Runtime.from_numpy(x)
    eng.quantize(xb, K, K, Mp, T, act32=0)
    xp = np.zeros((Mp, K), np.float32)
    xp[:T] = x
    raq, rasc, rabsum = orc.quantize_act(xp, act32=False)
    assert np.array_equal(eng.aq.read(np.int8, Mp * K).reshape(Mp, K), raq)
    assert np.array_equal(eng.asc.read(np.uint32, Mp * K // 256).reshape(K // 256, Mp), rasc.view(np.uint32))
    rows = Mp if T > 8 else T
    cb = az.Runtime.alloc(rows * N * 4).fill(0xFFFFFFFF)
    with pytest.raises(az.ArczError):
        eng.matmul("m", w, Mp, cb, N, 0, 0, act32=True)          # the chunk has per-256 scales
    eng.matmul("m", w, Mp, cb, N, 0, 0, act32=False)
    y = cb.read(np.float32, rows * N).reshape(rows, N)[:T]
    ref = orc.matmul_ref(qtype, W, N, K, raq[:T], np.ascontiguousarray(np.repeat(rasc, 8, axis=0)))
    assert np.isfinite(y).all() and rel_err_rows(y, ref).max() <= TOL
    for b in (cb, xb):
        b.free()
    w.free()


@pytest.mark.parametrize("T,Mp,N,K,acc", [(1100, 1104, 392, 512, 0), (1030, 1040, 640, 768, 1), (760, 768, 520, 1024, 2),
                                          (2050, 2064, 136, 256, 1), (300, 384, 388, 5120, 0)])
def test_gemm_per_256_scales_integer_sums(rt, T, Mp, N, K, acc):
    """act32 = 0 on chunks of at least 256 token rows of Q4_K: the form of the 128 x 128 kernel that adds a superblock's
    block sums up as integers (sc * I) and applies sa * d once per four blocks.  Against the double-accumulated
    reference with the one scale on each of a superblock's eight blocks, the three epilogues, partly empty last tiles,
    run to run."""
    print(f"per-256 integer sums T={T} Mp={Mp} N={N} K={K} acc={acc}", flush=True)
    eng = az.Engine(Mp, K)
    W = make_weights(az.Q4_K, N, K, seed=75)
    x = make_acts(T, K, seed=76, outliers=True)
    c0 = np.random.default_rng(77).standard_normal((Mp, N)).astype(np.float32)
    w = eng.make_weight(az.Q4_K, N, K, W)
    xb = az.Runtime.from_numpy(x)
    eng.quantize(xb, K, K, Mp, T, act32=0)
    ys = []
    for _ in range(2):
        cb = az.Runtime.alloc(Mp * N * 4)
        cb.write(c0) if acc else cb.fill(0xFFFFFFFF)
        eng.matmul("test", w, Mp, cb, N, 0, acc, act32=False)
        ys.append(cb.read(np.float32, Mp * N).reshape(Mp, N))
        cb.free()
    xb.free(); w.free(); eng.close()
    assert np.array_equal(ys[0].view(np.uint32), ys[1].view(np.uint32))
    xp = np.zeros((Mp, K), np.float32)
    xp[:T] = x
    raq, rasc, _ = orc.quantize_act(xp, act32=False)
    ref = orc.matmul_ref(az.Q4_K, W, N, K, raq[:T], np.ascontiguousarray(np.repeat(rasc, 8, axis=0)[:, :T]))
    if acc == 1:
        ref = ref + c0[:T]
    elif acc == 2:
        g = c0[:T].astype(np.float64)
        ref = ref * (g / (1.0 + np.exp(-g)))
    y = ys[0][:T]
    assert np.isfinite(y).all() and mixed_err(y, ref) <= TOL
    if acc == 0:
        assert not ys[0][T:].any()


@pytest.mark.parametrize("qtype", [az.Q4_K, az.Q5_K])
@pytest.mark.parametrize("T,Mp,N,K,acc", [(1100, 1104, 392, 512, 0), (1100, 1104, 390, 512, 0), (1030, 1040, 640, 768, 1),
                                          (760, 768, 520, 1024, 2), (1200, 1216, 132, 256, 0),
                                          (2100, 2112, 392, 512, 0), (2050, 2064, 136, 256, 1), (2048, 2048, 256, 768, 2)])
def test_gemm_ready_made_scale_vectors(rt, monkeypatch, qtype, T, Mp, N, K, acc):
    """The 128 x 128 Q4_K / Q5_K kernel whose scale vectors are written by small kernels in front of it (token side: sa and
    sa * S; row side, from 256 token rows on when N is a multiple of 4: d * sc and -(dmin * mn), for Q4_K with the min
    term's factors as bf16 pieces for the matrix instruction) and go into LDS by DMA:
    chunks whose last token tile and last row tile are partly empty, so that the whole-row reads run into the next
    block's entries and past the arrays' ends; the three epilogues.  Against the oracle, and run to run."""
    print(f"ready-made scales {TYPE_NAMES[qtype]} T={T} Mp={Mp} N={N} K={K} acc={acc}", flush=True)
    monkeypatch.setenv("ARCZ_Q4_WM", "2")   # (the 128 x 128 tiles also where the launch rule would take 64 x 128)
    eng = az.Engine(Mp, K)            # (an engine of exactly this chunk: the arrays end where the chunk ends)
    W = make_weights(qtype, N, K, seed=71)
    x = make_acts(T, K, seed=72, outliers=True)
    c0 = np.random.default_rng(73).standard_normal((Mp, N)).astype(np.float32)
    y = run_gemm(eng, qtype, W, N, K, x, Mp, acc=acc, c_init=c0 if acc else None)[:T]
    y2 = run_gemm(eng, qtype, W, N, K, x, Mp, acc=acc, c_init=c0 if acc else None)[:T]
    eng.close()
    assert np.array_equal(y.view(np.uint32), y2.view(np.uint32))
    aq, asc, _ = quantize_padded(x, Mp)
    ref = orc.matmul_ref(qtype, W, N, K, aq[:T], np.ascontiguousarray(asc[:, :T]))
    if acc == 1:
        ref = ref + c0[:T]
    elif acc == 2:
        g = c0[:T].astype(np.float64)
        ref = ref * (g / (1.0 + np.exp(-g)))
    assert np.isfinite(y).all() and mixed_err(y, ref) <= TOL


@pytest.mark.parametrize("qtype,T,Mp,N,K", [(az.Q6_K, 257, 384, 1000, 768), (az.Q6_K, 130, 256, 392, 2048), (az.Q8_0, 300, 384, 520, 4096),
                                            (az.Q8_0, 129, 256, 3000, 512), (az.Q4_K, 300, 384, 5200, 512), (az.IQ3_S, 257, 384, 1000, 512)])
@pytest.mark.parametrize("acc", [0, 1, 2])
def test_gemm_padding_rows(rt, qtype, T, Mp, N, K, acc):
    """Token tiles that hold padding alone are left out of the launch: the rows from T on come out as the products of zero
    rows all the same (zeros, or what was there), with K shared out and not."""
    print(f"padding rows {TYPE_NAMES[qtype]} T={T} Mp={Mp} N={N} K={K} acc={acc}", flush=True)
    eng = az.Engine(Mp, K)
    W = make_weights(qtype, N, K, seed=85)
    x = make_acts(T, K, seed=86, outliers=True)
    c0 = np.random.default_rng(87).standard_normal((Mp, N)).astype(np.float32)
    y = run_gemm(eng, qtype, W, N, K, x, Mp, acc=acc, c_init=c0)
    eng.close()
    aq, asc, _ = quantize_padded(x, Mp)
    ref = orc.matmul_ref(qtype, W, N, K, aq[:T], np.ascontiguousarray(asc[:, :T]))
    if acc == 1:
        ref = ref + c0[:T]
    elif acc == 2:
        g = c0[:T].astype(np.float64)
        ref = ref * (g / (1.0 + np.exp(-g)))
    assert np.isfinite(y).all() and mixed_err(y[:T], ref) <= TOL
    assert np.array_equal(y[T:], c0[T:] if acc == 1 else np.zeros((Mp - T, N), np.float32))


@pytest.mark.parametrize("T,Mp,N,K,pieces", [(9, 16, 1, 256, 0), (63, 64, 129, 512, 0), (64, 64, 128, 768, 0), (65, 80, 127, 1024, 0),
                                             (300, 384, 520, 1280, 0), (130, 256, 390, 4096, 0), (100, 112, 260, 512, 2),
                                             (300, 300, 1030, 2048, 5)])
@pytest.mark.parametrize("acc,ldc,c_off", [(0, 0, 0), (1, 1, 0), (2, 8, 4)])
def test_gemm_q8_0_eight_waves(rt, monkeypatch, T, Mp, N, K, pieces, acc, ldc, c_off):
    """Q8_0 in tiles of eight waves that share out each superblock's blocks: one superblock and more than the stages hold,
    ragged last tiles, K in pieces besides, rows of whole vectors and not.  Against the oracle's formula, padding rows and the
    columns around the result, and run to run."""
    monkeypatch.setenv("ARCZ_Q8_WK", "1")   # (read when an engine is made)
    monkeypatch.setenv("ARCZ_Q4_SPLITK", str(pieces))
    print(f"eight waves T={T} Mp={Mp} N={N} K={K} pieces={pieces} acc={acc} ldc=N+{ldc + c_off} c_off={c_off}", flush=True)
    eng = az.Engine(Mp, K)
    W = make_weights(az.Q8_0, N, K, seed=111)
    x = make_acts(T, K, seed=112, outliers=True)
    ld = N + ldc + c_off
    c0 = np.random.default_rng(113).standard_normal((Mp, ld)).astype(np.float32)
    y, y2 = (run_gemm(eng, az.Q8_0, W, N, K, x, Mp, acc=acc, c_init=c0, ldc=ld, c_off=c_off) for _ in range(2))
    eng.close()
    assert np.array_equal(y.view(np.uint32), y2.view(np.uint32))
    aq, asc, absum = quantize_padded(x, Mp)
    c = c0[:, c_off:c_off + N]
    form = np.zeros((Mp, N), np.float64)
    form[:T] = orc.matmul_formula(az.Q8_0, 1, W, N, K, aq[:T], asc, absum)
    want = form + c if acc == 1 else form * (c.astype(np.float64) / (1.0 + np.exp(-c.astype(np.float64)))) if acc == 2 else form
    assert mixed_err(y[:T, c_off:c_off + N], want[:T]) <= TIGHT
    assert np.array_equal(y[T:, c_off:c_off + N], c[T:] if acc == 1 else np.zeros((Mp - T, N), np.float32))
    assert np.array_equal(y[:, :c_off], c0[:, :c_off]) and np.array_equal(y[:, c_off + N:], c0[:, c_off + N:])


@pytest.mark.parametrize("qtype,T,Mp,N,K,acc", [(az.Q3_K, 256, 256, 4096, 256, 0), (az.Q3_K, 300, 304, 3500, 1280, 1),
                                                (az.Q4_0, 257, 260, 12289, 256, 0), (az.Q4_0, 1000, 1024, 3200, 768, 2),
                                                (az.MXFP4, 385, 400, 8190, 512, 1), (az.IQ3_S, 390, 400, 8000, 1024, 0),
                                                (az.Q6_K, 1030, 1040, 7700, 256, 0), (az.Q6_K, 1024, 1024, 7810, 768, 1),
                                                (az.IQ3_XXS, 2049, 2052, 4100, 512, 0), (az.IQ3_XXS, 1025, 1040, 8100, 1024, 2)])
def test_gemm_on_digits(rt, monkeypatch, qtype, T, Mp, N, K, acc):
    """The GEMM of long chunks whose tokens and rows are written as digits first: one, two and three digits a weight, K
    shared out and not, ragged last tiles of tokens and rows, one superblock and odd numbers of them, the three epilogues.
    Against the oracle, and run to run."""
    monkeypatch.setenv("ARCZ_GEMM_DIGITS", "1")   # (read when an engine is made; the rule leaves the smallest to the int8 kernels)
    print(f"digits {TYPE_NAMES[qtype]} T={T} Mp={Mp} N={N} K={K} acc={acc}", flush=True)
    eng = az.Engine(Mp, K)
    W = make_weights(qtype, N, K, seed=81)
    x = make_acts(T, K, seed=82, outliers=True)
    c0 = np.random.default_rng(83).standard_normal((Mp, N)).astype(np.float32)
    y = run_gemm(eng, qtype, W, N, K, x, Mp, acc=acc, c_init=c0 if acc else None)[:T]
    y2 = run_gemm(eng, qtype, W, N, K, x, Mp, acc=acc, c_init=c0 if acc else None)[:T]
    eng.close()
    assert np.array_equal(y.view(np.uint32), y2.view(np.uint32))
    aq, asc, _ = quantize_padded(x, Mp)
    ref = orc.matmul_ref(qtype, W, N, K, aq[:T], np.ascontiguousarray(asc[:, :T]))
    if acc == 1:
        ref = ref + c0[:T]
    elif acc == 2:
        g = c0[:T].astype(np.float64)
        ref = ref * (g / (1.0 + np.exp(-g)))
    assert np.isfinite(y).all() and mixed_err(y, ref) <= TOL


@pytest.mark.parametrize("qtype,T,Mp,N,K", [(az.Q6_K, 20, 256, 1000, 768), (az.Q8_0, 20, 256, 3000, 512), (az.Q8_0, 60, 384, 256, 4096),
                                            (az.Q4_K, 20, 384, 5200, 512), (az.Q4_K, 130, 256, 392, 2048), (az.Q3_K, 100, 256, 4224, 2048),
                                            (az.Q4_K, 10, 16, 264, 1024), (az.Q5_K, 12, 16, 264, 6400), (az.IQ4_XS, 40, 256, 300, 512)])
def test_caller_quantized_rows_are_multiplied_as_given(rt, qtype, T, Mp, N, K):
    """set_activations takes all Mp rows from the caller: in a chunk of more than 8 tokens the rows from T on are multiplied
    like the others, whatever form the launch rule takes (tiles left out, K in pieces, digits, gemv_mm)."""
    print(f"caller's rows {TYPE_NAMES[qtype]} T={T} Mp={Mp} N={N} K={K}", flush=True)
    W = make_weights(qtype, N, K, seed=89)
    aq, asc, absum = orc.quantize_act(make_acts(Mp, K, seed=90, outliers=True))
    eng = az.Engine(Mp, K)
    w = eng.make_weight(qtype, N, K, W)
    cb = az.Runtime.alloc(Mp * N * 4).fill(0xFFFFFFFF)
    eng.set_activations(aq, asc, absum, K, Mp, T)
    eng.matmul("test", w, Mp, cb, N, 0, 0)
    y = cb.read(np.float32, Mp * N).reshape(Mp, N)
    for b in (cb, w):
        b.free()
    eng.close()
    assert np.isfinite(y).all() and rel_err_rows(y, orc.matmul_ref(qtype, W, N, K, aq, asc)).max() <= TOL


@pytest.mark.parametrize("qtype", [az.Q4_K, az.Q5_K, az.Q4_0, az.IQ4_XS, az.IQ4_NL, az.MXFP4, az.Q6_K, az.Q8_0, az.Q3_K, az.IQ3_S, az.IQ3_XXS])
@pytest.mark.parametrize("T,Mp,N,K", [(40, 48, 272, 768), (33, 48, 1040, 1024), (120, 128, 528, 1280), (24, 32, 256, 1280)])
def test_short_rows_in_pieces_of_a_superblock(rt, qtype, T, Mp, N, K):
    """Rows of three to five superblocks of few tiles: a piece of K each, on the int8 kernels (the product and its reduction), against
    the oracle, into a wider C; the reduction's other two epilogues on the same sums."""
    print(f"pieces of a superblock {TYPE_NAMES[qtype]} T={T} N={N} K={K}", flush=True)
    W = make_weights(qtype, N, K, seed=93)
    x = make_acts(T, K, seed=94, outliers=True)
    eng = az.Engine(Mp, K)
    eng.profile(True)
    y = run_gemm(eng, qtype, W, N, K, x, Mp, ldc=N + 5, c_off=3)
    eng.profile_collect()
    assert eng.profile_get("act_digits")[1] == 0 and eng.profile_get("test")[1] >= 2
    eng.profile(False)
    c0 = az.gen_normal(95, (Mp, N + 5))
    ya, ys = (run_gemm(eng, qtype, W, N, K, x, Mp, acc=acc, c_init=c0, ldc=N + 5, c_off=3) for acc in (1, 2))
    eng.close()
    y0, g = y[:, 3:3 + N], c0[:, 3:3 + N].astype(np.float64)
    want = y0.astype(np.float64) * (g / (1.0 + np.exp(-g)))
    assert np.array_equal(ya[:, 3:3 + N], y0 + c0[:, 3:3 + N])
    assert np.abs(ys[:, 3:3 + N] - want).max() <= 1e-5 * np.abs(want).max()   # (three f32 roundings and the exponential's)
    for other in (ya, ys):
        assert np.array_equal(np.delete(other, np.s_[3:3 + N], axis=1), np.delete(c0, np.s_[3:3 + N], axis=1))
    aq, asc, _ = quantize_padded(x, Mp)
    assert rel_err_rows(y[:T, 3:3 + N], orc.matmul_ref(qtype, W, N, K, aq[:T], asc)).max() <= TOL
    assert not y[T:, 3:3 + N].any()
    assert (np.delete(y, np.s_[3:3 + N], axis=1).view(np.uint32) == 0xFFFFFFFF).all()


@pytest.mark.parametrize("qtype,N,K,digits", [(az.Q4_0, 1024, 2048, 1), (az.Q4_0, 1023, 2048, 0), (az.MXFP4, 513, 4096, 1), (az.Q4_0, 4096, 768, 0),
                                              (az.Q3_K, 1024, 2048, 1), (az.Q3_K, 4096, 1024, 0), (az.IQ3_S, 1024, 4096, 1),
                                              (az.IQ3_S, 1023, 4096, 0)])
def test_smallest_matrices_that_keep_digits(rt, qtype, N, K, digits):
    """The sizes from which a weight's rows are kept as digits, by type and row length, and those below (41 tokens, which only kept
    digits take): which kernels ran, and the oracle."""
    T, Mp = 41, 48
    print(f"kept digits type={qtype} N={N} K={K}", flush=True)
    W = make_weights(qtype, N, K, seed=91)
    x = make_acts(T, K, seed=92, outliers=True)
    eng = az.Engine(Mp, K)
    eng.profile(True)
    y = run_gemm(eng, qtype, W, N, K, x, Mp)
    eng.profile_collect()
    assert eng.profile_get("act_digits")[1] == digits and eng.profile_get("keep_digits")[1] == digits
    eng.close()
    aq, asc, _ = quantize_padded(x, Mp)
    assert rel_err_rows(y[:T], orc.matmul_ref(qtype, W, N, K, aq[:T], asc)).max() <= TOL


@pytest.mark.parametrize("qtype,T,Mp,N,K", [(az.IQ4_XS, 241, 256, 816, 3072), (az.IQ4_NL, 65, 80, 1504, 2048), (az.Q5_K, 418, 512, 1888, 2048),
                                            (az.IQ4_XS, 56, 64, 1408, 1536)])
def test_kept_digits_left_for_even_pieces_of_k(rt, qtype, T, Mp, N, K):
    """Small matrices whose K goes in even pieces on the int8 kernels, which are then ahead of the kept digits: which kernels
    ran, and the oracle."""
    print(f"even pieces {TYPE_NAMES[qtype]} T={T} N={N} K={K}", flush=True)
    W = make_weights(qtype, N, K, seed=97)
    x = make_acts(T, K, seed=98, outliers=True)
    eng = az.Engine(Mp, K)
    eng.profile(True)
    y = run_gemm(eng, qtype, W, N, K, x, Mp)
    eng.profile_collect()
    assert eng.profile_get("keep_digits")[1] == 1 and eng.profile_get("act_digits")[1] == 0 and eng.profile_get("test")[1] == 2
    eng.close()
    aq, asc, _ = quantize_padded(x, Mp)
    assert rel_err_rows(y[:T], orc.matmul_ref(qtype, W, N, K, aq[:T], asc)).max() <= TOL


@pytest.mark.parametrize("env,digits,products", [({}, 1, None), ({"ARCZ_GEMM_DIGITS": "1", "ARCZ_Q4_SPLITK": "2"}, 1, 2), ({"ARCZ_GEMM_DIGITS": "0"}, 0, None), ({"ARCZ_Q4_SPLITK": "0"}, 1, 1),
                                                 ({"ARCZ_Q4_SPLITK": "2"}, 1, 2),
                                                 ({"ARCZ_GEMM_SPLIT": "3", "ARCZ_Q4_SPLITK": "0"}, 0, 4)])
def test_switches_of_the_gemm_on_digits(rt, monkeypatch, env, digits, products):
    """The launch-rule switches on a chunk that the digits take by rule: off, K in one piece, two pieces forced (the
    product and its reduction), and the int8 kernels in pieces of superblocks (one expansion and a launch a piece)."""
    T, N, K = 256, 4224, 2048
    print(f"digits switches {env}", flush=True)
    for k, v in env.items():
        monkeypatch.setenv(k, v)          # (read when an engine is made)
    W = make_weights(az.Q3_K, N, K, seed=87)
    x = make_acts(T, K, seed=88, outliers=True)
    eng = az.Engine(T, K)
    eng.profile(True)
    y = run_gemm(eng, az.Q3_K, W, N, K, x, T)
    eng.profile_collect()
    counts = [eng.profile_get(k)[1] for k in ("act_digits", "test")]
    eng.close()
    # (where the rule ends: the same outputs over shorter rows)
    eng = az.Engine(T, K)
    eng.profile(True)
    run_gemm(eng, az.Q3_K, make_weights(az.Q3_K, N, 1024, seed=86), N, 1024, x[:, :1024].copy(), T)
    eng.profile_collect()
    assert eng.profile_get("act_digits")[1] == (1 if env.get("ARCZ_GEMM_DIGITS") == "1" else 0)
    eng.close()
    aq, asc, _ = quantize_padded(x, T)
    assert np.isfinite(y).all() and rel_err_rows(y, orc.matmul_ref(az.Q3_K, W, N, K, aq, asc)).max() <= TOL
    assert counts[0] == digits and products in (None, counts[1]), counts


@pytest.mark.parametrize("qtype,T,N,K", [(az.Q4_0, 128, 4096, 2048), (az.Q3_K, 200, 4099, 2304), (az.Q6_K, 400, 4100, 4096), (az.IQ3_XXS, 200, 12300, 2048),
                                         (az.MXFP4, 65, 4225, 2048), (az.IQ4_XS, 90, 9001, 1024), (az.IQ4_NL, 300, 16500, 1024)])
def test_digits_of_rows_kept_with_the_weight(rt, qtype, T, N, K):
    """Matrices of 2^23 values and more keep their rows' digits: no matmul writes them, and shorter chunks are multiplied on
    digits.  Given back where an allocation finds no memory -- not while a recorded list names them --, the weight is
    multiplied all the same.  Against the oracle."""
    print(f"kept digits {TYPE_NAMES[qtype]} T={T} N={N} K={K}", flush=True)
    Mp = (T + 15) // 16 * 16 if T < 128 else (T + 127) // 128 * 128
    W = make_weights(qtype, N, K, seed=61)
    x = make_acts(T, K, seed=62, outliers=True)
    aq, asc, _ = quantize_padded(x, Mp)
    rows = np.r_[0:300, N - 300:N]
    Ws = np.ascontiguousarray(W.reshape(N, -1)[rows]).reshape(-1)
    ref = orc.matmul_ref(qtype, Ws, len(rows), K, aq[:T], np.ascontiguousarray(asc[:, :T]))
    eng = az.Engine(512, K)
    spare0 = az.lib.arcz_spare_bytes()
    w = eng.make_weight(qtype, N, K, W)
    spare1 = az.lib.arcz_spare_bytes()
    assert spare1 > spare0
    xb, cb = az.Runtime.from_numpy(x), az.Runtime.alloc(Mp * N * 4)

    def step():
        eng.quantize(xb, K, K, Mp, T)
        eng.matmul("test", w, Mp, cb, N, 0, 0)

    def out(f):
        cb.fill(0xFFFFFFFF)
        f()
        y = cb.read(np.float32, Mp * N).reshape(Mp, N)
        assert np.isfinite(y).all() and not y[T:].any() and rel_err_rows(y[:T, rows], ref).max() <= TOL
        return y.view(np.uint32)

    eng.profile(True)
    y = out(step)
    eng.profile_collect()
    assert eng.profile_get("act_digits")[1] == 1 and eng.profile_get("row_digits")[1] == 0
    eng.profile(False)
    lst = az.Runtime.record(step)
    try:
        az.lib.arcz_set_fake_oom(1)
        with pytest.raises(az.ArczError):
            az.Runtime.alloc(1024)                      # (every allocation fails once; what the list names stays)
        assert az.lib.arcz_spare_bytes() == spare1
        assert np.array_equal(out(lst.run), y)
        lst.free()
        lst = None
        az.Runtime.alloc(1024).free()
        assert az.lib.arcz_spare_bytes() == spare0
    finally:
        az.lib.arcz_set_fake_oom(0)
        if lst is not None:
            lst.free()
    out(step)
    for b in (xb, cb, w):
        b.free()
    eng.close()
    assert az.lib.arcz_spare_bytes() == spare0


def test_limits_of_kept_digits(rt):
    """Kept digits hold at most an eighth of the device's memory, over all engines, and leave a quarter of it free; a weight
    beyond that is multiplied without them.  An allocation that finds no memory takes back as many as it needs, the
    smallest that is large enough first, another allocator's request as many as make it; each weight's results agree
    before and after."""
    T = Mp = 256
    print("limits of kept digits", flush=True)
    sizes = [(4096, 2048), (8192, 2048), (12288, 2048)]
    Ws = [make_weights(az.Q4_0, n, k, seed=81 + i) for i, (n, k) in enumerate(sizes)]
    x = make_acts(T, 2048, seed=84)
    engs = [az.Engine(Mp, 2048) for _ in range(2)]
    xb, cb = az.Runtime.from_numpy(x), az.Runtime.alloc(Mp * 12288 * 4)
    base = az.lib.arcz_spare_bytes()
    each = [n * k // 32 * 28 for n, k in sizes]                    # (24 bytes of digits and a scale for a block of 32)

    def out(e, w):
        e.quantize(xb, 2048, 2048, Mp, T)
        e.profile(True)
        e.profile_reset()
        e.matmul("test", w, Mp, cb, w.N, 0, 0)
        e.profile_collect()
        return cb.read(np.float32, Mp * w.N).reshape(Mp, -1), e.profile_get("row_digits")[1] == 0 and e.profile_get("act_digits")[1] == 1

    def upload(total, free, order=(0, 1, 2)):
        az.lib.arcz_set_fake_mem(total, free)
        try:
            made = {i: engs[i % 2].make_weight(az.Q4_0, *sizes[i], Ws[i]) for i in order}
        finally:
            az.lib.arcz_set_fake_mem(0, 0)
        return [made[i] for i in range(3)]

    # the eighth holds the first and, uploaded next, the third; eight bytes fewer of memory: the second, uploaded last
    big, eighth = 1 << 40, base + each[0] + each[2]
    for total, kept in ((8 * eighth, [1, 0, 1]), (8 * eighth - 8, [1, 1, 0])):
        ws = upload(total, big, (0, 2, 1))
        assert az.lib.arcz_spare_bytes() - base == sum(b for b, k in zip(each, kept) if k)
        for w, k in zip(ws, kept):
            assert out(w.eng, w)[1] == bool(k)
            w.free()
        assert az.lib.arcz_spare_bytes() == base
    # a quarter stays free
    ws = upload(big, big // 4 + each[1])
    assert az.lib.arcz_spare_bytes() - base == each[0] + each[1]
    for w in ws:
        w.free()
    # taken back one by one
    ws = upload(0, 0)
    assert az.lib.arcz_spare_bytes() - base == sum(each)
    ys = [out(w.eng, w)[0] for w in ws]
    left = sum(each)
    for need, gone in ((each[0] + 1, 1), (each[2] * 2, 2), (64, 0)):
        az.lib.arcz_set_fake_oom(1)
        try:
            az.Runtime.alloc(need).free()
        finally:
            az.lib.arcz_set_fake_oom(0)
        left -= each[gone]
        assert az.lib.arcz_spare_bytes() - base == left
    for w, y in zip(ws, ys):
        z, kept = out(w.eng, w)
        assert not kept and rel_err_rows(z, y).max() <= 2e-5          # (the same block sums, f32 from there on)
        w.free()
    ws = upload(0, 0)
    assert az.Runtime.give_back(each[1]) == each[1] and az.Runtime.give_back(each[2] + 1) == each[0] + each[2]
    assert az.lib.arcz_spare_bytes() == base
    for b in (xb, cb, *ws):
        b.free()
    for e in engs:
        e.close()


def test_allocations_that_kept_digits_make_no_room_for(rt):
    """A request that is larger than what is free and what kept digits hold fails, and they stay; one byte fewer takes them."""
    N, K = 4096, 2048
    print("allocations that kept digits make no room for", flush=True)
    eng = az.Engine(256, K)
    spare0 = az.lib.arcz_spare_bytes()
    ws = [eng.make_weight(az.Q4_0, N, K, make_weights(az.Q4_0, N, K, seed=91 + i)) for i in range(2)]
    held = az.lib.arcz_spare_bytes()
    assert held > spare0
    with pytest.raises(az.ArczError):
        az.Runtime.alloc(1 << 50)
    assert az.lib.arcz_spare_bytes() == held
    for free in (999, 1000):
        az.lib.arcz_set_fake_mem(1 << 40, free)
        az.lib.arcz_set_fake_oom(1)   # (every allocation finds no memory once)
        try:
            if free == 999:
                with pytest.raises(az.ArczError):
                    az.Runtime.alloc(held + 1000)
                assert az.lib.arcz_spare_bytes() == held
            else:
                az.Runtime.alloc(held + 1000).free()
                assert az.lib.arcz_spare_bytes() < held
        finally:
            az.lib.arcz_set_fake_oom(0)
            az.lib.arcz_set_fake_mem(0, 0)
    for w in ws:
        w.free()
    eng.close()


@pytest.mark.parametrize("qtype,N,K", [(az.Q4_0, 4096, 2048), (az.Q4_K, 4100, 2304), (az.Q6_K, 4100, 4096)])
def test_planes_rewritten_under_kept_digits(rt, qtype, N, K):
    """A matrix whose rows are kept as digits, its planes asked for and rewritten: chunks multiply the new values, as the
    passes of few tokens do -- bit for bit a weight uploaded with them whose digits were dropped too.  While a recorded
    list names the digits the planes are not handed out, and the list goes on giving the old values."""
    T = Mp = 512
    print(f"planes rewritten {TYPE_NAMES[qtype]} N={N} K={K}", flush=True)
    W = [make_weights(qtype, N, K, seed=s) for s in (71, 72)]
    x = make_acts(T, K, seed=73)
    eng = az.Engine(Mp, K)
    spare0 = az.lib.arcz_spare_bytes()
    w = eng.make_weight(qtype, N, K, W[0])
    spare1 = az.lib.arcz_spare_bytes()
    assert spare1 > spare0
    xb, cb = az.Runtime.from_numpy(x), az.Runtime.alloc(Mp * N * 4)

    def step(v=None):
        eng.quantize(xb, K, K, Mp, T)
        eng.matmul("test", v or w, Mp, cb, N, 0, 0)

    def out(f=step):
        cb.fill(0xFFFFFFFF)
        f()
        return cb.read(np.uint32, Mp * N)

    y0 = out()
    lst = az.Runtime.record(step)
    assert not az.lib.arcz_weight_raw(w.h) and b"launch list" in az.lib.arcz_engine_error()
    assert az.lib.arcz_spare_bytes() == spare1 and np.array_equal(out(lst.run), y0) and np.array_equal(out(), y0)
    lst.free()
    az.lib.arcz_record_begin()
    assert not az.lib.arcz_weight_raw(w.h)
    az.lib.arcz_record_end(None)
    raw = az.binding.Buffer(az.lib.arcz_weight_raw(w.h), owner=False)
    assert raw.h and az.lib.arcz_spare_bytes() == spare0 and raw.size == az.planes_bytes(qtype, N, K)
    raw.write(az.repack_planes(qtype, N, K, W[1]))
    w1 = eng.make_weight(qtype, N, K, W[1])
    assert az.lib.arcz_weight_raw(w1.h)
    assert np.array_equal(out(), out(lambda: step(w1)))
    rows = np.r_[0:200, N - 200:N]
    y = out().view(np.float32).reshape(Mp, N)
    aq, asc, _ = quantize_padded(x, Mp)
    ref = orc.matmul_ref(qtype, np.ascontiguousarray(W[1].reshape(N, -1)[rows]).reshape(-1), len(rows), K, aq, asc)
    assert np.isfinite(y).all() and rel_err_rows(y[:, rows], ref).max() <= TOL
    for b in (w, w1, xb, cb):
        b.free()
    eng.close()


@pytest.mark.parametrize("qtype", [az.Q4_K, az.Q4_0, az.Q3_K, az.Q6_K])
@pytest.mark.parametrize("T,Mp,N,K,acc,pieces", [(17, 32, 8200, 1024, 0, 1), (33, 128, 4099, 2304, 2, 4), (150, 256, 4228, 2048, 1, 1), (193, 208, 33000, 256, 0, 1), (260, 384, 4096, 2560, 2, 3)])
def test_gemm_on_digits_tiles_of_64_tokens(rt, monkeypatch, qtype, T, Mp, N, K, acc, pieces):
    """Tiles of 64 tokens x 256 rows on the images of 128 and 128: at most 32 tokens and more in the last one, the second half of
    an image of tokens, an odd number of row tiles, K in pieces and not, padding rows and the columns beside C's, the three
    epilogues.  Against the oracle on the first and last rows, and run to run."""
    monkeypatch.setenv("ARCZ_GEMM_DIGITS", "1")
    monkeypatch.setenv("ARCZ_GEMM_D64", "1")
    if pieces > 1:
        monkeypatch.setenv("ARCZ_Q4_SPLITK", str(pieces))
    else:
        monkeypatch.setenv("ARCZ_Q4_SPLITK", "0")
    print(f"64-token tiles on digits {TYPE_NAMES[qtype]} T={T} Mp={Mp} N={N} K={K} acc={acc} pieces={pieces}", flush=True)
    ldc = N + 5
    W = make_weights(qtype, N, K, seed=41)
    x = make_acts(T, K, seed=42, outliers=True)
    c0 = np.random.default_rng(43).standard_normal((Mp, ldc)).astype(np.float32)
    eng = az.Engine(Mp, K)
    spare0 = az.lib.arcz_spare_bytes()
    w = eng.make_weight(qtype, N, K, W)
    assert az.lib.arcz_spare_bytes() > spare0   # (kept digits: the switch then names these tiles alone)
    xb, cb = az.Runtime.from_numpy(x), az.Runtime.alloc(Mp * ldc * 4)
    eng.quantize(xb, K, K, Mp, T)
    ys = []
    eng.profile(True)
    for _ in range(2):
        cb.write(c0)
        eng.matmul("test", w, Mp, cb, ldc, 0, acc)
        ys.append(cb.read(np.float32, Mp * ldc).reshape(Mp, ldc))
    eng.profile_collect()
    assert eng.profile_get("act_digits")[1] == 2
    for b in (xb, cb, w):
        b.free()
    eng.close()
    y = ys[0]
    assert np.array_equal(y.view(np.uint32), ys[1].view(np.uint32)) and np.array_equal(y[:, N:], c0[:, N:]) and np.isfinite(y).all()
    assert np.array_equal(y[T:, :N], c0[T:, :N] if acc == 1 else np.zeros((Mp - T, N), np.float32))
    rows = np.r_[0:200, N - 400:N]
    Ws = np.ascontiguousarray(W.reshape(N, -1)[rows]).reshape(-1)
    aq, asc, _ = quantize_padded(x, Mp)
    ref = orc.matmul_ref(qtype, Ws, len(rows), K, aq[:T], np.ascontiguousarray(asc[:, :T]))
    g = c0[:T, rows].astype(np.float64)
    ref = ref + g if acc == 1 else ref * (g / (1.0 + np.exp(-g))) if acc == 2 else ref
    assert mixed_err(y[:T, rows], ref) <= TOL


@pytest.mark.parametrize("qtype,T,N,K,ldc,acc", [(az.Q4_0, 300, 11653, 4096, 11660, 1), (az.Q4_K, 640, 13308, 2560, 13312, 2), (az.Q6_K, 130, 17501, 4096, 17501, 0)])
def test_gemm_on_digits_in_pieces_of_the_last_tiles(rt, monkeypatch, qtype, T, N, K, ldc, acc):
    """Tiles that full rounds of work-groups leave over go in pieces of K, the others whole (273, 520 and 274 tiles on a chip
    of 256 compute units): ragged rows and whole vectors, the three epilogues, run to run, the columns beside C's untouched.
    Against the oracle on the first and last rows."""
    monkeypatch.setenv("ARCZ_GEMM_D64", "0")   # (read when an engine is made)
    monkeypatch.setenv("ARCZ_GEMM_DIGITS", "1")
    print(f"last tiles in pieces {TYPE_NAMES[qtype]} T={T} N={N} K={K} acc={acc}", flush=True)
    Mp = (T + 127) // 128 * 128
    W = make_weights(qtype, N, K, seed=51)
    x = make_acts(T, K, seed=52, outliers=True)
    c0 = np.random.default_rng(53).standard_normal((Mp, ldc)).astype(np.float32)
    eng = az.Engine(Mp, K)
    w = eng.make_weight(qtype, N, K, W)
    xb, cb = az.Runtime.from_numpy(x), az.Runtime.alloc(Mp * ldc * 4)
    eng.quantize(xb, K, K, Mp, T)
    ys = []
    for i in range(2):
        cb.write(c0)
        eng.profile(i == 0)
        eng.matmul("test", w, Mp, cb, ldc, 0, acc)
        ys.append(cb.read(np.float32, Mp * ldc).reshape(Mp, ldc))
        if i == 0:
            eng.profile_collect()
            assert eng.profile_get("test")[1] == 2 and eng.profile_get("act_digits")[1] == 1
    for b in (xb, cb, w):
        b.free()
    eng.close()
    assert np.array_equal(ys[0].view(np.uint32), ys[1].view(np.uint32)) and np.array_equal(ys[0][:, N:], c0[:, N:])
    rows = np.r_[0:200, N - 400:N]
    Ws = np.ascontiguousarray(W.reshape(N, -1)[rows]).reshape(-1)
    aq, asc, _ = quantize_padded(x, Mp)
    ref = orc.matmul_ref(qtype, Ws, len(rows), K, aq[:T], np.ascontiguousarray(asc[:, :T]))
    g = c0[:T, rows].astype(np.float64)
    ref = ref + g if acc == 1 else ref * (g / (1.0 + np.exp(-g))) if acc == 2 else ref
    y = ys[0][:T, rows]
    assert np.isfinite(ys[0]).all() and mixed_err(y, ref) <= TOL


def _extreme_rows(qtype, N, K, rng):
    """Blocks of random bytes with the superblock's scale set to one (IQ3_XXS: four), so that all values are integers; a
    fifth of the Q6_K and Q3_K rows at the ends of their ranges: every value -32 or 31 times -128 or 127, -4 or 3 times -32
    or 31, in runs and alternating."""
    one = np.frombuffer(np.float16(4.0 if qtype == az.IQ3_XXS else 1.0).tobytes(), np.uint8)
    nsb = K // 256
    n = az.gguf_bytes(qtype, 1, 256)
    if qtype in (az.Q4_0, az.MXFP4):
        blk = rng.integers(0, 256, (N, nsb * 8, n // 8), dtype=np.uint8)
        if qtype == az.MXFP4:
            blk[..., 0] = 128
        else:
            blk[..., 0:2] = one
        return np.ascontiguousarray(blk).reshape(-1)
    blk = rng.integers(0, 256, (N, nsb, n), dtype=np.uint8)
    ends = np.arange(N) % 5 == 0
    fill = np.array([0x00, 0xFF, 0xAA, 0x55], np.uint8)[rng.integers(0, 4, (N, nsb))]
    if qtype == az.Q6_K:
        blk[ends, :, :192] = np.where(rng.integers(0, 2, (N, nsb)) == 1, fill, 0)[ends][..., None]
        blk[ends, :, 192:208] = np.where(rng.integers(0, 2, (N, nsb, 16)) == 1, 128, 127).astype(np.uint8)[ends]
        blk[..., 208:210] = one
    elif qtype == az.Q3_K:
        blk[ends, :, :96] = fill[ends][..., None]
        blk[ends, :, 96:108] = np.array([0x00, 0xFF], np.uint8)[rng.integers(0, 2, (N, nsb))][ends][..., None]
        blk[..., 108:110] = one
    else:
        blk[..., 0:2] = one
    return blk.reshape(-1)


@pytest.mark.parametrize("qtype,T,N", [(az.Q6_K, 1024, 7808), (az.Q3_K, 256, 4224), (az.IQ3_XXS, 1024, 8192), (az.IQ3_S, 256, 12288),
                                       (az.Q4_0, 256, 12288), (az.MXFP4, 256, 12288)])
def test_gemm_on_digits_block_sums_exact(rt, monkeypatch, qtype, T, N):
    """The GEMM on digits keeps every block sum exact, at the ends of the ranges too: a token has one block of values up to
    -128 (all ends, alternating ends, random ends, random) and zeros elsewhere, unit scales, so an output is one block's
    sum -- up to 32 x 128 x 4096 = 2^24, with whole and partial cancellation -- and has to be that integer."""
    monkeypatch.setenv("ARCZ_GEMM_DIGITS", "1")   # (read when an engine is made; the rule leaves the smallest to the int8 kernels)
    print(f"digits, exact block sums {TYPE_NAMES[qtype]} T={T} N={N}", flush=True)
    K = 512
    rng = np.random.default_rng(170 + qtype)
    W = _extreme_rows(qtype, N, K, rng)
    wi = orc.dequant_rows(qtype, W, N, K).astype(np.float64)
    assert np.array_equal(wi, np.round(wi))
    if qtype in (az.Q6_K, az.Q3_K):
        assert np.abs(wi).max() == (4096 if qtype == az.Q6_K else 128)
    aq = np.zeros((T, K // 32, 32), np.int8)
    for t in range(T):
        i = np.arange(32)
        v = [np.full(32, 127), np.full(32, -128), np.where(i & 1, 127, -127), np.where(i < 16, -128, 127), np.where(i & 2, -127, 127),
             np.where(rng.integers(0, 2, 32) == 1, 127, -128), rng.integers(-128, 128, 32), np.where(i & 1, 1, -128)][(t // (K // 32)) % 8]
        aq[t, t % (K // 32)] = v
    aq = aq.reshape(T, K)
    asc = np.ones((K // 32, T), np.float32)
    absum = np.ascontiguousarray(aq.reshape(T, K // 16, 16).sum(axis=2, dtype=np.int64).astype(np.int16).T)
    eng = az.Engine(T, K)
    w = eng.make_weight(qtype, N, K, W)
    eng.set_activations(aq, asc, absum, K, T, T)
    cb = az.Runtime.alloc(T * N * 4).fill(0xFFFFFFFF)
    eng.matmul("test", w, T, cb, N, 0, 0)
    y = cb.read(np.float32, T * N).reshape(T, N)
    for b in (cb, w):
        b.free()
    eng.close()
    want = aq.astype(np.float64) @ wi.T
    assert np.abs(want).max() <= 2 ** 24
    print(f"  largest sum {np.abs(want).max():.0f}, differing {int((y != want).sum())} of {y.size}", flush=True)
    assert np.array_equal(y, want.astype(np.float32))


@pytest.mark.parametrize("qtype", [az.Q4_K, az.Q5_K])
@pytest.mark.parametrize("T,Mp,N,K,acc", [(130, 144, 392, 512, 0), (257, 260, 390, 768, 1), (300, 384, 1029, 256, 2), (100, 112, 136, 5120, 0)])
def test_gemm_on_digits_with_a_minimum(rt, monkeypatch, qtype, T, Mp, N, K, acc):
    """Q4_K and Q5_K on digits: the values around their middle in one digit, the min term with what that leaves on the bf16
    instruction; K shared out and not, ragged last tiles, the three epilogues.  Tokens with a mean, where products and min
    term are both large, against 64 bits (measured up to 2.3e-7 of the result's norm; test_min_term_is_not_one_sided has the
    comparison with the int8 kernels)."""
    monkeypatch.setenv("ARCZ_GEMM_DIGITS", "1")
    print(f"digits with a minimum {TYPE_NAMES[qtype]} T={T} Mp={Mp} N={N} K={K} acc={acc}", flush=True)
    W = make_weights(qtype, N, K, seed=63)
    x = make_acts(T, K, seed=64, outliers=True) + np.float32(0.5)
    c0 = np.random.default_rng(65).standard_normal((Mp, N)).astype(np.float32)
    eng = az.Engine(Mp, K)
    y = run_gemm(eng, qtype, W, N, K, x, Mp, acc=acc, c_init=c0 if acc else None)
    eng.close()
    aq, asc, _ = quantize_padded(x, Mp)
    ref = (aq * np.repeat(asc.astype(np.float64).T, 32, axis=1)) @ orc.dequant_rows(qtype, W, N, K).astype(np.float64).T
    c64 = c0.astype(np.float64)
    ref = ref + c64 if acc == 1 else ref * (c64 / (1.0 + np.exp(-c64))) if acc == 2 else ref
    assert np.isfinite(y).all() and mixed_err(y, ref) <= TOL
    if acc == 0:
        assert np.linalg.norm(y - ref) <= 4e-7 * np.linalg.norm(ref) and not y[T:].any()


@pytest.mark.parametrize("qtype", [az.Q4_K, az.Q5_K])
@pytest.mark.parametrize("T,N,K", [(300, 2048, 4096), (200, 768, 17408), (31, 2048, 5120)])
def test_min_term_is_not_one_sided(rt, monkeypatch, qtype, T, N, K):
    """The min term's pieces on the bf16 instruction, which cuts products off towards zero: tokens with a mean, against 64 bits,
    K in one piece.  The results' errors have no mean of their own -- one piece by truncation leaves 0.5 - 3.1e-7 of the
    results' deviation, a mean of this many errors of 2 - 7e-7 with the tokens' and rows' own in common is below 3e-8 -- and
    their norm is no larger than with the int8 kernels, whose min term is an f32 instruction (to 2 %: other sums in f32)."""
    print(f"min term {TYPE_NAMES[qtype]} T={T} N={N} K={K}", flush=True)
    monkeypatch.setenv("ARCZ_Q4_SPLITK", "0")
    Mp = (T + 127) // 128 * 128
    W = make_weights(qtype, N, K, seed=61)
    x = make_acts(T, K, seed=62, outliers=True) + np.float32(0.5)
    aq, asc, _ = orc.quantize_act(x)
    ref = (aq * np.repeat(asc.astype(np.float64).T, 32, axis=1)) @ orc.dequant_rows64(qtype, W, N, K).T
    off = {}
    for digits, d64 in (("0", "0"), ("1", "0"), ("1", "1")):
        monkeypatch.setenv("ARCZ_GEMM_DIGITS", digits)   # (read when an engine is made)
        monkeypatch.setenv("ARCZ_GEMM_D64", d64)
        eng = az.Engine(Mp, K)
        e = run_gemm(eng, qtype, W, N, K, x, Mp)[:T] - ref
        eng.close()
        off[digits + d64] = np.linalg.norm(e) / np.linalg.norm(ref)
        mean = e.mean() / ref.std()
        print(f"  digits={digits} 64-token tiles={d64}: off {off[digits + d64]:.3g}, mean {mean:.2g}", flush=True)
        assert abs(mean) <= 3e-8
    assert max(off["10"], off["11"]) <= 1.02 * off["00"]


@pytest.mark.parametrize("qtype", [az.Q4_K, az.Q5_K])
def test_gemm_on_digits_with_a_minimum_exact(rt, monkeypatch, qtype):
    """... and exact where all is whole: scale and minimum one, random sub-scales and values, a token one block of values at
    the ends of the range; the largest products are 63 x 31 x 32 x 128 < 2^23."""
    monkeypatch.setenv("ARCZ_GEMM_DIGITS", "1")
    T, N, K = 256, 640, 512
    rng = np.random.default_rng(180 + qtype)
    blk = rng.integers(0, 256, (N, K // 256, az.gguf_bytes(qtype, 1, 256)), dtype=np.uint8)
    blk[..., 0:4] = np.frombuffer(np.array([1.0, 1.0], np.float16).tobytes(), np.uint8)
    W = blk.reshape(-1)
    wi = orc.dequant_rows(qtype, W, N, K).astype(np.float64)
    aq = np.zeros((T, K // 32, 32), np.int8)
    for t in range(T):
        i = np.arange(32)
        aq[t, t % (K // 32)] = [np.full(32, 127), np.full(32, -128), np.where(i & 1, 127, -127), rng.integers(-128, 128, 32)][(t // (K // 32)) % 4]
    aq = aq.reshape(T, K)
    absum = np.ascontiguousarray(aq.reshape(T, K // 16, 16).sum(axis=2, dtype=np.int64).astype(np.int16).T)
    eng = az.Engine(T, K)
    w = eng.make_weight(qtype, N, K, W)
    eng.set_activations(aq, np.ones((K // 32, T), np.float32), absum, K, T, T)
    cb = az.Runtime.alloc(T * N * 4).fill(0xFFFFFFFF)
    eng.matmul("test", w, T, cb, N, 0, 0)
    y = cb.read(np.float32, T * N).reshape(T, N)
    for b in (cb, w):
        b.free()
    eng.close()
    assert np.array_equal(y, (aq.astype(np.float64) @ wi.T).astype(np.float32))


@pytest.mark.parametrize("qtype,N,K", [(az.Q4_0, 4096, 2048), (az.Q5_K, 4100, 2304), (az.MXFP4, 4100, 4096)])
@pytest.mark.parametrize("T,rows", [(300, 384), (70, 80)])
def test_kept_digits_on_another_engine(rt, qtype, N, K, T, rows):
    """Engines share weights: one whose rows are kept as digits, on an engine that uploaded none (no room for its tokens'
    digits: the int8 kernels, bit for bit those of an upload without digits) and on one that keeps digits itself, of a
    smaller matrix in a shorter engine: the uploader's kernels and bits."""
    print(f"kept digits on another engine {TYPE_NAMES[qtype]} T={T} N={N} K={K}", flush=True)
    W = make_weights(qtype, N, K, seed=101)
    x = make_acts(T, K, seed=102, outliers=True)
    first, plain, own = az.Engine(512, max(K, 4096)), az.Engine(rows, K), az.Engine(rows, K)
    spare0 = az.lib.arcz_spare_bytes()
    w = first.make_weight(qtype, N, K, W)
    assert az.lib.arcz_spare_bytes() > spare0
    own.make_weight(az.Q4_0, 32768, 256, make_weights(az.Q4_0, 32768, 256, seed=103))
    w8 = first.make_weight(qtype, N, K, W)
    assert az.lib.arcz_weight_raw(w8.h)   # (handed out: without digits from here on)

    def out(e, v):
        xb, cb = az.Runtime.from_numpy(x), az.Runtime.alloc(rows * N * 4).fill(0xFFFFFFFF)
        e.quantize(xb, K, K, rows, T)
        e.profile(True)
        e.profile_reset()
        e.matmul("test", v, rows, cb, N, 0, 0)
        e.profile_collect()
        e.profile(False)
        y = cb.read(np.uint32, rows * N)
        for b in (xb, cb):
            b.free()
        return y, e.profile_get("act_digits")[1], e.profile_get("row_digits")[1]

    y, acts, made = out(first, w)
    assert made == 0 and (acts == 1 or T == 70)   # (of 70 tokens a type goes by price)
    z = out(own, w)
    assert z[1:] == (acts, 0) and np.array_equal(z[0], y)
    z, z8 = out(plain, w), out(plain, w8)
    assert z[1:] == z8[1:] == (0, 0) and np.array_equal(z[0], z8[0])
    aq, asc, _ = quantize_padded(x, rows)
    ref = orc.matmul_ref(qtype, W, N, K, aq, asc)
    for got in (y, z[0]):
        got = got.view(np.float32).reshape(rows, N)
        assert np.isfinite(got).all() and not got[T:].any() and rel_err_rows(got[:T], ref[:T]).max() <= TOL
    for e in (own, plain, first):
        e.close()


@pytest.mark.parametrize("qtype,T,N,K", [(az.Q4_0, 300, 12288, 512), (az.MXFP4, 512, 8192, 256), (az.Q6_K, 1024, 7808, 512), (az.Q3_K, 300, 4224, 2560)])
@pytest.mark.parametrize("before", [None, 256, 1024])
def test_weights_of_another_engine(rt, qtype, T, N, K, before):
    """Engines share weights: a matrix that an engine for single tokens uploaded, in a long chunk of an engine that
    uploaded none itself (no room for digits: the int8 kernels), or one with shorter or longer rows (room for panels of
    this one's rows, where these fill the chip, or for all).  Against the oracle."""
    print(f"another engine's {TYPE_NAMES[qtype]} T={T} N={N} K={K} before={before}", flush=True)
    small = az.Engine(16, K)
    W = make_weights(qtype, N, K, seed=96)
    w = small.make_weight(qtype, N, K, W)
    Mp = (T + 127) // 128 * 128
    eng = az.Engine(Mp, max(K, 1024))
    if before:   # (rows enough for the launch rule of every type)
        small_n = -(-8 * 1024 * 1024 // Mp) if qtype != az.Q3_K else -(-3 * 1024 * 1024 // Mp)
        eng.make_weight(qtype, small_n, before, make_weights(qtype, small_n, before, seed=95)).free()
    x = make_acts(T, K, seed=97, outliers=True)
    xb = az.Runtime.from_numpy(x)
    eng.quantize(xb, K, K, Mp, T)
    eng.profile(True)
    cb = az.Runtime.alloc(Mp * N * 4).fill(0xFFFFFFFF)
    if qtype == az.Q3_K and before is None:
        with pytest.raises(az.ArczError):   # (no room for the expansion that the int8 kernels take either)
            eng.matmul("test", w, Mp, cb, N, 0, 0)
        for b in (cb, xb, w, eng, small):
            b.close() if isinstance(b, az.Engine) else b.free()
        return
    eng.matmul("test", w, Mp, cb, N, 0, 0)
    y = cb.read(np.float32, Mp * N).reshape(Mp, N)
    for b in (cb, xb):
        b.free()
    w.free()
    eng.profile_collect()
    launches = eng.profile_get("row_digits")[1]
    eng.close()
    small.close()
    aq, asc, _ = quantize_padded(x, Mp)
    ref = orc.matmul_ref(qtype, W, N, K, aq[:T], np.ascontiguousarray(asc[:, :T]))
    assert np.isfinite(y).all() and rel_err_rows(y[:T], ref).max() <= TOL and not y[T:].any()
    # (256: half the room that rows of 512 values need, 32 row tiles x 8 token tiles for Q6_K, 85 x 3 for Q4_0; Q3_K, whose
    #  expansion has no room: 6 row tiles a panel, or 25)
    want = {None: 0, 256: {az.Q4_0: 0, az.MXFP4: 1, az.Q6_K: 2}, 1024: {az.Q4_0: 1, az.MXFP4: 1, az.Q6_K: 1}}[before]
    assert qtype == az.Q3_K or launches == (want[qtype] if before else 0)
    assert launches > 1 or qtype != az.Q3_K


@pytest.mark.parametrize("T,Mp,N,K,acc", [(1100, 1104, 392, 512, 0), (1030, 1040, 640, 768, 1), (760, 768, 520, 1024, 2),
                                          (300, 304, 132, 256, 0), (2050, 2064, 136, 256, 1)])
def test_gemm_tiles_of_256_tokens(rt, monkeypatch, T, Mp, N, K, acc):
    """The Q4_K kernel in tiles of 256 tokens x 128 rows, work-groups of 8 waves (ARCZ_Q4_WM=4, which an engine reads
    when it is made; not the default launch): the same arithmetic in the same order as the 128 x 128 kernel, so the same
    bits, on chunks whose last tiles are partly empty, with the three epilogues."""
    print(f"256-token tiles T={T} Mp={Mp} N={N} K={K} acc={acc}", flush=True)
    W = make_weights(az.Q4_K, N, K, seed=91)
    x = make_acts(T, K, seed=92, outliers=True)
    c0 = np.random.default_rng(93).standard_normal((Mp, N)).astype(np.float32)
    monkeypatch.setenv("ARCZ_Q4_WM", "2")
    eng = az.Engine(Mp, K)
    want = run_gemm(eng, az.Q4_K, W, N, K, x, Mp, acc=acc, c_init=c0 if acc else None)[:T]
    eng.close()
    monkeypatch.setenv("ARCZ_Q4_WM", "4")
    monkeypatch.setenv("ARCZ_Q4_WM_MIN", "256")
    eng = az.Engine(Mp, K)
    y = run_gemm(eng, az.Q4_K, W, N, K, x, Mp, acc=acc, c_init=c0 if acc else None)[:T]
    eng.close()
    assert np.array_equal(y.view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("wm", ["1", "0"])
@pytest.mark.parametrize("T,Mp,N,K,acc", [(1100, 1104, 392, 512, 0), (1100, 1104, 390, 512, 0), (1030, 1040, 640, 768, 1),
                                          (760, 768, 520, 1024, 2), (300, 304, 132, 256, 0), (257, 260, 1000, 2048, 0),
                                          (2050, 2064, 136, 256, 1)])
def test_gemm_tiles_of_64_tokens_on_ready_made_scales(rt, monkeypatch, wm, T, Mp, N, K, acc):
    """The Q4_K kernel in tiles of 64 tokens x 128 rows that takes all four scale vectors ready-made -- the launch
    rule's choice for chunks of a few rounds of work-groups (ARCZ_Q4_WM=0, the default; =1 always, =2 never; read when
    an engine is made) -- on chunks whose last tiles are partly empty, so that the whole-row reads run into the next
    block's entries and past the arrays' ends, with the three epilogues.  Against the oracle, and run to run."""
    print(f"64-token tiles T={T} Mp={Mp} N={N} K={K} acc={acc} ARCZ_Q4_WM={wm}", flush=True)
    W = make_weights(az.Q4_K, N, K, seed=91)
    x = make_acts(T, K, seed=92, outliers=True)
    c0 = np.random.default_rng(93).standard_normal((Mp, N)).astype(np.float32)
    monkeypatch.setenv("ARCZ_Q4_WM", wm)
    eng = az.Engine(Mp, K)            # (an engine of exactly this chunk: the arrays end where the chunk ends)
    y = run_gemm(eng, az.Q4_K, W, N, K, x, Mp, acc=acc, c_init=c0 if acc else None)[:T]
    y2 = run_gemm(eng, az.Q4_K, W, N, K, x, Mp, acc=acc, c_init=c0 if acc else None)[:T]
    eng.close()
    assert np.array_equal(y.view(np.uint32), y2.view(np.uint32))
    aq, asc, _ = quantize_padded(x, Mp)
    ref = orc.matmul_ref(az.Q4_K, W, N, K, aq[:T], np.ascontiguousarray(asc[:, :T]))
    if acc == 1:
        ref = ref + c0[:T]
    elif acc == 2:
        g = c0[:T].astype(np.float64)
        ref = ref * (g / (1.0 + np.exp(-g)))
    assert np.isfinite(y).all() and mixed_err(y, ref) <= TOL

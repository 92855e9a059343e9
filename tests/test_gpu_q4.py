"""GPU parity of the Q4_0 path: dequantization (bit-exact) and the GEMV
(error vs fp64 and vs the reference AVX2 order), through the C-ABI.

Tolerance for GEMV, written out: for every output row i,
    |y_i - y64_i| / sum_j |W_ij x_j|  <=  1e-5
where y64 is the fp64 dot product of the exactly dequantized weights.  At the
BASELINE shapes the maximum and the RMS of that statistic must also not
exceed the reference AVX2 accumulation order's own (oracle or_gemv_q4, which
is bit-identical to the reference's q_gemv_q4_f32_avx2).
"""
import ctypes as C

import numpy as np
import pytest

from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32)


def same_bits_nan(a, b):
    a, b = np.asarray(a, np.float32), np.asarray(b, np.float32)
    return bool(np.all((bits(a) == bits(b)) | (np.isnan(a) & np.isnan(b))))


class Gemv:
    """Device-resident W/x/y for repeated qh_gemv_q4_f32 calls."""

    def __init__(self, qa, W, M, N):
        self.qa, self.M, self.N = qa, M, N
        self.dW = qa.DeviceBuffer.from_numpy(np.ascontiguousarray(W))
        self.dx = qa.DeviceBuffer(N * 4)
        self.dy = qa.DeviceBuffer(M * 4)
        self.dr = qa.DeviceBuffer(M * 4)
        self.ws = qa.DeviceBuffer(qa.lib().qh_gemv_workspace_bytes(N))
        self.t = qa.q4_tensor(self.dW.ptr, M, N)

    def __call__(self, x, res=None):
        qa = self.qa
        self.dx.upload(np.ascontiguousarray(x, np.float32))
        if res is None:
            qa.check(qa.lib().qh_gemv_q4_f32(self.t.addr, self.dx.ptr, self.dy.ptr, self.ws.ptr, None), "gemv")
        else:
            self.dr.upload(np.ascontiguousarray(res, np.float32))
            qa.check(qa.lib().qh_gemv_q4_f32_add(self.t.addr, self.dx.ptr, self.dr.ptr, self.dy.ptr,
                                                 self.ws.ptr, None), "gemv_add")
        qa.check(qa.lib().qh_device_synchronize(), "sync")
        return self.dy.download(np.float32, (self.M,))


def stats(y, y64, cond):
    r = np.abs(y.astype(np.float64) - y64) / np.maximum(cond, 1e-300)
    return float(r.max()), float(np.sqrt(np.mean(r * r)))


# ----------------------------------------------------------------- dequant --

@pytest.mark.parametrize("case", [1, 2, 3, 4])
def test_dequant_block_public_golden(qa, case):
    from test_oracle import load_golden
    blk, exp = load_golden(case)
    out = orc.aligned_empty((32,), np.float32)
    b = orc.aligned_copy(blk)
    qa.lib().q_dequantize_q4_0_block_avx2_public(b.ctypes.data, out.ctypes.data)
    assert np.array_equal(out, exp)
    assert same_bits_nan(out, orc.dequant(blk))  # FMA form, +0 where (q-8)*s is -0


def test_dequant_public_null_is_silent(qa):
    out = orc.aligned_empty((32,), np.float32)
    qa.lib().q_dequantize_q4_0_block_avx2_public(None, out.ctypes.data)
    qa.lib().q_dequantize_q4_0_block_avx2_public(out.ctypes.data, None)


def test_dequant_device_bitexact_random_and_adversarial(qa):
    from test_oracle import ADV_PATTERNS, ADV_SCALES, adv_block
    rng = orc.rng_for(101)
    W = orc.gen_q4(333, 4096, rng).reshape(-1)
    adv = np.concatenate([adv_block(s, p, rng) for s in ADV_SCALES for p in ADV_PATTERNS])
    blob = np.concatenate([W, adv])
    nb = blob.size // 20
    d_in = qa.DeviceBuffer.from_numpy(blob)
    d_out = qa.DeviceBuffer(nb * 128)
    qa.check(qa.lib().qh_dequantize_q4_0(d_in.ptr, d_out.ptr, nb, None), "dequant")
    qa.check(qa.lib().qh_device_synchronize())
    got = d_out.download(np.float32, (nb * 32,))
    assert same_bits_nan(got, orc.dequant(blob))


# Wave and workgroup edges (64 and 256 blocks) and both sides of the size past
# which the stores are non-temporal.
@pytest.mark.parametrize("nb", [1, 2, 63, 64, 65, 255, 256, 257, 1000, 262144, 262145, 262209, 906876, 906877, 906941, 1813752,
                                1813753, 1813817])
def test_dequant_block_counts_bitexact(qa, nb):
    rng = orc.rng_for(103, nb)
    blob = orc.gen_q4(nb, 32, rng).reshape(-1)
    d_in = qa.DeviceBuffer.from_numpy(blob)
    guard = np.full(64, 7.5, np.float32)
    d_out = qa.DeviceBuffer.from_numpy(np.concatenate([np.full(nb * 32, np.nan, np.float32), guard]))
    qa.check(qa.lib().qh_dequantize_q4_0(d_in.ptr, d_out.ptr, nb, None), "dequant")
    qa.check(qa.lib().qh_device_synchronize())
    got = d_out.download(np.float32, (nb * 32 + 64,))
    assert same_bits_nan(got[:nb * 32], orc.dequant(blob))
    assert np.array_equal(got[nb * 32:], guard)


# -------------------------------------------------------------------- GEMV --

# Shapes exercising every launch configuration (nblk <= 64, <= 128, <= 256,
# > 256 with one and several K-chunks), row tails and column tails.
TAIL_SHAPES = [(1, 32), (3, 96), (17, 160), (5, 224), (64, 2048), (33, 2080), (16, 4096),
               (4097, 4096), (19, 8192), (7, 8224), (40, 14336), (9, 16416), (3, 65536)]


@pytest.mark.parametrize("M,N", TAIL_SHAPES)
def test_gemv_shapes_vs_fp64(qa, M, N):
    rng = orc.rng_for(102, M, N)
    W = orc.gen_q4(M, N, rng)
    x = orc.gen_f32(N, rng)
    y64, cond = orc.gemv_f64(W, M, N, x)
    y = Gemv(qa, W, M, N)(x)
    mx, _ = stats(y, y64, cond)
    assert mx <= 1e-5, f"max rel-to-condition error {mx:.3e}"


# BASELINE configs 1-3 (config 2 = the Llama-3-8B per-layer set).
CONFIG_SHAPES = {
    "c1_4096x4096": (4096, 4096),
    "c2_wk_1024x4096": (1024, 4096),
    "c2_gate_14336x4096": (14336, 4096),
    "c2_down_4096x14336": (4096, 14336),
}


@pytest.mark.parametrize("name", list(CONFIG_SHAPES))
def test_gemv_config_shapes_vs_fp64_and_avx2(qa, name):
    M, N = CONFIG_SHAPES[name]
    rng = orc.rng_for(103, M, N)
    W = orc.gen_q4(M, N, rng)
    x = orc.gen_f32(N, rng)
    y64, cond = orc.gemv_f64(W, M, N, x)
    y = Gemv(qa, W, M, N)(x)
    y_avx2 = orc.gemv(W, M, N, x)
    mx, rms = stats(y, y64, cond)
    amx, arms = stats(y_avx2, y64, cond)
    # the plain relative error, over the outputs whose magnitude is at least
    # the median (outputs that cancel to ~0 have no meaningful plain error)
    big = np.abs(y64) >= np.median(np.abs(y64))
    plain = float(np.max(np.abs(y[big].astype(np.float64) - y64[big]) / np.abs(y64[big])))
    aplain = float(np.max(np.abs(y_avx2[big].astype(np.float64) - y64[big]) / np.abs(y64[big])))
    print(f"{name}: gpu max {mx:.3e} rms {rms:.3e} plain(>=median) {plain:.3e} | "
          f"avx2 max {amx:.3e} rms {arms:.3e} plain(>=median) {aplain:.3e}")
    assert mx <= 1e-5
    assert mx <= amx and rms <= arms
    assert plain <= 1e-5


def test_gemv_lm_head_vs_fp64(qa):
    M, N = 128256, 4096
    rng = orc.rng_for(104)
    W = orc.gen_q4(M, N, rng)
    x = orc.gen_f32(N, rng)
    y64, cond = orc.gemv_f64(W, M, N, x)
    y = Gemv(qa, W, M, N)(x)
    mx, rms = stats(y, y64, cond)
    assert mx <= 1e-5
    assert int(np.argmax(y)) == int(np.argmax(y64))


def test_gemv_residual_epilogue_and_determinism(qa):
    M, N = 4096, 14336
    rng = orc.rng_for(105)
    W = orc.gen_q4(M, N, rng)
    x = orc.gen_f32(N, rng)
    r = orc.gen_f32(M, rng)
    g = Gemv(qa, W, M, N)
    y1 = g(x)
    y2 = g(x)
    assert np.array_equal(bits(y1), bits(y2))
    ya = g(x, res=r)
    assert np.array_equal(bits(ya), bits((r + y1).astype(np.float32)))


def test_gemv_compat_host_entry(qa):
    """q_gemv_q4_f32_avx2 with host pointers, as the reference's callers use it."""
    lib = qa.lib()
    for M, N in [(1, 32), (7, 224), (128, 1024), (1024, 8192)]:
        rng = orc.rng_for(106, M, N)
        W = orc.aligned_copy(orc.gen_q4(M, N, rng).reshape(-1))
        x = orc.aligned_copy(orc.gen_f32(N, rng))
        y = orc.aligned_empty((M,), np.float32)
        t = qa.q4_tensor(W.ctypes.data, M, N)
        assert lib.q_gemv_q4_f32_avx2(t.addr, x.ctypes.data, y.ctypes.data) == 0
        y64, cond = orc.gemv_f64(W.reshape(M, -1), M, N, x)
        assert stats(y, y64, cond)[0] <= 1e-5


SCALES = [1e-10, 1e10, 0.0, -1.0, float(np.finfo(np.float32).tiny), float(np.finfo(np.float32).max)]
INPUTS = ["zeros", "ones", "neg", "large", "small", "inf", "nan", "rand"]
PATTERNS = [0x88, 0xFF, 0x00, "alt", "rand"]


def make_input(kind, N, rng):
    return {"zeros": np.zeros(N), "ones": np.ones(N), "neg": -np.ones(N), "large": np.full(N, 1e10),
            "small": np.full(N, 1e-10), "inf": np.full(N, np.inf), "nan": np.full(N, np.nan),
            "rand": rng.random(N) * 2 - 1}[kind].astype(np.float32)


def scalar_ref(W, M, N, x):
    """The reference test's own scalar GEMV (tests/test_matmul.c:10-46):
    weight = ((float)q - 8.0f) * scale; sum += weight * x, in float32."""
    q = orc.q4_nibbles(W).astype(np.float32)
    s = np.repeat(orc.q4_scales(W), 32, axis=1).astype(np.float32)
    with np.errstate(all="ignore"):
        w = (q - np.float32(8.0)) * s
        out = np.zeros(M, np.float32)
        for j in range(N):
            out = (out + w[:, j] * x[j]).astype(np.float32)
    return out


def test_gemv_extreme_values(qa):
    """Cases of reference tests/test_matmul_adversarial.c:341-558 run with
    real strides (the reference's own copies leave nb[0] = 0 and never reach
    the math).  Acceptance restates that file's rule: where the reference
    test's scalar GEMV is finite, the result must match it within abs 1.5e-4
    or rel 1e-4; NaN/Inf inputs must give non-finite outputs; where the
    scalar reference itself overflows in float32 (scale FLT_MAX), any result
    is accepted, as there (the GPU's exact integer dot may return the exact,
    finite value)."""
    from test_oracle import adv_block
    M, N = 4, 128
    rng = orc.rng_for(107)
    checked = 0
    for sc in SCALES:
        for pat in PATTERNS:
            W = np.stack([np.concatenate([adv_block(sc, pat, rng) for _ in range(N // 32)]) for _ in range(M)])
            g = Gemv(qa, W, M, N)
            for kind in INPUTS:
                x = make_input(kind, N, rng)
                y = g(x)
                yr = scalar_ref(W, M, N, x)
                if kind in ("inf", "nan"):
                    assert not np.isfinite(y).any(), (sc, pat, kind, y)
                elif np.isfinite(yr).all():
                    err = np.abs(y.astype(np.float64) - yr)
                    ok = (err <= 1.5e-4) | (err <= 1e-4 * np.abs(yr))
                    assert ok.all(), (sc, pat, kind, y, yr)
                checked += 1
    assert checked == len(SCALES) * len(PATTERNS) * len(INPUTS)


def test_gemv_tiny_and_mixed_magnitude_inputs(qa):
    M, N = 64, 4096
    rng = orc.rng_for(108)
    W = orc.gen_q4(M, N, rng)
    g = Gemv(qa, W, M, N)
    for x in (orc.gen_f32(N, rng) * np.float32(1e-38),            # subnormal range
              orc.gen_f32(N, rng) * np.float32(1e30),
              np.where(rng.random(N) < 0.05, 1e6, 1e-6).astype(np.float32) * orc.gen_f32(N, rng)):
        y64, cond = orc.gemv_f64(W, M, N, x)
        assert stats(g(x), y64, cond)[0] <= 1e-5


# Input widths around every launch-shape boundary of the fp32-input GEMV
# (in-kernel digit conversion up to 512 blocks, prepare + GEMV above).
F32_WIDTHS = [32, 2048, 2080, 4096, 4128, 8192, 8224, 14336, 14368, 16384, 16416]


def special_input(N, rng):
    """N(0,1) with whole blocks of zeros, subnormals, huge values and a
    block mixing magnitudes 2^-60..2^60."""
    x = orc.gen_f32(N, rng)
    nb = N // 32
    if nb >= 4:
        x[0:32] = 0.0
        x[32:64] = rng.standard_normal(32).astype(np.float32) * np.float32(1e-40)
        x[64:96] = rng.standard_normal(32).astype(np.float32) * np.float32(3e37)
        x[96:128] = (rng.standard_normal(32) * 2.0 ** rng.integers(-60, 60, 32)).astype(np.float32)
    return x


@pytest.mark.parametrize("N", F32_WIDTHS)
def test_gemv_f32_multi_bitexact_vs_prepared(qa, N):
    """qh_gemv_q4_f32_multi (digit planes made inside the GEMV) must equal
    qh_gemv_prepare + qh_gemv_q4_f32_prepared bit for bit, with 1-3
    matrices, residuals, and NaN/Inf blocks (non-finite rows match too)."""
    lib = qa.lib()
    rng = orc.rng_for(109, N)
    Ms = [37, 8, 130][: 1 + (N // 32) % 3]
    Ws = [orc.gen_q4(M, N, rng) for M in Ms]
    dW = [qa.DeviceBuffer.from_numpy(np.ascontiguousarray(W)) for W in Ws]
    ts = [qa.q4_tensor(d.ptr, M, N) for d, M in zip(dW, Ms)]
    tp = (C.c_void_p * len(ts))(*[t.addr for t in ts])
    dx = qa.DeviceBuffer(N * 4)
    ya = [qa.DeviceBuffer(M * 4) for M in Ms]
    yb = [qa.DeviceBuffer(M * 4) for M in Ms]
    rs = [qa.DeviceBuffer.from_numpy(orc.gen_f32(M, rng)) for M in Ms]
    ws = qa.DeviceBuffer(lib.qh_gemv_workspace_bytes(N))
    yap = (C.c_void_p * len(Ms))(*[b.ptr for b in ya])
    ybp = (C.c_void_p * len(Ms))(*[b.ptr for b in yb])
    rsp = (C.c_void_p * len(Ms))(*[b.ptr for b in rs])
    inputs = [orc.gen_f32(N, rng), special_input(N, rng)]
    if N >= 256:
        bad = special_input(N, rng)
        bad[160 + 5] = np.nan
        bad[192 + 31] = np.inf
        inputs.append(bad)
    for x in inputs:
        for res in (None, rsp):
            dx.upload(x)
            qa.check(lib.qh_gemv_q4_f32_multi(tp, res, yap, len(Ms), dx.ptr, None, None), "multi")
            qa.check(lib.qh_gemv_prepare(dx.ptr, N, ws.ptr, None), "prepare")
            qa.check(lib.qh_gemv_q4_f32_prepared(tp, res, ybp, len(Ms), ws.ptr, None), "prepared")
            qa.check(lib.qh_device_synchronize(), "sync")
            for a, b, M in zip(ya, yb, Ms):
                assert same_bits_nan(a.download(np.float32, (M,)), b.download(np.float32, (M,))), (N, M)
    # Accuracy of the one-launch path itself.
    y64, cond = orc.gemv_f64(Ws[0], Ms[0], N, inputs[0])
    dx.upload(inputs[0])
    qa.check(lib.qh_gemv_q4_f32_multi(tp, None, yap, len(Ms), dx.ptr, None, None), "multi")
    qa.check(lib.qh_device_synchronize(), "sync")
    assert stats(ya[0].download(np.float32, (Ms[0],)), y64, cond)[0] <= 1e-5


# The persistent kernel's launch shapes between those widths: one-wave rows of
# 3 block columns, K split over 4 to 16 waves (each at its widest and one block
# past it), and the first width of the tile-per-workgroup kernel.
@pytest.mark.parametrize("N", [6144, 6176, 10240, 10272, 12288, 12320, 20480, 20512, 24576, 24608, 28672, 28704,
                               32768, 32800])
def test_gemv_launch_shape_edges(qa, N):
    test_gemv_f32_multi_bitexact_vs_prepared(qa, N)


# Activation outliers meeting zero weights (nibble 8 in every row): one
# channel, one column of every block, 2/3/4/6 equal outliers in one block or
# in every block, and four outliers of mixed sizes (mag .. mag/1000), at
# 1e3, 1e4 and 1e5 times the N(0,1) rest.  The shapes cover every launch
# form (in-kernel conversion by lane quads, wave-local conversion, prepared
# digits, the generic kernel).
OUTLIER_SHAPES = [(512, 4096), (256, 14336), (256, 2048), (128, 8192), (64, 32768)]


@pytest.mark.parametrize("M,N", OUTLIER_SHAPES)
def test_gemv_activation_outliers_vs_fp64_and_avx2(qa, M, N):
    """Blocks where outliers set the digit step take the GEMV's second digit
    level, so the other elements keep their full precision: max <= 1e-5 at
    every width, and at the BASELINE widths (N >= 4096, the rule of the
    config-shape test above) max and RMS of the error statistic no worse
    than the reference AVX2 order's.  Narrower inputs are held to twice the
    AVX2 order's: there both errors are the fp32 rounding of a few dozen
    terms (N = 2048 measured 2.1e-8 vs 1.8e-8).  The prepared-digit path
    gives the same bits as the in-kernel conversion."""
    from adversarial import CASES, Layout, apply_case, set_nibble8
    lib = qa.lib()
    rng = orc.rng_for(110, M, N)
    lay = Layout(N, rng)
    W = set_nibble8(orc.gen_q4(M, N, rng), lay.zero_columns())
    g = Gemv(qa, W, M, N)
    yp = qa.DeviceBuffer(M * 4)
    tp = (C.c_void_p * 1)(g.t.addr)
    ypp = (C.c_void_p * 1)(yp.ptr)
    base = orc.gen_f32(N, rng)
    bad = []
    for kind, n, mag in CASES:
        x = apply_case(base, lay, kind, n, mag)
        y = g(x)
        y64, cond = orc.gemv_f64(W, M, N, x)
        mx, rms = stats(y, y64, cond)
        amx, arms = stats(orc.gemv(W, M, N, x), y64, cond)
        print(f"{M}x{N} {kind}:{n} {mag:.0e}: gpu max {mx:.2e} rms {rms:.2e} | avx2 max {amx:.2e} rms {arms:.2e}")
        f = 1 if N >= 4096 else 2
        if not (mx <= 1e-5 and mx <= f * amx and rms <= f * arms):
            bad.append((kind, n, mag, mx, amx, rms, arms))
        qa.check(lib.qh_gemv_prepare(g.dx.ptr, N, g.ws.ptr, None), "prepare")
        qa.check(lib.qh_gemv_q4_f32_prepared(tp, None, ypp, 1, g.ws.ptr, None), "prepared")
        qa.check(lib.qh_device_synchronize(), "sync")
        assert same_bits_nan(yp.download(np.float32, (M,)), y), (kind, n, mag)
    assert not bad, bad


# Level-2 digits in the same launch shapes.
@pytest.mark.parametrize("M,N", [(96, 6144), (96, 10240), (64, 20480), (48, 28672)])
def test_gemv_activation_outliers_launch_shapes(qa, M, N):
    test_gemv_activation_outliers_vs_fp64_and_avx2(qa, M, N)

"""Operator-level parity: HIP kernels (through the C ABI) vs the oracle.

Bars: bit-exact for the activation quantizer, integer block sums, embedding,
RoPE (host libm sin/cos table), residual add and argmax; float kernels within
the tolerance written at each assert, relative to the magnitude of the terms
summed (the reference's own bound style, src/kernels/matmul.rs:315-335).
"""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

sq = pytest.importorskip("sqhip")
from sqhip import ops  # noqa: E402
from sqhip.ops import DeviceArray  # noqa: E402


A32_SKIP = ("f32-activation kernels (BF16, SQUIRREL_F32_ACTS) are switched off after a GPU "
            "memory fault in a BF16 model prefill whose cause is not identified yet")


def rng(seed):
    return np.random.default_rng(seed)


def quant_weights(wtype, rows, k, seed, scale=0.02):
    """GGUF blocks for a rows x k matrix, built with the oracle's quantizer
    (Q8_0) or the ggml Q4_0 rule (Q4_0) or RNE bf16."""
    x = (rng(seed).standard_normal((rows, k)) * scale).astype(np.float32)
    if wtype == O.Q8_0:
        return O.quantize_row_q8_0(x).reshape(rows, k // 32), x
    if wtype == O.Q4_0:
        xb = x.reshape(-1, 32)
        idx = np.argmax(np.abs(xb), axis=1)
        mx = xb[np.arange(xb.shape[0]), idx]
        d = (mx / np.float32(-8)).astype(np.float32)
        inv = np.where(d != 0, np.float32(1) / np.where(d != 0, d, 1), 0).astype(np.float32)
        q = np.minimum(15, np.trunc(xb * inv[:, None] + np.float32(8.5)).astype(np.int32))
        blk = np.zeros(xb.shape[0], O.BLOCK_Q4_0)
        blk["d"] = d.astype(np.float16).view(np.uint16)
        blk["qs"] = (q[:, :16] | (q[:, 16:] << 4)).astype(np.uint8)
        return blk.reshape(rows, k // 32), x
    u = x.view(np.uint32)
    b = ((u + 0x7FFF + ((u >> 16) & 1)) >> 16).astype(np.uint16)
    return b.reshape(rows, k), x


# ---------------------------------------------------------------- quantizer

def quantizer_inputs():
    r = rng(1)
    rows = [r.standard_normal(4096).astype(np.float32) * 3,
            (r.standard_normal(2048) * 1e-3).astype(np.float32)]
    # The reference's edge cases (dot_prod.rs:629-654): all-zero block,
    # negative absmax, +-0.5 ties, f32::MAX/2 (scale overflows f16).
    src = (np.sin(np.arange(32 * 6, dtype=np.float32) * np.float32(0.37)) * 4 - 0.5).astype(np.float32)
    src[32:64] = 0
    src[64] = -100
    src[96] = 0.5
    src[97] = -0.5
    src[128] = np.finfo(np.float32).max / 2
    rows.append(src)
    # exact ties after scaling, tiny values, subnormals, NaN / inf entries
    t = np.zeros(32 * 8, np.float32)
    t[:32] = np.arange(32, dtype=np.float32) - 15.5
    t[32:64] = np.float32(127.0) * (np.arange(32, dtype=np.float32) / 31) - 63.5
    t[64:96] = np.float32(1e-40) * np.arange(32, dtype=np.float32)
    t[96:128] = np.float32(1e-30) * (np.arange(32, dtype=np.float32) - 16)
    t[128] = np.nan
    t[129:160] = 1.0
    t[160] = np.inf
    t[161:192] = -2.0
    t[192:224] = np.float32(65504.0 * 127) * (r.random(32).astype(np.float32) - 0.5)
    t[224:256] = r.standard_normal(32).astype(np.float32) * 1e5
    rows.append(t)
    return rows


@pytest.mark.parametrize("case", range(4))
def test_quantize_row_bit_exact(case):
    x = quantizer_inputs()[case]
    got = ops.quantize_row_q8_0(DeviceArray.from_numpy(x))
    want = O.quantize_row_q8_0(x)
    assert np.array_equal(got["d"], want["d"]), "scales differ"
    assert np.array_equal(got["qs"], want["qs"]), "quants differ"


# ---------------------------------------------------------------- integer sums

@pytest.mark.parametrize("wtype", [O.Q8_0, O.Q4_0])
@pytest.mark.parametrize("k", [2048, 8192])
def test_block_isums_bit_exact(wtype, k):
    w, _ = quant_weights(wtype, 4, k, seed=k + wtype)
    a = rng(5).standard_normal(k).astype(np.float32)
    aq = O.quantize_row_q8_0(a)
    W = ops.Weight(wtype, w, 4, k)
    d_aq = DeviceArray.from_numpy(aq)
    for row in (0, 3):
        got = ops.block_isums(d_aq, W, row)
        want = O.block_isums(aq, w[row], wtype)
        assert np.array_equal(got, want)


def test_q4_int_dot_exact_on_integers():
    """q4_int_dot_exact_on_integers (dot_prod.rs:774-803) on the device."""
    qs = np.array([((i % 16) << 4) | (15 - i % 16) for i in range(16)], np.uint8)
    w = np.zeros((1, 1), O.BLOCK_Q4_0)
    w["d"] = np.float16(1.0).view(np.uint16)
    w["qs"][0, 0] = qs
    a = np.zeros(1, O.BLOCK_Q8_0)
    a["d"] = np.float16(1.0).view(np.uint16)
    a["qs"][0] = np.arange(32, dtype=np.int32) - 16
    expected = 0
    for j in range(16):
        lo, hi = int(qs[j] & 15) - 8, int(qs[j] >> 4) - 8
        expected += int(a["qs"][0][j]) * lo + int(a["qs"][0][j + 16]) * hi
    W = ops.Weight(O.Q4_0, w, 1, 32)
    assert int(ops.block_isums(DeviceArray.from_numpy(a), W, 0)[0]) == expected


# ---------------------------------------------------------------- linear

SHAPES = [(2048, 2048), (2048, 512), (2048, 8192), (8192, 2048), (96, 9), (128, 7)]


def term_mag(x, w_f32):
    return np.abs(x.astype(np.float64)) @ np.abs(w_f32.astype(np.float64)).T


@pytest.mark.parametrize("wtype", [O.Q8_0, O.Q4_0, O.BF16])
@pytest.mark.parametrize("k,n", SHAPES)
@pytest.mark.parametrize("m", [1, 5, 67, 200])
@pytest.mark.parametrize("f32_acts", [False, True])
def test_linear_matches_oracle(wtype, k, n, m, f32_acts):
    if wtype == O.BF16 and f32_acts:
        pytest.skip("BF16 always uses f32 activations")
    if wtype == O.BF16 or f32_acts:
        pytest.skip(A32_SKIP)
    w, _ = quant_weights(wtype, n, k, seed=31 * k + n + wtype)
    x = (rng(k + n).standard_normal((m, k)) * 1.5).astype(np.float32)
    W = ops.Weight(wtype, w, n, k)
    out = DeviceArray((m, n))
    ops.linear(DeviceArray.from_numpy(x), W, out, f32_acts=f32_acts)
    got = out.numpy()
    mode = O.W8A32 if (f32_acts or wtype == O.BF16) else O.W8A8
    want = O.linear(x, wtype, w, n, mode)
    wf = np.stack([O.dequantize(wtype, w[i], k) for i in range(n)])
    mag = term_mag(x, wf)
    err = np.abs(got.astype(np.float64) - want)
    # Same per-block terms, different summation order: f32 rounding of a sum
    # of |terms| <= mag is bounded by ~k*eps*mag; 4e-6 * mag covers k <= 8192
    # with the tree orders used on both sides.
    assert np.all(err <= 4e-6 * mag + 1e-6), float((err / (mag + 1e-30)).max())


@pytest.mark.parametrize("k", [2048, 8192])
@pytest.mark.parametrize("tile", ["64x128", "128x64", "128"])
def test_matmul_ragged_tiles_match_oracle(tile, k, monkeypatch):
    """Q8_0 weights on ragged tiles (1000 prompt rows: 7 full 128-row tiles
    and 104 rows; 4000 columns: 31 full 128-column tiles and 32): rows of the
    first, the inner and the last tile, every column, within 4e-6 of the sum
    of |terms| of the oracle (matmul.rs:133-171), and all of it bit for bit
    what 64 x 64 tiles give (the same terms in the same order)."""
    m, n = 1000, 4000
    w, _ = quant_weights(O.Q8_0, n, k, seed=91)
    x = (rng(5).standard_normal((m, k)) * 1.5).astype(np.float32)
    W = ops.Weight(O.Q8_0, w, n, k)
    d_x = DeviceArray.from_numpy(x)
    outs = {}
    for t in (tile, "64"):
        monkeypatch.setenv("SQUIRREL_GEMM_TILE", t)
        out = DeviceArray((m, n))
        ops.gemm_counters(reset=True)
        ops.linear(d_x, W, out)
        wide = ops.gemm_tile64x128_launches()
        got = ops.gemm_counters(reset=True)
        assert got["launches"] == 1 and got["split_launches"] == 0, got
        assert (got["tile128_launches"], got["tile128x64_launches"], wide) == (t == "128", t == "128x64", t == "64x128")
        outs[t] = out.numpy()
    rows = np.array([0, 31, 32, 127, 128, 500, 895, 896, 959, 960, 991, 992, 999])
    want = O.linear(x[rows], O.Q8_0, w, n, O.W8A8)
    wf = np.stack([O.dequantize(O.Q8_0, w[i], k) for i in range(n)])
    assert np.all(np.abs(outs[tile][rows].astype(np.float64) - want) <= 4e-6 * term_mag(x[rows], wf) + 1e-6)
    assert np.array_equal(outs[tile], outs["64"])


@pytest.mark.parametrize("wtype", [O.Q8_0, O.Q4_0])
@pytest.mark.parametrize("m,k,n", [(131, 2080, 16416), (300, 160, 10000)])
def test_matmul_wide_ragged_input_takes_64_row_tiles(wtype, m, k, n):
    """Matrices of 8192 and more rows and an input whose last 128-row tile
    would be mostly empty take 64 x 128 tiles with no tiling pinned: last tiles
    of 32 and 16 columns, of 3 and 44 rows, and odd counts of blocks (65, 5),
    against the oracle as above."""
    w, _ = quant_weights(wtype, n, k, seed=5 + m)
    x = (rng(m).standard_normal((m, k)) * 1.5).astype(np.float32)
    out = DeviceArray((m, n))
    ops.gemm_counters(reset=True)
    ops.linear(DeviceArray.from_numpy(x), ops.Weight(wtype, w, n, k), out)
    wide = ops.gemm_tile64x128_launches()
    c = ops.gemm_counters(reset=True)
    assert c["launches"] == 1 and c["split_launches"] == 0 and wide == 1, (c, wide)
    rows = np.array(sorted({0, 31, 32, 63, 64, 127, 128, m - 1}))
    want = O.linear(x[rows], wtype, w, n, O.W8A8)
    wf = np.stack([O.dequantize(wtype, w[i], k) for i in range(n)])
    assert np.all(np.abs(out.numpy()[rows].astype(np.float64) - want) <= 4e-6 * term_mag(x[rows], wf) + 1e-6)


@pytest.mark.parametrize("wtype", [O.Q8_0, O.Q4_0])
def test_matmul_tiles_agree(wtype, monkeypatch):
    """The prefill matmul's four tile shapes (64 x 64, 64 x 128, 128 x 64 and
    128 x 128, wavefronts of one to four 32 x 32 tiles) fold the same
    per-block terms in the same order for every output, so without a K split
    they agree bit for bit; the 128 x 128 result also matches the oracle
    (matmul.rs:133-171)."""
    m, k, n = 1024, 2048, 4096      # 1024, 512, 512 and 256 tiles: no shape splits K
    w, _ = quant_weights(wtype, n, k, seed=77 + wtype)
    x = (rng(3).standard_normal((m, k)) * 1.5).astype(np.float32)
    W = ops.Weight(wtype, w, n, k)
    d_x = DeviceArray.from_numpy(x)
    outs = {}
    for tile in ("64", "64x128", "128x64", "128"):
        monkeypatch.setenv("SQUIRREL_GEMM_TILE", tile)
        out = DeviceArray((m, n))
        ops.gemm_counters(reset=True)
        ops.linear(d_x, W, out)
        assert ops.gemm_tile64x128_launches() == (1 if tile == "64x128" else 0)
        got = ops.gemm_counters(reset=True)
        assert got["launches"] == 1 and got["split_launches"] == 0, got
        assert got["tile128_launches"] == (1 if tile == "128" else 0), got
        assert got["tile128x64_launches"] == (1 if tile == "128x64" else 0), got
        outs[tile] = out.numpy()
    assert np.array_equal(outs["64"], outs["128"])
    assert np.array_equal(outs["64x128"], outs["128"])
    assert np.array_equal(outs["128x64"], outs["128"])
    rows = np.arange(0, m, 97)
    want = O.linear(x[rows], wtype, w, n, O.W8A8)
    wf = np.stack([O.dequantize(wtype, w[i], k) for i in range(n)])
    err = np.abs(outs["128"][rows].astype(np.float64) - want)
    assert np.all(err <= 4e-6 * term_mag(x[rows], wf) + 1e-6)


@pytest.mark.parametrize("wtype", [O.Q8_0, O.Q4_0])
@pytest.mark.parametrize("m,k,n,pin", [
    (2, 2048, 2048, None), (13, 2048, 3072, None), (32, 8192, 2048, None), (29, 128, 7, None),
    (7, 512, 1000, None), (45, 2048, 512, "rows"), (200, 1024, 96, "rows"),
    (16, 2048, 16384, None), (8, 512, 16416, None),
])
def test_matmul_rows_kernel_matches_oracle(wtype, m, k, n, pin, monkeypatch):
    """The few-rows prefill matmul (inputs of at most 32 rows, or pinned with
    SQUIRREL_GEMM_TILE=rows): 32-row tiles, K split over the workgroup's
    wavefronts and summed in wavefront order.  Ragged rows and columns, K of
    one load batch (128), several row tiles when pinned, two column tiles per
    workgroup on the widest matrices (16384 and 16416 rows, the latter with a
    half-empty last pair) and a K split over workgroups at K = 8192; every
    output within 4e-6 of its sum of |terms| of the oracle
    (matmul.rs:133-171)."""
    if pin:
        monkeypatch.setenv("SQUIRREL_GEMM_TILE", pin)
    w, _ = quant_weights(wtype, n, k, seed=101 + m)
    x = (rng(m).standard_normal((m, k)) * 1.5).astype(np.float32)
    W = ops.Weight(wtype, w, n, k)
    out = DeviceArray((m, n))
    ops.gemm_counters(reset=True)
    ops.linear(DeviceArray.from_numpy(x), W, out)
    c = ops.gemm_counters(reset=True)
    assert c["launches"] == 1 and c["rows_launches"] == 1, c
    assert c["split_launches"] == (1 if k == 8192 else 0), c
    got = out.numpy().astype(np.float64)
    rows = np.arange(0, m, max(1, m // 9))
    want = O.linear(x[rows], wtype, w, n, O.W8A8)
    wf = np.stack([O.dequantize(wtype, w[i], k) for i in range(n)])
    err = np.abs(got[rows] - want)
    assert np.all(err <= 4e-6 * term_mag(x[rows], wf) + 1e-6), float(err.max())


@pytest.mark.parametrize("wtype", [O.Q8_0, O.Q4_0])
@pytest.mark.parametrize("pin", [None, "64", "64x128", "128x64", "128"])
@pytest.mark.parametrize("m,k,n", [
    (33, 32, 1), (63, 96, 33), (65, 160, 100), (97, 224, 129), (128, 64, 64), (131, 2048, 300), (257, 288, 65),
    (2, 4128, 40),
])
def test_matmul_fragment_order_edges(wtype, pin, m, k, n, monkeypatch):
    """Operands in fragment order on every tile shape: last tiles of 1 to 31
    rows and columns, one block of K, odd block counts (an unpaired last
    scale), K that is not whole groups of four blocks, K splits with a short
    last part; every output within 4e-6 of its sum of |terms| of the oracle
    (matmul.rs:133-171), as in the tests of the other shapes."""
    if pin:
        monkeypatch.setenv("SQUIRREL_GEMM_TILE", pin)
    w, _ = quant_weights(wtype, n, k, seed=7 + m)
    x = (rng(m + k).standard_normal((m, k)) * 1.5).astype(np.float32)
    out = DeviceArray((m, n))
    ops.gemm_counters(reset=True)
    ops.linear(DeviceArray.from_numpy(x), ops.Weight(wtype, w, n, k), out)
    assert ops.gemm_tile64x128_launches() == (1 if pin == "64x128" else 0)
    got = out.numpy().astype(np.float64)
    want = O.linear(x, wtype, w, n, O.W8A8)
    wf = np.stack([O.dequantize(wtype, w[i], k) for i in range(n)])
    assert np.all(np.abs(got - want) <= 4e-6 * term_mag(x, wf) + 1e-6)


def test_matmul_rows_kernel_inf_activation_scale():
    """An activation block of f32::MAX/2 has a Q8_0 scale that overflows
    binary16 to inf (dot_prod.rs:629-654): that row's outputs are +-inf or
    NaN, as the oracle's, element for element, and the other rows match the
    oracle within the usual bound."""
    m, k, n = 4, 256, 64
    w, _ = quant_weights(O.Q8_0, n, k, seed=5)
    x = (rng(6).standard_normal((m, k))).astype(np.float32)
    x[1, 224:256] = np.float32(np.finfo(np.float32).max / 2)   # the last block of row 1
    W = ops.Weight(O.Q8_0, w, n, k)
    out = DeviceArray((m, n))
    ops.gemm_counters(reset=True)
    ops.linear(DeviceArray.from_numpy(x), W, out)
    assert ops.gemm_counters(reset=True)["rows_launches"] == 1
    got = out.numpy().astype(np.float64)
    want = O.linear(x, O.Q8_0, w, n, O.W8A8)
    assert not np.all(np.isfinite(want[1]))
    fin = np.isfinite(want)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(got[~fin & ~np.isnan(want)], want[~fin & ~np.isnan(want)])
    wf = np.stack([O.dequantize(O.Q8_0, w[i], k) for i in range(n)])
    mag = term_mag(x, wf)
    assert np.all(np.abs(got[fin] - want[fin]) <= 4e-6 * mag[fin] + 1e-6)


@pytest.mark.parametrize("tile", ["64", "128x64", "128", "rows"])
def test_matmul_subnormal_activation_scales(tile, monkeypatch):
    """Activation rows of magnitude about 1e-4 have Q8_0 block scales below
    binary16's smallest normal (6.1e-5): the matrix-core kernels form the
    scale product sa * sw from f16 operands, so a flush of subnormal inputs
    would zero these outputs.  Every output must match the oracle within
    4e-6 of its sum of |terms|, with no absolute floor, on each tiling."""
    m, k, n = 256, 2048, 4096
    w, _ = quant_weights(O.Q8_0, n, k, seed=91)
    r = rng(5)
    x = (r.standard_normal((m, k)) * (1e-4 * r.uniform(0.5, 2.0, (m, 1)))).astype(np.float32)
    aq = O.quantize_row_q8_0(x.reshape(-1))
    sa = aq["d"].view(np.float16).astype(np.float32)
    assert np.all(sa < 6.1e-5) and np.all(sa > 0)
    W = ops.Weight(O.Q8_0, w, n, k)
    monkeypatch.setenv("SQUIRREL_GEMM_TILE", tile)
    out = DeviceArray((m, n))
    ops.gemm_counters(reset=True)
    ops.linear(DeviceArray.from_numpy(x), W, out)
    c = ops.gemm_counters(reset=True)
    assert c["tile128_launches"] == (1 if tile == "128" else 0) and \
        c["tile128x64_launches"] == (1 if tile == "128x64" else 0) and \
        c["rows_launches"] == (1 if tile == "rows" else 0), c
    got = out.numpy().astype(np.float64)
    rows = np.arange(0, m, 13)
    want = O.linear(x[rows], O.Q8_0, w, n, O.W8A8)
    wf = np.stack([O.dequantize(O.Q8_0, w[i], k) for i in range(n)])
    mag = term_mag(x[rows], wf)
    err = np.abs(got[rows] - want)
    assert np.all(mag > 0)
    assert np.all(err <= 4e-6 * mag), float((err / mag).max())


@pytest.mark.parametrize("wtype", [O.Q8_0, O.Q4_0])
@pytest.mark.parametrize("m,k,rows", [(2, 128, (7, 100, 33)), (32, 2048, (2048, 512, 512)), (9, 512, (512, 128)),
                                      (5, 256, (64, 1, 32, 31)), (32, 2048, (8192, 8192)), (3, 96, (40, 50))])
def test_linear_shared_one_launch_equals_separate(wtype, m, k, rows):
    """Matrices that share an input of at most 32 rows run as one launch where
    each would run unsplit on single tiles, else apart: every output equals
    the separate call's, bit for bit."""
    x = DeviceArray.from_numpy(rng(m).standard_normal((m, k)).astype(np.float32))
    Ws = [ops.Weight(wtype, quant_weights(wtype, n, k, seed=n)[0], n, k) for n in rows]
    outs = [DeviceArray((m, n)) for n in rows]
    ops.linear_shared(x, Ws, outs)
    for W, n, o in zip(Ws, rows, outs):
        alone = DeviceArray((m, n))
        ops.linear(x, W, alone)
        assert np.array_equal(alone.numpy(), o.numpy())


@pytest.mark.parametrize("wtype", [O.Q8_0, O.Q4_0, O.BF16])
def test_linear_shared_matches_separate(wtype):
    """fused_matches_separate_calls (matmul.rs:257-279): bit-equal."""
    if wtype == O.BF16:
        pytest.skip(A32_SKIP)
    k = 2048
    dims = [2048, 512, 512]
    ws = [quant_weights(wtype, n, k, seed=n + i)[0] for i, n in enumerate(dims)]
    Ws = [ops.Weight(wtype, w, n, k) for w, n in zip(ws, dims)]
    x = DeviceArray.from_numpy(rng(9).standard_normal((3, k)).astype(np.float32))
    fused = [DeviceArray((3, n)) for n in dims]
    ops.linear_shared(x, Ws, fused)
    for W, f, n in zip(Ws, fused, dims):
        sep = DeviceArray((3, n))
        ops.linear(x, W, sep)
        assert np.array_equal(sep.numpy(), f.numpy())


# ---------------------------------------------------------------- pointwise

def test_rms_norm_hand_computed():
    """matches_hand_computed (rms_norm.rs:86-98) and weight_scales_output."""
    x = DeviceArray.from_numpy(np.array([[1, 2, 3, 4]], np.float32))
    out = DeviceArray((1, 4))
    ops.rms_norm(x, DeviceArray.from_numpy(np.ones(4, np.float32)), out, 0.0)
    rms = np.sqrt(np.float32(7.5))
    assert np.allclose(out.numpy()[0], np.array([1, 2, 3, 4]) / rms, atol=1e-5)
    ops.rms_norm(x, DeviceArray.from_numpy(np.full(4, 2, np.float32)), out, 0.0)
    assert np.allclose(out.numpy()[0], 2 * np.array([1, 2, 3, 4]) / rms, atol=1e-5)
    z = DeviceArray.from_numpy(np.zeros((1, 4), np.float32))
    ops.rms_norm(z, DeviceArray.from_numpy(np.ones(4, np.float32)), out, 1e-5)
    assert np.all(np.isfinite(out.numpy())) and np.all(out.numpy() == 0)


@pytest.mark.parametrize("dim", [2048, 512, 100])
def test_rms_norm_matches_oracle(dim):
    x = (rng(dim).standard_normal((7, dim)) * 2).astype(np.float32)
    w = (1 + 0.1 * rng(1).standard_normal(dim)).astype(np.float32)
    out = DeviceArray((7, dim))
    ops.rms_norm(DeviceArray.from_numpy(x), DeviceArray.from_numpy(w), out, 1e-5)
    want = O.rms_norm(x, w, 1e-5)
    # Only the sum of squares is reordered: relative error ~ dim * eps.
    assert np.allclose(out.numpy(), want, rtol=2e-6, atol=1e-7)


def test_rope_rows_bit_exact():
    inv = O.rope_inv_freq(64, 500000.0)
    t = rng(3).standard_normal((9, 2048)).astype(np.float32)
    d = DeviceArray.from_numpy(t)
    ops.rope_rows(d, 4090, inv)
    st, want = O.rope_rows(t, 4090, inv)
    assert st == 0
    assert np.array_equal(d.numpy(), want)


def test_silu_mul_add():
    x = (rng(4).standard_normal(5000) * 8).astype(np.float32)
    x[:4] = [0.0, -100.0, 100.0, -0.0]
    d = DeviceArray.from_numpy(x)
    ops.silu(d)
    want = O.silu(x)
    # device expf vs glibc expf: each within ~1 ulp, so a few ulps apart
    assert np.allclose(d.numpy(), want, rtol=1e-6, atol=1e-38)
    a, b = x, x[::-1].copy()
    o = DeviceArray(a.shape)
    ops.elementwise_mul(DeviceArray.from_numpy(a), DeviceArray.from_numpy(b), o)
    assert np.array_equal(o.numpy(), a * b)
    da = DeviceArray.from_numpy(a)
    ops.elementwise_add(da, DeviceArray.from_numpy(b))
    assert np.array_equal(da.numpy(), a + b)


def test_softmax_known_values():
    """known_values / sums_to_one / survives_large_values (softmax.rs:39-65)."""
    o = DeviceArray(3)
    ops.softmax(DeviceArray.from_numpy(np.array([1, 2, 3], np.float32)), o)
    assert np.allclose(o.numpy(), [0.09003057, 0.24472847, 0.66524096], atol=1e-6)
    o2 = DeviceArray(2)
    ops.softmax(DeviceArray.from_numpy(np.array([100, 101], np.float32)), o2)
    v = o2.numpy()
    assert np.all(np.isfinite(v)) and abs(v.sum() - 1) < 1e-6 and v[1] > v[0]
    with pytest.raises(sq.KernelError) as e:
        ops.softmax(DeviceArray(0), DeviceArray(0))
    assert e.value.kind == "EmptyInput"


# ---------------------------------------------------------------- attention

def sdpa_dev(q, k, v, seq_q, seq_k, nh, nkv, hd):
    out = DeviceArray(q.size)
    ops.sdpa_cached(DeviceArray.from_numpy(q), DeviceArray.from_numpy(k), DeviceArray.from_numpy(v), out,
                    nh, nkv, hd)
    return out.numpy()


def test_sdpa_reference_known_answers():
    """The five attention tests of attention.rs:84-171 on the device."""
    q = np.array([0.5, -1.0, 2.0, 0.25], np.float32)
    v = np.array([7.0, 8.0, 9.0, 10.0], np.float32)
    assert np.allclose(sdpa_dev(q, q, v, 1, 1, 1, 1, 4), v, atol=1e-5)
    q = np.array([1.0, 0.0, 0.5, 0.5], np.float32)
    k = np.array([1.0, 0.0, 0.0, 1.0], np.float32)
    va = np.array([3.0, 4.0, 99.0, -99.0], np.float32)
    vb = np.array([3.0, 4.0, -42.0, 1234.0], np.float32)
    oa, ob = sdpa_dev(q, k, va, 2, 2, 1, 1, 2), sdpa_dev(q, k, vb, 2, 2, 1, 1, 2)
    assert np.allclose(oa[:2], ob[:2], atol=1e-5) and np.allclose(oa[:2], [3, 4], atol=1e-5)
    q = np.array([1, 0, 1, 0, 0, 1, 0, 1], np.float32)
    k = np.array([1.0, 1.0, 0.5, -0.5], np.float32)
    v = np.array([10.0, 20.0, 30.0, 40.0], np.float32)
    o = sdpa_dev(q, k, v, 1, 1, 4, 2, 2)
    assert np.allclose(o[0:2], o[2:4], atol=1e-5) and np.allclose(o[4:6], o[6:8], atol=1e-5)
    q = np.array([0.1, 0.2, 0.3, 0.4], np.float32)
    k = np.array([1.0, 0.0, -1.0, 2.0], np.float32)
    v = np.array([5.0, 6.0, 7.0, 8.0], np.float32)
    assert np.allclose(sdpa_dev(q, k, v, 1, 1, 2, 2, 2), v, atol=1e-5)
    with pytest.raises(sq.KernelError) as e:
        sdpa_dev(np.zeros(6, np.float32), np.zeros(6, np.float32), np.zeros(6, np.float32), 1, 1, 3, 2, 2)
    assert e.value.kind == "ShapeMismatch"


@pytest.mark.parametrize("seq_q,seq_k", [(1, 1), (1, 37), (1, 300), (1, 4096), (200, 200), (64, 300), (5, 5)])
@pytest.mark.parametrize("nh,nkv", [(32, 8), (8, 2), (4, 4)])
@pytest.mark.parametrize("attn", ["auto", "split"])
def test_sdpa_model_kernels_match_oracle(seq_q, seq_k, nh, nkv, attn, monkeypatch):
    """The model's attention kernels against the oracle: decode (one query),
    and the prefill kernel the size selects (auto: fp32 matrix instructions
    up to 192 keys, split-f16 beyond) or the split-f16 kernel at every size
    (SQUIRREL_ATTN_F32=0)."""
    if attn == "split":
        monkeypatch.setenv("SQUIRREL_ATTN_F32", "0")
    hd = 64
    r = rng(seq_q * 1000 + seq_k + nh)
    q = r.standard_normal(seq_q * nh * hd).astype(np.float32)
    k = r.standard_normal(seq_k * nkv * hd).astype(np.float32)
    v = r.standard_normal(seq_k * nkv * hd).astype(np.float32)
    got = sdpa_dev(q, k, v, seq_q, seq_k, nh, nkv, hd)
    st, want = O.sdpa(q, k, v, seq_q, seq_k, nh, nkv, hd)
    assert st == 0
    # Online softmax vs two-pass: outputs are convex combinations of v rows
    # (|v| ~ 1); rounding differences stay at a few f32 ulps of the scale.
    assert np.allclose(got, want, rtol=1e-5, atol=2e-6), float(np.abs(got - want).max())


@pytest.mark.parametrize("seq_k", [2, 63, 64, 65, 128, 129, 1000, 4095, 4097, 8200])
@pytest.mark.parametrize("nh,nkv", [(32, 8), (4, 2), (8, 1), (3, 3)])
def test_sdpa_decode_tile_edges(seq_k, nh, nkv):
    """One query over key counts around the 64-position tiles, the merge's 64
    tiles per round and its 16 loads in flight, for every GQA group size; the
    rows past the keys (the same buffers' next tile, infinite and NaN) do not
    reach the result.  The bound of the test above: outputs are convex
    combinations of v rows."""
    hd = 64
    r = rng(seq_k + nh)
    q = r.standard_normal(nh * hd).astype(np.float32) * 2
    k = r.standard_normal(seq_k * nkv * hd).astype(np.float32)
    v = r.standard_normal(seq_k * nkv * hd).astype(np.float32)
    st, want = O.sdpa(q, k, v, 1, seq_k, nh, nkv, hd)
    assert st == 0

    class Head:  # the first seq_k rows of a longer buffer
        def __init__(self, rows, past):
            self.buf = DeviceArray.from_numpy(np.concatenate([rows, np.full(64 * nkv * hd, past, np.float32)]))
            self.ptr, self.size = self.buf.ptr, rows.size

    for past_k, past_v in ((np.inf, np.inf), (np.nan, np.nan)):
        out = DeviceArray(q.size)
        ops.sdpa_cached(DeviceArray.from_numpy(q), Head(k, past_k), Head(v, past_v), out, nh, nkv, hd)
        got = out.numpy()
        assert np.allclose(got, want, rtol=1e-5, atol=2e-6), float(np.abs(got - want).max())
    # an infinite last row reaches the output as infinities, not NaN
    v[-nkv * hd:] = np.inf
    got = sdpa_dev(q, k, v, 1, seq_k, nh, nkv, hd)
    assert np.all(np.isposinf(got))


@pytest.mark.parametrize("scale", [1e-3, 1.0, 6.0])
def test_prefill_attention_split_f16_within_f32_noise(scale, monkeypatch):
    """The prefill attention's split-f16 products (hi + 2^-11 lo halves of
    every f32 operand) against the oracle, beside the fp32 matrix kernel
    (SQUIRREL_ATTN_F32=1) on the same inputs: over operand magnitudes from
    1e-3 (f16 subnormal hi halves) to 6 (sharp softmax rows), the split
    kernel's largest error stays within a small multiple of the fp32
    kernel's, i.e. within f32 rounding noise."""
    seq_q, seq_k, nh, nkv, hd = 130, 300, 8, 2, 64
    r = rng(int(scale * 1000) + 7)
    q = (r.standard_normal(seq_q * nh * hd) * scale).astype(np.float32)
    k = (r.standard_normal(seq_k * nkv * hd) * scale).astype(np.float32)
    v = (r.standard_normal(seq_k * nkv * hd) * scale).astype(np.float32)
    st, want = O.sdpa(q, k, v, seq_q, seq_k, nh, nkv, hd)
    assert st == 0
    monkeypatch.setenv("SQUIRREL_ATTN_F32", "0")
    got = sdpa_dev(q, k, v, seq_q, seq_k, nh, nkv, hd)
    monkeypatch.setenv("SQUIRREL_ATTN_F32", "1")
    ref = sdpa_dev(q, k, v, seq_q, seq_k, nh, nkv, hd)
    e_split = float(np.abs(got - want).max()) / scale
    e_f32 = float(np.abs(ref - want).max()) / scale
    print(f"scale {scale}: max error / scale: split {e_split:.3e}, fp32 {e_f32:.3e}")
    assert np.isfinite(got).all()
    assert e_split <= max(4 * e_f32, 2e-6), (e_split, e_f32)


def test_prefill_attention_large_operands(monkeypatch):
    """Operands up to 3e4 (beyond f16's range before the split kernel's 2^-8
    scaling) stay finite and match the oracle: the softmax rows are then
    nearly one-hot, so the output is a v row to f32 rounding."""
    monkeypatch.setenv("SQUIRREL_ATTN_F32", "0")
    seq_q, seq_k, nh, nkv, hd = 70, 70, 4, 4, 64
    r = rng(99)
    q = r.standard_normal(seq_q * nh * hd).astype(np.float32)
    k = r.standard_normal(seq_k * nkv * hd).astype(np.float32)
    v = r.standard_normal(seq_k * nkv * hd).astype(np.float32)
    q[::97] = 3e4
    k[::89] = -2e4
    v[::83] = 3e4
    st, want = O.sdpa(q, k, v, seq_q, seq_k, nh, nkv, hd)
    assert st == 0
    got = sdpa_dev(q, k, v, seq_q, seq_k, nh, nkv, hd)
    assert np.isfinite(got).all()
    assert np.allclose(got, want, rtol=1e-5, atol=1e-5 * 3e4), float(np.abs(got - want).max())


def test_sdpa_generic_head_dims():
    for hd, nh, nkv, sq_, sk in [(4, 2, 1, 3, 5), (32, 4, 2, 1, 9), (128, 2, 2, 4, 4)]:
        r = rng(hd)
        q = r.standard_normal(sq_ * nh * hd).astype(np.float32)
        k = r.standard_normal(sk * nkv * hd).astype(np.float32)
        v = r.standard_normal(sk * nkv * hd).astype(np.float32)
        got = sdpa_dev(q, k, v, sq_, sk, nh, nkv, hd)
        st, want = O.sdpa(q, k, v, sq_, sk, nh, nkv, hd)
        assert st == 0 and np.allclose(got, want, rtol=1e-5, atol=2e-6)


# ---------------------------------------------------------------- greedy / embed

@pytest.mark.parametrize("case", range(7))
def test_greedy_matches_oracle(case):
    r = rng(case)
    nan = np.float32(np.nan)
    cases = [
        np.array([0.1, -2.3, 5.7, 4.0], np.float32),                      # picks_max_index
        np.array([1.0, nan, 3.0, 2.0], np.float32),                       # ignores_nan
        np.array([3.0, 1.0, 3.0, 2.0, 3.0, 0.0], np.float32),             # ties -> last
        np.array([5.0, nan, 1.0], np.float32),                            # NaN hands over the lead
        np.array([1.0, 3.0, nan], np.float32),                            # trailing NaN wins
        r.standard_normal(128256).astype(np.float32),
        np.round(r.standard_normal(128256) * 2).astype(np.float32),       # many exact ties
    ]
    x = cases[case]
    assert ops.greedy(DeviceArray.from_numpy(x)) == O.greedy(x)


def test_log_softmax_at_closed_forms():
    """log p(idx) of the perplexity harness (perplexity.rs:112-117) on inputs
    whose value is known in closed form, and on a vocabulary-sized row
    against scipy's log-softmax (an independent formulation), in f64."""
    from scipy.special import log_softmax
    ls = lambda x, i: ops.log_softmax_at(DeviceArray.from_numpy(np.asarray(x, np.float32)), i)  # noqa: E731
    assert abs(ls(np.full(1000, 3.7), 17) - (-np.log(1000.0))) < 1e-12
    x = np.array([0.0, -np.inf, -np.inf, np.log(3.0)], np.float32)
    assert abs(ls(x, 0) - np.log(1.0 / (1.0 + float(np.exp(np.float64(np.float32(np.log(3.0)))))))) < 1e-12
    assert ls(x, 1) == -np.inf
    assert abs(ls([1e30, 1e30], 1) - np.log(0.5)) < 1e-15
    assert np.isnan(ls([1.0, np.nan, 2.0], 0))            # exp(NaN - max) poisons the sum
    a, b, k, n = 2.5, -1.25, 37, 4096
    x = np.full(n, b, np.float32)
    x[:k] = a
    want = (a - a) - np.log(k + (n - k) * np.exp(b - a))
    assert abs(ls(x, 3) - want) < 1e-12
    r = rng(5)
    x = (r.standard_normal(128256) * 3).astype(np.float32)
    ref = log_softmax(x.astype(np.float64))
    for i in (0, 1, 77777, 128255, int(np.argmax(x))):
        assert abs(ls(x, i) - ref[i]) < 1e-11
    with pytest.raises(sq.SqError):
        ls(x, 128256)


def test_linear_from_several_threads():
    """Calls share a pool of scratch blocks: threads that multiply inputs of
    different sizes at once, over and over, each get the results of a call
    made alone, bit for bit."""
    import threading
    cases = []
    for i, (m, k, n) in enumerate([(1, 2048, 512), (9, 512, 300), (40, 1024, 256), (130, 256, 2048)]):
        w, _ = quant_weights(O.Q8_0, n, k, seed=40 + i)
        W = ops.Weight(O.Q8_0, w, n, k)
        x = DeviceArray.from_numpy((rng(i).standard_normal((m, k))).astype(np.float32))
        alone = DeviceArray((m, n))
        ops.linear(x, W, alone)
        cases.append((W, x, alone.numpy(), [DeviceArray((m, n)) for _ in range(12)]))
    errors = []

    def work(W, x, want, outs):
        try:
            for o in outs:
                ops.linear(x, W, o)
            for o in outs:
                assert np.array_equal(o.numpy(), want)
        except BaseException as e:  # noqa: BLE001
            errors.append(e)

    threads = [threading.Thread(target=work, args=c) for c in cases]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors


@pytest.mark.parametrize("n", [1, 255, 2047, 2048, 2049, 4097, 512 * 2048 + 5])
def test_log_softmax_at_chunk_edges(n):
    """Rows of one partial chunk, whole chunks and chunks longer than the
    workgroup's; a first chunk that is -inf throughout adds nothing."""
    x = (rng(n).standard_normal(n) * 4).astype(np.float32)
    x[:min(n - 1, 2048)] = -np.inf
    mx = np.float64(x.max())
    lse = np.log(np.exp(x.astype(np.float64) - mx).sum())
    d = DeviceArray.from_numpy(x)
    for i in {n - 1, max(0, n - 2), n // 2}:
        want = np.float64(x[i]) - mx - lse
        got = ops.log_softmax_at(d, i)
        # f64 sums of at most 2^20 terms
        assert got == want or abs(got - want) < 1e-11
    if n > 4096:
        x[n - 3] = np.inf
        assert np.isnan(ops.log_softmax_at(DeviceArray.from_numpy(x), 0))
    assert np.isnan(ops.log_softmax_at(DeviceArray.from_numpy(np.full(n, -np.inf, np.float32)), 0))


@pytest.mark.parametrize("wtype", [O.Q8_0, O.Q4_0, O.BF16])
def test_embed_bit_exact(wtype):
    if wtype == O.BF16:
        pytest.skip(A32_SKIP)
    vocab, dim = 300, 2048
    w, _ = quant_weights(wtype, vocab, dim, seed=11 + wtype)
    toks = np.array([0, 299, 17, 17, 150], np.uint32)
    out = DeviceArray((toks.size, dim))
    ops.embed(DeviceArray.from_numpy(toks), ops.Weight(wtype, w, vocab, dim), out)
    want = O.embed(toks, wtype, w, dim, vocab)
    assert np.array_equal(out.numpy(), want)


@pytest.mark.parametrize("bad", [300, 2**31, 2**32 - 1])
def test_embed_id_past_the_table_is_an_error(bad):
    """A token id past the table that reaches the kernel from device memory
    is an error status, as the reference's slice index panics
    (embedding.rs:43-44).  The kernel clamps the row it reads, so the launch
    stays in bounds, and raises the error word the host turns into the
    status."""
    vocab, dim = 300, 2048
    w, _ = quant_weights(O.Q8_0, vocab, dim, seed=11)
    table = ops.Weight(O.Q8_0, w, vocab, dim)
    out = DeviceArray((3, dim))
    ops.embed(DeviceArray.from_numpy(np.array([3, 299, 0], np.uint32)), table, out)
    with pytest.raises(sq.SqError) as e:
        ops.embed(DeviceArray.from_numpy(np.array([3, bad, 0], np.uint32)), table, out)
    assert e.value.code == 22 and "embedding table" in str(e.value)

"""GPU parity of the batched q4/q8 contraction on the matrix cores (`q4nx_gemm`) against the
oracle, for row counts from one (decode) to prefill lengths.

Bars: max|Δ|/max|ref| < 1e-5 against the float64 oracle with cosine > 0.9999999 for every
row (the reference's GEMV gate, designs/granite_gemv/granite_gemv.py:335, and its per-token
check of the batched design, granite_gemv32.py:279-288); one-hot rows reproduce the
float32 dequantised column bit-for-bit; split-K launches are bit-reproducible.
"""

import numpy as np
import pytest
import torch

from llmnputest_amd import ops, synth
from oracle import q4nx_oracle as qo

pytestmark = pytest.mark.gpu

REL = 1e-5
COS = 0.9999999


def _tiles(kind, n, k, seed):
    rng = np.random.default_rng(seed)
    t = synth.q4_tiles(rng, n, k) if kind == "q4" else synth.q8_tiles(rng, n, k)
    return t.reshape(-1, t.shape[-1]), rng


def _dev_u8(a, dev):
    return torch.from_numpy(np.ascontiguousarray(a).reshape(-1)).to(dev)


def _dev_bf16(bits, dev):
    return torch.from_numpy(np.ascontiguousarray(bits, dtype=np.uint16).view(np.int16)).to(dev).view(torch.bfloat16)


def _check_rows(y, ref):
    """Every row on its own, then the whole block."""
    for i in range(ref.shape[0]):
        rel, cos = qo.metrics(y[i], ref[i])
        assert rel < REL and cos > COS, (i, rel, cos)


@pytest.mark.parametrize("kind", ["q4", "q8"])
@pytest.mark.parametrize("m,n,k", [
    (1, 128, 512),
    (5, 128, 512),       # partial m-tile
    (16, 256, 768),
    (17, 256, 2560),     # two m-tiles, one of one row
    (33, 128, 1024),     # K split over two waves, two m-tiles per wave
    (64, 192, 768),
    (65, 256, 1024),     # prefill blocks: 128 rows per workgroup
    (200, 512, 2560),
    (8, 2560, 8192),     # down_proj shape, batch 8: split K across workgroups
])
def test_gemm_parity(dev, kind, m, n, k):
    raw, rng = _tiles(kind, n, k, 11 + m)
    x = synth.random_bf16(rng, (m, k))
    y = ops.gemm(_dev_u8(raw, dev), kind, _dev_bf16(x, dev), n // 32, k // 256).cpu().numpy()
    ref = qo.gemv(raw, kind, x, n // 32, k // 256, acc=np.float64)
    _check_rows(y, ref)


@pytest.mark.parametrize("kind", ["q4", "q8"])
def test_gemm_onehot_exact(dev, kind):
    """Row i of x is the unit vector e_{k_i}: row i of y is column k_i of the float32
    dequantised matrix, bit for bit (code * d + m rounds once, as tools/q4nx.py:127-137)."""
    n, k = 96, 1024
    raw, _ = _tiles(kind, n, k, 2)
    cols = [0, 1, 7, 8, 31, 32, 255, 256, 511, 777, 1000, 1023, 5, 600, 64, 130, 900]
    x = np.zeros((len(cols), k), np.float32)
    x[np.arange(len(cols)), cols] = 1.0
    y = ops.gemm(_dev_u8(raw, dev), kind, _dev_bf16(qo.bf16_round(x), dev), n // 32,
                 k // 256).cpu().numpy()
    wm = qo.dequant_matrix(raw, kind, n // 32, k // 256)
    for i, kk in enumerate(cols):
        assert np.array_equal(y[i].view(np.uint32), wm[:, kk].view(np.uint32)), kk


@pytest.mark.parametrize("scale", [1e-30, 1e-3, 1e4, 1e30])
def test_gemm_activation_range(dev, scale):
    """bf16 x enters the matrix cores unchanged: any bf16 range is exact input."""
    m, n, k = 24, 256, 2560
    raw, rng = _tiles("q4", n, k, 8)
    xf = rng.standard_normal((m, k)).astype(np.float32) * np.float32(scale)
    xf[:, ::97] *= np.float32(1e-6)
    x = qo.bf16_round(xf)
    y = ops.gemm(_dev_u8(raw, dev), "q4", _dev_bf16(x, dev), n // 32, k // 256).cpu().numpy()
    ref = qo.gemv(raw, "q4", x, n // 32, k // 256, acc=np.float64)
    _check_rows(y, ref)


def test_gemm_heavy_tailed(dev):
    """Student-t(2) activations: a few entries dwarf the rest."""
    m, n, k = 12, 512, 8192
    raw, rng = _tiles("q4", n, k, 9)
    x = qo.bf16_round(rng.standard_t(2.0, (m, k)).astype(np.float32))
    y = ops.gemm(_dev_u8(raw, dev), "q4", _dev_bf16(x, dev), n // 32, k // 256).cpu().numpy()
    ref = qo.gemv(raw, "q4", x, n // 32, k // 256, acc=np.float64)
    _check_rows(y, ref)


def test_gemm_residual_strided_x(dev):
    """x rows with a stride longer than K, and a residual added once."""
    m, n, k = 40, 256, 1536
    raw, rng = _tiles("q4", n, k, 10)
    xfull = synth.random_bf16(rng, (m, k + 64))
    xd = _dev_bf16(xfull, dev)[:, :k]
    res = rng.standard_normal((m, n)).astype(np.float32)
    y = ops.gemm(_dev_u8(raw, dev), "q4", xd, n // 32, k // 256,
                 residual=torch.from_numpy(res).to(dev)).cpu().numpy()
    ref = qo.gemv(raw, "q4", np.ascontiguousarray(xfull[:, :k]), n // 32, k // 256,
                  acc=np.float64) + res
    _check_rows(y, ref)


@pytest.mark.parametrize("parts", [1, 2, 3, 5])
@pytest.mark.parametrize("n,m", [(2560, 3), (2560, 30), (2560, 100),
                                 (512, 3), (512, 12)])   # 16 tile-rows: row-block workgroups
def test_gemm_ksplit_deterministic(dev, parts, m, n):
    """Any split of K gives the oracle's result, and the same bits on every call (with 16
    tile-rows and one m-tile the parts are row-block workgroups, two per tile-row)."""
    k = 8192
    raw, rng = _tiles("q4", n, k, 12)
    w = _dev_u8(raw, dev)
    x = synth.random_bf16(rng, (m, k))
    xd = _dev_bf16(x, dev)
    pol = ops.Policy(gemm_ksplit=parts)
    y1 = ops.gemm(w, "q4", xd, n // 32, k // 256, policy=pol).cpu().numpy()
    y2 = ops.gemm(w, "q4", xd, n // 32, k // 256, policy=pol).cpu().numpy()
    assert np.array_equal(y1.view(np.uint32), y2.view(np.uint32))
    ref = qo.gemv(raw, "q4", x, n // 32, k // 256, acc=np.float64)
    _check_rows(y1, ref)


@pytest.mark.parametrize("parts", [1, 3])
def test_gemm_q8_rowblock_split(dev, parts):
    """q8 tiles on row-block workgroups (16 tile-rows, 3 rows), whole and with K in 3 parts:
    each workgroup stages the scales and its block's 4096 code bytes (the last load of lanes
    32..63 lands in the slot's padding)."""
    n, k, m = 512, 8192, 3
    raw, rng = _tiles("q8", n, k, 15)
    x = synth.random_bf16(rng, (m, k))
    y = ops.gemm(_dev_u8(raw, dev), "q8", _dev_bf16(x, dev), n // 32, k // 256,
                 policy=ops.Policy(gemm_ksplit=parts)).cpu().numpy()
    _check_rows(y, qo.gemv(raw, "q8", x, n // 32, k // 256, acc=np.float64))


@pytest.mark.parametrize("kind", ["q4", "q8"])
def test_gemm_matches_gemv_batch(dev, kind):
    """For the batch sizes both paths take, the two agree to the oracle's bar."""
    n, k, b = 1024, 2560, 8
    raw, rng = _tiles(kind, n, k, 13)
    w = _dev_u8(raw, dev)
    x = synth.random_bf16(rng, (b, k))
    xd = _dev_bf16(x, dev)
    y_mma = ops.gemm(w, kind, xd, n // 32, k // 256).cpu().numpy()
    y_vec = ops.gemv(w, kind, xd, n // 32, k // 256).cpu().numpy()
    ref = qo.gemv(raw, kind, x, n // 32, k // 256, acc=np.float64)
    _check_rows(y_mma, ref)
    _check_rows(y_vec, ref)


def test_gemm_q8_lm_head_prefill(dev):
    """The tied lm_head shape of the granite-3B step (q8 2560 -> 100352) over 48 prompt rows,
    checked against the oracle on a slice of the vocabulary."""
    n, k, m = 100352, 2560, 48
    rng = np.random.default_rng(14)
    raw = synth.q8_tiles(rng, n, k).reshape(-1, qo.Q8_TILE_BYTES)
    x = synth.random_bf16(rng, (m, k))
    y = ops.gemm(_dev_u8(raw, dev), "q8", _dev_bf16(x, dev), n // 32, k // 256).cpu().numpy()
    lo, hi = 96 * 32, 160 * 32   # tile-rows 96..159
    k_t = k // 256
    ref = qo.gemv(raw[lo // 32 * k_t: hi // 32 * k_t], "q8", x, (hi - lo) // 32, k_t,
                  acc=np.float64)
    _check_rows(y[:, lo:hi], ref)


# ------------------------------------------------------------------ prompt blocks
# From 65 rows a launch goes to the fp16-operand kernel, whose workgroup tile (rows, tile-rows, K
# parts) the library chooses by the workgroups each would give and names in a query. One shape per
# tile, ragged both ways where it can be:
TILE_SHAPES = {
    "q4": {(32, 1, 8): (65, 32, 1024), (32, 2, 4): (129, 2080, 1024), (64, 2, 4): (257, 2080, 1280),
           (64, 2, 2): (449, 2592, 1024), (64, 4, 1): (1500, 2464, 1024),
           (128, 8, 1): (4100, 4128, 768), (128, 8, 2): (1900, 4320, 2304)},
    "q8": {(32, 1, 8): (65, 32, 1024), (32, 2, 4): (129, 2080, 1024), (64, 2, 4): (257, 2080, 1280),
           (64, 2, 2): (449, 2592, 1024), (64, 4, 1): (1500, 2464, 1024),
           (128, 4, 1): (2900, 2208, 1024)},
}
EVERY_TILE = [(kind, t, *shape) for kind, d in TILE_SHAPES.items() for t, shape in d.items()]


def _tile(kind, m, n, k):
    """The tile of a prompt block (None: the batched kernel takes it)."""
    from llmnputest_amd import _lib
    v = _lib.lib().q4nx_gemm_prompt_tile(ops.KIND[kind], n // 32, k // 256, m)
    return (v >> 16, v >> 8 & 255, v & 255) if v else None


@pytest.mark.parametrize("kind", ["q4", "q8"])
@pytest.mark.parametrize("m,n,k", [
    (4100, 2016, 512),   # 63 tile-rows: the last workgroup's fourth wave has none; ragged rows
    (2048, 4096, 1024),
    (1544, 8192, 768),   # ragged rows, a partial chunk of groups (3 K-tiles)
    (3100, 4064, 512),   # 127 tile-rows: the last workgroup's last wave has none
])
def test_gemm_prefill_parity(dev, kind, m, n, k):
    """Every row against the float64 oracle at the GEMV bar."""
    assert _tile(kind, m, n, k) == ((64, 4, 1) if kind == "q4" else (128, 4, 1))
    raw, rng = _tiles(kind, n, k, 21 + m)
    x = synth.random_bf16(rng, (m, k))
    y = ops.gemm(_dev_u8(raw, dev), kind, _dev_bf16(x, dev), n // 32, k // 256).cpu().numpy()
    ref = qo.gemv(raw, kind, x, n // 32, k // 256, acc=np.float64)
    _check_rows(y, ref)


def test_gemm_prefill_long_k(dev):
    """K = 8192 (16 tiles per wave and K part): every row at the GEMV bar."""
    m, n, k = 2048, 4096, 8192
    assert _tile("q4", m, n, k) == (128, 8, 2)
    raw, rng = _tiles("q4", n, k, 23)
    x = synth.random_bf16(rng, (m, k))
    y = ops.gemm(_dev_u8(raw, dev), "q4", _dev_bf16(x, dev), n // 32, k // 256).cpu().numpy()
    ref = qo.gemv(raw, "q4", x, n // 32, k // 256, acc=np.float64)
    _check_rows(y, ref)


@pytest.mark.parametrize("kind", ["q4", "q8"])
@pytest.mark.parametrize("n,m", [(2048, 4096), (8192, 1536)])
def test_gemm_prefill_onehot_exact(dev, kind, n, m):
    """One-hot rows reproduce the float32 dequantised column bit for bit: the operand d c - o (q4)
    or q under its scale (q8) is exact, and so is its sum with the minimum term."""
    k = 1024
    assert _tile(kind, m, n, k) == ((64, 4, 1) if kind == "q4" else (128, 4, 1))
    raw, _ = _tiles(kind, n, k, 3)
    cols = np.arange(m) * 5 % k
    x = np.zeros((m, k), np.float32)
    x[np.arange(m), cols] = 1.0
    y = ops.gemm(_dev_u8(raw, dev), kind, _dev_bf16(qo.bf16_round(x), dev), n // 32,
                 k // 256).cpu().numpy()
    wm = qo.dequant_matrix(raw, kind, n // 32, k // 256)
    assert np.array_equal(y.view(np.uint32), wm[:, cols].T.copy().view(np.uint32))


@pytest.mark.parametrize("dist", ["student_t2", "outliers"])
def test_gemm_prefill_heavy_tailed(dev, dist):
    """Heavy-tailed activations on the three large tiles: a few entries dwarf the rest of their
    32-K group, so the group sums S carry most of the minimum term and the scaled code sums
    cancel against it."""
    for m, n, k, tile in ((1536, 8192, 1024, (64, 4, 1)), (2048, 2048, 1024, (64, 4, 1)),
                          (2100, 4128, 2304, (128, 8, 1)), (1900, 4320, 2304, (128, 8, 2))):
        assert _tile("q4", m, n, k) == tile
        raw, rng = _tiles("q4", n, k, 31 + m)
        if dist == "student_t2":
            xf = rng.standard_t(2.0, (m, k)).astype(np.float32)
        else:
            xf = rng.standard_normal((m, k)).astype(np.float32)
            hit = rng.random((m, k)) < 1e-3
            xf[hit] *= np.float32(1e4)
        x = qo.bf16_round(xf)
        y = ops.gemm(_dev_u8(raw, dev), "q4", _dev_bf16(x, dev), n // 32, k // 256).cpu().numpy()
        ref = qo.gemv(raw, "q4", x, n // 32, k // 256, acc=np.float64)
        _check_rows(y, ref)


@pytest.mark.parametrize("scale", [1e-30, 1e30])
@pytest.mark.parametrize("m,n,k,tile", [(4096, 2048, 512, (64, 4, 1)), (4100, 4128, 768, (128, 8, 1)),
                                        (1900, 4320, 2304, (128, 8, 2))])
def test_gemm_prefill_activation_range_residual_stride(dev, scale, m, n, k, tile):
    """Extreme activation ranges, rows with a stride longer than K and a residual."""
    assert _tile("q4", m, n, k) == tile
    raw, rng = _tiles("q4", n, k, 14)
    xf = rng.standard_normal((m, k + 64)).astype(np.float32) * np.float32(scale)
    xfull = qo.bf16_round(xf)
    xd = _dev_bf16(xfull, dev)[:, :k]
    res = rng.standard_normal((m, n)).astype(np.float32) * np.float32(scale)
    y = ops.gemm(_dev_u8(raw, dev), "q4", xd, n // 32, k // 256,
                 residual=torch.from_numpy(res).to(dev)).cpu().numpy()
    ref = qo.gemv(raw, "q4", np.ascontiguousarray(xfull[:, :k]), n // 32, k // 256,
                  acc=np.float64) + res
    _check_rows(y, ref)


@pytest.mark.parametrize("kind", ["q4", "q8"])
@pytest.mark.parametrize("m,n,k", [(2048, 4096, 256), (1536, 8192, 512), (2048, 4096, 768),
                                   (4100, 4128, 256), (4100, 4128, 512), (4100, 4128, 768)])
def test_gemm_prefill_short_k(dev, kind, m, n, k):
    """One to three K-tiles per tile-row: the loads of tiles past the last and the steps of x past
    the end all stay unused (the last three: the 128-row tile with its first wave of K alone)."""
    assert _tile(kind, m, n, k) == ((128, 4, 1) if kind == "q8" else
                                    (128, 8, 1) if m == 4100 else (64, 4, 1))
    raw, rng = _tiles(kind, n, k, 41 + k)
    x = synth.random_bf16(rng, (m, k))
    y = ops.gemm(_dev_u8(raw, dev), kind, _dev_bf16(x, dev), n // 32, k // 256).cpu().numpy()
    ref = qo.gemv(raw, kind, x, n // 32, k // 256, acc=np.float64)
    _check_rows(y, ref)


def test_gemm_prefill_without_workspace(dev):
    """A prompt block with no workspace (NULL, 0), or one too small for the fp16 operands, runs on
    the batched kernel instead: every row at the same bar."""
    from llmnputest_amd import _lib
    m, n, k = 2048, 4096, 512
    assert _tile("q4", m, n, k) is not None
    raw, rng = _tiles("q4", n, k, 43)
    x = synth.random_bf16(rng, (m, k))
    w, xd = _dev_u8(raw, dev), _dev_bf16(x, dev)
    ref = qo.gemv(raw, "q4", x, n // 32, k // 256, acc=np.float64)
    need = _lib.lib().q4nx_gemm_ws_bytes(4, n // 32, k // 256, m, None)
    small = torch.empty(need // 2, dtype=torch.uint8, device=dev)
    for wp, wn in ((None, 0), (small.data_ptr(), small.numel())):
        y = torch.full((m, n), float("nan"), dtype=torch.float32, device=dev)
        _lib.call("q4nx_gemm", 4, w.data_ptr(), n // 32, k // 256, xd.data_ptr(), k, m,
                  y.data_ptr(), n, None, wp, wn, None, ops._stream())
        _check_rows(y.cpu().numpy(), ref)


# ------------------------------------------------------------------ q4 prompt blocks on fp16 operands
# The operands d (B + c) + A are exact and the sums fp32, so every row is held to the GEMV bar; minima unrelated to the scales (every other case here has
# m = -8 d) make the minimum term carry a full share of the result.

def _free_minima(raw, rng):
    m = synth.f32_to_bf16_bits((rng.standard_normal((raw.shape[0], 256)) * 0.1).astype(np.float32))
    raw = raw.copy()
    raw[:, 512:1024] = m.view(np.uint8).reshape(raw.shape[0], 512)
    return raw


@pytest.mark.parametrize("m,n,k", [
    (65, 32, 768),        # 32 x 1: one tile-row, five of eight K parts empty
    (66, 64, 1024),       # the pre-pass's last row length of a wave per row, of 256 threads, and
    (67, 64, 4096),       # the first of 512
    (67, 64, 4352),
    (80, 544, 2816),      # 32 x 1: 11 K-tiles over eight parts of two, the last ones empty
    (129, 2080, 768),     # 32 x 2 (325 workgroups of 32 x 1): a last workgroup with one tile-row
    (257, 2080, 1280),    # 64 x 2 in four parts: five K-tiles in parts of two, one empty
    (449, 2592, 768),     # 64 x 2 in two parts, ragged rows
    (1500, 2464, 256),    # 64 x 4: one K-tile, fewer steps than the ring holds ahead
    (3900, 2016, 2048),   # 128 x 8 in two parts, ragged rows, a last workgroup of seven tile-rows
    (130, 128, 8448),     # rows longer than the pre-pass keeps in registers
])
def test_gemm_fp16_operands_parity(dev, m, n, k):
    raw, rng = _tiles("q4", n, k, 51 + m)
    raw = _free_minima(raw, rng)
    x = synth.random_bf16(rng, (m, k))
    res = rng.standard_normal((m, n)).astype(np.float32)
    w, xd = _dev_u8(raw, dev), _dev_bf16(x, dev)
    y = ops.gemm(w, "q4", xd, n // 32, k // 256, residual=torch.from_numpy(res).to(dev))
    rows = np.unique(np.concatenate([np.arange(0, m, max(1, m // 48)), [m - 1]]))
    ref = qo.gemv(raw, "q4", x[rows], n // 32, k // 256, acc=np.float64) + res[rows]
    _check_rows(y.cpu().numpy()[rows], ref)
    ssq = torch.full((m, n // 16), float("nan"), device=dev)
    y2 = ops.gemv_ex(w, "q4", xd, n // 32, k // 256, residual=torch.from_numpy(res).to(dev),
                     ssq_out=ssq)
    assert torch.equal(y, y2)
    want = y2.double().view(m, -1, 16).square().sum(-1)
    # 16 squares added in fp32: 16 roundings of 2^-24 at most
    assert ((ssq.double() - want).abs() <= 16 * 2.0 ** -24 * want).all()


@pytest.mark.parametrize("m,n,k", [
    (65, 32, 768),        # 32 x 1: one tile-row, five of eight K parts empty
    (66, 64, 1024),       # the pre-pass's last row length of a wave per row, of 256 threads, and
    (67, 64, 4096),       # the first of 512
    (67, 64, 4352),
    (80, 544, 2816),      # 32 x 1: 11 K-tiles over eight parts of two, the last ones empty
    (129, 2080, 768),     # 32 x 2: a last workgroup with one tile-row
    (257, 2080, 1280),    # 64 x 2 in four parts: five K-tiles in parts of two, one empty
    (449, 2592, 768),     # 64 x 2 in two parts, ragged rows
    (1500, 2464, 256),    # 64 x 4 (480 workgroups): one K-tile, fewer steps than the ring's
    (2900, 2208, 1024),   # 128 x 4, ragged rows, a last workgroup of one tile-row
    (70, 131104, 256),    # 128 x 4, row blocks first: weights beyond the L2s, 1025 groups (no
                          # multiple of eight), one tile-row in the last
    (130, 66592, 512),    # the same with two row blocks
    (130, 128, 8448),     # rows longer than the pre-pass keeps in registers
])
def test_gemm_q8_fp16_operands_parity(dev, m, n, k):
    """q8 on every tile of the fp16-operand kernel and on both orders of its workgroups."""
    raw, rng = _tiles("q8", n, k, 151 + m)
    x = synth.random_bf16(rng, (m, k))
    res = rng.standard_normal((m, n)).astype(np.float32)
    w, xd, rd = _dev_u8(raw, dev), _dev_bf16(x, dev), torch.from_numpy(res).to(dev)
    y = ops.gemm(w, "q8", xd, n // 32, k // 256, residual=rd)
    rows = np.unique(np.concatenate([np.arange(0, m, max(1, m // (48 if n < 4096 else 4))), [m - 1]]))
    ref = qo.gemv(raw, "q8", x[rows], n // 32, k // 256, acc=np.float64) + res[rows]
    _check_rows(y.cpu().numpy()[rows], ref)
    ssq = torch.full((m, n // 16), float("nan"), device=dev)
    y2 = ops.gemv_ex(w, "q8", xd, n // 32, k // 256, residual=rd, ssq_out=ssq)
    assert torch.equal(y, y2)
    want = y2.double().view(m, -1, 16).square().sum(-1)
    # 16 squares added in fp32: 16 roundings of 2^-24 at most
    assert ((ssq.double() - want).abs() <= 16 * 2.0 ** -24 * want).all()


@pytest.mark.parametrize("kind,m,n,k", [("q8", 256, 4096, 512), ("q8", 257, 4096, 512),
                                        ("q4", 96, 2048, 512), ("q4", 97, 2048, 512),
                                        ("q4", 200, 512, 512), ("q4", 200, 512, 768),
                                        ("q4", 90, 16384, 512), ("q4", 90, 16416, 512),
                                        ("q4", 128, 16384, 256), ("q4", 300, 16448, 256),
                                        ("q8", 512, 4096, 256), ("q8", 513, 4096, 256)])
def test_gemm_short_k_either_side(dev, kind, m, n, k):
    """Both sides of the short-K line between the batched and the fp16-operand kernel."""
    raw, rng = _tiles(kind, n, k, 7 + m)
    x = synth.random_bf16(rng, (m, k))
    y = ops.gemm(_dev_u8(raw, dev), kind, _dev_bf16(x, dev), n // 32, k // 256).cpu().numpy()
    _check_rows(y, qo.gemv(raw, kind, x, n // 32, k // 256, acc=np.float64))


def test_gemm_q8_fp16_operands_range(dev):
    """q8 scales over the whole bf16 exponent range between a tile's columns, zero scales, code
    -128, rows of very different size; infinities and NaN stay in their rows."""
    m, n, k = 72, 96, 768
    raw, rng = _tiles("q8", n, k, 61)
    raw = raw.copy()
    e = (10.0 ** rng.uniform(-25, 25, (1, 1, 32))).astype(np.float32)   # one size per column
    v = qo.bf16_to_f32(raw[:, :512].copy().view(np.uint16)).reshape(-1, 8, 32) * e
    v[:, :, 5] = 0.0
    raw[:, :512] = synth.f32_to_bf16_bits(v.reshape(-1, 256).astype(np.float32)).view(
        np.uint8).reshape(-1, 512)
    raw[:, 512::97] = 0x80
    xf = rng.standard_normal((m, k)).astype(np.float32)
    xf *= (10.0 ** rng.uniform(-6, 6, (m, 1))).astype(np.float32)
    xf[3] = 0.0
    x = qo.bf16_round(xf)
    w, xd = _dev_u8(raw, dev), _dev_bf16(x, dev)
    y = ops.gemm(w, "q8", xd, n // 32, k // 256).cpu().numpy().astype(np.float64)
    ref = qo.gemv(raw, "q8", x, n // 32, k // 256, acc=np.float64)
    assert (y[3] == 0).all() and (y[:, 5] == 0).all() and (y[:, 37] == 0).all()
    # each output against its own terms' size, K roundings of 2^-24 at most
    wabs = np.abs(qo.dequant_matrix(raw, "q8", n // 32, k // 256).astype(np.float64))
    size = np.abs(qo.bf16_to_f32(x).astype(np.float64)) @ wabs.T
    assert (np.abs(y - ref) <= k * 2.0 ** -24 * size).all()
    bad = xd.clone()
    bad[7, 100], bad[20, 3], bad[64, 511] = float("inf"), float("nan"), float("-inf")
    yb = ops.gemm(w, "q8", bad, n // 32, k // 256).cpu().numpy()
    hit = np.zeros(m, bool)
    hit[[7, 20, 64]] = True
    assert not np.isfinite(yb[hit]).any()
    assert np.array_equal(yb[~hit].view(np.uint32), y[~hit].astype(np.float32).view(np.uint32))


def test_gemm_fp16_operands_range(dev):
    """Scales over the whole bf16 exponent range between a tile's columns, zero scales and
    minima, all-zero rows and rows of very different size, exactly as the 64-bit result has
    them; an infinity or a NaN in a row of x reaches every output of that row and no other."""
    m, n, k = 72, 96, 768
    raw, rng = _tiles("q4", n, k, 61)
    raw = _free_minima(raw, rng)
    e = (10.0 ** rng.uniform(-25, 25, (1, 8, 32))).astype(np.float32)   # one size per column
    for p in (0, 512):
        v = qo.bf16_to_f32(raw[:, p:p + 512].copy().view(np.uint16)).reshape(-1, 8, 32) * e[:, :1]
        v[:, :, 5] = 0.0
        raw[:, p:p + 512] = synth.f32_to_bf16_bits(v.reshape(-1, 256).astype(np.float32)).view(
            np.uint8).reshape(-1, 512)
    xf = rng.standard_normal((m, k)).astype(np.float32)
    xf *= (10.0 ** rng.uniform(-6, 6, (m, 1))).astype(np.float32)
    xf[3] = 0.0
    x = qo.bf16_round(xf)
    w, xd = _dev_u8(raw, dev), _dev_bf16(x, dev)
    y = ops.gemm(w, "q4", xd, n // 32, k // 256).cpu().numpy().astype(np.float64)
    ref = qo.gemv(raw, "q4", x, n // 32, k // 256, acc=np.float64)
    assert (y[3] == 0).all() and (y[:, 5] == 0).all() and (y[:, 37] == 0).all()
    # columns differ by up to 2^166: each output against its own terms' size, K roundings of
    # 2^-24 at most
    wabs = np.abs(qo.dequant_matrix(raw, "q4", n // 32, k // 256).astype(np.float64))
    size = np.abs(qo.bf16_to_f32(x).astype(np.float64)) @ (wabs.T + 16 * wabs.max(1))
    assert (np.abs(y - ref) <= k * 2.0 ** -24 * size).all()
    bad = xd.clone()
    bad[7, 100], bad[20, 3], bad[64, 511] = float("inf"), float("nan"), float("-inf")
    yb = ops.gemm(w, "q4", bad, n // 32, k // 256).cpu().numpy()
    hit = np.zeros(m, bool)
    hit[[7, 20, 64]] = True
    assert not np.isfinite(yb[hit]).any()
    assert np.array_equal(yb[~hit].view(np.uint32), y[~hit].astype(np.float32).view(np.uint32))


@pytest.mark.parametrize("batch,n,k,norm", [
    (65, 96, 256, False),      # 32 x 1 pairs
    (67, 64, 4352, True),      # 512 threads per row of x
    (200, 1312, 768, True),    # 32 x 2 pairs (287 workgroups of 32 x 1)
    (300, 2080, 2816, True),   # 64 x 2 pairs in two parts
    (1300, 2464, 512, True),   # 128 x 4 pairs, ragged both ways
])
def test_gate_up_fp16_operands(dev, batch, n, k, norm):
    """[RMSNorm, gate, up, SwiGLU] on the fp16-operand kernel: the fp32 gate and up values at the
    GEMV bar on the prologue's own bf16 output, h their SwiGLU's rounding."""
    rng = np.random.default_rng(71 + batch)
    g = _free_minima(synth.q4_tiles(rng, n, k).reshape(-1, qo.Q4_TILE_BYTES), rng)
    u = synth.q4_tiles(rng, n, k).reshape(-1, qo.Q4_TILE_BYTES)
    xn = torch.empty((batch, k), dtype=torch.bfloat16, device=dev)
    raw_out = torch.empty((batch, 2 * n), dtype=torch.float32, device=dev)
    kw = {}
    if norm:
        h = (rng.standard_normal((batch, k)) * 5).astype(np.float32)
        x = torch.from_numpy(h).to(dev)
        kw = dict(norm_w=_dev_bf16(synth.random_bf16(rng, k), dev), xn_out=xn,
                  ssq_in=x.view(batch, -1, 16).square().sum(-1).contiguous())
    else:
        x = _dev_bf16(synth.random_bf16(rng, (batch, k)), dev)
        xn.copy_(x)
    h_out = ops.gate_up_swiglu(_dev_u8(g, dev), _dev_u8(u, dev), n // 32, k // 256, x,
                               raw_out=raw_out, **kw)
    if norm:   # the prologue against the batched kernel's: the same bits
        xn2 = torch.empty_like(xn)
        ops.gate_up_swiglu(_dev_u8(g, dev), _dev_u8(u, dev), n // 32, k // 256, x,
                           policy=ops.Policy(gemm_ksplit=1), **dict(kw, xn_out=xn2))
        assert torch.equal(xn, xn2)
    rows = np.unique(np.concatenate([np.arange(0, batch, max(1, batch // 32)), [batch - 1]]))
    xb = xn.view(torch.int16).cpu().numpy().view(np.uint16)[rows]
    got = raw_out.cpu().numpy()
    _check_rows(got[rows, :n], qo.gemv(g, "q4", xb, n // 32, k // 256, acc=np.float64))
    _check_rows(got[rows, n:], qo.gemv(u, "q4", xb, n // 32, k // 256, acc=np.float64))
    narrow = lambda t: t.to(torch.bfloat16).double()
    gv, uv = narrow(raw_out[:, :n]), narrow(raw_out[:, n:])
    want = (gv / (1 + torch.exp(-gv)) * uv)
    # one bf16 rounding (2^-9 of the value's binade) and the fp32 formula's own few ulps
    assert ((h_out.double() - want).abs() <= want.abs() * (2.0 ** -8 + 2.0 ** -20) + 1e-38).all()


@pytest.mark.parametrize("kind", ["q4", "q8"])
@pytest.mark.parametrize("off,odd", [(1, 0), (0, 1), (1, 1), (2, 2)])
def test_prompt_block_outputs_at_any_float(dev, kind, off, odd):
    """y and residual `off` floats past an aligned address, rows N + odd floats apart, as
    q4nx_gemv_ex takes them: every row at the GEMV bar, the floats between the rows untouched. q4
    pairs that no 8-byte access may touch give the batched kernel's bits (the call without a
    workspace)."""
    from llmnputest_amd import _lib
    m, n, k = 200, 2592, 768         # (no K split on the batched kernel)
    raw, rng = _tiles(kind, n, k, 91)
    x = synth.random_bf16(rng, (m, k))
    res = rng.standard_normal((m, n)).astype(np.float32)
    w, xd = _dev_u8(raw, dev), _dev_bf16(x, dev)
    code, ld = ops.KIND[kind], n + odd
    rd = torch.zeros(off + m * ld, device=dev)
    rd[off:].view(m, ld)[:, :n] = torch.from_numpy(res).to(dev)

    def call(ws, out, ssq, o, stride, r):
        _lib.call("q4nx_gemv_ex", code, w.data_ptr(), n // 32, k // 256, xd.data_ptr(), k, None, 0.0,
                  None, m, out.data_ptr() + 4 * o, stride, r, ssq.data_ptr(), None,
                  ws.buf.data_ptr() if ws else None, ws.buf.numel() if ws else 0, None,
                  ops._stream())
    ws = ops.Workspace(16 << 20, device=dev)
    y = torch.full((off + m * ld,), -7.0, device=dev)
    ssq = torch.zeros((m, n // 16), device=dev)
    call(ws, y, ssq, off, ld, rd.data_ptr() + 4 * off)
    got = y[off:].view(m, ld)
    _check_rows(got[:, :n].cpu().numpy(),
                qo.gemv(raw, kind, x, n // 32, k // 256, acc=np.float64) + res)
    assert (y[:off] == -7).all() and (got[:, n:] == -7).all()
    flat = torch.from_numpy(res).to(dev)
    want, wssq = torch.empty((m, n), device=dev), torch.empty_like(ssq)
    pair = kind == "q8" or (off % 2 == 0 and odd % 2 == 0)
    call(ws if pair else None, want, wssq, 0, n, flat.data_ptr())
    assert torch.equal(got[:, :n], want) and torch.equal(ssq, wssq)


@pytest.mark.parametrize("off", [1, 2])
def test_prompt_gate_up_raw_out_at_any_float(dev, off):
    """raw_out of [gate, up] `off` floats past an aligned address: the bits of the batched kernel
    where no 8-byte access may touch it, else those of the aligned call."""
    from llmnputest_amd import _lib
    m, n, k = 200, 6176, 512
    raw, rng = _tiles("q4", n, k, 92)
    w, xd = _dev_u8(raw, dev), _dev_bf16(synth.random_bf16(rng, (m, k)), dev)
    ws = ops.Workspace(32 << 20, device=dev)
    out = []
    for o, work in ((off, True), (0, off % 2 == 0)):
        h = torch.zeros((m, n), dtype=torch.bfloat16, device=dev)
        r = torch.zeros(o + m * 2 * n, device=dev)
        _lib.call("q4nx_gate_up_swiglu", w.data_ptr(), w.data_ptr(), n // 32, k // 256,
                  xd.data_ptr(), k, None, 0.0, None, m, h.data_ptr(), n, r.data_ptr() + 4 * o, None,
                  ws.buf.data_ptr() if work else None, ws.buf.numel() if work else 0, None,
                  ops._stream())
        out.append((h, r[o:]))
    assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1])


@pytest.mark.parametrize("m,n,k", [(500, 8192, 2560), (1000, 4096, 4096), (900, 2560, 8192),
                                   (1500, 2560, 8192), (2048, 8192, 2560), (2048, 8192, 1024),
                                   (2048, 12288, 768), (300, 4096, 1280)])
@pytest.mark.parametrize("mean", [0.0, 0.5])
def test_prompt_blocks_as_exact_as_batched(dev, m, n, k, mean):
    """Prompt blocks that ran on the batched kernel ([gate, up], and projections that also give
    sums of squares) are no further from the 64-bit result on the fp16-operand kernel: the 2-norm
    of the difference, against that of the batched kernel (the same call without a workspace)."""
    from llmnputest_amd import _lib
    g = torch.Generator(device=dev)
    g.manual_seed(m)
    from llmnputest_amd.granite import random_q4_tiles
    w = random_q4_tiles(n, k, g, dev)
    x = (torch.randn((m, k), device=dev, generator=g) + mean).to(torch.bfloat16)
    wm = ops.dequant(w, "q4", n // 32, k // 256, out_dtype=torch.float32, untile=True).double()
    ref = x.double() @ wm.t().contiguous()
    ws = ops.Workspace(96 << 20, device=dev)
    gu, pl = [], []
    for wp, wn in ((ws.buf.data_ptr(), ws.buf.numel()), (None, 0)):
        h = torch.empty((m, n), dtype=torch.bfloat16, device=dev)
        raw = torch.empty((m, 2 * n), device=dev)
        _lib.call("q4nx_gate_up_swiglu", w.data_ptr(), w.data_ptr(), n // 32, k // 256, x.data_ptr(),
                  k, None, 0.0, None, m, h.data_ptr(), n, raw.data_ptr(), None, wp, wn, None,
                  ops._stream())
        y = torch.empty((m, n), device=dev)
        ssq = torch.empty((m, n // 16), device=dev)
        _lib.call("q4nx_gemv_ex", 4, w.data_ptr(), n // 32, k // 256, x.data_ptr(), k, None, 0.0, None,
                  m, y.data_ptr(), n, None, ssq.data_ptr(), None, wp, wn, None, ops._stream())
        gu.append(((raw[:, :n].double() - ref).norm() / ref.norm()).item())
        pl.append(((y.double() - ref).norm() / ref.norm()).item())
    assert gu[0] <= gu[1] and pl[0] <= pl[1], (gu, pl)


@pytest.mark.parametrize("m,n,k", [
    (2100, 4128, 2304),   # 128 x 8 in one part (289 workgroups), ragged both ways, nine K-tiles
    (4100, 4000, 256),    # the same (528), one K-tile
    (1900, 4320, 2304),   # 128 x 8 in two parts (255 workgroups), five and four K-tiles
    (2000, 4064, 8448),   # the same, rows longer than the pre-pass keeps in registers
])
def test_gemm_large_tiles_parity(dev, m, n, k):
    """The 128-row q4 tiles, plain and with sums of squares (which may take another tile)."""
    raw, rng = _tiles("q4", n, k, 51 + m)
    raw = _free_minima(raw, rng)
    x = synth.random_bf16(rng, (m, k))
    res = rng.standard_normal((m, n)).astype(np.float32)
    w, xd, rd = _dev_u8(raw, dev), _dev_bf16(x, dev), torch.from_numpy(res).to(dev)
    rows = np.unique(np.concatenate([np.arange(0, m, max(1, m // 32)), [m - 1]]))
    ref = qo.gemv(raw, "q4", x[rows], n // 32, k // 256, acc=np.float64) + res[rows]
    _check_rows(ops.gemm(w, "q4", xd, n // 32, k // 256, residual=rd).cpu().numpy()[rows], ref)
    ssq = torch.full((m, n // 16), float("nan"), device=dev)
    y = ops.gemv_ex(w, "q4", xd, n // 32, k // 256, residual=rd, ssq_out=ssq)
    _check_rows(y.cpu().numpy()[rows], ref)
    want = y.double().view(m, -1, 16).square().sum(-1)
    assert ((ssq.double() - want).abs() <= 16 * 2.0 ** -24 * want).all()


@pytest.mark.parametrize("batch,n,k", [
    (1000, 3616, 2304),        # 128 x 4 pairs in two parts (232), ragged both ways, nine K-tiles
    (900, 1984, 1280),         # 64 x 4 pairs (240), five K-tiles
    (1700, 2592, 256),         # the same, one K-tile
])
def test_gate_up_large_tiles(dev, batch, n, k):
    test_gate_up_fp16_operands(dev, batch, n, k, False)


# ------------------------------------------------------------------ any range within a row or column
# Under one power of two per row of x and per column of the weights an fp16 operand reaches some
# 2^30 below the largest entry. Where both a row's and a column's 32-K groups lie further apart than
# 2^10 the kernel adds the tile up with the groups' own fp32 scales.

def _group_scaled(raw, f):
    """Tiles with the scales (and minima) of every 32-K group divided by the power of two f[group]."""
    q4 = raw.shape[1] == qo.Q4_TILE_BYTES
    kt = f.size // 8
    out = raw.copy()
    for p in range(2 if q4 else 1):
        v = qo.bf16_to_f32(raw[:, 512 * p:512 * p + 512].copy().view(np.uint16)).astype(np.float64)
        v = v.reshape(-1, kt, 8, 32) / f.reshape(1, kt, 8, 1)
        out[:, 512 * p:512 * p + 512] = synth.f32_to_bf16_bits(
            v.astype(np.float32).reshape(raw.shape[0], 256)).view(np.uint8).reshape(-1, 512)
    return out


def _close_per_output(y, raw, kind, x, n_t, k_t, rows, d_weight):
    """|y - ref| against the size of the output's own terms, 24 roundings of 2^-24: |x| on |w| and,
    for q4, on the codes' offset times the group's own scale."""
    w = qo.dequant_matrix(raw, kind, n_t, k_t).astype(np.float64)
    xf = qo.bf16_to_f32(x[rows]).astype(np.float64)
    size = np.abs(xf) @ (np.abs(w) + d_weight).T
    err = np.abs(y[rows].astype(np.float64) - xf @ w.T)
    assert (err <= 24 * 2.0 ** -24 * size).all(), float((err / size).max() * 2 ** 24)


ANY_RANGE = [
    (80, 544, 2816),      # 32 x 1, eight K parts
    (129, 2080, 768),     # 32 x 2, four parts
    (257, 2080, 1280),    # 64 x 2, four parts
    (449, 2592, 768),     # 64 x 2, two parts
    (130, 128, 8448),     # rows longer than the pre-pass keeps in registers
    (1500, 2464, 256),    # 64 x 4
    (2100, 4128, 768),    # 128 rows
    (1900, 4320, 2304),   # 128 x 8, two parts (q4)
    (2100, 4128, 2304),   # 128 x 8, one part (q4)
]


@pytest.mark.parametrize("kind", ["q4", "q8"])
@pytest.mark.parametrize("m,n,k,spread", [(*c, s) for c in ANY_RANGE for s in (4, 10, 11, 30, 70)
                                          if c[0] < 1000 or s in (10, 11, 70)])
def test_prompt_blocks_any_range(dev, kind, m, n, k, spread):
    """Groups of the weights up to 2^spread apart, x the other way round in two rows of three (every
    group contributes as much) and as it was in the third."""
    raw, rng = _tiles(kind, n, k, 300 + m + spread)
    f = 2.0 ** (rng.integers(0, spread + 1, k // 32) - spread // 2)
    f[:2] = 2.0 ** (spread - spread // 2), 2.0 ** -(spread // 2)
    raw = _group_scaled(raw, f)
    xf = rng.standard_normal((m, k))
    xf[np.arange(m) % 3 < 2] *= np.repeat(f, 32)
    x = qo.bf16_round(xf.astype(np.float32))
    y = ops.gemm(_dev_u8(raw, dev), kind, _dev_bf16(x, dev), n // 32, k // 256).cpu().numpy()
    rows = np.unique(np.concatenate([np.arange(0, m, max(1, m // 12)), [m - 2, m - 1]]))
    ones = raw.copy()      # the group scales alone: every code 1 (and no minimum), times 16
    if kind == "q4":
        ones[:, 512:1024], ones[:, 1024:] = 0, 0x11
        d = 16 * np.abs(qo.dequant_matrix(ones, kind, n // 32, k // 256).astype(np.float64))
    else:
        d = 0.0
    _close_per_output(y, raw, kind, x, n // 32, k // 256, rows, d)


@pytest.mark.parametrize("kind", ["q4", "q8"])
def test_prompt_block_outlier_on_pruned_group(dev, kind):
    """An entry 1e12 times the rest on a group whose weights are all zero leaves the others' sum."""
    m, n, k = 200, 2592, 1024
    raw, rng = _tiles(kind, n, k, 17)
    raw = raw.copy().reshape(n // 32, k // 256, -1)
    for p in range(2 if kind == "q4" else 1):          # group 3 of K-tile 1
        raw[:, 1, 512 * p + 64 * 3:512 * p + 64 * 4] = 0
    raw = raw.reshape(-1, raw.shape[-1])
    xf = rng.standard_normal((m, k)).astype(np.float32)
    xf[::2, 256 + 96 + 5] = 1e12
    x = qo.bf16_round(xf)
    y = ops.gemm(_dev_u8(raw, dev), kind, _dev_bf16(x, dev), n // 32, k // 256).cpu().numpy()
    _check_rows(y, qo.gemv(raw, kind, x, n // 32, k // 256, acc=np.float64))


@pytest.mark.parametrize("own", [True, False])
@pytest.mark.parametrize("batch,n,k", [(65, 96, 1024), (300, 2080, 2816), (900, 1984, 1280),
                                       (1000, 3616, 2304)])
def test_gate_up_any_range_norm(dev, own, batch, n, k):
    """[RMSNorm, gate, up] with the norm's weights and the tiles' scales 2^40 apart the other way
    round, the normalised rows taken by the caller or not: raw_out per output, h from raw_out."""
    rng = np.random.default_rng(400 + batch)
    f = 2.0 ** (rng.integers(0, 41, k // 32) - 20)
    g = _group_scaled(synth.q4_tiles(rng, n, k).reshape(-1, qo.Q4_TILE_BYTES), f)
    u = _group_scaled(synth.q4_tiles(rng, n, k).reshape(-1, qo.Q4_TILE_BYTES), f)
    h = rng.standard_normal((batch, k)).astype(np.float32)
    h[1::3] /= np.repeat(f, 32)[None].astype(np.float32)   # rows that come out narrow
    x = torch.from_numpy(h).to(dev)
    nw = synth.f32_to_bf16_bits(np.repeat(f, 32).astype(np.float32))
    kw = dict(norm_w=_dev_bf16(nw, dev), ssq_in=x.view(batch, -1, 16).square().sum(-1).contiguous())
    raw_out = torch.empty((batch, 2 * n), device=dev)
    xn = torch.zeros((batch, k), dtype=torch.bfloat16, device=dev)
    wg, wu = _dev_u8(g, dev), _dev_u8(u, dev)
    out = ops.gate_up_swiglu(wg, wu, n // 32, k // 256, x, raw_out=raw_out, **kw,
                             **({} if own else {"xn_out": xn}))
    if own:      # the rows it normalised, from a call that gives them
        ops.gate_up_swiglu(wg, wu, n // 32, k // 256, x, xn_out=xn, **kw)
    xb = xn.view(torch.int16).cpu().numpy().view(np.uint16)
    rows = np.unique(np.concatenate([np.arange(0, batch, max(1, batch // 12)), [1, 4, batch - 1]]))
    got = raw_out.cpu().numpy()
    for w, o in ((g, 0), (u, n)):
        ones = w.copy()
        ones[:, 512:1024], ones[:, 1024:] = 0, 0x11
        d = 16 * np.abs(qo.dequant_matrix(ones, "q4", n // 32, k // 256).astype(np.float64))
        _close_per_output(got[:, o:o + n], w, "q4", xb, n // 32, k // 256, rows, d)
    narrow = lambda t: t.to(torch.bfloat16).double()
    gv, uv = narrow(raw_out[:, :n]), narrow(raw_out[:, n:])
    want = gv / (1 + torch.exp(-gv)) * uv
    assert ((out.double() - want).abs() <= want.abs() * (2.0 ** -8 + 2.0 ** -20) + 1e-38).all()


@pytest.mark.parametrize("kind", ["q4", "q8"])
@pytest.mark.parametrize("m,n,k,parts", [(2048, 8192, 512, 1), (2048, 8192, 512, 3), (100, 2560, 2560, 1)])
def test_prompt_block_keeps_its_kernel_under_a_ksplit(dev, kind, m, n, k, parts):
    """gemm_ksplit 1, and any on a projection that fills the chip by itself: the bits of the default
    policy's kernel (which the batched kernel's differ from)."""
    from llmnputest_amd import _lib
    raw, rng = _tiles(kind, n, k, 77)
    w, xd = _dev_u8(raw, dev), _dev_bf16(synth.random_bf16(rng, (m, k)), dev)
    want = ops.gemm(w, kind, xd, n // 32, k // 256)
    assert torch.equal(ops.gemm(w, kind, xd, n // 32, k // 256, policy=ops.Policy(gemm_ksplit=parts)), want)
    y = torch.empty_like(want)
    _lib.call("q4nx_gemm", ops.KIND[kind], w.data_ptr(), n // 32, k // 256, xd.data_ptr(), k, m,
              y.data_ptr(), n, None, None, 0, None, ops._stream())
    assert not torch.equal(y, want)


# ------------------------------------------------------------------ every tile

def _onehot_rows(m, k, dev):
    cols = torch.from_numpy(np.arange(m) * 7 % k).to(dev)
    x = torch.zeros((m, k), dtype=torch.bfloat16, device=dev)
    x[torch.arange(m, device=dev), cols] = 1.0
    return x, cols


def _onehot_check(y, raw, kind, n, k, cols, dev, rows=0):
    """Rows of y against the columns `cols` of the float32 dequantised matrix: the same bits; where a
    q4 minimum is below 2^-14 of 8 d (its bits end past the two terms of u) or is added on top of
    the codes' sum (minima other than -8 d on the 128-row tiles) to 2^-22 of 8 d, m and the value."""
    column = lambda r: ops.dequant(_dev_u8(r, dev), kind, n // 32, k // 256, out_dtype=torch.float32,
                                   untile=True)[:, cols].t()
    want = column(raw)
    if kind == "q8":
        assert torch.equal(y, want)
        return
    lo, hi = raw.copy(), raw.copy()
    lo[:, 1024:], hi[:, 1024:], hi[:, 512:1024] = 0, 0x11, 0     # the minimum; the scale
    m, d8 = column(lo).abs(), 8 * column(hi).abs()
    far = (m < 2.0 ** -14 * d8) | ((m != d8) & (rows == 128))
    assert torch.equal(torch.where(far, want, y), want)
    assert ((y - want).abs()[far] <= 2.0 ** -22 * (m + d8 + want.abs())[far]).all()


@pytest.mark.parametrize("kind,tile,m,n,k,minima", [(*c, v) for c in EVERY_TILE
                                                    for v in ("zero_point", "free")
                                                    if c[0] == "q4" or v == "zero_point"])
def test_every_tile_onehot_exact(dev, kind, tile, m, n, k, minima):
    """One-hot rows on every tile (the K parts that do not hold the entry add zeros)."""
    assert _tile(kind, m, n, k) == tile
    raw, rng = _tiles(kind, n, k, 500 + m)
    if minima == "free":
        raw = _free_minima(raw, rng)
    x, cols = _onehot_rows(m, k, dev)
    y = ops.gemm(_dev_u8(raw, dev), kind, x, n // 32, k // 256)
    _onehot_check(y, raw, kind, n, k, cols, dev, tile[0])


@pytest.mark.parametrize("batch,n,k", [
    (65, 96, 1024),            # 32 x 1 pairs
    (200, 1312, 768),          # 32 x 2
    (300, 2080, 2816),         # 64 x 2 in two parts
    (900, 1984, 1280),         # 64 x 4
    (1000, 3616, 2304),        # 128 x 4 in two parts
])
def test_gate_up_onehot_exact(dev, batch, n, k):
    """The same for the gate and the up values of [gate, up]."""
    rng = np.random.default_rng(600 + batch)
    w = [synth.q4_tiles(rng, n, k).reshape(-1, qo.Q4_TILE_BYTES) for _ in range(2)]
    w[1] = _free_minima(w[1], rng)
    x, cols = _onehot_rows(batch, k, dev)
    raw_out = torch.empty((batch, 2 * n), device=dev)
    ops.gate_up_swiglu(_dev_u8(w[0], dev), _dev_u8(w[1], dev), n // 32, k // 256, x, raw_out=raw_out)
    for t, o in ((w[0], 0), (w[1], n)):
        _onehot_check(raw_out[:, o:o + n], t, "q4", n, k, cols, dev, 128 if batch == 1000 else 64)


@pytest.mark.parametrize("kind", ["q4", "q8"])
@pytest.mark.parametrize("m,n,k", [(65, 96, 1024), (70, 64, 2560), (300, 2080, 4096),
                                   (449, 2592, 4352), (1500, 2464, 512)])
def test_prompt_block_norm_prologue(dev, kind, m, n, k):
    """A projection with its RMSNorm in the pre-pass (4, 1 and 1 rows per workgroup of 256, 256 and
    512 threads) gives the bits of the projection of the rows that [RMSNorm, gate, up] normalises."""
    raw, rng = _tiles(kind, n, k, 700 + m)
    w = _dev_u8(raw, dev)
    x = torch.from_numpy((rng.standard_normal((m, k)) * 3).astype(np.float32)).to(dev)
    kw = dict(norm_w=_dev_bf16(synth.random_bf16(rng, k), dev),
              ssq_in=x.view(m, -1, 16).square().sum(-1).contiguous())
    xn = torch.zeros((m, k), dtype=torch.bfloat16, device=dev)
    gate = _dev_u8(synth.q4_tiles(rng, 32, k), dev)
    ops.gate_up_swiglu(gate, gate, 1, k // 256, x, xn_out=xn, **kw)
    y = ops.gemv_ex(w, kind, x, n // 32, k // 256, **kw)
    assert _tile(kind, m, n, k) is not None
    assert torch.equal(y, ops.gemm(w, kind, xn, n // 32, k // 256))
    xb = xn.view(torch.int16).cpu().numpy().view(np.uint16)
    rows = np.unique(np.concatenate([np.arange(0, m, max(1, m // 24)), [m - 1]]))
    _check_rows(y.cpu().numpy()[rows], qo.gemv(raw, kind, xb[rows], n // 32, k // 256, acc=np.float64))


@pytest.mark.parametrize("m,n,k,gateup", [
    (130, 26272, 2304, False),    # 64 x 4: 821 tile-rows, no multiple of eight tiles
    (300, 26272, 2304, False),    # 128 x 8
    (130, 13088, 2304, True),     # [gate, up]: 409 pairs
    (1030, 13088, 2304, True),
])
def test_q4_weights_beyond_the_l2(dev, m, n, k, gateup):
    """q4 weights of more than 32 MB: row blocks first within an XCD's share of the tiles."""
    g = torch.Generator(device=dev)
    g.manual_seed(m)
    from llmnputest_amd.granite import random_q4_tiles
    w = [random_q4_tiles(n, k, g, dev) for _ in range(1 + gateup)]
    assert sum(t.numel() for t in w) > 32 << 20
    x = torch.randn((m, k), device=dev, generator=g).to(torch.bfloat16)
    if gateup:
        y = torch.full((m, 2 * n), float("nan"), device=dev)
        ops.gate_up_swiglu(w[0], w[1], n // 32, k // 256, x, raw_out=y)
    else:
        y = ops.gemm(w[0], "q4", x, n // 32, k // 256)
    for i, t in enumerate(w):
        wm = ops.dequant(t, "q4", n // 32, k // 256, out_dtype=torch.float32, untile=True).double()
        ref = x.double() @ wm.t().contiguous()
        err = (y[:, i * n:(i + 1) * n].double() - ref).abs()
        assert (err <= REL * ref.abs().amax(1, keepdim=True)).all()

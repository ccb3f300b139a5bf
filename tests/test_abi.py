"""The C ABI without a GPU: the library loads, exports every function include/q4nx_hip.h
declares, rejects bad arguments with the documented codes (mirroring the reference's
CPU-forceable failures: wrong tile size, K not a multiple of 256, bad factoring), and its
host-side RoPE table equals the oracle's."""

import ctypes as C
import re
from pathlib import Path

import numpy as np
import pytest

from llmnputest_amd import _lib
from oracle import decode_oracle as do

HEADER = Path(__file__).resolve().parents[1] / "include" / "q4nx_hip.h"
ERR_ARG, ERR_SHAPE, ERR_WS = -1, -2, -3


def declared():
    text = re.sub(r"/\*.*?\*/", "", HEADER.read_text(), flags=re.S)
    return sorted(set(re.findall(r"\b(q4nx_\w+)\s*\(", text)))


def test_header_symbols_exported():
    h = C.CDLL(str(_lib.LIB_PATH))
    names = declared()
    assert len(names) >= 20
    missing = [n for n in names if not hasattr(h, n)]
    assert not missing, missing
    assert set(names) == set(_lib.SIGNATURES), set(names) ^ set(_lib.SIGNATURES)
    assert _lib.lib().q4nx_abi_version() == 2


def rc_msg(name, *args):
    rc = getattr(_lib.lib(), name)(*args)
    return rc, _lib.lib().q4nx_last_error().decode()


def pol(**kw):
    return C.byref(_lib.Policy(**kw))


def test_policy_defaults_and_validation():
    p = _lib.Policy()
    assert (p.mfma_rows_q4, p.mfma_rows_q8, p.rowblock, p.gemv_ksplit, p.gemv_tiles_per_wave,
            p.gemm_ksplit, p.attn_mfma) == (2, 2, 1, 0, 0, 0, 1)
    fake = C.c_void_p(0x10000)
    for bad in ({"gemv_ksplit": 9}, {"gemv_tiles_per_wave": 3}, {"gemm_ksplit": -1},
                {"attn_mfma": 2}, {"rowblock": 5}, {"mfma_rows_q4": -1}):
        rc, msg = rc_msg("q4nx_gemv_q4", fake, fake, fake, 8, 10, 1, 2560, 256, None, None, 0,
                         pol(**bad), None)
        assert rc == ERR_ARG and "policy" in msg, bad
        assert _lib.lib().q4nx_gemv_ws_bytes(4, 80, 32, 1, pol(**bad)) == 0   # queries: 0
        assert _lib.lib().q4nx_gqa_decode_splits(1, 40, 8, 2048, pol(**bad)) == 0


def test_gemv_argument_errors():
    fake = C.c_void_p(0x10000)       # aligned, never dereferenced: validation fails first
    rc, msg = rc_msg("q4nx_gemv_q4", None, fake, fake, 8, 10, 1, 2560, 256, None, None, 0, None,
                     None)
    assert rc == ERR_ARG and "weights" in msg
    rc, msg = rc_msg("q4nx_gemv_q4", C.c_void_p(0x10001), fake, fake, 8, 10, 1, 2560, 256,
                     None, None, 0, None, None)
    assert rc == ERR_ARG                                   # misaligned tiles
    rc, msg = rc_msg("q4nx_gemv_q4", fake, fake, fake, 0, 10, 1, 2560, 256, None, None, 0, None,
                     None)
    assert rc == ERR_SHAPE and "n_tile_rows" in msg
    rc, msg = rc_msg("q4nx_gemv_q8", fake, fake, fake, 8, 4, 9, 1024, 256, None, None, 0,
                     pol(mfma_rows_q8=0), None)                 # VALU kernel only: batch <= 8
    assert rc == ERR_SHAPE and "batch" in msg
    rc, msg = rc_msg("q4nx_gemv_q4", fake, fake, fake, 8, 10, 1, 2000, 256, None, None, 0, None,
                     None)
    assert rc == ERR_SHAPE and "x_stride" in msg           # K = 2560 does not fit a 2000 row
    rc, msg = rc_msg("q4nx_gemv_ex", 5, fake, 8, 10, fake, 2560, None, C.c_float(1e-5), None, 1,
                     fake, 256, None, None, None, None, 0, None, None)
    assert rc == ERR_ARG and "kind" in msg
    rc, msg = rc_msg("q4nx_gemv_ex", 4, fake, 8, 10, fake, 2560, None, C.c_float(1e-5), fake, 1,
                     fake, 256, None, None, None, None, 0, None, None)
    assert rc == ERR_ARG and "ssq_in" in msg               # partial sums without a norm


def test_floor_and_tiles_per_wave_errors():
    """The weight-stream floors validate as the GEMV does; a K-tiles-per-wave request that
    would need more than 16 waves in a row-block workgroup is refused before any launch."""
    fake = C.c_void_p(0x10000)
    rc, msg = rc_msg("q4nx_gemv_q4_null", None, fake, fake, 8, 10, None)
    assert rc == ERR_ARG and "w must" in msg
    rc, msg = rc_msg("q4nx_gemv_q4_null", fake, fake, fake, 8, 65, None)
    assert rc == ERR_SHAPE and "k_tiles" in msg
    rc, msg = rc_msg("q4nx_gemv_q4_null", fake, fake, fake, 0, 10, None)
    assert rc == ERR_SHAPE and "n_tile_rows" in msg
    rc, msg = rc_msg("q4nx_stream_read", fake, 24, fake, None)
    assert rc == ERR_SHAPE and "multiple of 16" in msg
    rc, msg = rc_msg("q4nx_stream_read", C.c_void_p(0x10008), 32, fake, None)
    assert rc == ERR_ARG
    # K = 8192 (32 K-tiles) at one K-tile per wave would need 32 waves
    rc, msg = rc_msg("q4nx_gemv_q4", fake, fake, fake, 80, 32, 1, 8192, 2560, None, None, 0,
                     pol(gemv_tiles_per_wave=1), None)
    assert rc == ERR_ARG and "16 waves" in msg


def test_fused_and_attention_argument_errors():
    fake = C.c_void_p(0x10000)
    rc, msg = rc_msg("q4nx_qkv_rope", fake, fake, fake, 40, 7, 10, fake, 2560, None,
                     C.c_float(1e-5), None, 1, fake, fake, 512, fake, fake, fake, 8 * 512 * 64,
                     512 * 64, None, None, None, 0, None, None)
    assert rc == ERR_SHAPE and "n_kv_heads" in msg         # 40 % 7 != 0
    rc, msg = rc_msg("q4nx_gqa_decode", fake, fake, fake, fake, None, 1, 40, 8, 128, fake, 512,
                     8 * 512 * 64, 512 * 64, C.c_float(0.125), 0, None, 0, None, None)
    assert rc == ERR_SHAPE and "head_dim" in msg
    rc, msg = rc_msg("q4nx_gqa_decode", fake, fake, fake, fake, None, 1, 40, 8, 64, fake, 4096,
                     8 * 4096 * 64, 4096 * 64, C.c_float(0.125), 8, None, 0, None, None)
    assert rc == ERR_WS and "workspace" in msg
    rc, msg = rc_msg("q4nx_embed", 8, fake, fake, fake, None, 100, 2560, 1, None)
    assert rc == ERR_SHAPE                                 # q8 tiles: vocab not a multiple of 32
    rc, msg = rc_msg("q4nx_embed", 16, fake, fake, fake, None, 100, 2500, 1, None)
    assert rc == ERR_SHAPE                                 # hidden not a multiple of 256
    rc, msg = rc_msg("q4nx_embed", 5, fake, fake, fake, None, 128, 2560, 1, None)
    assert rc == ERR_ARG and "kind" in msg
    rc, msg = rc_msg("q4nx_dequant_q4", fake, None, 1, 1, 0, 0, None)
    assert rc == ERR_ARG
    rc, msg = rc_msg("q4nx_decode_advance_embed", fake, 64, fake, fake, fake, None, fake, 0, 65,
                     8, fake, 1024, 512, fake, None, None)
    assert rc == ERR_SHAPE and "batch" in msg              # at most 64 sequences
    rc, msg = rc_msg("q4nx_decode_advance_embed", fake, 64, fake, fake, fake, None, fake, 0, 1,
                     8, fake, 1000, 512, fake, None, None)
    assert rc == ERR_SHAPE                                 # q8 tiles: vocab not a multiple of 32
    rc, msg = rc_msg("q4nx_decode_advance_embed", fake, 64, fake, fake, fake, None, fake, 0, 1,
                     8, None, 1024, 512, fake, None, None)
    assert rc == ERR_ARG and "table" in msg


def test_attention_record_splits_and_errors():
    """Split policies (host-only queries) and the argument checks of the attention records and
    the o-projection that merges them, which all return before any launch."""
    lib = _lib.lib()
    fake = C.c_void_p(0x10000)
    for lmax, auto in ((640, 5), (2176, 9), (4160, 16)):   # the 3B decode shapes
        assert lib.q4nx_gqa_decode_splits(1, 40, 8, lmax, None) == auto
        assert lib.q4nx_gqa_decode_records_splits(1, 40, 8, lmax, None) == min(auto, 12)
    assert lib.q4nx_gqa_decode_splits(1, 40, 8, 32768, None) == 32
    valu = pol(attn_mfma=0)                                  # VALU policy: up to 64 splits
    assert lib.q4nx_gqa_decode_splits(1, 40, 8, 32768, valu) == 64
    assert lib.q4nx_gqa_decode_records_splits(1, 40, 8, 32768, valu) == 12
    assert lib.q4nx_gqa_decode_splits(1, 40, 8, 0, None) == 0       # invalid shapes: 0
    assert lib.q4nx_gqa_decode_records_splits(0, 40, 8, 64, None) == 0
    rc, msg = rc_msg("q4nx_gqa_decode_records", fake, fake, fake, 1, 40, 8, 64, fake, 512,
                     8 * 512 * 64, 512 * 64, C.c_float(0.125), 0, fake, 1 << 20, None, None)
    assert rc == ERR_ARG and "n_split" in msg               # the count must be given
    rc, msg = rc_msg("q4nx_gqa_decode_records", fake, fake, fake, 1, 40, 8, 64, fake, 512,
                     8 * 512 * 64, 512 * 64, C.c_float(0.125), 4, fake, 4096, None, None)
    assert rc == ERR_WS and "workspace" in msg              # 4 splits need 64 KB + 43,520 B
    rc, msg = rc_msg("q4nx_gemv_attn_q4", fake, 80, fake, 10, 44, 4, fake, None, None, None)
    assert rc == ERR_SHAPE and "query heads" in msg         # 11 K-tiles
    rc, msg = rc_msg("q4nx_gemv_attn_q4", fake, 80, fake, 10, 40, 7, fake, None, None, None)
    assert rc == ERR_SHAPE                                   # 40 % 7 != 0
    rc, msg = rc_msg("q4nx_gemv_attn_q4", fake, 80, fake, 19, 40, 8, fake, None, None, None)
    assert rc == ERR_SHAPE and "n_split" in msg             # more than the merge holds
    rc, msg = rc_msg("q4nx_gemv_attn_q4", fake, 80, C.c_void_p(0x10008), 10, 40, 8, fake, None,
                     None, None)
    assert rc == ERR_ARG and "16-byte" in msg               # misaligned records


def test_policies_are_per_call():
    """Two policies used side by side, also from racing threads (ctypes drops the GIL in the
    call), each get their own answer: the library keeps no setting between calls."""
    import threading
    lib = _lib.lib()
    pm, pv = _lib.Policy(), _lib.Policy(attn_mfma=0)
    bad = []

    def worker(i):
        for n in range(2000):
            p = pm if (i + n) % 2 else pv
            want = 32 if p is pm else 64
            if lib.q4nx_gqa_decode_splits(1, 40, 8, 32768, C.byref(p)) != want:
                bad.append((i, n))
            ws = lib.q4nx_gemv_ws_bytes(4, 80, 32, 1, C.byref(p))
            if ws != 0:                       # one row of q4 on the row-block kernels
                bad.append(("ws", ws))

    threads = [threading.Thread(target=worker, args=(i,)) for i in range(8)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad, bad[:5]
    # the general VALU kernel's split needs a workspace; the row-block one does not
    assert lib.q4nx_gemv_ws_bytes(4, 80, 32, 1, pol(rowblock=0)) == 65536 + 80 * 3 * 32 * 4
    assert lib.q4nx_gemv_ws_bytes(4, 80, 32, 1, None) == 0


def test_gemm_argument_errors():
    fake = C.c_void_p(0x10000)
    rc, msg = rc_msg("q4nx_gemm", 3, fake, 8, 10, fake, 2560, 4, fake, 256, None, None, 0, None,
                     None)
    assert rc == ERR_ARG and "kind" in msg
    rc, msg = rc_msg("q4nx_gemm", 4, fake, 8, 10, fake, 2560, 0, fake, 256, None, None, 0, None,
                     None)
    assert rc == ERR_SHAPE and "m_rows" in msg
    rc, msg = rc_msg("q4nx_gemm", 4, fake, 8, 10, fake, 2564, 4, fake, 256, None, None, 0, None,
                     None)
    assert rc == ERR_SHAPE and "x_stride" in msg            # not a multiple of 8
    rc, msg = rc_msg("q4nx_gemm", 4, fake, 8, 10, fake, 2560, 4, fake, 128, None, None, 0, None,
                     None)
    assert rc == ERR_SHAPE and "y_stride" in msg            # N = 256 does not fit
    rc, msg = rc_msg("q4nx_gemm", 8, fake, 8, 10, fake, 2560, 4, C.c_void_p(0x10004), 256,
                     None, None, 0, None, None)
    assert rc == ERR_ARG and "y" in msg                     # misaligned output
    rc, msg = rc_msg("q4nx_gemm", 4, fake, 8, 10, fake, 2560, 4, fake, 256, None, None, 0,
                     pol(gemm_ksplit=9), None)
    assert rc == ERR_ARG and "policy" in msg


def test_ws_queries():
    lib = _lib.lib()
    general = pol(rowblock=0)
    # 80 tile-rows do not fill the GPU: the general VALU kernel splits K 3 ways, partials
    # [80][3][1][32] fp32; the row-block kernels (the default at one row) need nothing
    assert lib.q4nx_gemv_ws_bytes(4, 80, 32, 1, general) == 65536 + 80 * 3 * 32 * 4
    assert lib.q4nx_gemv_ws_bytes(4, 80, 32, 1, None) == 0
    assert lib.q4nx_gemv_ws_bytes(4, 256, 10, 1, general) == 0   # enough tile-rows: no split
    # batch 9 runs on the matrix cores: no split, room for 9 normalised rows
    assert lib.q4nx_gemv_ws_bytes(4, 256, 10, 9, None) == 65536 + 9 * 2560 * 2
    # 56 heads of 2 tile-rows, batch 2 on the VALU kernel: 5 parts of 2 K-tiles,
    # [56][5][batch 2][64]; on the matrix cores (the default from 2 rows) the heads run whole
    # on 112 row-block workgroups: no split records, room for the normalised rows of 2560
    # bf16. Up to 8 rows the query also sizes for the VALU kernel, whose records are larger.
    assert lib.q4nx_qkv_rope_ws_bytes(40, 8, 10, 2, pol(mfma_rows_q4=0)) == 65536 + 56 * 5 * 2 * 64 * 4
    assert lib.q4nx_qkv_rope_ws_bytes(40, 8, 10, 2, None) == 65536 + 56 * 5 * 2 * 64 * 4
    assert lib.q4nx_qkv_rope_ws_bytes(40, 8, 10, 12, None) == 65536 + 12 * 2560 * 2
    assert lib.q4nx_qkv_rope_ws_bytes(40, 8, 10, 1, None) == 0     # one row: row-block kernel
    # q8 lm_head at one row: the row-block kernel (the default) needs nothing; on the matrix
    # cores 3136 workgroups, no split, one normalised row
    assert lib.q4nx_gemv_ws_bytes(8, 3136, 10, 1, None) == 0
    assert lib.q4nx_gemv_ws_bytes(8, 3136, 10, 1, pol(mfma_rows_q8=1)) == 65536 + 2560 * 2
    assert lib.q4nx_gate_up_ws_bytes(256, 10, 1, None) == 0
    assert lib.q4nx_gqa_decode_ws_bytes(1, 40, 8, 64, None) == 0  # one split: no workspace
    big = lib.q4nx_gqa_decode_ws_bytes(1, 40, 8, 32768, pol(attn_mfma=0))   # 64 splits
    assert big == 65536 + 8 * 64 * 5 * 68 * 4
    # batched contraction: 80 tile-rows x 1 block of 16 rows, one tile-row per workgroup of
    # up to 16 waves: 32 K-tiles in 2 parts
    assert lib.q4nx_gemm_ws_bytes(4, 80, 32, 8, None) == 65536 + 80 * 2 * 16 * 32 * 4
    assert lib.q4nx_gemm_ws_bytes(4, 256, 10, 8, None) == 0      # 256 workgroups: no split
    # 512 rows: 40 pairs of tile-rows x 4 blocks of 128 rows, split 2 ways
    assert lib.q4nx_gemm_ws_bytes(4, 80, 32, 512, None) == 65536 + 160 * 2 * 128 * 64 * 4
    assert lib.q4nx_gemm_ws_bytes(5, 80, 32, 8, None) == 0


@pytest.mark.parametrize("max_pos,theta", [(4096, 10000.0), (64, 500000.0)])
def test_rope_table_host(max_pos, theta):
    tab = np.empty((max_pos, 2, 32), np.float32)
    _lib.call("q4nx_rope_table_host", tab.ctypes.data, max_pos, 64, C.c_double(theta))
    ref = do.rope_table(max_pos, 64, theta)
    assert np.abs(tab - ref).max() <= 6e-8
    assert np.array_equal(tab[0, 0], np.ones(32, np.float32)) and not tab[0, 1].any()


def test_rope_table_host_closed_forms():
    """The C table's frequencies pinned by closed forms, independent of the oracle:
    pair i turns by pos * theta^(-2i/64), i.e. pos/10, pos/100, pos/1000 for i = 8, 16, 24
    at theta = 10^4 and pos/1000 for i = 16 at theta = 10^6."""
    from tests.pins import check_rope_frequencies

    def c_table(max_pos, hd, theta):
        tab = np.empty((max_pos, 2, hd // 2), np.float32)
        _lib.call("q4nx_rope_table_host", tab.ctypes.data, max_pos, hd, C.c_double(theta))
        return tab
    check_rope_frequencies(c_table)


def test_prompt_workspace_queries_ask_for_what_is_used():
    """Prompt blocks that the batched kernel takes (a named K split, a short K) ask for its own
    workspace only; gemm_ksplit=1 and projections that fill the chip ask as by default."""
    f, g = _lib.lib().q4nx_gemm_ws_bytes, _lib.lib().q4nx_gemm_prompt_ws_bytes
    q4, q8 = 4, 8
    full = f(q4, 256, 10, 2048, None)
    assert full == g(q4, 256, 10, 2048) > 10 << 20
    for parts in (1, 2, 8):
        assert f(q4, 256, 10, 2048, pol(gemm_ksplit=parts)) >= full
    assert f(q4, 80, 10, 100, pol(gemm_ksplit=1)) == g(q4, 80, 10, 100) > 0
    # 80 groups of one row block in two parts: counters and 2 x 128 x 32 floats each, no more
    assert f(q4, 80, 10, 100, pol(gemm_ksplit=2)) <= 65536 + 80 * 2 * 128 * 64 * 4
    assert g(q8, 16, 2, 1000) == 0 and f(q8, 16, 2, 1000, None) == 0
    assert g(q4, 64, 2, 96) == 0 and g(q4, 64, 2, 97) > 0
    # K <= 512 stays on the batched kernel up to a number of its workgroups, not of rows alone
    assert g(q4, 512, 2, 96) == 0 and g(q4, 3136, 2, 96) > 0 and g(q4, 3136, 2, 65) > 0
    assert g(q4, 256, 1, 256) == 0 and g(q4, 512, 1, 300) > 0 and g(q4, 32, 1, 6000) == 0
    assert g(q8, 128, 1, 512) == 0 and g(q8, 128, 1, 513) > 0
    t = _lib.lib().q4nx_gemm_prompt_tile
    assert t(q4, 80, 32, 333) == 64 << 16 | 2 << 8 | 4 and t(q4, 80, 32, 64) == 0
    assert t(q8, 7760, 4, 512) == 128 << 16 | 4 << 8 | 1 and t(3, 80, 32, 333) == 0
    # [gate, up] under a named split is the batched kernel's: its normalised rows alone
    h = _lib.lib().q4nx_gate_up_ws_bytes
    assert h(256, 10, 500, pol(gemm_ksplit=1)) == 65536 + 500 * 2560 * 2 < h(256, 10, 500, None)

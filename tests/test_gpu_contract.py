# SPDX-License-Identifier: Apache-2.0
"""GPU tests of the boundary contract and the drop-in.

- BF16 matrices (bf16_n, src/10_compute/dsv4_matmul.c:88-113) and FP8 rows
  of 8192 bytes (wo_b, src/00_base/dsv4_weights.h:68) run through the C ABI
  against the oracle and the reference's own golden outputs.
- A host-pointer call returns 0 only when the GPU produced the whole result:
  a kernel that meets a value its arithmetic cannot carry raises a status bit
  and the call returns -1 (the reference's GPU convention,
  src/80_prefill/dsv4_prefill_vk.h:37-41), and the next good call returns 0.
- The many-token seam scales each activation row by a power of two before
  its fp16 MFMA, so huge and tiny rows keep the 1e-3 contract row by row.
- The reference-named library (libdsv4_amd.so) runs one decode layer's matrix
  sequence (src/70_decode/dsv4_layer_attn.c:21-106, dsv4_layer.c:52) at real
  shapes with E8M0 FP8, BF16 and FP4 weights.
- The grouped MoE's permutation matches the reference's counting sort
  (src/80_prefill/dsv4_prefill_union.c:30-51) index for index."""
import numpy as np
import pytest
import torch

import pyoracle as P
from conftest import REL_L2_TOL, bits, golden, max_abs, rel_l2
from test_gpu_decode import DEV, Resident, check_close

pytestmark = pytest.mark.gpu


def bf16_bits(a):
    """fp32 -> bf16 bits, round to nearest even."""
    u = np.ascontiguousarray(a, np.float32).view(np.uint32).astype(np.uint64)
    return ((u + 0x7FFF + ((u >> 16) & 1)) >> 16).astype(np.uint16)


class ResidentBf16:
    """A BF16 matrix registered with the library: weights only, s = NULL."""

    def __init__(self, lib, pkg, W, rows, cols):
        self.W = np.ascontiguousarray(W, np.uint16)
        lib.check(lib.register(self.W), "register")
        self.lib = lib
        self.desc = pkg.qmat(pkg.DSV4_WBF16, self.W.ctypes.data, None, rows, cols, 0, 0)
        self.hm = P.HostMat(pkg.DSV4_WBF16, self.W, None, rows, cols, 0, 0)

    def drop(self):
        self.lib.unregister(self.W)


def check_bf16(got, want):
    """bf16_n's fp64 sums in bf16_n's order and its one final rounding: bit
    for bit the reference's result (a sum beyond the fp32 range is inf in
    both; NaN where the reference has NaN)."""
    got, want = np.asarray(got, np.float32), np.asarray(want, np.float32)
    nan = np.isnan(want)
    assert np.array_equal(np.isnan(got), nan)
    diff = np.nonzero(bits(got[~nan]) != bits(want[~nan]))[0]
    assert diff.size == 0, f"{diff.size} of {want.size} differ, first at {diff[0]}: " \
        f"{got[~nan][diff[0]]!r} vs {want[~nan][diff[0]]!r}"


def e4m3_codes(rng, n):
    b = rng.integers(0, 256, n).astype(np.uint8)
    b[(b & 0x7F) == 0x7F] &= 0xFE          # no NaN codes
    return b


# ---------------------------------------------------------------- BF16 ----

def test_bf16_golden_through_abi(lib, pkg):
    g = golden("bf16")
    rows, cols, nt = (int(v) for v in g["dims"])
    m = ResidentBf16(lib, pkg, g["W"], rows, cols)
    got = lib.mmq_n(m.desc, g["x"], nt)
    check_bf16(got, g["y"])
    m.drop()


@pytest.mark.parametrize("rows,cols,nt", [
    (256, 4096, 1),      # router gate (src/70_decode/dsv4_layer.c:52)
    (1024, 4096, 2),     # compressor wkv / wgate
    (64, 4096, 1),       # indexer weights_proj
    (512, 4096, 40),     # a prefill block of 40 tokens
    (1000, 8192, 1),     # 16 KiB rows
    (33, 136, 3),        # ragged: rows not a multiple of the wave's, 136 columns
])
def test_bf16_gemv_shapes(lib, pkg, oracle, rows, cols, nt):
    rng = np.random.default_rng(rows * 7 + cols + nt)
    W = bf16_bits(rng.standard_normal(rows * cols).astype(np.float32) * 0.02)
    x = rng.standard_normal(nt * cols).astype(np.float32)
    m = ResidentBf16(lib, pkg, W, rows, cols)
    got = lib.mmq_n(m.desc, x, nt)
    check_bf16(got, oracle.bf16_n(W, x, rows, cols, nt))
    m.drop()


@pytest.mark.parametrize("rows,cols,nt", [(7, 8, 3), (64, 4104, 3), (96, 72, 5)])
def test_bf16_gemv_special_values(lib, pkg, oracle, rows, cols, nt):
    """Sums that overflow to +-inf, inf times zero and NaN inputs, tail
    columns past the last 16-column group, 8 columns: the fp64 chains in
    bf16_n's order give the reference's inf, NaN and finite bits."""
    rng = np.random.default_rng(rows + cols * 3 + nt)
    Wf = rng.standard_normal(rows * cols).astype(np.float32)
    Wf[::11] *= 1e36
    Wf[5] = 0.0
    W = bf16_bits(Wf)
    x = rng.standard_normal(nt * cols).astype(np.float32) * 1e3
    x[3] = np.inf                  # token 0
    x[cols + 1] = np.nan           # token 1
    x[-1] = -3e38                  # the last token
    m = ResidentBf16(lib, pkg, W, rows, cols)
    got = lib.mmq_n(m.desc, x, nt)
    want = oracle.bf16_n(W, x, rows, cols, nt)
    assert np.isinf(want).any() and np.isnan(want).any() and np.isfinite(want).any()
    check_bf16(got, want)
    m.drop()


@pytest.mark.parametrize("rows,cols,nt", [
    (9215, 72, 1), (9216, 1032, 1), (9223, 4096, 1),      # the rows form from 9216 rows, one token
    (12287, 136, 3), (12301, 1096, 4), (12288, 24, 2),    # and from 12288 for two to four
    (5, 4104, 4), (6, 8192, 5), (30, 8184, 8), (4, 16, 1),      # small form: one and two parts of columns
    (2048, 264, 4), (2052, 264, 4), (1021, 264, 8),       # small form's and GEMM's sides of the three rounds
    (17, 4104, 529), (3100, 264, 9), (3073, 520, 17), (3085, 8, 32),
    (2049, 72, 1), (2050, 512, 1), (2051, 520, 1), (4099, 1024, 1), (3075, 1032, 1), (3073, 2048, 1),   # a wave per four rows
    (5121, 136, 2), (5122, 1016, 2), (3077, 16, 1),
    (65537, 136, 2), (65541, 272, 3), (65536, 1016, 4), (65539, 8, 1), (14337, 520, 2),   # rows form, four steps in flight
    (4097, 80, 3), (12290, 1024, 2), (33, 504, 3), (34, 1032, 2)])                # and eight; small form of short rows
def test_bf16_forms(lib, pkg, oracle, rows, cols, nt):
    """Each form of the BF16 matvec at its edges: rows and tokens past the
    last tile, one to three 16-column groups past the last 64, trailing 8
    columns, no whole group; bit for bit bf16_n."""
    rng = np.random.default_rng(rows * 11 + cols * 3 + nt)
    W = bf16_bits(rng.standard_normal(rows * cols).astype(np.float32) * np.float32(0.02))
    x = rng.standard_normal(nt * cols).astype(np.float32)
    x[::7] *= np.float32(2.0 ** 40)        # products far apart, so that the order of the sums shows
    x[::11] *= np.float32(2.0 ** -40)
    m = ResidentBf16(lib, pkg, W, rows, cols)
    check_bf16(lib.mmq_n(m.desc, x, nt), oracle.bf16_n(W, x, rows, cols, nt))
    m.drop()


# ------------------------------------------------------- wide FP8 rows ----

@pytest.mark.parametrize("rows,nt", [(4096, 1), (1024, 1), (512, 3), (512, 40)])
def test_fp8_e8m0_8192_wide_rows(lib, pkg, oracle, rows, nt):
    """wo_b: FP8 [4096 x 8192] with E8M0 128x128 scales; nt = 1 takes the
    chunk-pair matvec (two or one 8-row tiles per workgroup), nt = 3 the
    block-scaled MFMA GEMV with 16 chunks per wave, 40 the fp16 seam."""
    cols = 8192
    rng = np.random.default_rng(rows + nt)
    W = e4m3_codes(rng, rows * cols)
    S = rng.integers(112, 121, (rows // 128) * (cols // 128)).astype(np.uint8)
    x = rng.standard_normal(nt * cols).astype(np.float32)
    m = Resident(lib, pkg, pkg.DSV4_WFP8, W, S, rows, cols, 128, 128)
    check_close(lib.mmq_n(m.desc, x, nt), oracle.fp8_n(W, S, x, rows, cols, 128, 128, nt))
    m.drop()


@pytest.mark.parametrize("nt", [1, 2])
def test_fp4_16384_wide_rows(lib, pkg, oracle, nt):
    rows, cols = 96, 16384
    rng = np.random.default_rng(nt)
    W = rng.integers(0, 256, rows * cols // 2).astype(np.uint8)
    S = rng.integers(118, 128, rows * cols // 32).astype(np.uint8)
    x = rng.standard_normal(nt * cols).astype(np.float32)
    m = Resident(lib, pkg, pkg.DSV4_WFP4, W, S, rows, cols, 1, 32)
    check_close(lib.mmq_n(m.desc, x, nt), oracle.fp4_n(W, S, x, rows, cols, 1, 32, nt))
    m.drop()


@pytest.mark.parametrize("nt", [1, 3])
def test_wider_rows_take_the_generic_matvec(lib, pkg, oracle, nt):
    """FP8 rows of 8,320 bytes (beyond the fast kernels' 8 KiB) run on the
    generic matvec, against the oracle."""
    rows, cols = 48, 8320
    rng = np.random.default_rng(8320 + nt)
    W = e4m3_codes(rng, rows * cols)
    S = rng.integers(112, 121, (rows // 128 + 1) * (cols // 128)).astype(np.uint8)
    x = rng.standard_normal(nt * cols).astype(np.float32)
    m = Resident(lib, pkg, pkg.DSV4_WFP8, W, S, rows, cols, 128, 128)
    check_close(lib.mmq_n(m.desc, x, nt), oracle.fp8_n(W, S, x, rows, cols, 128, 128, nt))
    m.drop()


def test_wider_bf16_rows_decline(lib, pkg):
    rows, cols = 4, 8200
    W = np.zeros(rows * cols, np.uint16)
    d = pkg.qmat(pkg.DSV4_WBF16, W.ctypes.data, None, rows, cols, 0, 0)
    assert lib.mmq_n_rc(d, np.zeros(cols, np.float32)) == -1
    assert "16384" in lib.error()


@pytest.mark.parametrize("fmt,rows,cols,blk_r,blk_c,nt", [
    ("fp8", 40, 300, 1, 64, 1),        # per-row scales, ragged last block
    ("fp8", 37, 1000, 3, 100, 3),      # three-row scale blocks, rows not a multiple
    ("fp8f", 130, 512, 128, 64, 2),    # fp32 scales, 64-wide blocks
    ("fp4", 33, 200, 2, 16, 2),        # 16-wide FP4 blocks
    ("fp4", 20, 4096, 1, 64, 1),       # 64-wide FP4 blocks
    ("fp4", 9, 34, 4, 30, 4),          # blocks that start on odd columns
])
def test_generic_geometry_shapes(lib, pkg, oracle, fmt, rows, cols, blk_r, blk_c, nt):
    """Block geometries the fast kernels do not take (the reference's generic
    bodies) through the drop-in, host and device entry points, against the
    oracle's generic bodies."""
    rng = np.random.default_rng(rows * 31 + cols + blk_c)
    nsc = ((rows + blk_r - 1) // blk_r) * ((cols + blk_c - 1) // blk_c)
    if fmt == "fp4":
        W = rng.integers(0, 256, rows * cols // 2).astype(np.uint8)
        S = rng.integers(120, 133, nsc).astype(np.uint8)
        wdt = pkg.DSV4_WFP4
        want_of = lambda x: oracle.fp4_n(W, S, x, rows, cols, blk_r, blk_c, nt)
    elif fmt == "fp8":
        W = e4m3_codes(rng, rows * cols)
        S = rng.integers(112, 121, nsc).astype(np.uint8)
        wdt = pkg.DSV4_WFP8
        want_of = lambda x: oracle.fp8_n(W, S, x, rows, cols, blk_r, blk_c, nt)
    else:
        W = e4m3_codes(rng, rows * cols)
        S = (rng.random(nsc) * 0.01 + 1e-3).astype(np.float32)
        wdt = pkg.DSV4_WFP8_F32S
        want_of = lambda x: oracle.fp8f_n(W, S, x, rows, cols, blk_r, blk_c, nt)
    x = rng.standard_normal(nt * cols).astype(np.float32)
    m = Resident(lib, pkg, wdt, W, S, rows, cols, blk_r, blk_c)
    want = want_of(x)
    check_close(lib.mmq_n(m.desc, x, nt), want)
    # the device entry point on device copies
    dW = torch.from_numpy(W).to(DEV)
    dS = torch.from_numpy(S.view(np.uint8)).to(DEV)
    dx = torch.from_numpy(x).to(DEV)
    dy = torch.full((nt * rows,), float("nan"), device=DEV)
    dd = pkg.qmat(wdt, dW.data_ptr(), dS.data_ptr(), rows, cols, blk_r, blk_c)
    lib.mmq_n_dev(dy.data_ptr(), dx.data_ptr(), dd, nt)
    torch.cuda.synchronize()
    got = dy.cpu().numpy()
    check_close(got, want)
    assert np.array_equal(bits(got), bits(lib.mmq_n(m.desc, x, nt)))
    m.drop()


# ------------------------------------------------- MFMA GEMV token groups ----

@pytest.mark.parametrize("nt", [8, 16, 31])
@pytest.mark.parametrize("fmt", ["fp4", "fp8", "fp8f"])
def test_mmq_n_token_groups(lib, pkg, oracle, nt, fmt):
    """8..31 tokens: the block-scaled MFMA GEMV in groups of up to four
    tokens per MFMA (the last group partial)."""
    rows, cols = 384, 4096
    rng = np.random.default_rng(nt * 3 + len(fmt))
    w = (rng.standard_normal((rows, cols)) * 0.02).astype(np.float32)
    x = rng.standard_normal(nt * cols).astype(np.float32)
    if fmt == "fp4":
        W, S = oracle.quant_fp4_mx(w)
        m = Resident(lib, pkg, pkg.DSV4_WFP4, W, S, rows, cols, 1, 32)
        want = oracle.fp4_n(W, S, x, rows, cols, 1, 32, nt)
    elif fmt == "fp8":
        W = e4m3_codes(rng, rows * cols)
        S = rng.integers(112, 121, (rows // 128) * (cols // 128)).astype(np.uint8)
        m = Resident(lib, pkg, pkg.DSV4_WFP8, W, S, rows, cols, 128, 128)
        want = oracle.fp8_n(W, S, x, rows, cols, 128, 128, nt)
    else:
        W, S = oracle.quant_fp8_blk128(w)
        m = Resident(lib, pkg, pkg.DSV4_WFP8_F32S, W, S, rows, cols, 128, 128)
        want = oracle.fp8f_n(W, S, x, rows, cols, 128, 128, nt)
    check_close(lib.mmq_n(m.desc, x, nt), want)
    m.drop()


@pytest.mark.parametrize("fmt,rows,cols,nt", [
    ("fp8", 200, 1024, 7),      # rows past the last whole 16-row tile; one token group per workgroup
    ("fp8f", 4096, 2048, 29),   # 256 row blocks: 8 groups walked four per workgroup, the last of one token
    ("fp8", 2048, 4096, 27),    # 128 row blocks: 14 two-token groups in parts of 4, 4, 4 and 2
    ("fp4", 72, 8192, 13),      # five row blocks, one-token groups: one group per workgroup
])
def test_mmq_n_presplit_shapes(lib, pkg, oracle, fmt, rows, cols, nt):
    """From five tokens the MFMA GEMV splits x once and walks the token
    groups with the weights held: ragged rows, many and few row blocks,
    against the oracle, and bit for bit the same per token as the same
    tokens in calls of two to four tokens, which split x inside the matvec
    (a token's MFMA steps do not depend on the other tokens)."""
    rng = np.random.default_rng(rows + cols + nt)
    w = (rng.standard_normal((rows, cols)) * 0.02).astype(np.float32)
    x = rng.standard_normal(nt * cols).astype(np.float32)
    if fmt == "fp4":
        W, S = oracle.quant_fp4_mx(w)
        m = Resident(lib, pkg, pkg.DSV4_WFP4, W, S, rows, cols, 1, 32)
        want = oracle.fp4_n(W, S, x, rows, cols, 1, 32, nt)
    elif fmt == "fp8":
        W = e4m3_codes(rng, rows * cols)
        S = rng.integers(112, 121, ((rows + 127) // 128) * (cols // 128)).astype(np.uint8)
        m = Resident(lib, pkg, pkg.DSV4_WFP8, W, S, rows, cols, 128, 128)
        want = oracle.fp8_n(W, S, x, rows, cols, 128, 128, nt)
    else:
        W, S = oracle.quant_fp8_blk128(w)
        m = Resident(lib, pkg, pkg.DSV4_WFP8_F32S, W, S, rows, cols, 128, 128)
        want = oracle.fp8f_n(W, S, x, rows, cols, 128, 128, nt)
    got = lib.mmq_n(m.desc, x, nt)
    check_close(got, want)
    got = got.reshape(nt, rows)
    xs = x.reshape(nt, cols)
    sizes = [4] * (nt // 4) + ([nt % 4] if nt % 4 else [])
    if sizes[-1] == 1:                                     # one token would take the single-token matvec
        sizes[-2:] = [3, 2]
    t0 = 0
    for n in sizes:
        part = lib.mmq_n(m.desc, np.ascontiguousarray(xs[t0:t0 + n].reshape(-1)), n).reshape(n, rows)
        assert np.array_equal(bits(part), bits(got[t0:t0 + n])), f"tokens {t0}..{t0 + n - 1}"
        t0 += n
    m.drop()


@pytest.mark.parametrize("fmt,rows,cols,nt", [
    ("bf16", 5, 128, 1),             # 20 bytes out: no multiple of 16
    ("bf16", 1, 8, 3),
    ("fp8", 128, 4096, 256),         # x fills the host calls' staging exactly
    ("fp8", 128, 4096, 257),         # and no longer fits
    ("fp8", 4096, 128, 257),         # y no longer fits
])
def test_host_call_staging(lib, pkg, oracle, fmt, rows, cols, nt):
    """A host-pointer call's bits are the device-pointer call's, whatever part
    of its operands goes through the pinned staging."""
    rng = np.random.default_rng(rows + cols + nt)
    x = rng.standard_normal(nt * cols).astype(np.float32)
    if fmt == "bf16":
        W = (rng.standard_normal(rows * cols).astype(np.float32).view(np.uint32) >> 16).astype(np.uint16)
        m = ResidentBf16(lib, pkg, W, rows, cols)
        dS = None
    else:
        W, S = oracle.quant_fp8_blk128((rng.standard_normal((rows, cols)) * 0.02).astype(np.float32))
        m = Resident(lib, pkg, pkg.DSV4_WFP8_F32S, W, S, rows, cols, 128, 128)
        dS = torch.from_numpy(np.ascontiguousarray(S)).cuda()
    dW = torch.from_numpy(np.ascontiguousarray(W).view(np.uint8)).cuda()
    dx, dy = torch.from_numpy(x).cuda(), torch.empty(nt * rows, device="cuda")
    d = pkg.qmat(m.desc.wdt, dW.data_ptr(), dS.data_ptr() if dS is not None else None, rows, cols, m.desc.blk_r,
                 m.desc.blk_c)
    lib.mmq_n_dev(dy.data_ptr(), dx.data_ptr(), d, nt)
    torch.cuda.synchronize()
    for _ in range(2):
        got = lib.mmq_n(m.desc, x, nt)
        assert np.array_equal(bits(got).reshape(-1), bits(dy.cpu().numpy()))
    m.drop()


# ------------------------------------------------------ seam GEMM (FP8) ----

def _fp8_resident(lib, pkg, oracle, fmt, rng, rows, cols):
    if fmt == "fp8":
        W = e4m3_codes(rng, rows * cols)
        S = rng.integers(112, 121, (rows // 128) * (cols // 128)).astype(np.uint8)
        m = Resident(lib, pkg, pkg.DSV4_WFP8, W, S, rows, cols, 128, 128)
        return m, lambda x, nt: oracle.fp8_n(W, S, x, rows, cols, 128, 128, nt)
    w = (rng.standard_normal((rows, cols)) * 0.02).astype(np.float32)
    W, S = oracle.quant_fp8_blk128(w)
    m = Resident(lib, pkg, pkg.DSV4_WFP8_F32S, W, S, rows, cols, 128, 128)
    return m, lambda x, nt: oracle.fp8f_n(W, S, x, rows, cols, 128, 128, nt)


# matrices and token counts that take the seam GEMM, by the dispatch rule (test_choice.py asks it)
@pytest.mark.parametrize("rows,cols,nt", [
    (3200, 256, 1280),    # two reduction blocks, ten full token tiles, a 128-row feature tail
    (2432, 512, 1337),    # four blocks, a partial token tile and a feature tail
    (2560, 1280, 1700),   # ten blocks, whole feature tiles
])
@pytest.mark.parametrize("fmt", ["fp8", "fp8f"])
def test_seam_gemm_shapes(lib, pkg, oracle, rows, cols, nt, fmt):
    """Many tokens on FP8 weights: the GEMM-shaped seam kernel
    (128 x 256 tiles, fp16 tokens, weights decoded in registers) against the
    oracle, every token within 1e-3."""
    rng = np.random.default_rng(rows + cols + nt + len(fmt))
    m, want_of = _fp8_resident(lib, pkg, oracle, fmt, rng, rows, cols)
    x = rng.standard_normal(nt * cols).astype(np.float32)
    got = lib.mmq_n(m.desc, x, nt).reshape(nt, rows)
    want = want_of(x, nt).reshape(nt, rows)
    for t in range(nt):
        e = rel_l2(got[t], want[t])
        assert e <= REL_L2_TOL, f"token {t}: rel L2 {e:.3e}"
    m.drop()


@pytest.mark.parametrize("fmt", ["fp8", "fp8f"])
def test_seam_gemm_bits_equal_grouped_form(lib, pkg, oracle, fmt):
    """The seam kernel (1700 tokens of 2560 x 1280) and the dense tiles, which
    have the grouped kernel's order (1290 tokens of the same matrix), run the
    same MFMA steps and block promotions: every one of the first 1290 tokens'
    outputs is bit for bit the same in both, including rows beyond fp16 (|x|
    1e5) and below its normal range (1e-9)."""
    rows, cols, nt, few = 2560, 1280, 1700, 1290
    rng = np.random.default_rng(128 + len(fmt))
    m, _ = _fp8_resident(lib, pkg, oracle, fmt, rng, rows, cols)
    x = rng.standard_normal((nt, cols)).astype(np.float32)
    x[0] *= 1e5
    x[1] *= 1e-9
    x[2] = 0.0
    x = np.ascontiguousarray(x.reshape(-1))
    big = lib.mmq_n(m.desc, x, nt).reshape(nt, rows)
    small = lib.mmq_n(m.desc, np.ascontiguousarray(x[:few * cols]), few).reshape(few, rows)
    assert np.array_equal(bits(big[:few]), bits(small))
    m.drop()


@pytest.mark.parametrize("fmt", ["fp8", "fp8f"])
@pytest.mark.parametrize("rows,cols,tokens", [
    (2048, 128, (32, 33, 129, 257, 300, 513, 600, 1000, 1290, 4096)),     # every tile height, then 128 x 256
    (2176, 640, (32, 47, 300, 500, 700, 1290, 2050)),                      # rows no multiple of eight tiles, then a feature tail
    (4224, 384, (40, 500, 700, 1337)),                                     # three blocks, the tallest dense tiles, seam
    (1024, 8192, (33, 600)),                                               # the longest rows of the dense tiles
    (128, 8448, (40, 300, 1290)),                                          # past 8192 bytes: the generic matvec throughout
])
def test_seam_tile_sizes_same_bits(lib, pkg, oracle, rows, cols, tokens, fmt):
    """The forms of the FP8 seam give a token the same bits: the dense tiles of
    16 to 96 tokens and the 128 x 256 tiles."""
    rng = np.random.default_rng(rows + cols + len(fmt))
    m, want_of = _fp8_resident(lib, pkg, oracle, fmt, rng, rows, cols)
    x = rng.standard_normal((tokens[-1], cols)).astype(np.float32)
    x[0] *= 1e5
    x[1] *= 1e-9
    x[2] = 0.0
    x = np.ascontiguousarray(x)
    got = {n: lib.mmq_n(m.desc, np.ascontiguousarray(x[:n].reshape(-1)), n).reshape(n, rows) for n in tokens}
    want = want_of(np.ascontiguousarray(x[:17].reshape(-1)), 17).reshape(17, rows)
    for t in range(17):
        assert rel_l2(got[tokens[0]][t], want[t]) <= REL_L2_TOL, t
    for n, y in got.items():
        assert np.array_equal(bits(y), bits(got[tokens[-1]][:n])), n
    m.drop()


@pytest.mark.parametrize("fmt", ["fp8", "fp8f"])
def test_fp8_16_token_tiles_ring_depths(lib, pkg, oracle, fmt):
    """FP8 weights, 32 to a few hundred tokens: the dense tiles of 32 tokens
    (150 tokens x 4096 rows; a three-stage ring) and of 16 (the first 96 tokens
    alone; four stages). Against the oracle, and the shared tokens bit for bit
    the same in both."""
    rows, cols, nt, nt_small = 4096, 1024, 150, 96
    rng = np.random.default_rng(150 + len(fmt))
    m, want_of = _fp8_resident(lib, pkg, oracle, fmt, rng, rows, cols)
    x = rng.standard_normal(nt * cols).astype(np.float32)
    got = lib.mmq_n(m.desc, x, nt).reshape(nt, rows)
    want = want_of(x, nt).reshape(nt, rows)
    for t in range(nt):
        e = rel_l2(got[t], want[t])
        assert e <= REL_L2_TOL, f"token {t}: rel L2 {e:.3e}"
    small = lib.mmq_n(m.desc, np.ascontiguousarray(x[:nt_small * cols]), nt_small).reshape(nt_small, rows)
    assert np.array_equal(bits(small), bits(got[:nt_small]))
    m.drop()


# ------------------------------------------------ 0 means the whole result ----

def test_scale_byte_outside_fp16_range_returns_minus1(lib, pkg, oracle):
    """An FP4 scale byte of 150 cannot be decoded exactly into the fp16 seam
    (nt >= 32): the call returns -1 with the reason. The same matrix at nt =
    1 takes the block-scaled MFMA, which uses the byte as is: 0 and exact. A
    good call after the bad one returns 0."""
    rows, cols = 256, 512
    rng = np.random.default_rng(150)
    W = rng.integers(0, 256, rows * cols // 2).astype(np.uint8)
    S = rng.integers(120, 128, rows * cols // 32).astype(np.uint8)
    S[37] = 150
    m = Resident(lib, pkg, pkg.DSV4_WFP4, W, S, rows, cols, 1, 32)
    x = rng.standard_normal(64 * cols).astype(np.float32)
    assert lib.mmq_n_rc(m.desc, x, 64) == -1
    assert "104..140" in lib.error()
    check_close(lib.mmq_n(m.desc, x[:cols], 1), oracle.fp4_n(W, S, x[:cols], rows, cols, 1, 32, 1))
    S2 = S.copy()
    S2[37] = 127
    m2 = Resident(lib, pkg, pkg.DSV4_WFP4, W.copy(), S2, rows, cols, 1, 32)
    check_close(lib.mmq_n(m2.desc, x, 64), oracle.fp4_n(W, S2, x, rows, cols, 1, 32, 64))
    assert lib.status() == 0            # the _dev word saw nothing
    m.drop()
    m2.drop()


@pytest.mark.parametrize("fmt,nt", [("fp8f", 40), ("fp4", 40), ("fp8f", 1288)])     # dense tiles, grouped, dense
def test_seam_large_and_tiny_rows(lib, pkg, oracle, fmt, nt):
    """The nt >= 32 seam on rows an unscaled fp16 cast would break: |x| up to
    1e5 (beyond fp16), rows scaled by 1e-9 (below fp16's normal range), an
    all-zero row and a row of fp32 subnormals; every row within 1e-3."""
    rows, cols = 256, 1024
    rng = np.random.default_rng(5)
    w = (rng.standard_normal((rows, cols)) * 0.02).astype(np.float32)
    x = rng.standard_normal((nt, cols)).astype(np.float32)
    x[0] *= 1e5
    x[1, ::97] = 1e5
    x[2] *= 1e-9
    x[3] = 0.0
    x[4] = (rng.standard_normal(cols) * 1e-39).astype(np.float32)
    x[5] *= 3e4
    x = np.ascontiguousarray(x.reshape(-1))
    if fmt == "fp4":
        W, S = oracle.quant_fp4_mx(w)
        m = Resident(lib, pkg, pkg.DSV4_WFP4, W, S, rows, cols, 1, 32)
        want = oracle.fp4_n(W, S, x, rows, cols, 1, 32, nt)
    else:
        W, S = oracle.quant_fp8_blk128(w)
        m = Resident(lib, pkg, pkg.DSV4_WFP8_F32S, W, S, rows, cols, 128, 128)
        want = oracle.fp8f_n(W, S, x, rows, cols, 128, 128, nt)
    got = lib.mmq_n(m.desc, x, nt).reshape(nt, rows)
    want = want.reshape(nt, rows)
    assert np.all(np.isfinite(got))
    assert np.array_equal(got[3], np.zeros(rows, np.float32))
    for t in range(nt):
        if t == 3:
            continue
        e = rel_l2(got[t], want[t])
        assert e <= REL_L2_TOL, f"row {t}: rel L2 {e:.3e} (max abs {max_abs(got[t], want[t]):.3e})"
    m.drop()


def test_grouped_swiglu_beyond_fp16_returns_minus1(lib, pkg, oracle):
    """Unclamped SwiGLU (limit 0) of gate and up values in the hundreds gives
    mid values past 65504, which the grouped path's fp16 operand cannot hold:
    -1 with the reason. With the reference's clamp (limit 10) every mid is
    at most 100 and the same call returns 0 with finite output. (Its accuracy
    is not checked here: gate and up of standard deviation 320 carry the fp16
    activations' absolute error of ~0.1 into the few up values inside the
    clamp; the clamp itself is checked against the oracle at realistic
    magnitudes in test_gpu_swiglu.py.)"""
    hidden, inter, ne, n, topk = 256, 128, 4, 8, 2
    rng = np.random.default_rng(65504)
    ex, keep = [], []
    for e in range(ne):
        mats = []
        for (r, c), sig in (((inter, hidden), 20.0), ((inter, hidden), 20.0), ((hidden, inter), 0.02)):
            W, S = oracle.quant_fp4_mx((rng.standard_normal((r, c)) * sig).astype(np.float32))
            mats.append(Resident(lib, pkg, pkg.DSV4_WFP4, W, S, r, c, 1, 32))
        keep += mats
        ex.append(mats)
    descs = [pkg.ExpertW(m[0].desc, m[1].desc, m[2].desc) for m in ex]
    idx = np.stack([rng.choice(ne, topk, replace=False) for _ in range(n)]).astype(np.int32)
    w = np.full((n, topk), 0.5, np.float32)
    x = rng.standard_normal((n, hidden)).astype(np.float32)
    with pytest.raises(pkg.Dsv4Error, match="fp16 range"):
        lib.moe_grouped(descs, idx, w, x, None, 0.0)
    got = lib.moe_grouped(descs, idx, w, x, None, 10.0)
    assert np.all(np.isfinite(got))
    assert lib.status() == 0
    for m in keep:
        m.drop()


# ------------------------------------------------------------ drop-in ----

def test_drop_in_decode_layer_sequence(lib, pkg, oracle):
    """One decode layer's matrices through the reference-named dsv4_mmq of
    libdsv4_amd.so, in the order src/70_decode/dsv4_layer_attn.c:21-106 and
    dsv4_layer.c:52 call them, at DeepSeek-V4-Flash shapes
    (src/00_base/dsv4_weights.h:44-112): E8M0 FP8 projections, BF16
    compressor / indexer / router matrices, the eight wo_a group slices of one
    [8192 x 4096] arena (dsv4_wo_a_group), the 8192-wide wo_b, and the FP8
    shared and FP4 routed experts through dsv4_expert_forward. Each output
    within 1e-3 of the oracle. Every matrix is first checked through the C
    ABI (which returns -1 instead of aborting), so an unsupported matrix
    fails this test rather than ending the process."""
    mirror = pkg.Mirror()
    rng = np.random.default_rng(4242)
    keep = []

    def fp8(rows, cols):
        W = e4m3_codes(rng, rows * cols)
        S = rng.integers(112, 120, (rows // 128) * (cols // 128)).astype(np.uint8)
        m = Resident(lib, pkg, pkg.DSV4_WFP8, W, S, rows, cols, 128, 128)
        keep.append(m)
        return m

    def bf16(rows, cols):
        W = bf16_bits(rng.standard_normal(rows * cols).astype(np.float32) * 0.02)
        m = ResidentBf16(lib, pkg, W, rows, cols)
        keep.append(m)
        return m

    def run(m, x):
        assert lib.mmq_n_rc(m.desc, x, 1) == 0, lib.error()
        got = mirror.mmq(m.desc, x)
        want = oracle.mmq_n(m.hm, np.ascontiguousarray(x, np.float32), 1)
        check_close(got, want)
        return got

    x = rng.standard_normal(4096).astype(np.float32)
    qr = run(fp8(1024, 4096), x)                        # wq_a
    run(fp8(32768, 1024), qr)                           # wq_b
    run(fp8(512, 4096), x)                              # wkv
    run(bf16(1024, 4096), x)                            # comp.wkv (ratio 4: coff 2)
    run(bf16(1024, 4096), x)                            # comp.wgate
    run(fp8(8192, 1024), qr)                            # idx.wq_b
    run(bf16(64, 4096), x)                              # idx.weights_proj
    wo_a = fp8(8192, 4096)                              # 8 groups of [1024 x 4096]
    o = rng.standard_normal(8 * 4096).astype(np.float32)
    ogrp = []
    for gi in range(8):
        sl = pkg.qmat(pkg.DSV4_WFP8, wo_a.W.ctypes.data + gi * 1024 * 4096,
                      wo_a.S.ctypes.data + gi * (1024 // 128) * (4096 // 128), 1024, 4096, 128, 128)
        hs = P.HostMat(pkg.DSV4_WFP8, wo_a.W[gi * 1024 * 4096:(gi + 1) * 1024 * 4096],
                       wo_a.S[gi * 8 * 32:(gi + 1) * 8 * 32], 1024, 4096, 128, 128)
        xs = o[gi * 4096:(gi + 1) * 4096]
        assert lib.mmq_n_rc(sl, xs, 1) == 0, lib.error()
        got = mirror.mmq(sl, xs)
        check_close(got, oracle.mmq_n(hs, np.ascontiguousarray(xs), 1))
        ogrp.append(got)
    run(fp8(4096, 8192), np.concatenate(ogrp))          # wo_b
    run(bf16(256, 4096), x)                             # moe.gate

    def expert(wdt, sig):
        mats = []
        for (r, c) in ((2048, 4096), (2048, 4096), (4096, 2048)):
            w = (rng.standard_normal((r, c)) * sig).astype(np.float32)
            if wdt == pkg.DSV4_WFP4:
                W, S = oracle.quant_fp4_mx(w)
                mats.append(Resident(lib, pkg, wdt, W, S, r, c, 1, 32))
            else:
                W = e4m3_codes(rng, r * c)
                S = rng.integers(110, 116, (r // 128) * (c // 128)).astype(np.uint8)
                mats.append(Resident(lib, pkg, wdt, W, S, r, c, 128, 128))
        keep.extend(mats)
        return pkg.ExpertW(mats[0].desc, mats[1].desc, mats[2].desc), \
            P.HostExpert(mats[0].hm, mats[1].hm, mats[2].hm)

    for wdt in (pkg.DSV4_WFP8, pkg.DSV4_WFP4):          # shared, routed
        d, h = expert(wdt, 0.02)
        assert lib.expert_forward(d, x, 10.0) is not None
        check_close(mirror.expert_forward(d, x, 10.0), oracle.expert_forward(h, x, 10.0))
    for m in keep:
        m.drop()


# -------------------------------------------------------- permutation ----

@pytest.mark.parametrize("n,topk,ne,zipf", [
    (64, 6, 256, 1.1), (4096, 6, 256, 1.1), (1000, 8, 1024, None), (5, 2, 3, None), (1, 1, 1, None),
    (45000, 6, 256, 1.1),    # 264 chunks of 1024 pairs: two chunks per workgroup
])
def test_route_matches_union_prepare(lib, oracle, n, topk, ne, zipf):
    """ex_off, ex_tok and ex_k of the device counting sort equal the
    reference's union_prepare index for index; pos inverts it."""
    rng = np.random.default_rng(n + topk + ne)
    p = None
    if zipf:
        p = 1.0 / np.arange(1, ne + 1) ** zipf
        p /= p.sum()
    idx = np.stack([rng.choice(ne, topk, replace=False, p=p) for _ in range(n)]).astype(np.int32)
    P_ = n * topk
    di = torch.from_numpy(idx.reshape(-1)).to(DEV)
    off = torch.full((ne + 1,), -7, dtype=torch.int32, device=DEV)
    tok = torch.full((P_,), -7, dtype=torch.int32, device=DEV)
    kk = torch.full((P_,), -7, dtype=torch.int32, device=DEV)
    pos = torch.full((P_,), -7, dtype=torch.int32, device=DEV)
    lib.moe_route_dev(off.data_ptr(), tok.data_ptr(), kk.data_ptr(), pos.data_ptr(), di.data_ptr(),
                      n, topk, ne)
    torch.cuda.synchronize()
    assert lib.status() == 0
    cnt, w_off, w_tok, w_k, _ = oracle.union_prepare(idx, ne)
    assert np.array_equal(off.cpu().numpy(), w_off)
    assert np.array_equal(np.diff(off.cpu().numpy()), cnt)
    assert np.array_equal(tok.cpu().numpy(), w_tok)
    assert np.array_equal(kk.cpu().numpy(), w_k)
    pp = pos.cpu().numpy()
    pairs = np.arange(P_)
    assert np.array_equal(w_tok[pp], pairs // topk)
    assert np.array_equal(w_k[pp], pairs % topk)


def test_route_bad_id_counting_pass(lib, oracle):
    """A bad id among 6,000 pairs (six chunks of 1024, the two-launch form):
    status bit 0, its pos -1, and every good pair placed as union_prepare
    places the ids with the bad one left out."""
    rng = np.random.default_rng(6000)
    n, topk, ne = 1000, 6, 64
    idx = np.stack([rng.choice(ne, topk, replace=False) for _ in range(n)]).astype(np.int32)
    idx[777, 3] = ne + 5
    P_ = n * topk
    di = torch.from_numpy(idx.reshape(-1)).to(DEV)
    off = torch.full((ne + 1,), -7, dtype=torch.int32, device=DEV)
    tok, kk, pos = (torch.full((P_,), -7, dtype=torch.int32, device=DEV) for _ in range(3))
    lib.status()
    lib.moe_route_dev(off.data_ptr(), tok.data_ptr(), kk.data_ptr(), pos.data_ptr(), di.data_ptr(),
                      n, topk, ne)
    torch.cuda.synchronize()
    assert lib.status() & 1
    pp = pos.cpu().numpy()
    assert pp[777 * topk + 3] == -1
    flat = idx.reshape(-1)
    good = np.flatnonzero(flat < ne)
    order = good[np.argsort(flat[good], kind="stable")]
    o = off.cpu().numpy()
    assert np.array_equal(np.diff(o), np.bincount(flat[good], minlength=ne))
    got_tok, got_k = tok.cpu().numpy()[:len(order)], kk.cpu().numpy()[:len(order)]
    assert np.array_equal(got_tok, order // topk) and np.array_equal(got_k, order % topk)
    assert np.array_equal(pp[order], np.arange(len(order)))


def test_route_bad_id(lib):
    idx = np.array([[0, 1], [2, 9], [1, 0]], np.int32)
    di = torch.from_numpy(idx.reshape(-1)).to(DEV)
    off = torch.empty(4, dtype=torch.int32, device=DEV)
    tok, kk, pos = (torch.full((6,), -7, dtype=torch.int32, device=DEV) for _ in range(3))
    lib.moe_route_dev(off.data_ptr(), tok.data_ptr(), kk.data_ptr(), pos.data_ptr(), di.data_ptr(),
                      3, 2, 3)
    torch.cuda.synchronize()
    assert lib.status() & 1
    pp = pos.cpu().numpy()
    assert pp[3] == -1
    assert np.array_equal(off.cpu().numpy(), [0, 2, 4, 5])
    t, k = tok.cpu().numpy(), kk.cpu().numpy()
    assert list(t[:5]) == [0, 2, 0, 2, 1] and list(k[:5]) == [0, 1, 1, 0, 0]

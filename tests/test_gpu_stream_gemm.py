"""GPU parity of the decode-batch GEMM over load-time packed matrices of the six block formats (vx_qweight_pack): the packed
copy dequantises to the reference's values bit for bit, the products match the CPU oracle's MatMulQ4_0 / Q8_0 / Q4_K / Q6_K / Q5_0 / Q5_K
(backend/cpu/cpu.go:842-911) to float32 summation order on every cut of the matrix the planner makes, a row's bits
do not depend on the batch it sits in (2 .. 32 rows; 33 .. 64 rows), and the fused decode blocks give the oracle's
layer with packed weights."""
import os
import subprocess
import sys

import numpy as np
import pytest

from oracle import numerics as nx
from oracle import quantize as qz

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def be():
    from vexel_amd.backend import HipBackend
    b = HipBackend(0)
    yield b
    b.close()


def _close(got, want, rtol, atol, what=""):
    err = np.abs(got.astype(np.float64) - want.astype(np.float64))
    lim = atol + rtol * np.abs(want.astype(np.float64))
    assert np.all(err <= lim), "%s: max err %.3e (limit %.3e at worst element)" % (
        what, err.max(), lim.reshape(-1)[err.argmax()])


FMTS = [nx.FMT_Q4_0, nx.FMT_Q8_0, nx.FMT_Q6_K, nx.FMT_Q4_K, nx.FMT_Q5_0, nx.FMT_Q5_K]


def _packed(be, w, n, k, fmt=nx.FMT_Q4_0):
    dw = be.upload(w, permanent=True)
    qw = be.qweight(fmt, dw, n, k)
    assert be.qweight_pack(qw)
    assert be.qweight_is_packed(qw)
    return dw, qw


@pytest.mark.parametrize("fmt", FMTS)
@pytest.mark.parametrize("n,k", [(16, 256), (48, 1024), (1040, 512)])
def test_packed_copy_dequantises_bit_exact(be, n, k, fmt):
    rng = np.random.default_rng(n + k)
    w = qz.random_quant(fmt, rng, n, k)
    if fmt == nx.FMT_Q5_0:
        w.reshape(-1)[2:22] = rng.integers(0, 256, 20, dtype=np.uint8)     # arbitrary fifth bits and nibbles in one block
    elif fmt == nx.FMT_Q5_K:
        w.reshape(-1)[4:176] = rng.integers(0, 256, 172, dtype=np.uint8)   # arbitrary scale / min fields, fifth bits and nibbles
    elif fmt == nx.FMT_Q4_K:
        w.reshape(-1)[4:144] = rng.integers(0, 256, 140, dtype=np.uint8)   # arbitrary scale / min fields and codes in one super-block
    elif fmt == nx.FMT_Q6_K:
        w.reshape(-1)[0:208] = rng.integers(0, 256, 208, dtype=np.uint8)   # arbitrary codes and scale bytes in one super-block
    else:
        w.reshape(-1)[2:34] = rng.integers(0, 256, 32, dtype=np.uint8)   # every code position carries arbitrary codes
    dw, qw = _packed(be, w, n, k, fmt)
    dst = be.alloc(n * k * 4)
    be.dequantize_packed(qw, dst)
    got = be.download(dst, (n * k,), np.float32)
    want = nx.dequantize(fmt, w, n * k)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
    be.free(dw)
    assert not be.qweight_is_packed(qw)                          # the copy goes with the matrix
    be.reset_pool()


def test_pack_refuses_other_formats_and_shapes(be):
    rng = np.random.default_rng(0)
    w = qz.random_quant(nx.FMT_BF16, rng, 32, 256)
    dw = be.upload(w, permanent=True)
    assert not be.qweight_pack(be.qweight(nx.FMT_BF16, dw, 32, 256))
    assert not be.qweight_pack(be.qweight(nx.FMT_Q4_0, dw, 24, 256))     # rows not a multiple of 16
    assert not be.qweight_pack(be.qweight(nx.FMT_Q4_0, dw, 32, 128))     # K not a multiple of 256
    be.free(dw)


# (n, k): one tile; K slices of one and two half chunks per wave; slices with an odd share of half chunks;
# more tiles than workgroups in a slice; a 7B down-projection's K
@pytest.mark.parametrize("n,k", [(16, 256), (80, 1024), (96, 2048), (1040, 2304), (4112, 512), (64, 4352), (208, 11008)])
@pytest.mark.parametrize("m", [2, 5, 16, 17, 32, 33, 48, 64])
@pytest.mark.parametrize("fmt", FMTS)
def test_matmul_packed_vs_oracle(be, n, k, m, fmt):
    rng = np.random.default_rng(n * 7 + k + m)
    w = qz.random_quant(fmt, rng, n, k)
    a = (rng.standard_normal((m, k)) * (1.0 + 3.0 * (rng.random((1, k)) < 0.1))).astype(np.float32)
    want = nx.matmul_quant(fmt, a, w, m, n, k)
    dw, qw = _packed(be, w, n, k, fmt)
    da = be.upload(a)
    dout = be.alloc(m * n * 4)
    be.matmul_quant(fmt, da, dw, dout, None, m, n, k)
    got = be.download(dout, (m, n), np.float32)
    scale = np.abs(want).max()
    _close(got, want, 2e-5, 2e-6 * scale + 1e-7, "packed matmul %dx%dx%d" % (m, n, k))
    # the unpacked path on the same inputs: float32 summation order apart
    be.qweight_unpack(qw)
    be.matmul_quant(fmt, da, dw, dout, None, m, n, k)
    plain = be.download(dout, (m, n), np.float32)
    _close(got, plain, 0, 3e-6 * scale + 1e-7, "packed vs unpacked")
    be.free(dw)
    be.reset_pool()


# Workgroups of five and six tiles (1285 over 256 compute units): groups of one, two and four tiles between two barriers with an odd one at
# the end, units asked for past a workgroup's last tile, sums added up a group later
@pytest.mark.parametrize("m", [16, 32, 64])
@pytest.mark.parametrize("fmt", FMTS)
def test_matmul_packed_several_groups_a_workgroup(be, m, fmt):
    n, k = 16 * 1285, 256
    rng = np.random.default_rng(m + fmt)
    w = qz.random_quant(fmt, rng, n, k)
    a = rng.standard_normal((m, k)).astype(np.float32)
    want = nx.matmul_quant(fmt, a, w, m, n, k)
    dw, _ = _packed(be, w, n, k, fmt)
    da, dout = be.upload(a), be.alloc(m * n * 4)
    be.matmul_quant(fmt, da, dw, dout, None, m, n, k)
    _close(be.download(dout, (m, n), np.float32), want, 2e-5, 2e-6 * np.abs(want).max() + 1e-7, "%d rows" % m)
    be.free(dw)
    be.reset_pool()


# more than 64 rows: the kernel whose waves own weight tiles and share the activation through LDS
# (n, k): fewer tiles than a workgroup's waves own; tiles not a multiple of a wave's; many K slices; a long K
@pytest.mark.parametrize("n,k", [(16, 256), (80, 1024), (1040, 2304), (4112, 512), (208, 11008)])
@pytest.mark.parametrize("m", [65, 96, 130, 256])
@pytest.mark.parametrize("fmt", FMTS)
def test_matmul_packed_many_rows_vs_oracle(be, n, k, m, fmt):
    rng = np.random.default_rng(n * 5 + k + m)
    w = qz.random_quant(fmt, rng, n, k)
    a = (rng.standard_normal((m, k)) * (1.0 + 3.0 * (rng.random((1, k)) < 0.1))).astype(np.float32)
    want = nx.matmul_quant(fmt, a, w, m, n, k)
    dw, qw = _packed(be, w, n, k, fmt)
    da = be.upload(a)
    dout = be.alloc(m * n * 4)
    be.matmul_quant(fmt, da, dw, dout, None, m, n, k)
    got = be.download(dout, (m, n), np.float32)
    scale = np.abs(want).max()
    _close(got, want, 2e-5, 2e-6 * scale + 1e-7, "packed matmul %dx%dx%d" % (m, n, k))
    res = rng.standard_normal((m, n)).astype(np.float32)
    dres = be.upload(res)
    be.matmul_quant(fmt, da, dw, dout, dres, m, n, k)
    assert np.array_equal(be.download(dout, (m, n), np.float32).view(np.uint32), (res + got).view(np.uint32))
    be.qweight_unpack(qw)
    be.matmul_quant(fmt, da, dw, dout, None, m, n, k)
    plain = be.download(dout, (m, n), np.float32)
    _close(got, plain, 0, 3e-6 * scale + 1e-7, "packed vs unpacked")
    be.free(dw)
    be.reset_pool()


@pytest.mark.parametrize("kind", ["largest", "smallest", "mixed"])
@pytest.mark.parametrize("m", [3, 33, 65])
@pytest.mark.parametrize("fmt", FMTS)
def test_matmul_packed_with_scales_at_their_limits(be, fmt, m, kind):
    """The kernels multiply scales into f16 operands: the largest integer scales and codes, f16's smallest subnormal as
    the block scale, and block scales from one end of f16 to the other within a row. Bound per output, against float64:
    the activation's two parts and the product of the two lower parts are each below 2^-22 of a term, and a term passes at
    most 16 float32 additions at the size of the sum of all terms: 2 * 2^-22 + 16 * 2^-24 of that sum."""
    rng = np.random.default_rng(fmt * 100 + m)
    n, k = 48, 512
    elems, size = nx.BLOCK_ELEMS[fmt], nx.BLOCK_BYTES[fmt]
    b = rng.integers(0, 256, (n, k // elems, size), dtype=np.uint8)
    if kind == "largest" and elems == 256:
        if fmt == nx.FMT_Q6_K:
            b[..., 192:208] = np.where(rng.random(b[..., 192:208].shape) < 0.5, 0x80, 0x7F)
        else:
            b[..., 4:16] = 0xFF
    shape = b.shape[:2] + (1,)
    d = {"largest": np.full(shape, 0.01), "smallest": np.full(shape, 2.0 ** -24), "mixed": 2.0 ** rng.uniform(-24, 15, shape)}[kind]
    if kind == "largest" and elems == 32:
        d = np.full(shape, 65504.0)
    raw = d.astype(np.float16).view(np.uint8)
    if fmt == nx.FMT_Q6_K:
        b[..., 208:210] = raw
    else:
        b[..., 0:2] = raw
        if elems == 256:
            b[..., 2:4] = raw
    w = b.reshape(n, -1)
    a = rng.standard_normal((m, k)).astype(np.float32)
    deq = nx.dequantize(fmt, w, n * k).reshape(n, k).astype(np.float64)
    want, size_of = a.astype(np.float64) @ deq.T, np.abs(a.astype(np.float64)) @ np.abs(deq).T
    dw, _ = _packed(be, w, n, k, fmt)
    da, dout = be.upload(a), be.alloc(m * n * 4)
    be.matmul_quant(fmt, da, dw, dout, None, m, n, k)
    got = be.download(dout, (m, n), np.float32)
    if elems == 256 and fmt != nx.FMT_Q6_K:  # (the two terms d * sc * q and dmin * m are summed apart)
        size_of *= 2
    assert np.all(np.abs(got - want) <= (2 * 2.0 ** -22 + 16 * 2.0 ** -24) * size_of), np.max(np.abs(got - want) / size_of)
    be.free(dw)
    be.reset_pool()


def _balanced_k_quant(rng, fmt, n, k):
    """Weights as quantizing zero-mean ones gives them: codes bell-shaped about the middle, minima that take the middle off."""
    sb = (n, k // 256)
    b = rng.integers(0, 256, sb + (nx.BLOCK_BYTES[fmt],), dtype=np.uint8)
    d = (0.0005 * (1 + rng.random(sb + (1,)))).astype(np.float16)
    if fmt == nx.FMT_Q6_K:
        b[..., 208:210] = d.view(np.uint8)
        q = np.clip(np.rint(32 + 9 * rng.standard_normal(sb + (2, 4, 32))), 0, 63).astype(np.uint8)
        b[..., 0:128] = ((q[..., 0:2, :] & 15) | (q[..., 2:4, :] & 15) << 4).reshape(sb + (128,))
        h = q >> 4
        b[..., 128:192] = (h[..., 0, :] | h[..., 1, :] << 2 | h[..., 2, :] << 4 | h[..., 3, :] << 6).reshape(sb + (64,))
        b[..., 192:208] = (rng.integers(64, 128, sb + (16,)) * rng.choice([-1, 1], sb + (16,))).astype(np.int8).view(np.uint8)
        return b.reshape(n, -1)
    wide = fmt == nx.FMT_Q5_K
    b[..., 0:2], b[..., 2:4] = d.view(np.uint8), (d * np.float16(15.5 if wide else 7.5)).view(np.uint8)
    s = rng.integers(32, 64, sb + (8,)).astype(np.uint8)
    b[..., 4:8] = b[..., 8:12] = (s[..., :4] & 63) | (s[..., 4:] >> 4) << 6
    b[..., 12:16] = (s[..., 4:] & 15) | (s[..., 4:] & 15) << 4
    z = rng.standard_normal(sb + (8, 32))
    q = np.clip(np.rint(15.5 + 7 * z if wide else 7.5 + 3.5 * z), 0, 31 if wide else 15).astype(np.uint8)
    b[..., 16 + 32 * wide:] = ((q[..., 0::2, :] & 15) | (q[..., 1::2, :] & 15) << 4).reshape(sb + (128,))
    if wide:
        b[..., 16:48] = np.bitwise_or.reduce((q >> 4) << np.arange(8, dtype=np.uint8)[:, None], axis=-2)
    return b.reshape(n, -1)


def _exact_k_quant(fmt, w, n, k):
    """The weights in float64 (gguf.Dequantize rounds d * sc * q - dmin * m to float32)."""
    sb = (n, k // 256)
    b = w.reshape(sb + (-1,))
    half = lambda x: np.ascontiguousarray(x).view(np.float16).astype(np.float64)
    if fmt == nx.FMT_Q6_K:
        q = np.empty(sb + (2, 4, 32))
        lo, hi = b[..., 0:128].reshape(sb + (2, 2, 32)), b[..., 128:192].reshape(sb + (2, 1, 32))
        q[..., 0:2, :], q[..., 2:4, :] = lo & 15, lo >> 4
        q += (((hi >> np.array([0, 2, 4, 6], dtype=np.uint8)[:, None]) & 3) << 4) - 32.0
        sc = np.ascontiguousarray(b[..., 192:208]).view(np.int8).astype(np.float64)
        return (half(b[..., 208:210])[..., None] * sc[..., None] * q.reshape(sb + (16, 16))).reshape(n, k)
    wide = fmt == nx.FMT_Q5_K
    s = b[..., 4:16].astype(np.int64)
    sc = np.concatenate([s[..., 0:4] & 63, (s[..., 8:12] & 15) | (s[..., 0:4] >> 6) << 4], -1)
    mn = np.concatenate([s[..., 4:8] & 63, (s[..., 8:12] >> 4) | (s[..., 4:8] >> 6) << 4], -1)
    qs = b[..., 16 + 32 * wide:].reshape(sb + (4, 32))
    q = np.stack([qs & 15, qs >> 4], axis=-2).reshape(sb + (8, 32)).astype(np.float64)
    if wide:
        q += ((b[..., None, 16:48] >> np.arange(8, dtype=np.uint8)[:, None]) & 1) * 16.0
    return (half(b[..., 0:2])[..., None] * sc[..., None] * q - half(b[..., 2:4])[..., None] * mn[..., None]).reshape(n, k)


# Relative error (2-norm) of the products against float64, in 1e-7, for one row, for 2 .. 64 rows and for more: what kernels leave that
# put d * sc on every block's own sum and take the minima off block by block, the largest measured on these matrices (2.87, 2.58 and 2.60;
# 5.27, 2.56 and 2.67; 5.20, 1.05 and 1.25), and 1 to 5 % for the seed. With the scales in the operands no precision is given away.
ROUNDING = {nx.FMT_Q4_K: (2.9, 2.7, 2.73), nx.FMT_Q5_K: (5.4, 2.7, 2.8), nx.FMT_Q6_K: (5.3, 1.1, 1.3)}


# both ends of the streaming kernel and of its four-tile form; 65 and more rows in few and in many slices of K
@pytest.mark.parametrize("n,k", [(2048, 2048), (512, 4096)])
@pytest.mark.parametrize("m", [1, 2, 32, 33, 64, 65, 200])
@pytest.mark.parametrize("fmt", [nx.FMT_Q4_K, nx.FMT_Q5_K, nx.FMT_Q6_K])
def test_scales_in_the_operands_round_no_more_than_scales_on_the_sums(be, fmt, m, n, k):
    rng = np.random.default_rng(1000 * fmt + m + k)
    w = _balanced_k_quant(rng, fmt, n, k)
    deq = _exact_k_quant(fmt, w, n, k)
    a = rng.standard_normal((max(m, 24 // m * m), k)).astype(np.float32)  # (24 rows at least: the error of one scatters)
    dw, _ = _packed(be, w, n, k, fmt)
    got = np.empty((len(a), n), dtype=np.float32)
    for r in range(0, len(a), m):
        da, dout = be.upload(a[r:r + m]), be.alloc(m * n * 4)
        be.matmul_quant(fmt, da, dw, dout, None, m, n, k)
        got[r:r + m] = be.download(dout, (m, n), np.float32)
    want = a.astype(np.float64) @ deq.T
    err = np.linalg.norm(got - want) / np.linalg.norm(want)
    be.free(dw)
    be.reset_pool()
    assert err <= ROUNDING[fmt][0 if m == 1 else 1 if m <= 64 else 2] * 1e-7, err


# What the same sum left in six slices of K, whose waves' sums were added one by one (1.122e-7 and 1.148e-7 measured), and 1 % for the
# seed: 131072 sums scatter by a third of that. Eleven slices added so left 1.16e-7 and 1.19e-7.
@pytest.mark.parametrize("fmt,bound", [(nx.FMT_Q4_0, 1.134e-7), (nx.FMT_Q8_0, 1.16e-7)])
def test_many_slices_of_a_deep_matrix_round_no_more_than_few(be, fmt, bound):
    rng = np.random.default_rng(fmt)
    m, n, k = 32, 4096, 11008
    w = qz.random_quant(fmt, rng, n, k)
    a = rng.standard_normal((m, k)).astype(np.float32)
    dw, _ = _packed(be, w, n, k, fmt)
    da, dout = be.upload(a), be.alloc(m * n * 4)
    be.matmul_quant(fmt, da, dw, dout, None, m, n, k)
    got = be.download(dout, (m, n), np.float32)
    want = a.astype(np.float64) @ nx.dequantize(fmt, w, n * k).reshape(n, k).astype(np.float64).T
    err = np.linalg.norm(got - want) / np.linalg.norm(want)
    be.free(dw)
    be.reset_pool()
    assert err <= bound, err


@pytest.mark.parametrize("fmt", FMTS)
def test_matmul_packed_many_rows_independent_of_batch(be, fmt):
    """A row has the same bits in any batch with the same number of 64-row groups (the K slicing depends on that
    number beside the matrix' shape): 65 .. 128 rows here."""
    rng = np.random.default_rng(12)
    n, k = 208, 4096
    w = qz.random_quant(fmt, rng, n, k)
    a = rng.standard_normal((128, k)).astype(np.float32)
    dw, qw = _packed(be, w, n, k, fmt)
    da = be.upload(a)

    def batch(first, rows):
        d = be.alloc(rows * n * 4)
        be.matmul_quant(fmt, da + first * k * 4, dw, d, None, rows, n, k)
        return be.download(d, (rows, n), np.float32)

    full = batch(0, 128)
    for first, rows in ((0, 65), (11, 90), (40, 88), (1, 127)):
        part = batch(first, rows)
        assert np.array_equal(part.view(np.uint32), full[first:first + rows].view(np.uint32)), (first, rows)
    be.free(dw)
    be.reset_pool()


@pytest.mark.parametrize("fmt", FMTS)
def test_matmul_packed_rows_independent_of_batch(be, fmt):
    """A row has the same bits in a batch of 2, of 16, of 17 and of 32 rows (the cut of the matrix depends on its
    shape and the device only; 16 rows and fewer run the one-tile form of the kernel), and in a batch of 33, of 40
    and of 64 rows (four activation tiles a step: K is cut into narrower slices there)."""
    rng = np.random.default_rng(11)
    n, k = 208, 4096
    w = qz.random_quant(fmt, rng, n, k)
    a = rng.standard_normal((64, k)).astype(np.float32)
    dw, qw = _packed(be, w, n, k, fmt)
    da = be.upload(a)

    def batch(first, rows):
        d = be.alloc(rows * n * 4)
        be.matmul_quant(fmt, da + first * k * 4, dw, d, None, rows, n, k)
        return be.download(d, (rows, n), np.float32)

    full = batch(0, 32)
    for first, rows in ((0, 2), (5, 2), (30, 2), (0, 16), (3, 17), (16, 16), (9, 7)):
        part = batch(first, rows)
        assert np.array_equal(part.view(np.uint32), full[first:first + rows].view(np.uint32)), (first, rows)
    full64 = batch(0, 64)
    for first, rows in ((0, 33), (20, 40), (31, 33), (7, 57)):
        part = batch(first, rows)
        assert np.array_equal(part.view(np.uint32), full64[first:first + rows].view(np.uint32)), (first, rows)
    scale = np.abs(full).max()
    _close(full64[:32], full, 0, 3e-6 * scale, "a row in 64 against the same row in 32")
    res = rng.standard_normal((32, n)).astype(np.float32)
    dres, d = be.upload(res), be.alloc(32 * n * 4)
    be.matmul_quant(fmt, da, dw, d, dres, 32, n, k)
    assert np.array_equal(be.download(d, (32, n), np.float32).view(np.uint32), (res + full).view(np.uint32))
    be.free(dw)
    be.reset_pool()


def test_default_configuration_takes_the_kernels_the_benchmark_reports(be):
    """With no environment switch set, a packed matrix runs the streaming kernel at 2 .. 64 rows and the many-rows
    kernel beyond, one row the matrix-vector kernel, and an unpacked matrix the kernels over the GGUF rows: the paths
    bench.py times are the paths a default process takes."""
    if [k for k in os.environ if k.startswith("VEXEL_HIP_")]:
        pytest.skip("a VEXEL_HIP_* switch is set: this is not the default configuration")
    rng = np.random.default_rng(21)
    n, k = 256, 4096
    w = qz.random_quant(nx.FMT_Q4_0, rng, n, k)
    a = rng.standard_normal((256, k)).astype(np.float32)
    dw, qw = _packed(be, w, n, k)
    da, dout = be.upload(a), be.alloc(256 * n * 4)
    for m, want in ((1, "qmatvec_kernel"), (2, "qstream_kernel"), (32, "qstream_kernel"), (64, "qstream_kernel"),
                    (65, "qtiles_kernel"), (256, "qtiles_kernel")):
        be.matmul_quant(nx.FMT_Q4_0, da, dw, dout, None, m, n, k)
        assert be.last_matmul_kernel() == want, (m, be.last_matmul_kernel())
    be.qweight_unpack(qw)
    for m, want in ((1, "qmatvec_kernel"), (32, "qgemm_wave_kernel"), (256, "qgemm_kernel")):
        be.matmul_quant(nx.FMT_Q4_0, da, dw, dout, None, m, n, k)
        assert be.last_matmul_kernel() == want, (m, be.last_matmul_kernel())
    be.free(dw)
    be.reset_pool()


def test_rewriting_the_matrix_drops_the_packed_copy(be):
    rng = np.random.default_rng(5)
    n, k, m = 64, 512, 8
    w1, w2 = qz.random_quant(nx.FMT_Q4_0, rng, n, k), qz.random_quant(nx.FMT_Q4_0, rng, n, k)
    a = rng.standard_normal((m, k)).astype(np.float32)
    dw, qw = _packed(be, w1, n, k)
    da, dout = be.upload(a), be.alloc(m * n * 4)
    be.to_device(dw, w2)                                         # new rows under the same address
    assert not be.qweight_is_packed(qw)
    be.matmul_q4_0(da, dw, dout, m, n, k)
    want = nx.matmul_quant(nx.FMT_Q4_0, a, w2, m, n, k)
    _close(be.download(dout, (m, n), np.float32), want, 2e-5, 2e-6 * np.abs(want).max() + 1e-7, "after rewrite")
    be.free(dw)
    be.reset_pool()


@pytest.mark.parametrize("fmt", FMTS)
@pytest.mark.parametrize("rows", [2, 7, 32, 64])
@pytest.mark.parametrize("hq,hk,d,hidden,ffn", [(8, 8, 64, 512, 1024), (8, 2, 128, 1024, 2816), (32, 32, 128, 4096, 1024)])
def test_fused_decode_blocks_with_packed_weights(be, rows, hq, hk, d, hidden, ffn, fmt):
    """RMSNorm -> Q|K|V -> RoPE -> KV store (one launch with the table of angles) and Wo -> residual -> RMSNorm ->
    gate|up -> SiLU*up -> down -> residual on packed weights against the oracle's operators."""
    rng = np.random.default_rng(rows + hq + hidden)
    bs, nblocks, theta, eps = 16, 8, 10000.0, 1e-5
    qd, kvd = hq * d, hk * d
    quant = {nx.FMT_Q4_0: qz.quantize_q4_0, nx.FMT_Q8_0: qz.quantize_q8_0, nx.FMT_Q5_0: qz.quantize_q5_0}.get(fmt)
    if fmt in (nx.FMT_Q6_K, nx.FMT_Q4_K, nx.FMT_Q5_K):
        mk = lambda n, k: qz.random_quant(fmt, rng, n, k, std=0.05).reshape(-1)
    else:
        mk = lambda n, k: quant((rng.standard_normal((n, k)) * 0.05).astype(np.float32)).reshape(-1)
    raw = {"wq": (mk(qd, hidden), qd, hidden), "wk": (mk(kvd, hidden), kvd, hidden), "wv": (mk(kvd, hidden), kvd, hidden),
           "wo": (mk(hidden, qd), hidden, qd), "w1": (mk(ffn, hidden), ffn, hidden), "w3": (mk(ffn, hidden), ffn, hidden),
           "w2": (mk(hidden, ffn), hidden, ffn)}
    dev, qws = {}, {}
    for name, (w, n, k) in raw.items():
        dev[name], qws[name] = _packed(be, w, n, k, fmt)
    x = rng.standard_normal((rows, hidden)).astype(np.float32)
    nw_attn = (1.0 + 0.1 * rng.standard_normal(hidden)).astype(np.float32)
    nw_ffn = (1.0 + 0.1 * rng.standard_normal(hidden)).astype(np.float32)
    positions = rng.integers(0, 100, rows).astype(np.int32)
    slots = rng.permutation(nblocks * bs)[:rows].astype(np.int32)
    per_block = 2 * bs * kvd
    pool0 = nx.f32_to_f16_array(rng.standard_normal(nblocks * per_block).astype(np.float32))

    # oracle
    h = nx.rmsnorm(x, nw_attn, rows, hidden, eps)
    q = nx.matmul_quant(fmt, h, raw["wq"][0], rows, qd, hidden)
    kk = nx.matmul_quant(fmt, h, raw["wk"][0], rows, kvd, hidden)
    vv = nx.matmul_quant(fmt, h, raw["wv"][0], rows, kvd, hidden)
    want_q, want_k = nx.rope_positions(q, kk, d, hq, hk, positions, d, theta, False)
    attn = rng.standard_normal((rows, qd)).astype(np.float32)
    x1 = nx.add(x, nx.matmul_quant(fmt, attn, raw["wo"][0], rows, hidden, qd))
    h2 = nx.rmsnorm(x1, nw_ffn, rows, hidden, eps)
    g = nx.matmul_quant(fmt, h2, raw["w1"][0], rows, ffn, hidden)
    u = nx.matmul_quant(fmt, h2, raw["w3"][0], rows, ffn, hidden)
    want_x = nx.add(x1, nx.matmul_quant(fmt, nx.silu_mul(g, u), raw["w2"][0], rows, hidden, ffn))

    # GPU
    dx, dnw, dnf = be.upload(x, permanent=True), be.upload(nw_attn, permanent=True), be.upload(nw_ffn, permanent=True)
    dpos, dslots = be.upload(positions, permanent=True), be.upload(slots, permanent=True)
    dpool, dq = be.upload(pool0, permanent=True), be.alloc_permanent(rows * qd * 4)
    be.rope_table_prepare(dpos, rows, d, theta)
    be.decode_attn_qkv(dx, dnw, eps, False, qws["wq"], qws["wk"], qws["wv"], rows, dpos, dslots, dpool, True, hq, hk, d, bs,
                       theta, dq)
    got_q = be.download(dq, (rows, qd), np.float32)
    _close(got_q, want_q, 2e-4, 2e-5 * np.abs(want_q).max(), "Q")
    pool = nx.f16_to_f32_array(be.download(dpool, (nblocks * per_block,), np.uint16))
    for r in range(rows):
        blk, off = divmod(int(slots[r]), bs)
        gk = pool[blk * per_block + off * kvd: blk * per_block + (off + 1) * kvd]
        gv = pool[blk * per_block + bs * kvd + off * kvd: blk * per_block + bs * kvd + (off + 1) * kvd]
        _close(gk, nx.f16_to_f32_array(nx.f32_to_f16_array(want_k[r])), 2e-3, 2e-3 * np.abs(want_k).max(), "K row %d" % r)
        _close(gv, nx.f16_to_f32_array(nx.f32_to_f16_array(vv[r])), 2e-3, 2e-3 * np.abs(vv).max(), "V row %d" % r)
    dattn = be.upload(attn, permanent=True)
    be.decode_ffn(dattn, dx, qws["wo"], dnf, eps, qws["w1"], qws["w3"], qws["w2"], rows)
    got_x = be.download(dx, (rows, hidden), np.float32)
    _close(got_x, want_x, 2e-4, 2e-5 * np.abs(want_x).max(), "layer output")
    for p in list(dev.values()) + [dx, dnw, dnf, dpos, dslots, dpool, dq, dattn]:
        be.free(p)
    be.reset_pool()


@pytest.mark.parametrize("fqk", [nx.FMT_Q4_K, nx.FMT_Q5_K])
@pytest.mark.parametrize("rows", [2, 7, 17, 32, 40])
@pytest.mark.parametrize("hq,hk,d,hidden", [(8, 2, 128, 1024), (32, 32, 128, 4096), (32, 8, 128, 4096), (24, 1, 64, 2048)])
def test_fused_qkv_with_packed_v_in_q6_k(be, rows, hq, hk, d, hidden, fqk):
    """attn_q and attn_k in Q4_K or Q5_K beside attn_v in Q6_K, as the K-quant mixes of GGUF files hold them, all
    three packed: up to 32 rows one launch computes the three (row groups shared out between the two formats),
    beyond that V takes a launch of its own; either way RMSNorm -> Q|K|V -> RoPE -> KV store gives what the oracle's
    operators give."""
    import os
    rng = np.random.default_rng(rows * 31 + hq + hidden + fqk)
    bs, nblocks, theta, eps = 16, 8, 10000.0, 1e-5
    qd, kvd = hq * d, hk * d
    fm = {"wq": fqk, "wk": fqk, "wv": nx.FMT_Q6_K}
    shapes = {"wq": (qd, hidden), "wk": (kvd, hidden), "wv": (kvd, hidden)}
    raw = {n: qz.random_quant(fm[n], rng, *shapes[n], std=0.05).reshape(-1) for n in shapes}
    dev, qws = {}, {}
    for name in shapes:
        dev[name], qws[name] = _packed(be, raw[name], *shapes[name], fm[name])
    x = rng.standard_normal((rows, hidden)).astype(np.float32)
    nw = (1.0 + 0.1 * rng.standard_normal(hidden)).astype(np.float32)
    positions = rng.integers(0, 100, rows).astype(np.int32)
    slots = rng.permutation(nblocks * bs)[:rows].astype(np.int32)
    per_block = 2 * bs * kvd
    pool0 = nx.f32_to_f16_array(rng.standard_normal(nblocks * per_block).astype(np.float32))

    h = nx.rmsnorm(x, nw, rows, hidden, eps)
    q = nx.matmul_quant(fqk, h, raw["wq"], rows, qd, hidden)
    kk = nx.matmul_quant(fqk, h, raw["wk"], rows, kvd, hidden)
    vv = nx.matmul_quant(nx.FMT_Q6_K, h, raw["wv"], rows, kvd, hidden)
    want_q, want_k = nx.rope_positions(q, kk, d, hq, hk, positions, d, theta, False)

    dx, dnw = be.upload(x, permanent=True), be.upload(nw, permanent=True)
    dpos, dslots = be.upload(positions, permanent=True), be.upload(slots, permanent=True)
    dpool, dq = be.upload(pool0, permanent=True), be.alloc_permanent(rows * qd * 4)
    be.rope_table_prepare(dpos, rows, d, theta)
    be.decode_attn_qkv(dx, dnw, eps, False, qws["wq"], qws["wk"], qws["wv"], rows, dpos, dslots, dpool, True, hq, hk, d, bs,
                       theta, dq)
    if not [k for k in os.environ if k.startswith("VEXEL_HIP_")] and rows <= 32 and hidden % 1024 == 0:
        assert be.last_matmul_kernel() == "qstream_mixed_kernel", be.last_matmul_kernel()
    got_q = be.download(dq, (rows, qd), np.float32)
    _close(got_q, want_q, 2e-4, 2e-5 * np.abs(want_q).max(), "Q")
    pool = nx.f16_to_f32_array(be.download(dpool, (nblocks * per_block,), np.uint16))
    untouched = np.ones(nblocks * per_block, dtype=bool)
    for r in range(rows):
        blk, off = divmod(int(slots[r]), bs)
        ko, vo = blk * per_block + off * kvd, blk * per_block + bs * kvd + off * kvd
        untouched[ko:ko + kvd] = False
        untouched[vo:vo + kvd] = False
        _close(pool[ko:ko + kvd], nx.f16_to_f32_array(nx.f32_to_f16_array(want_k[r])), 2e-3, 2e-3 * np.abs(want_k).max(), "K row %d" % r)
        _close(pool[vo:vo + kvd], nx.f16_to_f32_array(nx.f32_to_f16_array(vv[r])), 2e-3, 2e-3 * np.abs(vv).max(), "V row %d" % r)
    assert np.array_equal(pool[untouched], nx.f16_to_f32_array(pool0)[untouched])
    for p in list(dev.values()) + [dx, dnw, dpos, dslots, dpool, dq]:
        be.free(p)
    be.reset_pool()


# Q|K|V rows over 2048 wide where the streaming launch and the one that finishes its rows take the place of the kernel that finishes its
# own (12288 x 4096, Q4_K also 13824 x 4608), and where they do not: small matrices, Q4_0 rows over 4096 wide. A captured step takes the
# same launches as one that is not, whatever ran before it.
@pytest.mark.parametrize("fmt,heads,hidden,streamed", [(nx.FMT_Q4_0, 32, 4096, True), (nx.FMT_Q8_0, 32, 4096, True), (nx.FMT_Q4_K, 36, 4608, True),
                                                       (nx.FMT_Q8_0, 20, 2560, False), (nx.FMT_Q4_0, 18, 2304, False), (nx.FMT_Q4_0, 34, 4352, False)])
@pytest.mark.parametrize("rows", [2, 17, 32])
def test_qkv_streamed_or_finished_in_one_launch(rows, fmt, heads, hidden, streamed):
    from vexel_amd.backend import HipBackend
    be = HipBackend(0)          # (scratch that no other test has grown)
    rng = np.random.default_rng(rows + hidden)
    d, bs, nblocks, theta, eps = 128, 16, 4, 10000.0, 1e-5
    n = heads * d
    raw = [qz.random_quant(fmt, rng, n, hidden) for _ in range(3)]
    qws = [_packed(be, w, n, hidden, fmt)[1] for w in raw]
    x, nw = rng.standard_normal((rows, hidden)).astype(np.float32), (1.0 + 0.1 * rng.standard_normal(hidden)).astype(np.float32)
    positions, slots = rng.integers(0, 100, rows).astype(np.int32), rng.permutation(nblocks * bs)[:rows].astype(np.int32)
    h = nx.rmsnorm(x, nw, rows, hidden, eps)
    q, k, v = (nx.matmul_quant(fmt, h, w, rows, n, hidden) for w in raw)
    want_q, want_k = nx.rope_positions(q, k, d, heads, heads, positions, d, theta, False)
    dx, dnw, dpos, dslots = (be.upload(a, permanent=True) for a in (x, nw, positions, slots))
    per_block = 2 * bs * n
    dpool, dq = be.alloc_permanent(nblocks * per_block * 2), be.alloc_permanent(rows * n * 4)

    def step():
        be.decode_attn_qkv(dx, dnw, eps, True, *qws, rows, dpos, dslots, dpool, True, heads, heads, d, bs, theta, dq)

    def check():
        got_q = be.download(dq, (rows, n), np.float32)
        _close(got_q, want_q, 2e-4, 2e-5 * np.abs(want_q).max(), "Q")
        bits = be.download(dpool, (nblocks * per_block,), np.uint16).reshape(nblocks, 2, bs, n)
        pool = nx.f16_to_f32_array(bits.ravel()).reshape(bits.shape)
        for part, want in enumerate((want_k, v)):
            got = pool[slots // bs, part, slots % bs]
            _close(got, nx.f16_to_f32_array(nx.f32_to_f16_array(want)), 2e-3, 2e-3 * np.abs(want).max(), "K" if part == 0 else "V")
        be.to_device(dq, np.full((rows, n), np.nan, dtype=np.float32))
        stored = bits[slots // bs, :, slots % bs]
        bits[slots // bs, :, slots % bs] = 0x7E00
        be.to_device(dpool, bits)
        return got_q, stored

    kernel = "qstream_kernel" if streamed else "qgemm_wave_kernel"
    be.rmsnorm_prepare(dx, dnw, None, rows, hidden, eps)
    be.sync()
    be.graph_begin_capture()    # (before any call has asked for scratch for slices' sums)
    be.rope_table_prepare(dpos, rows, d, theta)
    step()
    recorded = be.last_matmul_kernel()
    graph = be.graph_end_capture()
    assert recorded == kernel
    be.rope_table_prepare(dpos, rows, d, theta)
    step()
    assert be.last_matmul_kernel() == kernel
    eager = check()
    for _ in range(3):
        be.graph_launch(graph)
        be.sync()
        got = check()
        assert all(np.array_equal(a, b) for a, b in zip(got, eager))
    be.graph_destroy(graph)
    be.close()


@pytest.mark.parametrize("fmt", [nx.FMT_Q4_0, nx.FMT_Q8_0, nx.FMT_Q4_K])
def test_streamed_qkv_rows_do_not_depend_on_the_batch(be, fmt):
    rng = np.random.default_rng(11)
    heads, kv_heads, d, hidden, bs, nblocks, theta, eps = 36, 30, 128, 4096, 16, 4, 10000.0, 1e-5
    qd, kvd = heads * d, kv_heads * d
    dev, qws = zip(*[_packed(be, qz.random_quant(fmt, rng, n, hidden), n, hidden, fmt) for n in (qd, kvd, kvd)])
    x, nw = rng.standard_normal((32, hidden)).astype(np.float32), (1.0 + 0.1 * rng.standard_normal(hidden)).astype(np.float32)
    positions, slots = rng.integers(0, 100, 32).astype(np.int32), rng.permutation(nblocks * bs)[:32].astype(np.int32)
    dx, dnw, dpos, dslots = (be.upload(a, permanent=True) for a in (x, nw, positions, slots))
    per_block = 2 * bs * kvd
    dpool, dq = be.alloc_permanent(nblocks * per_block * 2), be.alloc_permanent(32 * qd * 4)
    want = None
    for rows in (32, 17, 16, 2):
        be.rope_table_prepare(dpos, rows, d, theta)
        be.decode_attn_qkv(dx, dnw, eps, False, *qws, rows, dpos, dslots, dpool, True, heads, kv_heads, d, bs, theta, dq)
        assert be.last_matmul_kernel() == "qstream_kernel"
        pool = be.download(dpool, (nblocks * per_block,), np.uint16).reshape(nblocks, 2, bs, kvd)
        got = be.download(dq, (rows, qd), np.float32), pool[slots // bs, :, slots % bs][:rows]
        want = want or got
        assert all(np.array_equal(a, b[:rows]) for a, b in zip(got, want)), rows
        be.fill_zero(dpool, nblocks * per_block * 2)
    for p in list(dev) + [dx, dnw, dpos, dslots, dpool, dq]:
        be.free(p)
    be.reset_pool()


def qkv_with_and_without_angles(rows_min):
    """(In a process of its own, whose VEXEL_HIP_ROWS_MIN is rows_min.)"""
    from vexel_amd.backend import HipBackend
    be = HipBackend(0)
    rng = np.random.default_rng(rows_min)
    hq, hk, d, hidden, bs, nblocks, theta, eps, fmt = 4, 2, 64, 512, 16, 8, 10000.0, 1e-5, nx.FMT_Q8_0
    dims = dict(wq=(hq * d, hidden), wk=(hk * d, hidden), wv=(hk * d, hidden))
    qw = {n: be.qweight(fmt, be.upload(qz.random_quant(fmt, rng, *v)), *v) for n, v in dims.items()}
    dnw, pool0 = be.upload(np.ones(hidden, dtype=np.float32)), np.zeros(nblocks * 2 * bs * hk * d, dtype=np.float16)
    for rows in (rows_min - 1, rows_min, 32):
        dx = be.upload(rng.standard_normal((rows, hidden)).astype(np.float32))
        dpos, dslots = be.upload(np.arange(rows, dtype=np.int32) * 5), be.upload(rng.permutation(nblocks * bs)[:rows].astype(np.int32))
        got = []
        for table in (True, False):
            dpool, dq = be.upload(pool0), be.alloc(rows * hq * d * 4)
            if table:
                be.rope_table_prepare(dpos, rows, d, theta)
            else:
                be.to_device(dpos, np.arange(rows, dtype=np.int32) * 5)   # (the table falls)
            be.decode_attn_qkv(dx, dnw, eps, False, qw["wq"], qw["wk"], qw["wv"], rows, dpos, dslots, dpool, True, hq, hk, d, bs, theta, dq)
            assert be.last_matmul_kernel() == ("qgemm_wave_kernel" if table or rows < rows_min else "qgemm_rows_kernel"), (rows, table)
            got.append((be.download(dq, (rows, hq * d), np.float32), be.download(dpool, pool0.shape, np.float16).astype(np.float32)))
        for a, b, rel in zip(*got, (2e-5, 2.0 ** -10)):               # (float32 sums in another order; rounded to f16)
            assert np.abs(b).max() > 0 and np.all(np.abs(a - b) <= rel * np.abs(b).max())
    be.close()


@pytest.mark.parametrize("rows_min", [3, 17])
def test_switch_for_many_rows_leaves_the_rows_that_are_finished_alone(rows_min):
    """VEXEL_HIP_ROWS_MIN moves batches to a kernel that leaves sums, also where a step's table of angles lets the Q|K|V launch finish its rows: those
    stay with the kernel that does."""
    r = subprocess.run([sys.executable, "-c", "import test_gpu_stream_gemm as t; t.qkv_with_and_without_angles(%d)" % rows_min],
                       cwd=os.path.dirname(os.path.abspath(__file__)), env=dict(os.environ, VEXEL_HIP_ROWS_MIN=str(rows_min), PYTHONPATH=ROOT),
                       capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr[-2000:]

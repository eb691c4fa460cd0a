"""GPU parity: the HIP path, called through the C ABI (chadslab_amd.ops -> ctypes -> libchadq.so), against the
CPU oracle on the same seeded inputs.  Bit-exact for unpack/pack/dequant and integer accumulation; rel-L2
<= 1e-3 for fp32 outputs and <= 1e-2 for bf16 outputs against the float64 ground truth (tolerances from the
benchmark statement).  Full benchmark shapes are covered too: the numpy oracle finishes them in seconds.
"""
import os

import numpy as np
import pytest
import torch

from oracle import chadq_oracle as O

pytestmark = pytest.mark.gpu

TOL_F32 = 1e-3   # fp32 out
TOL_BF16 = 1e-2  # bf16 out
GOLD = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")
DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    from chadslab_amd import _lib, ops as _ops

    assert torch.cuda.is_available(), "these tests need the GPU"
    _lib.load()  # raises if libchadq.so is missing: there is no fallback to hide behind
    return _ops


def rng(seed):
    return np.random.Generator(np.random.PCG64(seed))


def bits(t):
    return t.view(torch.int16).cpu().numpy().view(np.uint16)


def bf16_tensor(b):
    return torch.from_numpy(b.view(np.int16)).view(torch.bfloat16).to(DEV)


def i4_case(seed, m, n, k, integer_x=False):
    from chadslab_amd import QWeightInt4G32

    r = rng(seed)
    u = r.integers(0, 16, (n, k), dtype=np.uint8)
    packed = (u[:, 0::2] | (u[:, 1::2] << 4)).astype(np.uint8)
    s = r.lognormal(-5, 0.5, (n, k // 32)).astype(np.float16)
    x = r.integers(-8, 9, (m, k)).astype(np.float32) if integer_x else r.standard_normal((m, k)).astype(np.float32)
    xb = O.f32_to_bf16(x)
    qw = QWeightInt4G32(torch.from_numpy(packed).to(DEV), torch.from_numpy(s).to(DEV))
    return packed, s, xb, qw


def i8_case(seed, m, n, k):
    from chadslab_amd import QWeightInt8

    r = rng(seed)
    x = r.standard_normal((m, k)).astype(np.float32)
    w = r.integers(-127, 128, (n, k), dtype=np.int8)
    s = r.uniform(0.001, 0.02, n).astype(np.float32)
    return x, w, s, QWeightInt8(torch.from_numpy(w).to(DEV), torch.from_numpy(s).to(DEV))


# ------------------------------------------------------------------ unpack / pack / dequant: bit-exact
@pytest.mark.parametrize("nbytes", [0, 1, 15, 16, 17, 255, 256, 4096 + 7, 1 << 20])
def test_unpack_bit_exact(ops, nbytes):
    wp = rng(nbytes).integers(0, 256, nbytes, dtype=np.uint8)
    if nbytes >= 256:
        wp[:256] = np.arange(256)  # every byte value
    out = ops.unpack_int4(torch.from_numpy(wp).to(DEV)).cpu().numpy()
    assert np.array_equal(out, O.unpack_int4(wp[None])[0] if nbytes else np.zeros(0, np.int8))


def test_unpack_unaligned_view(ops):
    wp = rng(3).integers(0, 256, 1001, dtype=np.uint8)
    t = torch.from_numpy(wp).to(DEV)[1:]  # data pointer off 16-byte alignment
    assert np.array_equal(ops.unpack_int4(t).cpu().numpy(), O.unpack_int4(wp[None, 1:])[0])


def test_pack_roundtrip(ops):
    q = rng(4).integers(-8, 8, (33, 130), dtype=np.int8)
    p = ops.pack_int4(torch.from_numpy(q).to(DEV))
    assert np.array_equal(p.cpu().numpy(), O.pack_int4(q))
    assert np.array_equal(ops.unpack_int4(p).cpu().numpy(), q)


def test_dequant_exact(ops):
    packed, s, _, qw = i4_case(5, 1, 96, 256)
    assert np.array_equal(ops.dequantize(qw).cpu().numpy(), O.dequant_int4g32(packed, s))
    _, w, s8, q8 = i8_case(6, 1, 50, 70)
    assert np.array_equal(ops.dequantize(q8).cpu().numpy(), O.dequant_int8(w, s8))


def test_bench_probe_reads_every_byte():
    # the loads-only kernel bench.py times beside the GEMV lives in its own small library next to bench.py
    import ctypes

    path = os.path.join(os.path.dirname(GOLD.rstrip(os.sep)), os.pardir, "bench_probe.so")
    if not os.path.exists(path):
        pytest.skip("bench_probe.so has not been built (__graft_entry__.build() builds it)")
    lib = ctypes.CDLL(os.path.abspath(path))
    lib.bench_probe_read.restype = ctypes.c_int
    lib.bench_probe_read.argtypes = [ctypes.c_void_p, ctypes.c_int64, ctypes.c_void_p, ctypes.c_void_p]
    n = 5 * 16384 + 100  # the tail that does not fill 16 KiB is left alone
    data = rng(11).integers(0, 256, n, dtype=np.uint8)
    t = torch.from_numpy(data).to(DEV)
    out = torch.zeros(n // 16384, dtype=torch.int32, device=DEV)
    assert lib.bench_probe_read(t.data_ptr(), n, out.data_ptr(), torch.cuda.current_stream().cuda_stream) == 0
    want = np.bitwise_xor.reduce(data[:5 * 16384].view(np.uint32).reshape(5, -1), axis=1)
    assert np.array_equal(out.cpu().numpy().view(np.uint32), want)


# ------------------------------------------------------------------ golden fixtures
def test_golden_int4(ops):
    from chadslab_amd import QWeightInt4G32

    g = np.load(os.path.join(GOLD, "i4g32_n64_k128.npz"))
    qw = QWeightInt4G32(torch.from_numpy(g["packed"]).to(DEV), torch.from_numpy(g["scale"]).to(DEV))
    x = bf16_tensor(g["x_bf16"])
    assert np.array_equal(ops.unpack_int4(qw.packed).cpu().numpy(), g["q"])
    assert np.array_equal(ops.dequantize(qw).cpu().numpy(), g["dequant"])
    assert O.rel_l2(ops.qgemv(x, qw).cpu().numpy(), g["y_f64"]) <= TOL_F32
    assert O.rel_l2(O.bf16_to_f32(bits(ops.qgemm(x, qw))), g["y_f64"]) <= TOL_BF16


def test_golden_int8(ops):
    from chadslab_amd import QWeightInt8

    g = np.load(os.path.join(GOLD, "i8row_n64_k128.npz"))
    q8 = QWeightInt8(torch.from_numpy(g["w"]).to(DEV), torch.from_numpy(g["scale"]).to(DEV))
    assert O.rel_l2(ops.qgemv(torch.from_numpy(g["x_f32"]).to(DEV), q8).cpu().numpy(), g["y_f64"]) <= TOL_F32
    assert O.rel_l2(O.bf16_to_f32(bits(ops.qgemm(bf16_tensor(g["x_bf16"]), q8))), g["yb_f64"]) <= TOL_BF16


# ------------------------------------------------------------------ GEMV int4 (config 1)
@pytest.mark.parametrize("m", [1, 2, 3, 4, 5, 8, 16])
@pytest.mark.parametrize("n,k", [(64, 128), (33, 32), (100, 4160), (48, 12288), (257, 2048), (1000, 4096), (16, 8192)])
def test_gemv_int4_shapes(ops, m, n, k):
    packed, s, xb, qw = i4_case(100 + m + n + k, m, n, k)
    y = ops.qgemv(bf16_tensor(xb), qw).cpu().numpy()
    assert y.shape == (m, n) and np.isfinite(y).all()
    assert O.rel_l2(y, O.qgemm_int4g32_f64(xb, packed, s)) <= TOL_F32


@pytest.mark.parametrize("m", [1, 2, 3, 4, 5, 6, 7, 8, 9, 13, 16])
def test_gemv_int4_config1_full_size(ops, m):
    packed, s, xb, qw = i4_case(1001, m, 14336, 4096)
    y = ops.qgemv(bf16_tensor(xb), qw).cpu().numpy()
    assert O.rel_l2(y, O.qgemm_int4g32_f64(xb, packed, s)) <= TOL_F32


@pytest.mark.parametrize("m,n,k", [(1, 32768, 2048), (1, 8200, 1024), (2, 8192, 8192), (5, 9001, 4096), (3, 8192, 256),
                                   (1, 11008, 4096), (2, 12345, 512), (4, 20000, 512), (8, 28672, 512), (1, 5000, 2048),
                                   (7, 12345, 768)])
def test_gemv_int4_tall_matrices(ops, m, n, k):
    # 8192 rows and more take the kernels with 32- and 64-row workgroups (a ragged last workgroup included); row
    # counts that would end mid-round on the chip run with tiles of 6, 7, 12, 13 or 14 rows instead of 8 or 16
    packed, s, xb, qw = i4_case(3000 + n + k, m, n, k)
    y = ops.qgemv(bf16_tensor(xb), qw).cpu().numpy()
    assert np.isfinite(y).all() and O.rel_l2(y, O.qgemm_int4g32_f64(xb, packed, s)) <= TOL_F32


@pytest.mark.parametrize("m", [1, 4])
def test_gemv_int4_output_table_256000_rows(ops, m):
    # the decode step's output projection: 256000 rows of K = 2048 (the tallest matrix the benchmark has); the float64
    # truth and the integer brute force are formed 32000 rows at a time to keep the host's copies small
    from chadslab_amd import QWeightInt4G32

    n, k, step = 256000, 2048, 32000
    packed, s, xb, qw = i4_case(4100 + m, m, n, k)
    y = ops.qgemv(bf16_tensor(xb), qw).cpu().numpy()
    assert y.shape == (m, n) and np.isfinite(y).all()
    want = np.concatenate([O.qgemm_int4g32_f64(xb, packed[r: r + step], s[r: r + step]) for r in range(0, n, step)], axis=1)
    assert O.rel_l2(y, want) <= TOL_F32
    xi = O.f32_to_bf16(rng(4102).integers(-8, 9, (m, k)).astype(np.float32))
    yi = ops.qgemv(bf16_tensor(xi), QWeightInt4G32(qw.packed, torch.ones_like(qw.scale))).cpu().numpy()
    xf = O.bf16_to_f32(xi).astype(np.float64)  # small integers: float64 sums of their products are exact
    brute = np.concatenate([xf @ O.unpack_int4(packed[r: r + step]).astype(np.float64).T for r in range(0, n, step)], axis=1)
    assert np.abs(brute).max() < 2 ** 24 and np.array_equal(yi, brute.astype(np.float32))


@pytest.mark.parametrize("m,n,k", [(1, 14336, 4096), (2, 14336, 4096), (8, 512, 4096), (4, 96, 256), (2, 40, 96),
                                   (5, 14336, 4096), (8, 14336, 4096), (6, 300, 512), (7, 8192, 256),
                                   (9, 8192, 2048), (12, 14336, 4096), (16, 512, 4096), (16, 300, 512), (11, 64, 256)])
def test_gemv_int4_integer_accumulation_bit_exact(ops, m, n, k):
    from chadslab_amd import QWeightInt4G32

    packed, _, xb, qw = i4_case(7, m, n, k, integer_x=True)
    ones = QWeightInt4G32(qw.packed, torch.ones_like(qw.scale))
    y = ops.qgemv(bf16_tensor(xb), ones).cpu().numpy()
    brute = O.bf16_to_f32(xb).astype(np.int64) @ O.unpack_int4(packed).astype(np.int64).T
    assert np.abs(brute).max() < 2 ** 24
    assert np.array_equal(y.astype(np.int64), brute) and np.array_equal(y, brute.astype(np.float32))


def test_gemv_int4_row_consistency_and_linearity(ops):
    packed, s, xb, qw = i4_case(8, 8, 512, 4096)
    x = bf16_tensor(xb)
    y8 = ops.qgemv(x, qw).cpu().numpy()
    for r in (0, 3, 7):
        y1 = ops.qgemv(x[r:r + 1].contiguous(), qw).cpu().numpy()
        assert O.rel_l2(y1[0], y8[r]) <= 1e-6  # same products, possibly another summation order
    a = rng(9).integers(-64, 64, (1, 4096)).astype(np.float32)
    b = rng(10).integers(-64, 64, (1, 4096)).astype(np.float32)
    ya, yb, yab = (ops.qgemv(bf16_tensor(O.f32_to_bf16(v)), qw).cpu().numpy() for v in (a, b, a + b))
    assert O.rel_l2(yab, ya + yb) <= 1e-5


def test_gemv_int4_zero_weights_and_special_scales(ops):
    from chadslab_amd import QWeightInt4G32

    n, k = 64, 4096
    x = bf16_tensor(O.f32_to_bf16(rng(11).standard_normal((2, k)).astype(np.float32)))
    zero = QWeightInt4G32(torch.full((n, k // 2), 0x88, dtype=torch.uint8, device=DEV), torch.ones(n, k // 32, dtype=torch.float16, device=DEV))
    y = ops.qgemv(x, zero).cpu().numpy()
    # u = 8 everywhere: the 128+u offset must cancel; what is left is fp32 rounding of sums near 136*sum|x|,
    # about 1e-4 of the size a typical output has for these shapes (~300)
    assert np.abs(y).max() <= 2e-2
    # one-hot activation returns one dequantised column exactly
    packed, s, _, qw = i4_case(12, 1, n, k)
    d = O.dequant_int4g32(packed, s)
    for kk in (0, 31, 32, 2047, 4095):
        e = np.zeros((1, k), np.float32)
        e[0, kk] = 1.0
        assert np.array_equal(ops.qgemv(bf16_tensor(O.f32_to_bf16(e)), qw).cpu().numpy()[0], d[:, kk])


# K not a multiple of 256: the matrix cores take five rows and more (three of more than 4096 k), whole and part scale groups of a step
@pytest.mark.parametrize("m,n,k", [(5, 1, 32), (16, 65, 96), (7, 63, 1056), (16, 200, 4064), (3, 130, 4128), (5, 31, 4128), (3, 77, 8160),
                                   (16, 77, 8160)])
def test_gemv_int4_other_k_several_rows(ops, m, n, k):
    packed, s, xb, q4 = i4_case(80 + m, m, n, k)
    ref = O.qgemm_int4g32_f64(xb, packed, s)
    # every product is exact; what is left is the fp32 sum of at most k terms and the scales' products
    u = np.stack([packed & 15, packed >> 4], 2).reshape(n, k).astype(np.float64) - 8
    mag = np.abs(O.bf16_to_f32(xb)).astype(np.float64) @ (np.abs(u) * np.repeat(s.astype(np.float64), 32, 1)).T
    x = bf16_tensor(xb)
    y = ops.qgemv(x, q4).cpu().numpy()
    assert (np.abs(y - ref) <= (k / 8 + 8) * 2.0**-24 * mag).all()
    yb = ops.qlinear(x, q4, out_dtype=torch.bfloat16)
    assert (np.abs(O.bf16_to_f32(bits(yb)) - ref) <= 2.0**-8 * np.abs(ref) + (k / 8 + 8) * 2.0**-24 * mag).all()


# ------------------------------------------------------------------ GEMV int8 (config 0)
@pytest.mark.parametrize("m,n,k", [(1, 16384, 2048), (1, 64, 16), (3, 100, 1040), (2, 77, 4096), (16, 40, 256),
                                   # rows of 2049..8192 k (4 or 8 chunks per row), and beyond (the general kernel)
                                   (1, 5000, 4096), (2, 300, 3008), (1, 4500, 8192), (3, 33, 6000), (1, 50, 8208),
                                   (1, 9000, 1024), (2, 8200, 528)])
def test_gemv_int8(ops, m, n, k):
    x, w, s, q8 = i8_case(1000 if (n, k) == (16384, 2048) else 20 + n, m, n, k)
    y = ops.qgemv(torch.from_numpy(x).to(DEV), q8).cpu().numpy()
    assert O.rel_l2(y, O.qgemv_int8_f64(x, w, s)) <= TOL_F32


# K a multiple of 128 runs on the int8 matrix core (activations as three fixed-point digits per 2048 k), one pass over
# the weights for any M <= 16; other K keep the fp32 kernels
@pytest.mark.parametrize("m,n,k", [(1, 16384, 2048), (4, 16384, 2048), (5, 16384, 2048), (8, 16384, 2048), (9, 16384, 2048),
                                   (16, 16384, 2048), (1, 1, 128), (4, 63, 128), (5, 65, 256), (8, 129, 1152), (12, 200, 2176),
                                   (16, 77, 1920), (3, 4100, 4096), (7, 300, 6144), (16, 130, 8192), (2, 50, 10240),
                                   (13, 70, 12416)])
def test_gemv_int8_matrix_core(ops, m, n, k):
    x, w, s, q8 = i8_case(300 + m + n, m, n, k)
    y = ops.qgemv(torch.from_numpy(x).to(DEV), q8).cpu().numpy()
    assert O.rel_l2(y, O.qgemv_int8_f64(x, w, s)) <= TOL_F32


# 16, 32 or 64 weight rows to a workgroup: either side of each line, ragged, with less k than its waves have parts
@pytest.mark.parametrize("n", [4096, 4097, 8192, 8205])
@pytest.mark.parametrize("m,k", [(1, 128), (4, 2048), (6, 2176), (16, 4224)])
def test_gemv_int8_matrix_core_rows_per_workgroup(ops, m, n, k):
    x, w, s, q8 = i8_case(340 + m + n, m, n, k)
    y = ops.qgemv(torch.from_numpy(x).to(DEV), q8).cpu().numpy()
    ref = O.qgemv_int8_f64(x, w, s)
    # every element: fixed point drops at most 2^-21 of the row's largest |x| per product, the one rounding to fp32 and the scale 2^-23
    bound = 2.0**-21 * np.abs(x).max(1)[:, None] * (np.abs(w.astype(np.float64)).sum(1) * s)[None] + 2.0**-22 * np.abs(ref)
    assert (np.abs(y - ref) <= bound).all()


@pytest.mark.parametrize("m,n,k", [(2, 300, 2048), (2, 300, 2064), (1, 100, 4096), (5, 333, 4096), (8, 64, 2048), (16, 70, 6144),
                                   (11, 90, 128)])
def test_gemv_int8_integer_exact(ops, m, n, k):
    from chadslab_amd import QWeightInt8

    r = rng(21 + m)
    x = r.integers(-8, 9, (m, k)).astype(np.float32)
    w = r.integers(-128, 128, (n, k), dtype=np.int8)
    q8 = QWeightInt8(torch.from_numpy(w).to(DEV), torch.ones(n, device=DEV))
    y = ops.qgemv(torch.from_numpy(x).to(DEV), q8).cpu().numpy()
    assert np.array_equal(y.astype(np.int64), x.astype(np.int64) @ w.astype(np.int64).T)


def test_gemv_int8_rows_do_not_depend_on_their_neighbours(ops):
    """Row m of an M-row call equals the one-row call on x[m] bit for bit (per-row scales, exact integer sums), for
    every form of the matrix-core kernel (M <= 4, <= 8, <= 16) and across a 2048-k block boundary."""
    x, w, s, q8 = i8_case(77, 16, 333, 4096)
    xt = torch.from_numpy(x).to(DEV)
    one = torch.cat([ops.qgemv(xt[i:i + 1], q8) for i in range(16)]).cpu().numpy()
    for m in (3, 4, 7, 8, 11, 16):
        assert np.array_equal(ops.qgemv(xt[:m], q8).cpu().numpy(), one[:m]), m


def test_gemv_int8_outliers_zero_rows_and_non_finite_values(ops):
    x, w, s, q8 = i8_case(78, 6, 200, 4096)
    x[0, 17] = 3.0e6          # one huge value: the block's fixed-point scale follows it
    x[1, :] = 0.0             # an all-zero row
    x[2, 2048:] *= 1.0e-20    # a block of tiny values next to an ordinary one
    x[3, :] *= 1.0e15
    y = ops.qgemv(torch.from_numpy(x).to(DEV), q8).cpu().numpy()
    ref = O.qgemv_int8_f64(x, w, s)
    for m in range(6):
        assert O.rel_l2(y[m:m + 1], ref[m:m + 1]) <= TOL_F32 or not ref[m].any(), m
    assert not y[1].any()
    x[4, 3000] = np.inf
    x[5, 5] = np.nan
    y2 = ops.qgemv(torch.from_numpy(x).to(DEV), q8).cpu().numpy()
    assert np.isnan(y2[4]).all() and np.isnan(y2[5]).all()   # a non-finite activation makes its own row NaN ...
    assert np.array_equal(y2[:4], y[:4])                      # ... and no other


def test_gemv_int8_outlier_column_error_bound_per_element(ops):
    """The matrix-core int8 GEMV holds a block of 2048 activations in fixed point relative to the block's largest |x|:
    the header's bound |err| <= |s[n]| * sum over blocks of 2^-21 * max|x| * sum|W[n,k]| is checked element by element
    with one outlier column, in particular on output rows whose weight at the outlier is ZERO (there the outlier adds
    nothing to the exact result and the whole difference is the other elements' lost low bits).  chadq_gemv_i8row_fp32
    has no such term: the same inputs come out at fp32 accuracy."""
    m_rows, n, k = 5, 512, 4096
    x, w, s, _ = i8_case(781, m_rows, n, k)
    col = 17
    x[:, col] = 3.0e6 * np.array([1, -1, 1, 1, -1], np.float32)
    w[::2, col] = 0                              # every other output row ignores the outlier
    x[3, 2048 + 5] = -7.0e4                      # a second, smaller outlier in row 3's second block
    from chadslab_amd import QWeightInt8

    q8 = QWeightInt8(torch.from_numpy(w).to(DEV), torch.from_numpy(s).to(DEV))
    xt = torch.from_numpy(x).to(DEV)
    ref = O.qgemv_int8_f64(x, w, s)
    y = ops.qgemv(xt, q8).cpu().numpy().astype(np.float64)
    aw = np.abs(w.astype(np.float64))
    bound = np.zeros((m_rows, n))
    for b0 in range(0, k, 2048):
        bmax = np.abs(x[:, b0:b0 + 2048]).max(axis=1).astype(np.float64)            # [M]
        bound += 2.0 ** -21 * bmax[:, None] * aw[:, b0:b0 + 2048].sum(axis=1)[None, :]
    bound = np.abs(s.astype(np.float64))[None, :] * bound
    slack = 4e-7 * np.abs(ref) + 1e-30                                               # the fp32 roundings of the sums
    err = np.abs(y - ref)
    assert (err <= bound + slack).all(), float((err / (bound + slack)).max())
    # the bound is not vacuous: on the rows that ignore the outlier the error is a visible fraction of the result ...
    zero_rows = err[:, ::2] / (np.abs(ref[:, ::2]) + 1e-30)
    assert np.median(zero_rows) > 1e-3
    # ... and the fp32 form has none of it
    yf = ops.qgemv(xt, q8, fp32_elements=True).cpu().numpy().astype(np.float64)
    mag = (np.abs(x.astype(np.float64)) @ (aw * np.abs(s.astype(np.float64))[:, None]).T)  # sum of |terms|
    assert (np.abs(yf - ref) <= 1e-5 * mag).all()
    assert np.median(np.abs(yf[:, ::2] - ref[:, ::2]) / (np.abs(ref[:, ::2]) + 1e-30)) < 1e-5


@pytest.mark.parametrize("m,n,k", [(1, 16384, 2048), (2, 300, 4096), (5, 333, 2048), (16, 70, 6144), (3, 100, 1040)])
def test_gemv_int8_fp32_elements_entry_point(ops, m, n, k):
    x, w, s, q8 = i8_case(790 + m, m, n, k)
    y = ops.qgemv(torch.from_numpy(x).to(DEV), q8, fp32_elements=True).cpu().numpy()
    assert O.rel_l2(y, O.qgemv_int8_f64(x, w, s)) <= TOL_F32
    xi = rng(791 + m).integers(-2000, 2001, (m, k)).astype(np.float32)
    one = type(q8)(q8.w, torch.ones_like(q8.scale))
    yi = ops.qgemv(torch.from_numpy(xi).to(DEV), one, fp32_elements=True).cpu().numpy()
    want = xi.astype(np.int64) @ w.astype(np.int64).T
    ok = np.abs(want) < 2 ** 24
    assert np.array_equal(yi[ok].astype(np.int64), want[ok])
    xinf = x.copy()
    xinf[0, 3] = np.inf
    yinf = ops.qgemv(torch.from_numpy(xinf).to(DEV), q8, fp32_elements=True).cpu().numpy()
    nz = w[:, 3] != 0  # IEEE arithmetic element by element: inf * w is an infinity, inf * 0 a NaN
    assert np.isinf(yinf[0][nz]).all() and np.isnan(yinf[0][~nz]).all()
    assert np.isfinite(yinf[1:]).all()


def test_gemv_int8_integer_digit_sums_that_cancel_stay_exact(ops):
    """The matrix-core kernel sums three base-256 digits of the fixed-point activations separately and recombines
    D0 * 2^16 + D1 * 2^8 + D2.  Here the digit sums are far beyond 2^24 and cancel: x = 32768 (digits 1, -128, 0)
    against weights +64 and x = 32512 (digits 0, 127, 0) against weights -64, so D0 * 2^16 = 2.1e9 and D1 * 2^8 = -2.1e9
    while the result is 8.4e6 + small.  Recombined in float64 the result is the exact integer (fp32 recombination
    was off by up to 128 here)."""
    n, k = 64, 2048
    r = rng(795)
    w = np.zeros((n, k), np.int8)
    x = np.zeros((1, k), np.float32)
    x[0, 0:1024:2], x[0, 1:1024:2] = 32768.0, 32512.0
    w[:, 0:1024:2], w[:, 1:1024:2] = 64, -64
    w[:, 0:1024:2] += r.integers(-1, 2, (n, 512)).astype(np.int8)   # a little variety per output row
    x[0, 1024:1100] = r.integers(-50, 51, 76)                        # the other half of K: small integers
    w[:, 1024:1100] = r.integers(-127, 128, (n, 76))
    from chadslab_amd import QWeightInt8

    q8 = QWeightInt8(torch.from_numpy(w).to(DEV), torch.ones(n, device=DEV))
    want = x.astype(np.int64) @ w.astype(np.int64).T
    assert np.abs(want).max() < 2 ** 24 and np.abs(want).min() > 2 ** 22
    y = ops.qgemv(torch.from_numpy(x).to(DEV), q8).cpu().numpy()
    assert np.array_equal(y.astype(np.int64), want)


# ------------------------------------------------------------------ seeded random shapes (ragged edges of every kind)
def test_random_shapes_int4_gemv_and_gemm(ops):
    r = rng(4242)
    for case in range(36):
        m = int(r.choice([1, 2, 3, 4, 5, 7, 8, 9, 16, 17, 40, 130]))
        n = int(r.integers(1, 700)) if case % 3 else int(r.integers(8192, 9500))
        k = 32 * int(r.integers(1, 70))
        if n >= 8192:
            k = 32 * int(r.integers(1, 20))  # keep the float64 reference quick
        packed, s, xb, qw = i4_case(5000 + case, m, n, k)
        ref = O.qgemm_int4g32_f64(xb, packed, s)
        if m <= 16:
            y = ops.qgemv(bf16_tensor(xb), qw).cpu().numpy()
            assert y.shape == (m, n) and np.isfinite(y).all() and O.rel_l2(y, ref) <= TOL_F32, ("gemv", m, n, k)
        yb = O.bf16_to_f32(bits(ops.qgemm(bf16_tensor(xb), qw)))
        assert yb.shape == (m, n) and np.isfinite(yb).all() and O.rel_l2(yb, ref) <= TOL_BF16, ("gemm", m, n, k)


def test_random_shapes_int8(ops):
    r = rng(4243)
    for case in range(16):
        m = int(r.choice([1, 3, 8, 33, 129]))
        n = int(r.integers(1, 600))
        k = 16 * int(r.integers(1, 90))
        x, w, s, q8 = i8_case(6000 + case, m, n, k)
        xb = O.f32_to_bf16(x)
        yb = O.bf16_to_f32(bits(ops.qgemm(bf16_tensor(xb), q8)))
        assert O.rel_l2(yb, O.qgemm_int8_f64(xb, w, s)) <= TOL_BF16, ("gemm8", m, n, k)
        y1 = ops.qgemv(torch.from_numpy(x[:1]).to(DEV), q8).cpu().numpy()
        ref1 = (x[:1].astype(np.float64) @ (w.astype(np.float64) * s[:, None].astype(np.float64)).T)
        assert O.rel_l2(y1, ref1) <= TOL_F32, ("gemv8", n, k)
    # the GEMV at every M it takes: K a multiple of 128 (int8 matrix core, all three operand forms, one to six
    # 2048-blocks) and other K (fp32 kernels), ragged N
    for case in range(40):
        m = int(r.integers(1, 17))
        n = int(r.integers(1, 400)) if case % 4 else int(r.integers(8192, 8400))
        k = 128 * int(r.integers(1, 90)) if case % 2 else 16 * int(r.integers(1, 300))
        if n >= 8192:
            k = min(k, 2048)
        x, w, s, q8 = i8_case(7000 + case, m, n, k)
        y = ops.qgemv(torch.from_numpy(x).to(DEV), q8).cpu().numpy()
        assert y.shape == (m, n) and np.isfinite(y).all() and O.rel_l2(y, O.qgemv_int8_f64(x, w, s)) <= TOL_F32, ("gemv8", m, n, k)


# ------------------------------------------------------------------ prefill GEMM (config 2)
@pytest.mark.parametrize("m,n,k", [(512, 4096, 4096), (1, 64, 128), (37, 100, 96), (130, 70, 288), (5, 33, 32), (128, 64, 256), (200, 192, 1056)])
def test_gemm_int4(ops, m, n, k):
    packed, s, xb, qw = i4_case(1002 if m == 512 else 30 + m, m, n, k)
    y = O.bf16_to_f32(bits(ops.qgemm(bf16_tensor(xb), qw)))
    assert y.shape == (m, n)
    assert O.rel_l2(y, O.qgemm_int4g32_f64(xb, packed, s)) <= TOL_BF16


@pytest.mark.parametrize("m,n,k", [(512, 4096, 4096), (3, 40, 16), (129, 65, 272), (64, 128, 128)])
def test_gemm_int8(ops, m, n, k):
    x, w, s, q8 = i8_case(40 + m, m, n, k)
    xb = O.f32_to_bf16(x)
    y = O.bf16_to_f32(bits(ops.qgemm(bf16_tensor(xb), q8)))
    assert O.rel_l2(y, O.qgemm_int8_f64(xb, w, s)) <= TOL_BF16


@pytest.mark.parametrize("m,n,k", [(4096, 4096, 512), (3300, 3500, 256), (2817, 4099, 768), (8192, 1536, 1024)])
def test_gemm_int4_many_rows_tile(ops, m, n, k):
    # enough 256 x 256 tiles to cover the chip: these shapes run on the large-tile kernel (K a multiple of 256), with
    # ragged last tiles in both directions and, for n = 4099, rows the vector stores cannot take
    packed, s, xb, qw = i4_case(600 + m + n + k, m, n, k)
    y = O.bf16_to_f32(bits(ops.qgemm(bf16_tensor(xb), qw)))
    assert y.shape == (m, n) and np.isfinite(y).all()
    assert O.rel_l2(y, O.qgemm_int4g32_f64(xb, packed, s)) <= TOL_BF16


@pytest.mark.parametrize("m,n,k", [(385, 8200, 64), (641, 4100, 96), (1025, 4095, 32), (1024, 4096, 384), (897, 4223, 1312),  # some of each
                                   (3841, 3847, 32), (4096, 4097, 288), (3840, 4096, 256),                                # 256 x 256
                                   (17, 100, 32), (32, 515, 512), (33, 1000, 4352), (64, 64, 256), (63, 4097, 1056),      # 64 x 64, at most 64 rows
                                   (65, 100, 32), (128, 8192, 64), (129, 5440, 1056), (1000, 1000, 288), (2049, 447, 512)])   # and in one round
@pytest.mark.parametrize("weight", ["int4", "int8"])
def test_gemm_eight_wave_tiles_every_row_and_column(ops, weight, m, n, k):
    """The tiles of gemm_tile_q.hip at ragged ends of rows, columns and k (k of one, two and three steps, no multiple of a
    step or of a 256-k block of scales).  Every row and every column of the result is held to the bf16 bound by itself, so
    that one wrong row at the edge of a tile cannot hide in the norm of the whole."""
    if weight == "int4":
        packed, s, xb, qw = i4_case(620 + m + k, m, n, k)
        ref = O.qgemm_int4g32_f64(xb, packed, s)
    else:
        x, w, s, qw = i8_case(620 + m + k, m, n, k)
        xb = O.f32_to_bf16(x)
        ref = O.qgemm_int8_f64(xb, w, s)
    y = O.bf16_to_f32(bits(ops.qgemm(bf16_tensor(xb), qw)))
    err = (y - ref) ** 2
    for axis in (0, 1):
        assert np.sqrt(err.sum(axis=axis) / (ref ** 2).sum(axis=axis)).max() <= TOL_BF16


@pytest.mark.parametrize("m,n,k", [(69, 3963, 32), (555, 1697, 96), (193, 4000, 512), (190, 4097, 1056),
                                   (99, 8259, 32), (509, 3918, 96), (512, 4095, 512), (385, 5000, 1312),
                                   (259, 8306, 512), (259, 6663, 1312), (276, 8097, 768),
                                   (390, 8279, 32), (1159, 3291, 160), (386, 11008, 256), (577, 5500, 544),
                                   (588, 8210, 32), (635, 8317, 160), (600, 8300, 512), (513, 8193, 1312)])
@pytest.mark.parametrize("weight", ["int4", "int8"])
def test_gemm_tiles_between_64_and_256_rows(ops, weight, m, n, k):
    """Grids of one to a few rounds, where the rule by size weighs all tiles against each other, ragged in rows, columns and k; every row and
    column by itself, as above.  (Each tile at the sizes where it can go wrong: test_gemm_each_tile_by_itself.)"""
    test_gemm_eight_wave_tiles_every_row_and_column(ops, weight, m, n, k)


TILES = [("32x64", 256), ("64x64", 256), ("96x64", 128), ("128x64", 128), ("96x128", 128), ("128x128", 128), ("192x128", 64), ("256x128", 64),
         ("256x256", 64), ("short 32x64", 256), ("short 64x64", 256), ("short 128x128", 128), ("short 256x256", 64)]  # k of a step


@pytest.mark.parametrize("tile", range(len(TILES)), ids=[t[0] for t in TILES])
@pytest.mark.parametrize("weight", ["int4", "int8"])
def test_gemm_each_tile_by_itself(ops, weight, tile):
    """Every tile at ragged ends of rows and columns, whichever the rule by size would take: k of one step, of as many as there are stages, of
    more than the unrolled loop takes and in between, with and without a remainder; int4 scales that are not 16-byte aligned."""
    import ctypes

    from chadslab_amd import _lib

    name, step = TILES[tile]
    if name == "short 256x256" and weight == "int8":
        pytest.skip("not built: never the faster one")
    launch = _lib.load()["_ZN5chadq22gemm_tile_i4g32_launchEPKtPKhS1_PtiiiNS_8GemmTileEP12ihipStream_t" if weight == "int4" else
                         "_ZN5chadq22gemm_tile_i8row_launchEPKtPKaPKfPtiiiNS_8GemmTileEP12ihipStream_t"]
    launch.argtypes = [ctypes.c_void_p] * 4 + [ctypes.c_int] * 4 + [ctypes.c_void_p]
    bm, bn = (int(v) for v in name.split()[-1].split("x"))
    if weight == "int4":
        ks = [256, 512, 768, 1024, 2304, 2560] + [32, 96, step + 32, 2 * step + 160, 4 * step + 96, 9 * step + 32, 1056]
    else:
        ks = [step * i for i in (1, 2, 3, 4, 6, 9, 10)] + [16, 48, step + 16, 2 * step + 144, 4 * step + 80, 9 * step + 16]
    for i, k in enumerate(ks):
        m, n = ((bm + 3, bn + 5), (2 * bm - 1, 3), (bm, 2 * bn))[i % 3]
        seed = 660 + 100 * tile + i
        if weight == "int4":
            packed, s, xb, q = i4_case(seed, m, n, k)
            w, sc = q.packed, q.scale
            wv = O.bf16_to_f32(O.f32_to_bf16(O.dequant_int4g32(packed, s))).astype(np.float64)  # as the matrix cores get them
        else:
            xf, wn, s, q = i8_case(seed, m, n, k)
            xb = O.f32_to_bf16(xf)
            w, sc, wv = q.w, q.scale, wn * s.astype(np.float64)[:, None]
        xv = O.bf16_to_f32(xb).astype(np.float64)
        ref, mag = xv @ wv.T, np.abs(xv) @ np.abs(wv).T
        x = bf16_tensor(xb)
        scales = [sc]
        if weight == "int4" and k % 256 == 0:
            scales.append(torch.cat((sc.new_zeros(1), sc.reshape(-1)))[1:])
        for sv in scales:
            y = torch.full((m + 1, n), 7.0, dtype=torch.bfloat16, device=DEV)
            assert launch(x.data_ptr(), w.data_ptr(), sv.data_ptr(), y.data_ptr(), m, n, k, tile, torch.cuda.current_stream().cuda_stream) == 0
            assert bool((y[m] == 7).all()), ("a row too many", k)
            # the products are exact in fp32: the fp32 sum of at most k terms, the rounding to bf16
            assert (np.abs(O.bf16_to_f32(bits(y[:m])) - ref) <= 2.0**-8 * np.abs(ref) + (k / 8 + 8) * 2.0**-24 * mag).all(), (m, n, k)


@pytest.mark.parametrize("tile,gated,shapes", [
    ("32x64", False, [(1, 64, 256, 1), (31, 192, 768, 2), (32, 64, 2560, 8)]),
    ("64x64", False, [(33, 64, 256, 1), (64, 192, 768, 2), (67, 192, 1280, 2), (129, 512, 2560, 4), (300, 2048, 3072, 3), (193, 1000, 2048, 4)]),
    ("128x128", False, [(396, 9280, 256, 1), (515, 5248, 512, 1), (130, 7168, 768, 2), (129, 8192, 2560, 4), (385, 5120, 1792, 3)]),
    ("128x64", False, [(641, 8192, 1024, 1), (177, 7600, 2560, 1), (153, 6000, 3072, 2), (255, 2048, 4096, 3), (256, 2048, 16384, 4), (348, 3392, 3584, 3), (197, 7232, 256, 1), (193, 1472, 2048, 4)]),
    ("32x64", True, [(1, 512, 256), (32, 1024, 768)]),
    ("64x64", True, [(33, 512, 512), (70, 2560, 2048), (257, 512, 1024)]),
    ("128x64", True, [(208, 4160, 2304), (130, 6976, 1792), (335, 2880, 2304), (257, 5376, 1280)]),
    ("128x128", True, [(300, 32768, 256), (130, 12288, 768), (70, 16896, 512), (97, 20480, 2048)]),
    ("256x128", True, [(130, 20480, 256), (257, 32768, 512), (511, 16384, 768), (256, 32768, 2048)])])
def test_exact_products_of_each_tile(ops, tile, gated, shapes):
    """A prompt's products by themselves, every tile at ragged ends of its rows, one step and more than the unrolled loop takes, K splits of
    uneven length; element by element against float64.  The rule by size is asked which tile it is, so that a list goes with its tile.  The
    activations carry the factor 2^-5 that these products expect, a gated result has it too; both are exact here."""
    import ctypes

    from chadslab_amd import _lib

    lib = _lib.load()
    rule = lib["_ZN5chadq15gemm_exact_tileEiiiibPfPi"]
    rule.argtypes = [ctypes.c_int] * 4 + [ctypes.c_bool, ctypes.POINTER(ctypes.c_float), ctypes.POINTER(ctypes.c_int)]
    launch = lib["_ZN5chadq30gemm_exact_scaled_geglu_launchEPKtPKhS1_PtiiiP12ihipStream_t" if gated else
                 "_ZN5chadq28gemm_exact_scaled_f32_launchEPKtPKhS1_PfiiiiP12ihipStream_t"]
    launch.argtypes = [ctypes.c_void_p] * 4 + [ctypes.c_int] * (3 if gated else 4) + [ctypes.c_void_p]
    for i, (m, n, k, *splits) in enumerate(shapes):
        per = -(-(k // 256) // (splits[0] if splits else 1))
        parts = -(-(k // 256) // per)
        columns = ctypes.c_int()
        rows = rule(m, n, per, parts, gated, ctypes.byref(ctypes.c_float()), ctypes.byref(columns))
        assert "%dx%d" % (rows, columns.value) == tile, (m, n, k)
        g = torch.Generator(device=DEV)
        g.manual_seed(9700 + 10 * rows + columns.value + i)
        packed = torch.randint(0, 256, (n, k // 2), dtype=torch.uint8, device=DEV, generator=g)
        scale = torch.exp(torch.randn(n, k // 32, device=DEV, generator=g) * 0.5 - 4.0).half()
        x = torch.randn(m, k, device=DEV, generator=g).bfloat16()
        scaled = (x.float() * 2.0 ** -5).bfloat16()
        w = torch.stack([packed & 15, packed >> 4], 2).reshape(n, k).double().sub_(8.0).mul_(scale.double().repeat_interleave(32, 1))
        ref, mag = x.double() @ w.t(), x.double().abs() @ w.abs().t()
        # 32 products of a group, its sum among K / 32 of them, the waves' and the parts' sums; an ulp each, as the matrix cores may truncate
        err = (k / 32 + 48) * 2.0**-23 * mag
        s = torch.cuda.current_stream().cuda_stream
        if gated:
            y = torch.full((m + 1, n // 2), 7.0, dtype=torch.bfloat16, device=DEV)
            assert launch(scaled.data_ptr(), packed.data_ptr(), scale.data_ptr(), y.data_ptr(), m, n, k, s) == 0
            got = y[:m].double() * 32
            gate, up = ref[:, ::2], ref[:, 1::2]
            ref = torch.nn.functional.gelu(gate, approximate="tanh") * up
            # |gelu'| <= 1.13 and |gelu(g)| <= |g|; gelu itself to 2^-18 of its argument; the result rounded to bf16
            err = 2.0**-8 * ref.abs() + 1.2 * err[:, ::2] * up.abs() + gate.abs() * err[:, 1::2] + 2.0**-18 * (gate * up).abs()
        else:
            y = torch.full((parts * m + 1, n), 7.0, device=DEV)
            assert launch(scaled.data_ptr(), packed.data_ptr(), scale.data_ptr(), y.data_ptr(), m, n, k, parts, s) == 0
            got = y[:parts * m].view(parts, m, n).double().sum(0)
        assert bool((y[-1] == 7).all()), "a row too many"
        assert bool(((got - ref).abs() <= err).all()), (m, n, k, float(((got - ref).abs() / err).max()))


@pytest.mark.parametrize("more", [0, 1])
@pytest.mark.parametrize("weight", ["int4", "int8"])
def test_gemm_of_rows_beyond_the_tiles_offsets(ops, weight, more):
    """K of 2^22 and more: the 128 x 64 kernel of gemm_q_bf16.hip, with and without a remainder of its step."""
    m, n = 5, 3
    if weight == "int4":
        k = 2 ** 22 + 32 * more
        packed, s, xb, q = i4_case(690 + more, m, n, k)
        w = (np.stack([packed & 15, packed >> 4], 2).reshape(n, k) - 8.0) * np.repeat(s.astype(np.float64), 32, 1)
    else:
        k = 2 ** 22 + 16 * more
        xf, wn, s, q = i8_case(690 + more, m, n, k)
        xb = O.f32_to_bf16(xf)
        w = wn * s.astype(np.float64)[:, None]
    y = O.bf16_to_f32(bits(ops.qgemm(bf16_tensor(xb), q)))
    assert O.rel_l2(y, O.bf16_to_f32(xb).astype(np.float64) @ w.T) <= TOL_BF16


@pytest.mark.parametrize("n", [64, 128, 512])
def test_gemm_refuses_4_gib_of_activations_for_every_tile(ops, n):
    """One row below the limit is served and right in its last rows; at the limit the call is refused, whichever tile N picks."""
    from chadslab_amd import QWeightInt4G32, QWeightInt8

    m, k = 65536, 32768
    r = rng(640 + n)
    x = torch.zeros(m, k, dtype=torch.bfloat16, device=DEV)
    xb = O.f32_to_bf16(r.standard_normal((3, k)).astype(np.float32))
    x[-4:-1] = bf16_tensor(xb)
    packed = r.integers(0, 256, (n, k // 2), dtype=np.uint8)
    s = r.lognormal(-5, 0.5, (n, k // 32)).astype(np.float16)
    qw = QWeightInt4G32(torch.from_numpy(packed).to(DEV), torch.from_numpy(s).to(DEV))
    with pytest.raises(ValueError, match="4 GiB"):
        ops.qgemm(x, qw)
    with pytest.raises(ValueError, match="4 GiB"):
        ops.qgemm(x, QWeightInt8(torch.zeros(n, k, dtype=torch.int8, device=DEV), torch.ones(n, device=DEV)))
    y = ops.qgemm(x[:-1], qw)
    assert not bool(y[:-3].any()) and O.rel_l2(O.bf16_to_f32(bits(y[-3:])), O.qgemm_int4g32_f64(xb, packed, s)) <= TOL_BF16


def test_gemm_int4_many_rows_full_k_and_integer_exact(ops):
    from chadslab_amd import QWeightInt4G32

    # 4096 x 4096 x 4096: the float64 truth is formed for a sample of rows only (the oracle's full product would take
    # minutes); every row of the result is still checked for being finite
    m = n = k = 4096
    packed, s, xb, qw = i4_case(611, m, n, k)
    y = O.bf16_to_f32(bits(ops.qgemm(bf16_tensor(xb), qw)))
    assert np.isfinite(y).all()
    rows = rng(612).choice(m, 96, replace=False)
    rows[:4] = (0, 255, 256, 4095)
    assert O.rel_l2(y[rows], O.qgemm_int4g32_f64(xb[rows], packed, s)) <= TOL_BF16
    # integer activations and unit scales: every sum is an integer below 2^24, so fp32 accumulation is exact and the
    # only rounding is the final one to bf16
    xi = O.f32_to_bf16(rng(613).integers(-4, 5, (m, 1024)).astype(np.float32))
    pk, _, _, q1 = i4_case(614, 1, n, 1024)
    yi = bits(ops.qgemm(bf16_tensor(xi), QWeightInt4G32(q1.packed, torch.ones_like(q1.scale))))
    brute = O.bf16_to_f32(xi[rows]).astype(np.float64) @ O.unpack_int4(pk).astype(np.float64).T
    assert np.abs(brute).max() < 2 ** 24
    assert np.array_equal(yi[rows], O.f32_to_bf16(brute.astype(np.float32)))


def test_gemm_agrees_with_gemv_at_m8(ops):
    packed, s, xb, qw = i4_case(50, 8, 1024, 4096)
    x = bf16_tensor(xb)
    gemv = ops.qgemv(x, qw).cpu().numpy()
    gemm = O.bf16_to_f32(bits(ops.qgemm(x, qw)))
    assert O.rel_l2(gemm, gemv) <= TOL_BF16


def test_gemm_int4_integer_exact_when_scales_are_one(ops):
    from chadslab_amd import QWeightInt4G32

    packed, _, xb, qw = i4_case(51, 64, 128, 512, integer_x=True)
    ones = QWeightInt4G32(qw.packed, torch.ones_like(qw.scale))
    # |sum| <= 512*8*8 = 32768 needs 16 bits: bf16 output cannot hold it, so compare after rounding the
    # exact integer result to bf16 (fp32 accumulation of exact integers is exact)
    brute = (O.bf16_to_f32(xb).astype(np.int64) @ O.unpack_int4(packed).astype(np.int64).T).astype(np.float32)
    assert np.array_equal(bits(ops.qgemm(bf16_tensor(xb), ones)), O.f32_to_bf16(brute))


# ------------------------------------------------------------------ full benchmark sizes: properties that need no CPU reference
def test_full_size_properties_without_a_reference(ops):
    from chadslab_amd import QWeightInt4G32, QWeightInt8

    # config 1: rows of an M=8 product equal the M=1 products; integer inputs make linearity exact
    n, k = 14336, 4096
    packed, s, xb, qw = i4_case(1001, 8, n, k)
    x = bf16_tensor(xb)
    y8 = ops.qgemv(x, qw).cpu().numpy()
    for r in (0, 5):
        assert O.rel_l2(ops.qgemv(x[r:r + 1].contiguous(), qw).cpu().numpy()[0], y8[r]) <= 1e-6
    ones = QWeightInt4G32(qw.packed, torch.ones_like(qw.scale))
    a = rng(2).integers(-4, 5, (1, k)).astype(np.float32)
    b = rng(3).integers(-4, 5, (1, k)).astype(np.float32)
    ya, yb, yab = (ops.qgemv(bf16_tensor(O.f32_to_bf16(v)), ones).cpu().numpy() for v in (a, b, a + b))
    assert np.array_equal(yab, ya + yb)
    # config 2: the prefill kernel and the decode kernel agree on the rows they share
    packed2, s2, xb2, qw2 = i4_case(1002, 512, 4096, 4096)
    x2 = bf16_tensor(xb2)
    gemm = O.bf16_to_f32(bits(ops.qgemm(x2, qw2)))
    gemv = ops.qgemv(x2[100:108].contiguous(), qw2).cpu().numpy()
    assert O.rel_l2(gemm[100:108], gemv) <= TOL_BF16
    # ... and a permutation of the activation rows permutes the output rows, bit for bit
    perm = rng(4).permutation(512)
    gemm_p = bits(ops.qgemm(bf16_tensor(xb2[perm]), qw2))
    assert np.array_equal(gemm_p, bits(ops.qgemm(x2, qw2))[perm])
    # config 0: scaling a row's scale scales that output; integer inputs make linearity exact
    x0, w0, s0, q8 = i8_case(1000, 1, 16384, 2048)
    y0 = ops.qgemv(torch.from_numpy(x0).to(DEV), q8).cpu().numpy()
    q8b = QWeightInt8(q8.w, q8.scale * 2.0)
    assert np.array_equal(ops.qgemv(torch.from_numpy(x0).to(DEV), q8b).cpu().numpy(), 2.0 * y0)
    q1 = QWeightInt8(q8.w, torch.ones_like(q8.scale))
    ia = rng(5).integers(-8, 9, (1, 2048)).astype(np.float32)
    ib = rng(6).integers(-8, 9, (1, 2048)).astype(np.float32)
    za, zb, zab = (ops.qgemv(torch.from_numpy(v).to(DEV), q1).cpu().numpy() for v in (ia, ib, ia + ib))
    assert np.array_equal(zab, za + zb)


# ------------------------------------------------------------------ operator layer and error behaviour
def test_qlinear_dispatch(ops):
    packed, s, xb, qw = i4_case(60, 6, 128, 256)
    x = bf16_tensor(xb).reshape(2, 3, 256)
    y = ops.qlinear(x, qw)
    assert y.shape == (2, 3, 128) and y.dtype == torch.float32  # decode sizes come back in fp32
    assert O.rel_l2(y.reshape(6, 128).cpu().numpy(), O.qgemm_int4g32_f64(xb, packed, s)) <= TOL_F32
    packed, s, xb, qw = i4_case(61, 40, 128, 256)
    y = ops.qlinear(bf16_tensor(xb), qw)
    assert y.dtype == torch.bfloat16 and O.rel_l2(O.bf16_to_f32(bits(y)), O.qgemm_int4g32_f64(xb, packed, s)) <= TOL_BF16
    assert ops.qlinear(bf16_tensor(xb), qw, out_dtype=torch.float32).dtype == torch.float32


def test_errors_surface_as_exceptions(ops):
    from chadslab_amd import QWeightInt4G32, _lib

    _, _, xb, qw = i4_case(62, 1, 64, 128)
    with pytest.raises(ValueError):
        ops.qgemv(bf16_tensor(xb)[:, :96].contiguous(), qw)          # K mismatch
    with pytest.raises(ValueError):
        ops.qgemv(bf16_tensor(xb).float(), qw)                       # wrong dtype
    with pytest.raises(ValueError):
        ops.qgemv(bf16_tensor(np.zeros((17, 128), np.uint16)), qw)   # M beyond the GEMV's range
    lib = _lib.load()
    assert lib.chadq_gemv_i4g32(None, None, None, None, 1, 64, 128, None) == -1
    assert b"null" in lib.chadq_last_error()
    assert lib.chadq_gemv_i4g32(None, None, None, None, 1, 64, 100, None) == -2
    assert b"multiple of 32" in lib.chadq_last_error()
    assert lib.chadq_gemv_i4g32(None, None, None, None, 1, 0, 128, None) == 0  # empty output: nothing to do


# ------------------------------------------------------------------ MoE (config 3)
def _experts(seed, e, h, f):
    """e experts of random int4 group-32 weights: numpy tuples for the oracle and device containers for the ops."""
    from chadslab_amd import QWeightInt4G32

    r = rng(seed)
    host, dev = [], []
    for _ in range(e):
        hw, dw = [], []
        for (n, k) in ((f, h), (f, h), (h, f)):
            u = r.integers(0, 16, (n, k), dtype=np.uint8)
            p = (u[:, 0::2] | (u[:, 1::2] << 4)).astype(np.uint8)
            s = (r.lognormal(-5, 0.5, (n, k // 32)) * (0.6 if n == h else 1.0)).astype(np.float16)
            hw += [p, s]
            dw.append(QWeightInt4G32(torch.from_numpy(p).to(DEV), torch.from_numpy(s).to(DEV)))
        host.append(tuple(hw))
        dev.append(tuple(dw))
    return host, dev


@pytest.mark.parametrize("m", [1, 2, 3, 4, 5, 8, 9, 16])
@pytest.mark.parametrize("n,k", [(1000, 2048), (8197, 512), (515, 4352), (300, 96), (301, 4128)])
def test_qlinear_bf16_result_is_the_fp32_one_rounded(ops, m, n, k):
    """Every GEMV kernel (tall and short matrices, K % 256 != 0, K beyond the row kernels) with the bf16 store."""
    from chadslab_amd import QWeightInt4G32, QWeightInt8

    r = rng(6100 + m + n)
    x = torch.from_numpy(r.standard_normal((m, k)).astype(np.float32)).to(DEV)
    p = torch.from_numpy(r.integers(0, 256, (n, k // 2), dtype=np.uint8)).to(DEV)
    s = torch.from_numpy(r.lognormal(-5, 0.5, (n, k // 32)).astype(np.float16)).to(DEV)
    w8 = torch.from_numpy(r.integers(-127, 128, (n, k), dtype=np.int8)).to(DEV)
    s8 = torch.from_numpy(r.lognormal(-8, 0.5, n).astype(np.float32)).to(DEV)
    for xv, qw in ((x.to(torch.bfloat16), QWeightInt4G32(p, s)), (x, QWeightInt8(w8, s8))):
        y = ops.qlinear(xv, qw, out_dtype=torch.bfloat16)
        assert y.dtype == torch.bfloat16 and torch.equal(y, ops.qlinear(xv, qw).to(torch.bfloat16))


def test_native_calls_serve_plain_tensors_and_leave_the_rest_to_python(ops):
    """The C++ call takes exact, contiguous tensors of the right types and nothing else; both roads give the same bits, and what
    only Python serves (or refuses) still is."""
    from chadslab_amd import QWeightInt4G32, QWeightInt8, _lib

    native = _lib.native()
    _, _, xb, q4 = i4_case(31, 40, 96, 256)
    x = bf16_tensor(xb)
    x8, w8, s8, q8 = i8_case(32, 40, 96, 256)
    xf = torch.from_numpy(x8).to(DEV)
    for rows in (1, 16, 17, 40):  # the fp32 and bf16 GEMV, the GEMM
        for dt in (None, torch.bfloat16) if rows > 16 else (None, torch.float32, torch.bfloat16):
            y = native.linear(x[:rows], q4, dt)
            ref = ops.qgemm(x[:rows], q4) if rows > 16 else ops.qgemv(x[:rows], q4)
            assert y is not None and torch.equal(y, ref if dt is None else ref.to(dt))
            y8 = native.linear(x[:rows] if rows > 16 else xf[:rows], q8, dt)
            ref8 = ops.qgemm(x[:rows], q8) if rows > 16 else ops.qgemv(xf[:rows], q8)
            assert y8 is not None and torch.equal(y8, ref8 if dt is None else ref8.to(dt))
    wide = torch.cat([x, x], 1)
    strided = QWeightInt4G32(torch.cat([q4.packed, q4.packed], 1)[:, :128], q4.scale)
    for a, w, dt in ((wide[:, :256], q4, None), (x.view(4, 10, 256), q4, None), (x[:5], strided, None), (x, q4, torch.float32),
                     (x[:3], q4, torch.float16)):
        assert native.linear(a, w, dt) is None
        y = ops.qlinear(a, w, out_dtype=dt)
        a2 = a.reshape(-1, 256)
        ref = ops.qgemm(a2, w) if a2.shape[0] > 16 else ops.qgemv(a2, w)
        assert torch.equal(y.reshape(ref.shape), ref if dt is None else ref.to(dt))
    for a, w in ((x.float(), q4), (xf[:20], q8), (x[:, :128], q4), (x.cpu(), q4), (x[:2].half(), q8), (x[:0], q4)):
        assert native.linear(a, w, None) is None
        with pytest.raises(ValueError):
            ops.qlinear(a, w)
    with pytest.raises((TypeError, AttributeError)):
        ops.qlinear(x, q4.packed)

    class Mine(torch.Tensor):
        pass

    assert native.linear(x.as_subclass(Mine), q4, None) is None
    experts = [(i4_case(40 + i, 1, 256, 256)[3],) * 3 for i in range(4)]
    z = torch.randn(5, 4, device=DEV)
    y = native.moe_ffn(x[:5], z, experts, 2, True)
    assert y is not None and torch.equal(y, ops.moe_ffn(x[:5], z, tuple(experts), top_k=2))
    mixed = experts[:3] + [tuple(ops.to_tiles(w) for w in experts[3])]
    for a, logits, ex, k in ((x[:5], z.double(), experts, 2), (wide[:5, :256], z, experts, 2), (x[:5], z[:, :3], experts, 2), (x[:5], z, mixed, 2),
                             (x[:5], z, iter(experts), 2), (x[:5], z, experts, 5)):
        assert native.moe_ffn(a, logits, ex, k, True) is None
    assert torch.equal(ops.moe_ffn(wide[:5, :256], z, experts, top_k=2), y)


def test_dimensions_and_casts_of_qlinear_stay_on_the_native_call(ops, monkeypatch):
    """An x of any number of dimensions, strided or not, and a result of another type: the same bits as the product of the same rows,
    and the product itself is the native one."""
    _, _, xb, q4 = i4_case(33, 40, 96, 256)
    x = bf16_tensor(xb)
    x8, _, _, q8 = i8_case(34, 40, 96, 256)
    xf = torch.from_numpy(x8).to(DEV)
    cases = []
    for a, q in ((x, q4), (x[:1], q4), (x[:16], q4), (x, q8), (xf[:16], q8), (xf[:1], q8)):
        y = ops.qgemm(a, q) if a.shape[0] > 16 else ops.qgemv(a, q)
        half = ops.qlinear(a, q, out_dtype=torch.bfloat16)
        rows = a.shape[0]
        shapes = [(rows, 256), (1, rows, 256)] + [(rows // 4, 2, 2, 256)] * (rows % 4 == 0) + [(256,)] * (rows == 1)
        for shape in shapes:
            for dt in (None, torch.float32, torch.bfloat16, torch.float16, torch.float64):
                cases.append((a.view(shape), q, dt, (half if dt == torch.bfloat16 else y if dt is None else y.to(dt)).view(*shape[:-1], 96)))
    wide = torch.cat([x, x], 1)
    turned, part, parts = x.view(8, 5, 256).transpose(0, 1), wide[:, :256], wide.view(8, 5, 512)[..., 256:]
    for a in (turned, part, parts, part[:3]):  # strided
        rows = a.reshape(-1, 256).contiguous()
        cases.append((a, q4, None, (ops.qgemm if len(rows) > 16 else ops.qgemv)(rows, q4).view(*a.shape[:-1], 96)))

    def left(*args, **kw):
        raise AssertionError("the product went through Python")

    for name in ("_gemv", "qgemv", "qgemm"):
        monkeypatch.setattr(ops, name, left)
    for a, q, dt, ref in cases:
        y = ops.qlinear(a, q, out_dtype=dt)
        assert y.dtype == ref.dtype and torch.equal(y, ref), (a.shape, dt)


def test_moe_ffn_reads_renorm_as_int_does(ops):
    """0.5 is 0, None has no int: what is no bool and no int goes the way of int(renorm), whichever road serves the call."""
    from chadslab_amd import _lib

    experts = [(i4_case(44 + i, 1, 256, 256)[3],) * 3 for i in range(4)]
    x, z = torch.randn(5, 256, device=DEV).bfloat16(), torch.randn(5, 4, device=DEV)
    yes, no = (ops.moe_ffn(x, z, experts, renorm=v) for v in (True, False))
    assert not torch.equal(yes, no)
    for value, same in ((1, yes), (-3, yes), (0, no), (0.5, no), (1.5, yes), (np.bool_(True), yes), (torch.tensor(0), no)):
        assert torch.equal(ops.moe_ffn(x, z, experts, renorm=value), same), value
    for value in (0.5, None, "1", np.bool_(True), 2 ** 40):
        assert _lib.native().moe_ffn(x, z, experts, 2, value) is None
    with pytest.raises(TypeError):
        ops.moe_ffn(x, z, experts, renorm=None)


@pytest.mark.parametrize("status,error", [(-5, RuntimeError), (-6, RuntimeError)])
def test_native_calls_raise_a_device_error_at_the_first_attempt(ops, status, error):
    """An entry point that reports a failed launch (-5) or device (-6) is called once and its error is the one that is raised; a refused
    argument (any other status) is left to the Python road."""
    import ctypes

    from chadslab_amd import QWeightInt4G32, QWeightInt8, QWeightInt4G32Tiles, _lib

    native = _lib.native()
    calls = []
    product = ctypes.CFUNCTYPE(ctypes.c_int, *[ctypes.c_void_p] * 4, *[ctypes.c_int] * 3, ctypes.c_void_p)
    moe = ctypes.CFUNCTYPE(ctypes.c_int, *[ctypes.c_void_p] * 4, *[ctypes.c_int] * 6, ctypes.c_void_p, ctypes.c_size_t, ctypes.c_void_p)

    def fail(*args):
        calls.append(args)
        return status

    p, m = product(fail), moe(fail)
    real = {n: ctypes.cast(getattr(_lib.load(), n), ctypes.c_void_p).value for n in _lib._NATIVE_ENTRIES}
    fake = [real[n] if "workspace" in n else ctypes.cast(m if "moe" in n else p, ctypes.c_void_p).value for n in _lib._NATIVE_ENTRIES]
    q = QWeightInt4G32(torch.zeros(256, 128, dtype=torch.uint8, device=DEV), torch.ones(256, 8, dtype=torch.float16, device=DEV))
    x = torch.ones(3, 256, dtype=torch.bfloat16, device=DEV)
    try:
        native.bind(tuple(fake), (QWeightInt4G32, QWeightInt8, QWeightInt4G32Tiles), _lib.check)
        with pytest.raises(error, match="chadq_gemv_i4g32 failed"):
            ops.qlinear(x, q)
        assert len(calls) == 1
        with pytest.raises(error, match="chadq_moe_ffn_i4g32 failed"):
            ops.moe_ffn(x, torch.zeros(3, 1, device=DEV), [(q, q, q)], top_k=1)
        assert len(calls) == 2
        status = -2
        assert native.linear(x, q, None) is None and len(calls) == 3
    finally:
        _lib._native_lib = None
        _lib.native()
    assert torch.equal(ops.qlinear(x, q), torch.full((3, 256), -2048.0, device=DEV))


def test_moe_route_matches_oracle(ops):
    r = rng(70)
    logits = r.standard_normal((300, 8)).astype(np.float32)
    logits[5, 2] = logits[5, 6] = logits[5].max() + 1.0   # tie for first place
    logits[9, :] = 0.25                                    # all equal
    logits[11, 1] = logits[11, 3]                          # tie somewhere
    for top_k, renorm in ((2, True), (2, False), (1, True), (4, True)):
        idx, w = ops.moe_route(torch.from_numpy(logits).to(DEV), top_k, renorm)
        oi, ow = O.moe_route(logits, top_k, renorm)
        assert np.array_equal(idx.cpu().numpy(), oi)       # indices bit-exact
        assert np.allclose(w.cpu().numpy(), ow, rtol=2e-5, atol=1e-7)
    assert idx.cpu().numpy()[9].tolist() == [0, 1, 2, 3]


def test_moe_golden(ops):
    from chadslab_amd import QWeightInt4G32

    g = np.load(os.path.join(GOLD, "moe_t16_h64_f96_e4.npz"))
    experts = [tuple(QWeightInt4G32(torch.from_numpy(g["e%d_%s_p" % (i, n)]).to(DEV), torch.from_numpy(g["e%d_%s_s" % (i, n)]).to(DEV))
                     for n in "gud") for i in range(4)]
    y = ops.moe_ffn(bf16_tensor(g["x_bf16"]), torch.from_numpy(g["logits"]).to(DEV), experts, top_k=2, renorm=True)
    assert O.rel_l2(O.bf16_to_f32(bits(y)), O.bf16_to_f32(g["y_bf16"])) <= TOL_BF16


@pytest.mark.parametrize("t,h,f,e,top_k", [(256, 512, 1024, 8, 2), (37, 128, 160, 3, 1), (64, 256, 256, 1, 1), (130, 256, 512, 16, 4),
                                           (300, 256, 512, 2, 2), (33, 256, 768, 8, 2), (200, 512, 512, 3, 1),
                                           # more than 1024 pairs (the router sorts them in several passes) and more than
                                           # 4096 (its ranks go through memory instead of LDS)
                                           (400, 256, 256, 8, 4), (1200, 256, 256, 4, 4), (1100, 64, 96, 5, 4)])
def test_moe_ffn(ops, t, h, f, e, top_k):
    host, dev = _experts(80 + t, e, h, f)
    r = rng(81 + t)
    xb = O.f32_to_bf16(r.standard_normal((t, h)).astype(np.float32))
    logits = r.standard_normal((t, e)).astype(np.float32)
    y = O.bf16_to_f32(bits(ops.moe_ffn(bf16_tensor(xb), torch.from_numpy(logits).to(DEV), dev, top_k=top_k, renorm=True)))
    ref = O.bf16_to_f32(O.moe_qffn(xb, logits, host, top_k, True))
    assert np.isfinite(y).all() and O.rel_l2(y, ref) <= TOL_BF16
    # token order does not matter
    perm = r.permutation(t)
    yp = O.bf16_to_f32(bits(ops.moe_ffn(bf16_tensor(xb[perm]), torch.from_numpy(logits[perm]).to(DEV), dev, top_k=top_k, renorm=True)))
    assert np.array_equal(yp, y[perm])


def test_moe_ffn_empty_experts_and_one_crowded_expert(ops):
    # experts 2..7 get nothing, expert 0 gets every token (three token tiles of 96), expert 1 the second choice of most
    t, h, f, e = 250, 256, 512, 8
    host, dev = _experts(90, e, h, f)
    r = rng(91)
    xb = O.f32_to_bf16(r.standard_normal((t, h)).astype(np.float32))
    logits = r.standard_normal((t, e)).astype(np.float32)
    logits[:, 0] += 30.0
    logits[:, 1] += 15.0
    logits[:7, 1] -= 40.0  # a few tokens take some other expert second: tiles of very few rows
    y = O.bf16_to_f32(bits(ops.moe_ffn(bf16_tensor(xb), torch.from_numpy(logits).to(DEV), dev, top_k=2, renorm=True)))
    ref = O.bf16_to_f32(O.moe_qffn(xb, logits, host, 2, True))
    assert np.isfinite(y).all() and O.rel_l2(y, ref) <= TOL_BF16


def test_moe_ffn_random_shapes(ops):
    r = rng(4244)
    for case in range(8):
        e = int(r.integers(1, 9))
        top_k = int(r.integers(1, min(e, 4) + 1))
        t = int(r.integers(1, 300))
        if case % 2:  # shapes the expert kernel takes (multiples of 256) / shapes that go the general way
            h, f = 256 * int(r.integers(1, 4)), 256 * int(r.integers(1, 4))
        else:
            h, f = 32 * int(r.integers(1, 12)), 32 * int(r.integers(1, 12))
        host, dev = _experts(7000 + case, e, h, f)
        xb = O.f32_to_bf16(r.standard_normal((t, h)).astype(np.float32))
        logits = r.standard_normal((t, e)).astype(np.float32)
        y = O.bf16_to_f32(bits(ops.moe_ffn(bf16_tensor(xb), torch.from_numpy(logits).to(DEV), dev, top_k=top_k, renorm=bool(case & 2))))
        ref = O.bf16_to_f32(O.moe_qffn(xb, logits, host, top_k, bool(case & 2)))
        assert np.isfinite(y).all() and O.rel_l2(y, ref) <= TOL_BF16, (t, h, f, e, top_k)


def test_moe_config3_full_size(ops):
    t, h, f, e = 256, 4096, 14336, 8
    host, dev = _experts(1003, e, h, f)
    r = rng(1003)
    logits = r.standard_normal((t, e)).astype(np.float32)
    xb = O.f32_to_bf16(r.standard_normal((t, h)).astype(np.float32))
    y = O.bf16_to_f32(bits(ops.moe_ffn(bf16_tensor(xb), torch.from_numpy(logits).to(DEV), dev, top_k=2, renorm=True)))
    ref = O.bf16_to_f32(O.moe_qffn(xb, logits, host, 2, True))
    assert O.rel_l2(y, ref) <= TOL_BF16
    # the same experts in tile order: the matrix-core kernel for that order holds the dequantised weights in fp16 (the
    # row-major one in bf16), so the two agree within rounding, and each with the oracle
    tiled = [tuple(ops.to_tiles(m) for m in tr) for tr in dev]
    yt = O.bf16_to_f32(bits(ops.moe_ffn(bf16_tensor(xb), torch.from_numpy(logits).to(DEV), tiled, top_k=2, renorm=True)))
    assert np.isfinite(yt).all() and O.rel_l2(yt, ref) <= TOL_BF16
    assert O.rel_l2(yt, ref) <= O.rel_l2(y, ref) * 1.05 + 1e-4  # never less accurate than the bf16 form
    assert O.rel_l2(yt, y) <= 6e-3


# ------------------------------------------------------------------ tile order (load-time repack for the experts)
@pytest.mark.parametrize("n,k", [(32, 256), (64, 512), (96, 1280), (256, 4096), (14336, 4096), (4096, 14336)])
def test_repack_tiles_bit_exact_and_round_trip(ops, n, k):
    from chadslab_amd import QWeightInt4G32

    r = rng(5100 + n + k)
    p = r.integers(0, 256, (n, k // 2), dtype=np.uint8)
    s = r.integers(0, 65536, (n, k // 32), dtype=np.uint16)  # every bit pattern, NaNs included: the repack moves bytes
    qw = QWeightInt4G32(torch.from_numpy(p).to(DEV), torch.from_numpy(s).view(torch.float16).to(DEV))
    tl = ops.to_tiles(qw)
    wp_t, sc_t = O.tile_int4g32(p, s.view(np.float16))
    assert np.array_equal(tl.packed.cpu().numpy(), wp_t)
    assert np.array_equal(tl.scale.view(torch.int16).cpu().numpy().view(np.uint16), sc_t.view(np.uint16))
    back = ops.to_rows(tl)
    assert torch.equal(back.packed, qw.packed) and torch.equal(back.scale.view(torch.int16), qw.scale.view(torch.int16))


def test_repack_tiles_refuses_bad_shapes_and_aliasing(ops):
    from chadslab_amd import QWeightInt4G32, _lib

    for n, k in ((48, 256), (32, 128), (32, 288)):
        qw = QWeightInt4G32(torch.zeros(n, k // 2, dtype=torch.uint8, device=DEV), torch.zeros(n, k // 32, dtype=torch.float16, device=DEV))
        with pytest.raises(ValueError):
            ops.to_tiles(qw)
    lib = _lib.load()
    a = torch.zeros(32, 128, dtype=torch.uint8, device=DEV)
    sc = torch.zeros(32, 8, dtype=torch.float16, device=DEV)
    sc2 = torch.zeros_like(sc)
    assert lib.chadq_repack_i4g32_tiles(a.data_ptr(), sc.data_ptr(), a.data_ptr(), sc2.data_ptr(), 32, 256, None) == -2  # in place
    assert lib.chadq_repack_i4g32_tiles(a.data_ptr(), sc.data_ptr(), None, sc2.data_ptr(), 32, 256, None) == -1


@pytest.mark.parametrize("t,h,f,e,top_k", [(256, 512, 1024, 8, 2), (64, 256, 256, 1, 1), (130, 256, 512, 16, 4), (300, 256, 768, 2, 2),
                                           (1200, 256, 256, 4, 4), (200, 768, 1280, 3, 2), (96, 1024, 2048, 2, 1)])
def test_moe_ffn_tiled_agrees_with_row_major_and_oracle(ops, t, h, f, e, top_k):
    host, dev = _experts(8800 + t, e, h, f)
    r = rng(8801 + t)
    xb = O.f32_to_bf16(r.standard_normal((t, h)).astype(np.float32))
    logits = r.standard_normal((t, e)).astype(np.float32)
    y = bits(ops.moe_ffn(bf16_tensor(xb), torch.from_numpy(logits).to(DEV), dev, top_k=top_k, renorm=True))
    tiled = [tuple(ops.to_tiles(m) for m in tr) for tr in dev]
    yt = bits(ops.moe_ffn(bf16_tensor(xb), torch.from_numpy(logits).to(DEV), tiled, top_k=top_k, renorm=True))
    ref = O.bf16_to_f32(O.moe_qffn(xb, logits, host, top_k, True))
    assert np.isfinite(O.bf16_to_f32(yt)).all() and O.rel_l2(O.bf16_to_f32(yt), ref) <= TOL_BF16
    assert O.rel_l2(O.bf16_to_f32(yt), O.bf16_to_f32(y)) <= 6e-3  # fp16 against bf16 dequantised weights: rounding only
    # token order does not matter
    perm = r.permutation(t)
    yp = bits(ops.moe_ffn(bf16_tensor(xb[perm]), torch.from_numpy(logits[perm]).to(DEV), tiled, top_k=top_k, renorm=True))
    assert np.array_equal(yp, yt[perm])


@pytest.mark.parametrize("t,h,f,e,top_k", [(1, 256, 256, 1, 1), (4, 1024, 2048, 8, 2), (16, 768, 4352, 16, 4), (16, 2304, 1280, 4, 1), (17, 512, 2048, 4, 2), (8, 2048, 4096, 8, 2)])
def test_moe_ffn_few_tokens(ops, t, h, f, e, top_k):
    """Up to 16 tokens stream the weights exactly (17: the many-row kernels), both orders with the same sums: one and
    several blocks of 256 k per wave, block counts that four waves and the K splits do not divide, an expert with all
    tokens beside empty ones."""
    host, dev = _experts(9400 + t + h, e, h, f)
    r = rng(9401 + t + h)
    xb = O.f32_to_bf16(r.standard_normal((t, h)).astype(np.float32))
    logits = r.standard_normal((t, e)).astype(np.float32)
    logits[:, e - 1] += 20.0  # every token takes the last expert
    x, z = bf16_tensor(xb), torch.from_numpy(logits).to(DEV)
    tiled = [tuple(ops.to_tiles(m) for m in tr) for tr in dev]
    ref = O.bf16_to_f32(O.moe_qffn(xb, logits, host, top_k, True))
    y, yt = (bits(ops.moe_ffn(x, z, ex, top_k=top_k, renorm=True)) for ex in (dev, tiled))
    small = min(e, t * top_k) * h * f * 27 // 16 <= 64 << 20  # what the tile order sends to the same kernel
    if t <= 16 and small:
        # bf16 roundings of h (some flip one ulp against the oracle's float64) and of the result, weights exact
        assert np.array_equal(y, yt) and O.rel_l2(O.bf16_to_f32(y), ref) <= 2.0 ** -8
    for v in (y, yt):
        assert O.rel_l2(O.bf16_to_f32(v), ref) <= TOL_BF16


@pytest.mark.parametrize("t,h,f,e,top_k", [(4, 4096, 3584, 8, 2), (1, 512, 2816, 16, 4), (5, 2048, 7424, 3, 2), (2, 1536, 256, 2, 1), (9, 1024, 4864, 4, 4)])
def test_moe_ffn_few_tokens_activations_through_lds(ops, t, h, f, e, top_k):
    """Activations of an expert small enough for LDS, with few items to a workgroup; K splits of uneven length."""
    test_moe_ffn_few_tokens(ops, t, h, f, e, top_k)


@pytest.mark.parametrize("t,h,f,e,top_k,gate,down", [(6, 256, 12288, 8, 2, True, False), (16, 512, 8960, 16, 4, True, False), (16, 2560, 4096, 16, 8, False, True),
                                                     (5, 3328, 10496, 8, 2, True, True), (3, 2304, 9984, 16, 4, True, True)])
def test_moe_ffn_few_tokens_many_items_are_summed_as_one_by_one(ops, t, h, f, e, top_k, gate, down):
    """Where the activations go through LDS, in one of the two products or in both, every token's result has the bits of a call with that token
    alone, which reads them straight to registers: workgroups whose run of items crosses from one expert or K split to the next, K splits of
    uneven length, all tokens on the same experts and tokens spread over all of them."""
    import ctypes

    from chadslab_amd import QWeightInt4G32, _lib

    fn = _lib.load()["_ZN5chadq19moe_few_through_ldsEiiiii"]
    fn.restype = ctypes.c_bool
    parts = 4 if f >= 4096 else 2 if f >= 2048 else 1
    rule = [(fn(n, e, top_k, f // 16, h // 256), fn(n, e, top_k, h // 32 * parts, -(-(f // 256) // parts))) for n in (t, 1)]
    assert rule[0] == (gate, down) and rule[0] != rule[1]
    g = torch.Generator(device=DEV)
    g.manual_seed(9500 + t)

    def matrix(n, k):
        return QWeightInt4G32(torch.randint(0, 256, (n, k // 2), dtype=torch.uint8, device=DEV, generator=g),
                              torch.exp(torch.randn(n, k // 32, device=DEV, generator=g) * 0.5 - 5.0).half())

    experts = [(matrix(f, h), matrix(f, h), matrix(h, f)) for _ in range(e)]
    x = torch.randn(t, h, device=DEV, generator=g).bfloat16()
    z = torch.randn(t, e, device=DEV, generator=g)
    same = z.clone()
    same[:, -top_k:] += 30.0
    for logits in (z, same):
        y = ops.moe_ffn(x, logits, experts, top_k=top_k)
        assert bool(torch.isfinite(y).all()) and bool(y.any())
        differ = 0
        for i in range(t):
            one = ops.moe_ffn(x[i:i + 1], logits[i:i + 1], experts, top_k=top_k)
            differ += int((one[0].view(torch.int16) != y[i].view(torch.int16)).sum())
        assert differ == 0


@pytest.mark.parametrize("tiled", [False, True])
@pytest.mark.parametrize("t,h,f,e,top_k", [(2, 256, 256, 1, 1), (4, 256, 512, 2, 2), (4, 1280, 2304, 3, 2), (5, 256, 256, 1, 1), (5, 2560, 1280, 2, 1), (8, 512, 4352, 2, 2),
                                           (13, 1024, 768, 1, 1), (16, 768, 2816, 2, 2)])
def test_moe_ffn_up_to_four_tokens_and_more_have_the_bits_of_one(ops, t, h, f, e, top_k, tiled):
    """At most four tokens are summed with four scale groups side by side, more with one group after the other: the same order of additions,
    so a token's bits do not depend on how many came with it."""
    from chadslab_amd import QWeightInt4G32

    g = torch.Generator(device=DEV)
    g.manual_seed(9600 + t + h)

    def matrix(n, k):
        w = QWeightInt4G32(torch.randint(0, 256, (n, k // 2), dtype=torch.uint8, device=DEV, generator=g),
                           torch.exp(torch.randn(n, k // 32, device=DEV, generator=g) * 0.5 - 5.0).half())
        return ops.to_tiles(w) if tiled else w

    experts = [(matrix(f, h), matrix(f, h), matrix(h, f)) for _ in range(e)]
    x = torch.randn(t, h, device=DEV, generator=g).bfloat16()
    z = torch.randn(t, e, device=DEV, generator=g)
    y = ops.moe_ffn(x, z, experts, top_k=top_k)
    assert bool(torch.isfinite(y).all()) and bool(y.any())
    for i in range(t):
        one = ops.moe_ffn(x[i:i + 1], z[i:i + 1], experts, top_k=top_k)
        assert torch.equal(one[0].view(torch.int16), y[i].view(torch.int16)), i


@pytest.mark.parametrize("t,h,f,e,top_k", [(16, 256, 512, 5, 4), (13, 256, 512, 7, 5), (16, 512, 256, 16, 8), (16, 256, 256, 1, 1), (8, 512, 512, 16, 8),
                                           (1, 256, 256, 16, 8)])
def test_moe_ffn_few_tokens_routed_by_one_wave(ops, t, h, f, e, top_k):
    """64 pairs of token and expert and fewer take the one-wave router, 65 and more the general one; every expert hit or few, one alone."""
    test_moe_ffn_few_tokens(ops, t, h, f, e, top_k)


@pytest.mark.parametrize("t,h,f,e,top_k", [(20, 512, 1280, 4, 2), (33, 1024, 2816, 3, 2), (70, 768, 5632, 8, 1), (260, 512, 3328, 2, 2), (40, 1536, 2304, 16, 4),
                                           (200, 3072, 1280, 8, 4), (150, 2304, 1792, 8, 2), (120, 3072, 3328, 8, 1)])
def test_moe_ffn_down_products_in_uneven_k_splits(ops, t, h, f, e, top_k):
    """F that no power of two divides into parts of whole blocks, in both weight orders; 64 and 128 weight rows per wave."""
    test_moe_ffn_tiled_agrees_with_row_major_and_oracle(ops, t, h, f, e, top_k)


@pytest.mark.parametrize("big", [0.0, 3e37, -2.9e38])
def test_moe_ffn_few_tokens_large_activations(ops, big):
    """One activation near the top of bf16's range in some tokens (its gate weights have the scale 0, so that the gate stays
    moderate), h as large: every sum of the exact result is finite, so the result must be, in both orders, and rows of
    ordinary size beside such rows keep their accuracy."""
    from chadslab_amd import QWeightInt4G32

    t, h, f, e = 6, 512, 768, 2
    host, _ = _experts(9700, e, h, f)
    for gp, gs, up, us, dp, ds in host:
        gs[:, 3] = 0
        us[:] = us.astype(np.float32) * 2.0 ** -6 if big else us
        ds[:] = ds.astype(np.float32) * 2.0 ** -6 if big else ds
    dev = [tuple(QWeightInt4G32(torch.from_numpy(tr[2 * i]).to(DEV), torch.from_numpy(tr[2 * i + 1]).to(DEV)) for i in range(3)) for tr in host]
    r = rng(9701)
    x = r.standard_normal((t, h)).astype(np.float32)
    if big:
        x[::2, 3 * 32 + 5] = big
    xb = O.f32_to_bf16(x)
    logits = r.standard_normal((t, e)).astype(np.float32)
    ref = O.bf16_to_f32(O.moe_qffn(xb, logits, host, 2, True)).astype(np.float64)
    assert np.isfinite(ref).all()
    for ex in (dev, [tuple(ops.to_tiles(m) for m in tr) for tr in dev]):
        y = O.bf16_to_f32(bits(ops.moe_ffn(bf16_tensor(xb), torch.from_numpy(logits).to(DEV), ex, top_k=2, renorm=True))).astype(np.float64)
        for row in range(t):
            assert np.linalg.norm(y[row] - ref[row]) <= 2.0 ** -8 * np.linalg.norm(ref[row]), row


@pytest.mark.parametrize("outlier", [1e3, -1e5])
def test_moe_ffn_few_tokens_beside_an_outlier_of_zero_weight(ops, outlier):
    """One activation far larger than the others of its scale group, all gate and up weights at it 0: the others count as
    ever.  The group's zero-point term, 8 times the outlier, is added and taken off in fp32: 1e5 * 8 * 2^-24 = 0.05 against a
    gate of some 16 groups of sqrt(32) * 4.6 = 100, 5e-4, beside the two bf16 roundings."""
    from chadslab_amd import QWeightInt4G32

    t, h, f, e = 4, 512, 768, 2
    host, _ = _experts(9750, e, h, f)
    for gp, gs, up, us, dp, ds in host:
        for p in (gp, up):
            p[:, 50] = (p[:, 50] & 0xF0) | 8
    dev = [tuple(QWeightInt4G32(torch.from_numpy(tr[2 * i]).to(DEV), torch.from_numpy(tr[2 * i + 1]).to(DEV)) for i in range(3)) for tr in host]
    r = rng(9751)
    x = r.standard_normal((t, h)).astype(np.float32)
    x[:, 100] = outlier
    xb = O.f32_to_bf16(x)
    logits = r.standard_normal((t, e)).astype(np.float32)
    ref = O.bf16_to_f32(O.moe_qffn(np.where(np.arange(h) == 100, 0, xb).astype(xb.dtype), logits, host, 2, True))
    for ex in (dev, [tuple(ops.to_tiles(m) for m in tr) for tr in dev]):
        y = O.bf16_to_f32(bits(ops.moe_ffn(bf16_tensor(xb), torch.from_numpy(logits).to(DEV), ex, top_k=2, renorm=True)))
        assert O.rel_l2(y, ref) <= 2.0 ** -8


def test_moe_ffn_keeps_no_memory_per_size(ops):
    """A server whose batch varies: what a call has used is free again when the next one of another size begins."""
    _, dev = _experts(9900, 2, 256, 512)
    r = rng(9901)
    z = torch.from_numpy(r.standard_normal((80, 2)).astype(np.float32)).to(DEV)
    x = bf16_tensor(O.f32_to_bf16(r.standard_normal((80, 256)).astype(np.float32)))
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    for t in range(1, 81):
        ops.moe_ffn(x[:t], z[:t], dev, top_k=2)
        assert torch.cuda.memory_allocated() == before, t


def test_moe_ffn_tiled_wide_ranges_of_activations_and_scales(ops):
    """The tile-order kernels carry activations and dequantised weights as fp16: rows are scaled by a power of two first,
    so activations far outside fp16's range (and rows of very different magnitude side by side) must come out as the
    oracle has them, row by row; scales from fp16's smallest normal up to 32, negative and zero ones included."""
    t, h, f, e, top_k = 160, 512, 768, 4, 2
    host, dev = _experts(9100, e, h, f)
    r = rng(9101)
    # scales: magnitudes 2^-14 .. 2^5 for the gate/up matrices (|dequantised weight| up to 256), signs mixed, some zero
    host2, dev2 = [], []
    from chadslab_amd import QWeightInt4G32
    for tr in host:
        hw, dw = [], []
        for i in range(3):
            p, s = tr[2 * i], tr[2 * i + 1].astype(np.float32)
            if i < 2:
                mag = np.exp2(r.integers(-14, 6, s.shape)).astype(np.float32) * (1 + r.random(s.shape).astype(np.float32) * 0.99)
                sgn = np.where(r.random(s.shape) < 0.3, -1.0, 1.0).astype(np.float32)
                s = (mag * sgn * (r.random(s.shape) > 0.05)).astype(np.float32)
            s16 = s.astype(np.float16)
            hw += [p, s16]
            dw.append(QWeightInt4G32(torch.from_numpy(p).to(DEV), torch.from_numpy(s16).to(DEV)))
        host2.append(tuple(hw))
        dev2.append(tuple(dw))
    x = r.standard_normal((t, h)).astype(np.float32)
    x *= np.exp2(r.integers(-40, 41, (t, 1))).astype(np.float32)   # rows from 2^-40 to 2^40
    x[3] = 0.0                                                       # an all-zero row
    x[5, ::7] *= 2.0 ** 20                                           # a row with a few huge elements beside tiny ones
    xb = O.f32_to_bf16(x)
    logits = r.standard_normal((t, e)).astype(np.float32)
    tiled = [tuple(ops.to_tiles(m) for m in tr) for tr in dev2]
    with np.errstate(over="ignore", invalid="ignore"):
        ref = O.bf16_to_f32(O.moe_qffn(xb, logits, host2, top_k, True))
    y = O.bf16_to_f32(bits(ops.moe_ffn(bf16_tensor(xb), torch.from_numpy(logits).to(DEV), tiled, top_k=top_k, renorm=True)))
    fin = np.isfinite(ref).all(axis=1)
    assert fin.sum() >= t // 2                      # the case is not degenerate
    assert np.isfinite(y[fin]).all()
    for row in np.nonzero(fin)[0]:                  # row by row: every row has its own magnitude
        n = np.linalg.norm(ref[row].astype(np.float64))
        if n == 0:
            assert not y[row].any()
        else:
            assert np.linalg.norm((y[row] - ref[row]).astype(np.float64)) <= TOL_BF16 * n, row
    assert not np.isfinite(y[~fin]).all(axis=1).any() or not (~fin).any()  # rows the oracle overflows on overflow here too


def test_moe_ffn_tiled_refuses_mixed_and_unaligned_shapes(ops):
    host, dev = _experts(8900, 2, 256, 256)
    tiled = [tuple(ops.to_tiles(m) for m in tr) for tr in dev]
    x = torch.zeros(8, 256, dtype=torch.bfloat16, device=DEV)
    z = torch.zeros(8, 2, device=DEV)
    with pytest.raises(TypeError):
        ops.moe_ffn(x, z, [tiled[0], dev[1]], top_k=1)
    # H = 288 is a multiple of 32 (fine for the row-major entry point) but not of 256: the tiled one refuses it
    from chadslab_amd import _lib
    lib = _lib.load()
    need = lib.chadq_moe_ffn_i4g32_workspace_bytes(8, 288, 256, 1, 1)
    ws = torch.empty(max(need, 16), dtype=torch.uint8, device=DEV)
    arr = (_lib.MoeExpertI4G32 * 1)(_lib.MoeExpertI4G32(*[ws.data_ptr()] * 6))
    y = torch.empty(8, 288, dtype=torch.bfloat16, device=DEV)
    x2 = torch.zeros(8, 288, dtype=torch.bfloat16, device=DEV)
    z1 = torch.zeros(8, 1, device=DEV)
    assert lib.chadq_moe_ffn_i4g32_tiled(x2.data_ptr(), z1.data_ptr(), arr, y.data_ptr(), 8, 288, 256, 1, 1, 1, ws.data_ptr(), need, None) == -2


@pytest.mark.parametrize("m,n,k,shift", [(17, 512, 8192, 0), (32, 102, 8192, 0), (40, 257, 4128, 0), (48, 1024, 14336, 0), (64, 64, 4096, 1), (70, 513, 16384, 0), (100, 1000, 8160, 0),
                                         (128, 2048, 8192, 1), (300, 1024, 16384, 0), (200, 512, 5152, 0)])
def test_gemm_in_parts_of_k(ops, m, n, k, shift):
    """Products of few tiles and a long K, summed in parts: ragged rows and columns (columns that no four divide, too), K that 256 does not divide,
    parts of uneven length, scales that are not 16-byte aligned.  Weights rounded to bf16 in the reference as in the kernel: what is left
    is the rounding of the result, 2^-9 at most per element."""
    from chadslab_amd import QWeightInt4G32, QWeightInt8, _lib

    lib = _lib.load()
    g = torch.Generator(device=DEV)
    g.manual_seed(m + n)
    x = torch.randn(m, k, device=DEV, generator=g).bfloat16()
    p = torch.randint(0, 256, (n, k // 2), dtype=torch.uint8, device=DEV, generator=g)
    s = torch.exp(torch.randn(n * (k // 32) + shift, device=DEV, generator=g) * 0.5 - 5.0).half()[shift:].view(n, k // 32)
    w4 = ((torch.stack((p & 15, p >> 4), -1).reshape(n, k).float() - 8) * s.float().repeat_interleave(32, 1)).bfloat16().double()
    w = torch.randint(-127, 128, (n, k), dtype=torch.int8, device=DEV, generator=g)
    s8 = torch.exp(torch.randn(n, device=DEV, generator=g) * 0.5 - 8.0)
    stream = torch.cuda.current_stream().cuda_stream
    for qw, ref, sc, name in ((QWeightInt4G32(p, s), x.double() @ w4.t(), s, "chadq_gemm_i4g32_bf16"),
                              (QWeightInt8(w, s8), x.double() @ (w.double() * s8.double()[:, None]).t(), s8, "chadq_gemm_i8row_bf16")):
        need = lib.chadq_gemm_bf16_workspace_bytes(m, n, k, int(sc is s8))
        assert need >= 2 * 4 * m * n  # in parts
        y = ops.qgemm(x, qw)
        err = (y.double() - ref).norm(dim=1) / ref.norm(dim=1)
        assert float(err.max()) <= 2.0 ** -8, (name, float(err.max()))
        # scratch of any content gives the same bits; none, or too little, the product in one part
        wp = p if sc is s else w
        scratch = torch.full((need,), 0xFF, dtype=torch.uint8, device=DEV)
        got = [torch.empty_like(y) for _ in range(4)]
        for out, ptr, size in ((got[0], scratch.data_ptr(), need), (got[1], None, 0), (got[2], scratch.data_ptr(), need // 2 - 16)):
            assert getattr(lib, name + "_ws")(x.data_ptr(), wp.data_ptr(), sc.data_ptr(), out.data_ptr(), m, n, k, ptr, size, stream) == 0
        assert getattr(lib, name)(x.data_ptr(), wp.data_ptr(), sc.data_ptr(), got[3].data_ptr(), m, n, k, stream) == 0
        for a, b in ((got[0], y), (got[1], got[3])):
            assert torch.equal(a.view(torch.int16), b.view(torch.int16))
        assert float((got[2].double() - ref).norm() / ref.norm()) <= 2.0 ** -8
        assert getattr(lib, name + "_ws")(x.data_ptr(), wp.data_ptr(), sc.data_ptr(), got[0].data_ptr(), m, n, k, scratch.data_ptr() + 4, need, stream) == -3


@pytest.mark.parametrize("weight,tile,m,n,k", [
    ("int4", 0, 17, 2052, 7712), ("int4", 1, 66, 1776, 7232), ("int4", 1, 36, 1264, 14432), ("int4", 1, 167, 1184, 5152), ("int4", 1, 67, 2067, 3936),
    ("int4", 1, 51, 4096, 7200), ("int4", 3, 202, 2066, 7904), ("int4", 3, 219, 1440, 10432), ("int4", 3, 487, 768, 12832),
    ("int8", 0, 17, 2058, 7696), ("int8", 0, 19, 7040, 9888), ("int8", 1, 66, 1312, 5152), ("int8", 1, 67, 1538, 5248), ("int8", 1, 258, 1392, 7232),
    ("int8", 3, 196, 1673, 8432), ("int8", 3, 198, 1307, 7696)])
def test_gemm_in_parts_reaches_the_end_of_k(ops, weight, tile, m, n, k):
    """K that 256 does not divide, in a number of parts that divides K / 256 rounded down: parts of that many k each would end before K.  All three
    tiles that are split, remainders of 16 to 240 k (whose activations are eight times the others'), element by element against float64."""
    import ctypes

    from chadslab_amd import QWeightInt4G32, QWeightInt8, _lib

    rule = _lib.load()["_ZN5chadq16gemm_split_partsEiiibPNS_8GemmTileEPi"]
    rule.argtypes = [ctypes.c_int] * 3 + [ctypes.c_bool] + [ctypes.POINTER(ctypes.c_int)] * 2
    picked, span = ctypes.c_int(), ctypes.c_int()
    parts = rule(m, n, k, weight == "int4", ctypes.byref(picked), ctypes.byref(span))
    assert parts > 1 and k // 256 % parts == 0 and k % 256 and picked.value == tile
    g = torch.Generator(device=DEV)
    g.manual_seed(m + n + k)
    x = torch.randn(m, k, device=DEV, generator=g)
    x[:, k // 256 * 256:] *= 8
    x = x.bfloat16()
    if weight == "int4":
        p = torch.randint(0, 256, (n, k // 2), dtype=torch.uint8, device=DEV, generator=g)
        s = torch.exp(torch.randn(n, k // 32, device=DEV, generator=g) * 0.5 - 5.0).half()
        qw = QWeightInt4G32(p, s)
        w = ((torch.stack((p & 15, p >> 4), -1).reshape(n, k).float() - 8) * s.float().repeat_interleave(32, 1)).bfloat16().double()
    else:
        w = torch.randint(-127, 128, (n, k), dtype=torch.int8, device=DEV, generator=g)
        s = torch.exp(torch.randn(n, device=DEV, generator=g) * 0.5 - 8.0)
        qw = QWeightInt8(w, s)
        w = w.double() * s.double()[:, None]
    ref, mag = x.double() @ w.t(), x.double().abs() @ w.abs().t()
    y = ops.qgemm(x, qw)
    # the products are exact in fp32: the fp32 sum of at most k terms, the rounding to bf16
    err = ((y.double() - ref).abs() / (2.0 ** -8 * ref.abs() + (k / 8 + 8) * 2.0 ** -24 * mag)).max()
    assert float(err) <= 1, float(err)
    assert torch.equal(ops.qlinear(x, qw).view(torch.int16), y.view(torch.int16))


def test_gemm_in_parts_captured_in_a_graph(ops):
    """A captured product in parts gives the eager bits on every replay, with other products in between."""
    from chadslab_amd import QWeightInt8

    g = torch.Generator(device=DEV)
    g.manual_seed(5)
    x = torch.randn(40, 8192, device=DEV, generator=g).bfloat16()
    qw = QWeightInt8(torch.randint(-127, 128, (512, 8192), dtype=torch.int8, device=DEV, generator=g), torch.rand(512, device=DEV, generator=g) * 1e-3)
    want = ops.qlinear(x, qw)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = ops.qlinear(x, qw)
    for _ in range(4):
        y.zero_()
        graph.replay()
        other = ops.qlinear(x + 1, qw)
        torch.cuda.synchronize()
        assert torch.equal(y.view(torch.int16), want.view(torch.int16)) and not torch.equal(other, want)


@pytest.mark.parametrize("m,n,k", [(1, 512, 16384), (1, 100, 13056), (2, 77, 16384), (3, 512, 16640), (4, 33, 20480), (5, 512, 8192), (7, 256, 12544), (8, 1000, 16384), (9, 512, 8192),
                                   (12, 77, 10496), (16, 2048, 16384), (16, 16, 7168), (6, 1000, 12544), (6, 2100, 8448), (16, 4090, 16384), (13, 5000, 10496)])
def test_gemv_in_parts_of_k(ops, m, n, k):
    """Decode products of few weight rows and a long K, summed in parts: every kernel family, ragged rows, a last part that is shorter.  No further
    from float64 than in one part (int8: sums in float64 either way; int4: fp32, shorter chains), results in bf16 the same sums rounded once."""
    from chadslab_amd import QWeightInt4G32, QWeightInt8, _lib

    lib = _lib.load()
    g = torch.Generator(device=DEV)
    g.manual_seed(m + n)
    p = torch.randint(0, 256, (n, k // 2), dtype=torch.uint8, device=DEV, generator=g)
    s = torch.exp(torch.randn(n, k // 32, device=DEV, generator=g) * 0.5 - 5.0).half()
    w4 = (torch.stack((p & 15, p >> 4), -1).reshape(n, k).double() - 8) * s.double().repeat_interleave(32, 1)
    w = torch.randint(-127, 128, (n, k), dtype=torch.int8, device=DEV, generator=g)
    s8 = torch.exp(torch.randn(n, device=DEV, generator=g) * 0.5 - 8.0)
    xf = torch.randn(m, k, device=DEV, generator=g)
    stream = torch.cuda.current_stream().cuda_stream
    for x, qw, ref, sc, name in ((xf.bfloat16(), QWeightInt4G32(p, s), xf.bfloat16().double() @ w4.t(), s, "chadq_gemv_i4g32"),
                                 (xf, QWeightInt8(w, s8), xf.double() @ (w.double() * s8.double()[:, None]).t(), s8, "chadq_gemv_i8row")):
        int8 = sc is s8
        if n > 2048 and not int8:  # in one part
            continue
        need = lib.chadq_gemv_workspace_bytes(m, n, k, int(int8))
        assert need >= 2 * m * n * (8 if int8 else 4)  # in parts
        y, yb = ops.qgemv(x, qw), ops.qlinear(x, qw, out_dtype=torch.bfloat16)
        assert torch.equal(yb.view(torch.int16), y.bfloat16().view(torch.int16)) and torch.equal(ops.qlinear(x, qw).view(torch.int32), y.view(torch.int32))
        wp, one, again = w if int8 else p, torch.empty_like(y), torch.empty_like(y)
        assert getattr(lib, name)(x.data_ptr(), wp.data_ptr(), sc.data_ptr(), one.data_ptr(), m, n, k, stream) == 0
        off, off1 = (float((v.double() - ref).norm() / ref.norm()) for v in (y, one))
        assert off <= 1.1 * off1 + 2.0 ** -25 and off <= 1e-6, (name, off, off1)
        scratch = torch.full((need,), 0xFF, dtype=torch.uint8, device=DEV)
        ws = getattr(lib, name + "_ws")
        assert ws(x.data_ptr(), wp.data_ptr(), sc.data_ptr(), again.data_ptr(), m, n, k, 0, scratch.data_ptr(), need, stream) == 0
        assert torch.equal(again.view(torch.int32), y.view(torch.int32))
        for ptr, size in ((None, 0), (scratch.data_ptr(), need - 1)):  # none, or too little: one part
            assert ws(x.data_ptr(), wp.data_ptr(), sc.data_ptr(), again.data_ptr(), m, n, k, 0, ptr, size, stream) == 0
            assert torch.equal(again.view(torch.int32), one.view(torch.int32))
        assert ws(x.data_ptr(), wp.data_ptr(), sc.data_ptr(), again.data_ptr(), m, n, k, 0, scratch.data_ptr() + 4, need, stream) == -3

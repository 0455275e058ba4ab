"""GPU parity of the INT4 path against the oracle (bit-exact for quantize,
unpack/dequantize and the reference-order kernel; 1e-3 of max|y| per row for
the tiled GEMV, whose fp32 summation order differs).
Reference: src/quantize/int4.c:10-114."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from cogito_amd.capi import DeviceArray, last_error
from gpu_util import (host_quant_from_arrays, host_tensor, quant_host_arrays,
                      rel_err_rows, tensor_np)
from oracle_lib import oracle_matmul, oracle_quantize, ptr

pytestmark = pytest.mark.gpu
TOL = 1e-3          # north star: GEMV within 1e-3 relative (fp32 accumulate)


def _bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32)


@pytest.mark.parametrize("shape,gs", [((64, 128), 64), ((33, 7), 8), ((4096, 64), 128),
                                      ((3, 1000), 100)])
def test_quantize_bitexact(gpu, oracle, rng, shape, gs):
    w = rng.normal(0, 0.3, shape).astype(np.float32)
    w.ravel()[::97] = 0.0
    t = host_tensor(gpu, w)
    q = gpu.cg_quantize_int4(t, gs)
    assert q, last_error(gpu)
    data, scales = quant_host_arrays(q)
    odata, oscales = oracle_quantize(oracle, w, gs)
    np.testing.assert_array_equal(data, odata)
    np.testing.assert_array_equal(_bits(scales), _bits(oscales))
    gpu.cg_tensor_quant_free(q)
    gpu.cg_tensor_free(t)


def test_unpack_all_bytes_on_gpu(gpu, oracle):
    # all 256 bytes, flat and tiled layouts: dequantised values bit-exact
    K, N, gs = 256, 512, 64
    data = np.tile(np.arange(256, dtype=np.uint8), K * N // 2 // 256)
    rng = np.random.default_rng(7)
    scales = rng.uniform(0.005, 0.02, K * N // gs).astype(np.float32)
    exp = np.zeros(K * N, np.float32)
    oracle.orc_dequantize_int4(ptr(data), ptr(scales), K * N, gs, ptr(exp))
    hq, keep = host_quant_from_arrays(data, scales, K, N, gs)
    for layout in (1, 2, 3):
        dq = gpu.cgx_quant_to_device_layout(C.byref(hq), layout)
        assert dq, last_error(gpu)
        assert gpu.cgx_quant_layout(dq) == layout
        t = gpu.cg_dequantize(dq)
        assert t, last_error(gpu)
        got = tensor_np(gpu, t).ravel()
        np.testing.assert_array_equal(_bits(got), _bits(exp))
        gpu.cg_tensor_free(t)
        gpu.cg_tensor_quant_free(dq)
    # host-resident quant through the API
    t = gpu.cg_dequantize(C.byref(hq))
    np.testing.assert_array_equal(_bits(tensor_np(gpu, t).ravel()), _bits(exp))
    gpu.cg_tensor_free(t)


def _make_weight(oracle, rng, K, N, gs, config2=False):
    if config2:
        # nibbles uniform in [-8, 7], fp16-valued scales
        v = rng.integers(-8, 8, size=K * N)
        nib = (v & 0xF).astype(np.uint8)
        data = (nib[0::2] | (nib[1::2] << 4)).astype(np.uint8)
        scales = rng.uniform(0.005, 0.02, K * N // gs).astype(np.float16).astype(np.float32)
        return data, scales
    w = rng.normal(0, 0.02, (K, N)).astype(np.float32)
    return oracle_quantize(oracle, w, gs)


SHAPES = [(4096, 4096, 128), (256, 512, 64), (1024, 2048, 128), (4096, 1024, 128),
          (11008, 4096, 128), (256, 16, 16), (768, 2304, 128), (3072, 768, 128)]


@pytest.mark.parametrize("K,N,gs", SHAPES)
@pytest.mark.parametrize("M", [1, 2, 3, 4, 5, 8])
@pytest.mark.parametrize("layout,kernel", [(2, 1), (3, 3)], ids=["valu", "mfma"])
def test_gemv_tiled_vs_oracle(gpu, oracle, rng, K, N, gs, M, layout, kernel):
    if K * N > 4096 * 4096 and M not in (1, 5):
        pytest.skip("large shape: M=1 and M=5 only")
    _gemv_case(gpu, oracle, rng, K, N, gs, M, layout, kernel)


@pytest.mark.parametrize("K,N,gs,M", [(4096, 4096, 128, 16), (1024, 2048, 128, 12),
                                      (768, 2304, 128, 20), (4096, 22016, 128, 5),
                                      (4096, 32000, 128, 5), (4096, 8192, 64, 7),
                                      (256, 512, 16, 40)])
def test_gemv_mfma_more_rows_and_wide(gpu, oracle, rng, K, N, gs, M):
    # M > 8 (row chunks of 16), and N wide enough for 2 / 4 column tiles per block
    _gemv_case(gpu, oracle, rng, K, N, gs, M, 3, 3)


@pytest.mark.parametrize("K,N,gs,M", [(4096, 4096, 128, 40), (1024, 2048, 128, 32),
                                      (256, 512, 128, 100), (768, 1280, 256, 64),
                                      (1024, 1024, 128, 128), (512, 384, 128, 256),
                                      (4096, 32000, 128, 40), (256, 128, 128, 1)])
def test_gemm_mfma_vs_oracle(gpu, oracle, rng, K, N, gs, M):
    # the shared-A-tile GEMM (row blocks of up to 64 / 128 rows, split K)
    _gemv_case(gpu, oracle, rng, K, N, gs, M, 3, 4)


@pytest.mark.parametrize("K,N,gs,M", [(256, 128, 128, 48), (256, 128, 128, 49),
                                      (768, 3072, 128, 97), (4096, 4096, 128, 24),
                                      (4096, 4096, 128, 25), (11008, 4096, 128, 16),
                                      (11008, 4096, 128, 17), (1024, 640, 128, 65),
                                      (512, 768, 256, 50), (512, 704, 64, 70)])
def test_matmul_dispatch_by_rows(gpu, oracle, rng, K, N, gs, M):
    # either side of the lines between the GEMV and the GEMM, odd row counts,
    # an odd number of 128-column slots, a group that the GEMM does not take
    _gemv_case(gpu, oracle, rng, K, N, gs, M, 3, 0)


@pytest.mark.parametrize("K,N,gs,M", [
    (256, 64, 64, 49), (256, 96, 32, 49),   # one missing slot, one row block and a row
    (512, 32, 32, 70), (768, 704, 64, 97), (512, 864, 96, 64), (512, 576, 192, 65),
    (11008, 4096, 64, 17), (11008, 4096, 32, 33),   # 2 and 3 row tiles, K split
    (4096, 4096, 32, 24), (4096, 4096, 64, 25),     # either side of the GEMV
    (512, 336, 48, 70),                     # a group that the GEMM does not take
])
def test_matmul_narrow_groups(gpu, oracle, rng, K, N, gs, M):
    print(f"narrow groups K={K} N={N} gs={gs} M={M}", flush=True)
    _gemv_case(gpu, oracle, rng, K, N, gs, M, 3, 0)


def test_matmul_many_rows_wide_dynamic_range(gpu, oracle, rng):
    # rows of very different magnitudes, a zero row and values spanning many
    # binades through the default dispatch (the GEMM's per-row scaling)
    K, N, gs, M = 1024, 512, 128, 64
    data, scales = _make_weight(oracle, rng, K, N, gs)
    scales = scales.copy()
    scales[::7] *= 1e4
    scales[3::11] *= 1e-6
    x = (rng.normal(0, 1, (M, K)) * np.exp(rng.uniform(-20, 20, (M, K)))).astype(np.float32)
    x *= np.exp(rng.uniform(-30, 30, (M, 1))).astype(np.float32)
    x[2] = 0.0
    y_ref = oracle_matmul(oracle, x, data, scales, K, N, gs)
    hq, keep = host_quant_from_arrays(data, scales, K, N, gs)
    dq = gpu.cgx_quant_to_device_layout(C.byref(hq), 3)
    dx = DeviceArray.from_numpy(gpu, x)
    dy = DeviceArray(gpu, M * N * 4)
    assert gpu.cgx_matmul_int4_dev(dx.ptr, M, dq, dy.ptr) == 0, last_error(gpu)
    assert gpu.cgx_synchronize() == 0
    y = dy.numpy(np.float32, (M, N))
    assert np.all(y[2] == 0.0)
    rows = [i for i in range(M) if i != 2]
    assert rel_err_rows(y[rows], y_ref[rows]) <= TOL
    gpu.cg_tensor_quant_free(dq)


def _gemv64(x, data, scales, K, N, gs):
    w = np.empty(K * N, np.int8)
    w[0::2], w[1::2] = data & 15, data >> 4
    w = np.where(w > 7, w - 16, w).astype(np.float64).reshape(K, N)
    return x.astype(np.float64) @ (w * np.repeat(scales.reshape(K, N // gs), gs, 1))


# of a scale group's largest output, in a row: an operand of the GEMM is off by
# at most 2^-22 of itself (2.4e-7), the sums of up to 11008 products by less than
# ten times that; without the lo halves the error is 2^-11
GEMM_TOL = 3e-6


def check_groups(gpu, x, data, scales, K, N, gs):
    """The default dispatch against 64 bits, each scale group of a row held to
    its own largest value."""
    M = x.shape[0]
    hq, keep = host_quant_from_arrays(data, scales.ravel(), K, N, gs)
    dq = gpu.cgx_quant_to_device_layout(C.byref(hq), 3)
    dx, dy = DeviceArray.from_numpy(gpu, x), DeviceArray(gpu, M * N * 4)
    assert gpu.cgx_matmul_int4_dev(dx.ptr, M, dq, dy.ptr) == 0, last_error(gpu)
    assert gpu.cgx_synchronize() == 0
    y = dy.numpy(np.float32, (M, N // gs, gs))
    ref = _gemv64(x, data, scales, K, N, gs).reshape(M, N // gs, gs)
    err = np.abs(y - ref).max(axis=2) / np.abs(ref).max(axis=2)
    assert err.max() <= GEMM_TOL, err.max()
    gpu.cg_tensor_quant_free(dq)


@pytest.mark.parametrize("K,N,gs,M", [
    (256, 128, 128, 49), (768, 3072, 128, 97), (4096, 4096, 128, 25), (11008, 1024, 128, 70),
    (1024, 640, 128, 65), (512, 768, 256, 50), (256, 96, 32, 49), (768, 704, 64, 97),
    (512, 864, 96, 64), (4096, 2048, 32, 60), (4096, 2048, 64, 60)])
def test_matmul_many_rows_against_64_bits(gpu, rng, K, N, gs, M):
    print(f"GEMM against 64 bits M={M} K={K} N={N} gs={gs}", flush=True)
    data = rng.integers(0, 256, K * N // 2, dtype=np.uint8)
    scales = rng.uniform(0.005, 0.02, (K, N // gs)).astype(np.float32)
    check_groups(gpu, rng.normal(0, 1, (M, K)).astype(np.float32), data, scales, K, N, gs)


@pytest.mark.parametrize("gs", [128, 32])
def test_matmul_many_rows_rows_and_groups_far_apart(gpu, rng, gs):
    # rows up to 2^80 and groups of columns up to 2^40 apart, each pair to its
    # own size
    print(f"rows and groups far apart, groups of {gs}", flush=True)
    K, N, M = 1024, 512, 64
    data = rng.integers(0, 256, K * N // 2, dtype=np.uint8)
    scales = rng.uniform(0.005, 0.02, (K, N // gs))
    scales = (scales * np.exp2(rng.integers(-20, 21, N // gs))).astype(np.float32)
    x = rng.normal(0, 1, (M, K)) * np.exp2(rng.integers(-40, 41, (M, 1)))
    check_groups(gpu, x.astype(np.float32), data, scales, K, N, gs)


@pytest.mark.parametrize("gs", [128, 64, 32])
@pytest.mark.parametrize("kind", ["column group", "zero groups", "infinite scale"])
def test_matmul_many_rows_scales_far_apart(gpu, rng, kind, gs):
    """Columns whose scales lie far below the weight's largest keep their bits:
    each scale group is held to its own size.  A product of the split operands
    is off by 2^-22 of itself, sums of 1024 by a few 2^-24."""
    print(f"scales far apart: {kind}, groups of {gs}", flush=True)
    K, N, M, tol = 1024, 512, 64, 3e-6
    data = rng.integers(0, 256, K * N // 2, dtype=np.uint8)
    scales = rng.uniform(0.005, 0.02, (K, N // gs)).astype(np.float32)
    ok = np.ones(N // gs, bool)
    if kind == "column group":
        scales[:, 1::2] *= np.float32(1e-8)
    elif kind == "zero groups":            # scale 1 by the quantiser's rule
        scales *= np.float32(1e-7)
        scales[5] = scales[700, ::2] = scales[:, 1] = 1.0
        nib = data.reshape(K, N // gs, gs // 2)
        nib[5] = 0
        nib[700, ::2] = nib[:, 1] = 0
        ok[1] = False
    else:
        scales[3, 0] = np.inf
        ok[0] = False
    x = rng.normal(0, 1, (M, K)).astype(np.float32)
    ref = _gemv64(x, data, np.where(np.isinf(scales), 0, scales), K, N, gs)
    hq, keep = host_quant_from_arrays(data, scales.ravel(), K, N, gs)
    dq = gpu.cgx_quant_to_device_layout(C.byref(hq), 3)
    dx, dy = DeviceArray.from_numpy(gpu, x), DeviceArray(gpu, M * N * 4)
    assert gpu.cgx_matmul_int4_dev(dx.ptr, M, dq, dy.ptr) == 0, last_error(gpu)
    assert gpu.cgx_synchronize() == 0
    y = dy.numpy(np.float32, (M, N // gs, gs))[:, ok]
    ref = ref.reshape(M, N // gs, gs)[:, ok]
    err = np.abs(y - ref).max(axis=(0, 2)) / np.abs(ref).max(axis=(0, 2))
    assert err.max() <= tol, err
    gpu.cg_tensor_quant_free(dq)


def test_matmul_many_rows_under_capture(gpu, rng):
    # a captured product takes the path without scratch memory: every replay
    # on new inputs equals the eager GEMV, with larger eager products (which
    # grow the scratch) between the replays
    K, N, gs, M = 512, 256, 128, 64
    data = rng.integers(0, 256, K * N // 2, dtype=np.uint8)
    scales = rng.uniform(0.005, 0.02, K * N // gs).astype(np.float32)
    hq, keep = host_quant_from_arrays(data, scales, K, N, gs)
    dq = gpu.cgx_quant_to_device_layout(C.byref(hq), 3)
    dx, dy = DeviceArray(gpu, M * K * 4), DeviceArray(gpu, M * N * 4)
    de = DeviceArray(gpu, M * N * 4)
    assert gpu.cgx_graph_begin() == 0, last_error(gpu)
    rc = gpu.cgx_matmul_int4_dev(dx.ptr, M, dq, dy.ptr)
    g = gpu.cgx_graph_end()
    assert rc == 0 and g, last_error(gpu)
    for rep in range(3):
        x = rng.normal(0, 1, (M, K)).astype(np.float32)
        dx.upload(x)
        assert gpu.cgx_graph_launch(g) == 0 and gpu.cgx_synchronize() == 0, last_error(gpu)
        y = dy.numpy(np.float32, (M, N))
        assert gpu.cgx_matmul_int4_dev_kernel(dx.ptr, M, dq, de.ptr, 3) == 0, last_error(gpu)
        assert gpu.cgx_synchronize() == 0
        assert np.array_equal(y, de.numpy(np.float32, (M, N)))
        big = 128 * (rep + 2)
        bx, by = DeviceArray(gpu, big * K * 4), DeviceArray(gpu, big * N * 4)
        gpu.cgx_memset(bx.ptr, 0, big * K * 4)
        assert gpu.cgx_matmul_int4_dev(bx.ptr, big, dq, by.ptr) == 0, last_error(gpu)
        assert gpu.cgx_synchronize() == 0
    assert gpu.cgx_graph_free(g) == 0
    gpu.cg_tensor_quant_free(dq)


def _stream_case(gpu, oracle, rng, K, N, gs, M, min_units):
    """The persistent streaming GEMV (taken at K = 4096, up to 5 rows, once
    the output has min_units 32-column units per CU) against the oracle, and
    against the block-per-tile kernel on the same inputs (both carry the rows
    as hi + lo fp16: within 1e-5 of max|y| per row)."""
    # nibble bytes and fp16-valued scales drawn directly (a normal draw of a
    # 4096 x 128256 matrix would take 2 GiB)
    data = rng.integers(0, 256, K * N // 2, dtype=np.uint8)
    scales = rng.uniform(0.005, 0.02, K * N // gs).astype(np.float16).astype(np.float32)
    x = rng.normal(0, 1, (M, K)).astype(np.float32)
    y_ref = oracle_matmul(oracle, x, data, scales, K, N, gs)
    hq, keep = host_quant_from_arrays(data, scales, K, N, gs)
    dq = gpu.cgx_quant_to_device_layout(C.byref(hq), 3)
    assert dq, last_error(gpu)
    dx = DeviceArray.from_numpy(gpu, x)
    dy = DeviceArray(gpu, M * N * 4)
    old = gpu.cgx_gemv_stream_min_units(-1)
    ys = []
    try:
        for units in (min_units, 0):
            gpu.cgx_gemv_stream_min_units(units)
            for rep in range(2):         # a second call on the same buffers
                gpu.cgx_memset(dy.ptr, 0xFF, M * N * 4)
                assert gpu.cgx_matmul_int4_dev_kernel(dx.ptr, M, dq, dy.ptr, 3) == 0, \
                    last_error(gpu)
                assert gpu.cgx_synchronize() == 0, last_error(gpu)
                y = dy.numpy(np.float32, (M, N))
                assert np.all(np.isfinite(y))
                assert rel_err_rows(y, y_ref) <= TOL
            ys.append(y)
    finally:
        gpu.cgx_gemv_stream_min_units(old)
    assert rel_err_rows(ys[0], ys[1]) <= 1e-5
    gpu.cg_tensor_quant_free(dq)


@pytest.mark.parametrize("N,M", [(128256, 5), (65536, 1), (65536, 3)])
def test_gemv_stream_wide_vocab(gpu, oracle, rng, N, M):
    # the default dispatch: a 64k / 128k-column lm_head at 1-5 rows
    _stream_case(gpu, oracle, rng, 4096, N, 128, M, 8)


@pytest.mark.parametrize("N,gs,M", [(4096, 128, 5), (22016, 128, 2), (2048, 64, 4),
                                    (6144, 256, 1), (4160, 64, 5)])
def test_gemv_stream_forced(gpu, oracle, rng, N, gs, M):
    # every supported product through the streaming kernel: runs of one to
    # three units (odd runs end with an idle unit), groups of two units
    _stream_case(gpu, oracle, rng, 4096, N, gs, M, 1)


def test_gemv_mfma_wide_dynamic_range(gpu, oracle, rng):
    # activations spanning many binades, a zero row, huge and tiny scales:
    # the per-round power-of-two scaling keeps the fp16 terms in range
    K, N, gs, M = 1024, 512, 128, 4
    data, scales = _make_weight(oracle, rng, K, N, gs)
    scales = scales.copy()
    scales[::7] *= 1e4
    scales[3::11] *= 1e-6
    x = (rng.normal(0, 1, (M, K)) * np.exp(rng.uniform(-20, 20, (M, K)))).astype(np.float32)
    x[2] = 0.0
    y_ref = oracle_matmul(oracle, x, data, scales, K, N, gs)
    hq, keep = host_quant_from_arrays(data, scales, K, N, gs)
    dq = gpu.cgx_quant_to_device_layout(C.byref(hq), 3)
    dx = DeviceArray.from_numpy(gpu, x)
    dy = DeviceArray(gpu, M * N * 4)
    assert gpu.cgx_matmul_int4_dev_kernel(dx.ptr, M, dq, dy.ptr, 3) == 0, last_error(gpu)
    assert gpu.cgx_synchronize() == 0
    y = dy.numpy(np.float32, (M, N))
    assert np.all(y[2] == 0.0)
    keep_rows = [0, 1, 3]
    assert rel_err_rows(y[keep_rows], y_ref[keep_rows]) <= TOL
    gpu.cg_tensor_quant_free(dq)


def _gemv_case(gpu, oracle, rng, K, N, gs, M, layout, kernel):
    data, scales = _make_weight(oracle, rng, K, N, gs, config2=(K == 4096 and N == 4096))
    x = rng.normal(0, 1, (M, K)).astype(np.float32)
    y_ref = oracle_matmul(oracle, x, data, scales, K, N, gs)
    hq, keep = host_quant_from_arrays(data, scales, K, N, gs)
    dq = gpu.cgx_quant_to_device_layout(C.byref(hq), layout)
    assert dq and gpu.cgx_quant_layout(dq) == layout, last_error(gpu)
    dx = DeviceArray.from_numpy(gpu, x)
    dy = DeviceArray(gpu, M * N * 4)
    for rep in range(2):         # a second call on the same buffers
        gpu.cgx_memset(dy.ptr, 0xFF, M * N * 4)
        assert gpu.cgx_matmul_int4_dev_kernel(dx.ptr, M, dq, dy.ptr, kernel) == 0, \
            last_error(gpu)
        assert gpu.cgx_synchronize() == 0, last_error(gpu)
        y = dy.numpy(np.float32, (M, N))
        assert np.all(np.isfinite(y))
        assert rel_err_rows(y, y_ref) <= TOL
    gpu.cg_tensor_quant_free(dq)


@pytest.mark.parametrize("M,K,N,gs", [(1, 64, 64, 64), (5, 128, 96, 32), (3, 17, 10, 4),
                                      (2, 300, 130, 26)])
def test_generic_kernel_bitexact(gpu, oracle, rng, M, K, N, gs):
    w = rng.normal(0, 0.02, (K, N)).astype(np.float32)
    x = rng.normal(0, 1, (M, K)).astype(np.float32)
    data, scales = oracle_quantize(oracle, w, gs)
    y_ref = oracle_matmul(oracle, x, data, scales, K, N, gs)
    # host tensors + host quant through cg_matmul_int4 (reference-order kernel)
    hq, keep = host_quant_from_arrays(data, scales, K, N, gs)
    tx = host_tensor(gpu, x)
    ty = host_tensor(gpu, np.full((M, N), 7.0, np.float32))
    gpu.cg_matmul_int4(tx, C.byref(hq), ty)
    assert last_error(gpu) == "", last_error(gpu)
    np.testing.assert_array_equal(_bits(tensor_np(gpu, ty)), _bits(y_ref))
    gpu.cg_tensor_free(tx)
    gpu.cg_tensor_free(ty)


@pytest.mark.parametrize("M,K,N,gs", [
    (1, 63, 65, 3),                         # below one step: thread per output
    (1, 64, 1, 1), (2, 65, 63, 2), (3, 128, 64, 7), (5, 191, 129, 129),
    (513, 71, 33, 40), (514, 64, 64, 10 ** 6), (9, 130, 4160, 100),
])
def test_reference_order_matmul_edges(gpu, oracle, rng, M, K, N, gs):
    """Ragged steps, columns and rows, one row or two a block: bit for bit the
    reference's sums, signed zeros, infinities and NaN among the inputs."""
    print(f"flat M={M} K={K} N={N} gs={gs}", flush=True)
    w = rng.normal(0, 0.02, (K, N)).astype(np.float32)
    w.flat[0:min(gs, K * N // 2)] = 0.0     # a group of scale 0
    x = rng.normal(0, 1, (M, K)).astype(np.float32)
    x[0, 0], x[0, K - 1] = -0.0, 1e-42
    if M > 1:
        x[1, K // 2] = np.inf
    if M > 2:
        x[2, K - 1] = np.nan
    data, scales = oracle_quantize(oracle, w, gs)
    y_ref = oracle_matmul(oracle, x, data, scales, K, N, gs)
    hq, keep = host_quant_from_arrays(data, scales, K, N, gs)
    tx = host_tensor(gpu, x)
    ty = host_tensor(gpu, np.full((M, N), 7.0, np.float32))
    gpu.cgx_clear_error()
    gpu.cg_matmul_int4(tx, C.byref(hq), ty)
    assert last_error(gpu) == "", last_error(gpu)
    y = tensor_np(gpu, ty)
    np.testing.assert_array_equal(np.isnan(y), np.isnan(y_ref))
    num = ~np.isnan(y_ref)                  # a NaN's sign is not part of the contract
    np.testing.assert_array_equal(_bits(y[num]), _bits(y_ref[num]))
    gpu.cg_tensor_free(tx)
    gpu.cg_tensor_free(ty)


def test_gemv_api_host_io_device_weight(gpu, oracle, rng):
    K, N, gs = 512, 256, 128
    data, scales = _make_weight(oracle, rng, K, N, gs)
    x = rng.normal(0, 1, (1, K)).astype(np.float32)
    y_ref = oracle_matmul(oracle, x, data, scales, K, N, gs)
    hq, keep = host_quant_from_arrays(data, scales, K, N, gs)
    dq = gpu.cgx_quant_to_device(C.byref(hq))
    tx = host_tensor(gpu, x)
    ty = host_tensor(gpu, np.zeros((1, N), np.float32))
    gpu.cgx_clear_error()
    gpu.cg_gemv_int4(tx, dq, ty)
    assert last_error(gpu) == "", last_error(gpu)
    assert rel_err_rows(tensor_np(gpu, ty), y_ref) <= TOL
    gpu.cg_tensor_quant_free(dq)
    gpu.cg_tensor_free(tx)
    gpu.cg_tensor_free(ty)


def test_matmul_shape_mismatch_sets_error(gpu, rng):
    x = host_tensor(gpu, np.ones((2, 10), np.float32))
    w = host_tensor(gpu, np.ones((12, 8), np.float32))
    q = gpu.cg_quantize_int4(w, 8)
    y = host_tensor(gpu, np.zeros((2, 8), np.float32))
    gpu.cgx_clear_error()
    gpu.cg_matmul_int4(x, q, y)
    assert "shape mismatch" in last_error(gpu)
    for t in (x, w, y):
        gpu.cg_tensor_free(t)
    gpu.cg_tensor_quant_free(q)

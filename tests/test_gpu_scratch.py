"""GPU: calls whose faster path needs scratch memory, on a device that has none
for it: the path without it runs, the results are its results, and neither the
failed allocation nor the fallback touches the library's error."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from cogito_amd.capi import CgFlashAttnParams, DeviceArray, host_quant_from_arrays, last_error
from oracle_lib import ptr
from test_gpu_filter import verify_inputs

pytestmark = pytest.mark.gpu


@pytest.fixture()
def limit(gpu):
    yield gpu.cgx_scratch_limit
    gpu.cgx_scratch_limit(0)
    gpu.cgx_clear_error()


def earlier_error(gpu):
    assert gpu.cgx_event_record(99) == -1
    return last_error(gpu)


@pytest.mark.parametrize("K,N,gs,M", [(512, 256, 128, 64), (1024, 96, 32, 200)])
def test_linear_without_scratch(gpu, rng, limit, K, N, gs, M):
    print(f"linear without scratch M={M} K={K} N={N} gs={gs}", flush=True)
    data = rng.integers(0, 256, K * N // 2, dtype=np.uint8)
    scales = rng.uniform(0.005, 0.02, K * N // gs).astype(np.float32)
    hq, keep = host_quant_from_arrays(data, scales, K, N, gs)
    dq = gpu.cgx_quant_to_device_layout(C.byref(hq), 3)
    dx = DeviceArray.from_numpy(gpu, rng.normal(0, 1, (M, K)).astype(np.float32))
    dy, de = DeviceArray(gpu, M * N * 4), DeviceArray(gpu, M * N * 4)
    limit(1)
    err = earlier_error(gpu)
    assert gpu.cgx_matmul_int4_dev(dx.ptr, M, dq, dy.ptr) == 0, last_error(gpu)
    assert gpu.cgx_matmul_int4_dev_kernel(dx.ptr, M, dq, de.ptr, 3) == 0, last_error(gpu)
    assert gpu.cgx_synchronize() == 0, last_error(gpu)
    assert last_error(gpu) == err
    np.testing.assert_array_equal(dy.numpy(np.uint32, (M, N)), de.numpy(np.uint32, (M, N)))
    gpu.cg_tensor_quant_free(dq)


def test_flash_without_scratch(gpu, rng, limit):
    B, Nq, Nk, H, D = 1, 37, 90, 2, 64
    print("flash without scratch", flush=True)
    dev = [DeviceArray.from_numpy(gpu, rng.normal(0, 1, (B, n, H, D)).astype(np.float32))
           for n in (Nq, Nk, Nk)]
    outs = []
    old = gpu.cgx_flash_packed_min(-1)
    try:
        for mega, lim in ((1 << 30, 0), (0, 1)):
            o, l = DeviceArray(gpu, B * Nq * H * D * 4), DeviceArray(gpu, B * H * Nq * 4)
            gpu.cgx_flash_packed_min(mega)
            limit(lim)
            err = earlier_error(gpu)
            p = CgFlashAttnParams(Q=dev[0].ptr, K=dev[1].ptr, V=dev[2].ptr, O=o.ptr, batch_size=B,
                                  seqlen_q=Nq, seqlen_k=Nk, n_heads=H, n_heads_k=H, d_head=D,
                                  scale=0.125, mask_type=1, softmax_lse=l.ptr)
            gpu.cg_flash_attention_forward(C.byref(p))
            assert last_error(gpu) == err
            outs.append((o.numpy(np.uint32, (B * Nq * H * D,)), l.numpy(np.uint32, (B * H * Nq,))))
    finally:
        gpu.cgx_flash_packed_min(old)
    for a, b in zip(*outs):
        np.testing.assert_array_equal(a, b)


def test_filtered_verify_without_scratch_for_all_rows(gpu, oracle, rng, limit):
    B, gamma, V, T, k, p = 1, 4, 4001, 0.8, 0, 0.9
    print("filtered verify without scratch for all rows", flush=True)
    host = verify_inputs(oracle, rng, V, gamma, T, k, p, True)
    dev = [DeviceArray.from_numpy(gpu, a) for a in host]
    out, n, ap = (DeviceArray(gpu, 4 * c) for c in (gamma + 1, 1, gamma))
    # 16 bytes a value (probabilities, sorted ones, the sort's buffers), and a
    # buffer is a quarter larger than asked for: room for gamma + 1 rows, not
    # for 2 gamma + 1
    limit(7 * V * 16 * 5 // 4)
    err = earlier_error(gpu)
    assert gpu.cgx_verify_chain_batch_dev(*(d.ptr for d in dev), B, gamma, V, T, k, p, out.ptr,
                                          n.ptr, ap.ptr) == 0, last_error(gpu)
    assert gpu.cgx_synchronize() == 0, last_error(gpu)
    assert last_error(gpu) == err
    o, ap_o = np.zeros(gamma + 1, np.int32), np.zeros(gamma, np.float32)
    n_o = oracle.orc_verify_chain(*(ptr(a) for a in host), gamma, V, T, k, p, ptr(o), ptr(ap_o))
    assert n.numpy(np.int32, (1,))[0] == n_o
    np.testing.assert_array_equal(out.numpy(np.int32, (gamma + 1,))[:n_o + 1], o[:n_o + 1])
    np.testing.assert_array_equal(ap.numpy(np.uint32, (gamma,)), ap_o.view(np.uint32))

"""The register-streamed products of few rows (gemm_rows.hip) and the lines of the tile rule, against
the exact rule: each tile shape at partial tiles in M, N and K, both sides of each line, unaligned
output rows, and the device-pointer entry (whose bias and multipliers are not padded)."""

import ctypes as C

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    from taco_amd import hip
    return hip.HipDevice.open(0)


# (m, n, k): 16 x 16 tiles (fewer k-steps than waves, and a remainder), 16 x 32, 32 x 16, 32 x 32 and
# its line at 512 tiles, 64 x 32 and 64 x 64 (K above 2,048), 64 x 64 LDS tiles below and above
# 512 rows, and one past them
SHAPES = [(1, 1, 1), (5, 100, 70), (16, 4096, 330), (16, 4200, 130), (130, 700, 128), (32, 2050, 64),
          (200, 2300, 700), (250, 2033, 200), (256, 2065, 130), (300, 1500, 2112), (512, 2000, 2176),
          (512, 2064, 2176), (700, 3001, 130), (1000, 3600, 130)]


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_few_row_products(dev, m, n, k):
    from taco_amd import hip
    r = np.random.default_rng(m * 31 + n * 7 + k)
    a = r.integers(-128, 128, (m, k)).astype(np.int8)
    w = r.integers(-128, 128, (n, k)).astype(np.int8)
    assert np.array_equal(hip.matmul_i8(dev, w, a), O.matmul_i8(w, a))
    bias = r.integers(-(1 << 31), 1 << 31, n).astype(np.int32)
    mult = r.integers(-(1 << 31), 1 << 31, n).astype(np.int32)
    shift = int(r.integers(36, 56))
    want = O.linear_act_ref(w, a, bias, mult, shift)
    assert np.array_equal(hip.gemm_requant_i8(dev, w, a, bias, mult, shift), want)
    # the device-pointer entry
    m_pad, n_pad, k_pad = hip.gemm_layout(m, n, k)
    L, bufs = hip.lib(), []
    for x in (hip.gemm_pack(w, n_pad, k_pad), hip.gemm_pack(a, m_pad, k_pad), bias, mult, np.zeros((m, n), np.int8)):
        p = C.c_void_p()
        hip._check(L.hs_device_alloc(dev.h, x.nbytes, C.byref(p)))
        hip._check(L.hs_device_upload(dev.h, p, hip._ptr(x), x.nbytes))
        bufs.append(p)
    hip._check(L.hs_op_gemm_requant_i8_dev(dev.h, *bufs[:4], shift, m, n, k, bufs[4], None))
    got = np.zeros((m, n), np.int8)
    hip._check(L.hs_device_download(dev.h, hip._ptr(got), bufs[4], got.nbytes))
    for p in bufs:
        L.hs_device_free(dev.h, p)
    assert np.array_equal(got, want)

"""The register-streamed products of few rows (gemm_rows.hip), the 64 x 64 LDS tiles, and the lines of
the tile rules between them, against the exact rule: each tile shape at partial tiles in M, N and K, both
sides of each line, the general and the narrow rescale (the lines differ), output rows that are aligned and
that are not, and the device-pointer entry (whose bias and multipliers are not padded)."""

import ctypes as C

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    from taco_amd import hip
    return hip.HipDevice.open(0)


# (m, n, k). The tiles of a shape follow from the counts of tiles beside it.
SHAPES = [
    # fewer k-steps than waves, a remainder of them, partial tiles in every direction
    (1, 1, 1), (5, 100, 70), (16, 4096, 330), (200, 2300, 700), (250, 2033, 200), (300, 1500, 2112), (512, 2000, 2176),
    (64, 1024, 130), (64, 1025, 130),  # 256 and 260 of 16 x 16
    (16, 4097, 130),                   # 16 x 32 (one row of tiles)
    (64, 2048, 130), (64, 2049, 130),  # 256 and 258 of 32 x 16
    (256, 2048, 130), (256, 2064, 130), (256, 2065, 130),  # 512 and 520 of 32 x 32: the narrow rescale's line
    (256, 3072, 130), (256, 3088, 130), (256, 3073, 130),  # 768 and 776: the general one's
    (256, 1024, 2112), (256, 1040, 2112),  # K above 2,048: 256 and 264 of 32 x 32
    (512, 1024, 2112), (512, 1040, 2112),  # 256 and 264 of 64 x 32
    (512, 2048, 2112), (512, 2064, 2112), (512, 2065, 2112),  # 256 and 264 of 64 x 64; past it the LDS tiles
    (960, 3840, 130), (960, 3856, 130), (960, 3841, 130),  # more than 512 rows: 900 and 915 of 64 x 64 in LDS
    (640, 4096, 1040), (640, 4112, 1040), (640, 4083, 1040),  # K above 1,024: 640 and 650
    (700, 3001, 130),  # unaligned 64 x 64 LDS tiles of three k-steps, above 512 rows
]


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
    small = (bias >> 16).astype(np.int32)  # every sum and bias within i32: the narrow rescale
    assert np.array_equal(hip.gemm_requant_i8(dev, w, a, small, mult, shift),
                          O.linear_act_ref(w, a, small, mult, shift))
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


def test_unaligned_rows_take_the_tiles_of_aligned_ones(dev):
    """Outputs whose rows do not start at multiples of 16 bytes differ in the stores alone: with a 256 x 128
    tile for each, 256 x 4,099 x 6,400 took 67 us where its 64 x 64 tiles take 28, as those of the aligned
    256 x 4,112 x 6,400 do."""
    from taco_amd import hip
    L, m, k = hip.lib(), 256, 6400

    def ns(n):
        m_pad, n_pad, k_pad = hip.gemm_layout(m, n, k)
        bufs = []
        for x in (np.ones(n_pad * k_pad, np.int8), np.ones(m_pad * k_pad, np.int8), np.zeros(n, np.int32),
                  np.full(n, 1 << 30, np.int32), np.zeros(m * n, np.int8)):
            p = C.c_void_p()
            hip._check(L.hs_device_alloc(dev.h, x.nbytes, C.byref(p)))
            hip._check(L.hs_device_upload(dev.h, p, hip._ptr(x), x.nbytes))
            bufs.append(p)
        t, best = C.c_uint64(), 1 << 62
        for _ in range(8):
            hip._check(L.hs_op_gemm_requant_gpu_ns(dev.h, *bufs[:4], 38, m, n, k, bufs[4], 20, C.byref(t)))
            best = min(best, t.value)
        for p in bufs:
            L.hs_device_free(dev.h, p)
        return best

    assert ns(4099) < 1.6 * ns(4112)

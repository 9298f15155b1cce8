"""The one-launch decode attention at head dims 16, 32 and 128: caches at both sides of the line between
a wave and a workgroup per row-head and at the lines of 64-key blocks, full, ragged and one-key
contexts, clamped and unclamped scores, against the oracle; the split form past 1,024 keys, at head_dim
256, and at head_dim 128 past 128 keys from 1,025 row-heads on; and folds (prefill passes take the same
kernels) at those head dims against the CPU fast path, among them passes whose rows hold few and many
keys in the mean and one whose split partials take more than 1 GiB (rows in two chunks)."""

import ctypes as C

import numpy as np
import pytest

from oracle import oracle as O
from tests.conftest import splitmix_tokens

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hd,cap", [(16, 1), (16, 100), (16, 512), (16, 513), (16, 1024), (32, 64), (32, 191), (32, 256),
                                    (32, 257), (32, 512), (32, 520), (32, 1024), (128, 64), (128, 128), (128, 129),
                                    (128, 700), (128, 1024),
                                    (16, 1100), (32, 1087), (64, 2048), (128, 1025), (256, 1), (256, 200), (256, 1030)])
def test_decode_attention(hd, cap):
    check_decode(hd, cap, 7, 3)


@pytest.mark.parametrize("rows,heads", [(512, 2), (205, 5)])  # 1,024 row-heads in one launch, 1,025 split
def test_line_of_head_dim_128(rows, heads):
    check_decode(128, 129, rows, heads)


def check_decode(hd, cap, B, H):
    from taco_amd import hip
    dev, L = hip.HipDevice.open(0), hip.lib()
    r = np.random.default_rng(hd * 2000 + cap)
    q = r.integers(-128, 128, (B, H, hd)).astype(np.int8)
    kc, vc = (r.integers(-128, 128, (B, H, cap, hd)).astype(np.int8) for _ in range(2))
    ctx = np.minimum(cap, np.resize([1, cap, cap - 1 if cap > 1 else 1, 63, 64, 65, 1 + cap // 2], B)).astype(np.uint32)
    table = np.array([round(2 ** 30 * np.exp(-i / 256)) for i in range(8192)], np.int32)
    for score_s in (33, 8):
        want = O.attend_decode_ref(q, kc, vc, ctx, 1_400_000_000, score_s, 1_300_000_000, 53, table, 30)
        out, bufs = np.zeros((B, H * hd), np.int8), []
        for x in (q, kc, vc, ctx, table, out):
            p = C.c_void_p()
            hip._check(L.hs_device_alloc(dev.h, x.nbytes, C.byref(p)))
            hip._check(L.hs_device_upload(dev.h, p, hip._ptr(x), x.nbytes))
            bufs.append(p)
        hip._check(L.hs_op_attend_decode_dev(dev.h, *bufs[:4], B, H, hd, cap, 1_400_000_000, score_s, 1_300_000_000,
                                             53, bufs[4], len(table), 30, bufs[5], None))
        hip._check(L.hs_device_download(dev.h, hip._ptr(out), bufs[5], out.nbytes))
        for p in bufs:
            L.hs_device_free(dev.h, p)
        assert np.array_equal(out, want), score_s


# n rows in all, `before` of them in a pass of their own
@pytest.mark.parametrize("heads,hd,n,before,n_ctx", [
    (3, 16, 190, 0, 1024), (3, 32, 600, 0, 1024), (2, 128, 200, 0, 1024),
    (5, 128, 300, 0, 1024), (3, 128, 900, 500, 1024), (3, 128, 1100, 600, 2048), (4, 16, 1400, 0, 1 << 16)])
def test_folds(heads, hd, n, before, n_ctx):
    from taco_amd import hip, synth
    dev, V = hip.HipDevice.open(0), 500
    mb = synth.build_model(synth.Dims(1, heads, heads * hd, 256, vocab=V, n_ctx=n_ctx), seed=0xD135)
    hm, om = hip.HipModel.load(dev, mb), O.Model(mb)
    blk = np.array(splitmix_tokens(n, n, V - 1), np.uint32)
    batch = hip.HipBatch(hm, 1, n)
    inputs, queries = [(0, V - 1)] + [(0, int(t)) for t in blk[:-1]], [(0, int(t)) for t in blk]
    raw = [batch.run_coded_raw(inputs[a:b], queries[a:b], 32) for a, b in ((0, before), (before, n)) if b > a]
    assert np.array_equal(np.concatenate(raw), O.fast_window_intervals(om, blk, chunk=32))

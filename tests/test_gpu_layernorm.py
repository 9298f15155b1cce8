"""The single-precision LayerNorm (layernorm.hip) at the widths and row counts that select its
forms, through whole passes whose intervals must equal the CPU fast path's: 384 columns below and
above 4,096 rows, 640 to 2,048 columns, integer and fractional beta (version 2), and a model whose
residual updates pass 2^24, so that rows leave the 64-bit terms. The host helpers are checked against
128-bit arithmetic by native/ln_terms_check.cpp."""

import os
import subprocess
import tempfile

import numpy as np
import pytest

from oracle import oracle as O
from tests.conftest import splitmix_tokens

HERE = os.path.dirname(os.path.abspath(__file__))


def test_row_terms_and_elements_are_exact():
    src = os.path.join(HERE, "native", "ln_terms_check.cpp")
    with tempfile.TemporaryDirectory() as d:
        exe = os.path.join(d, "ln_terms_check")
        subprocess.run(["g++", "-O2", "-std=c++17", "-o", exe, src], check=True)
        out = subprocess.run([exe], capture_output=True, text=True, timeout=300)
        assert out.returncode == 0, out.stdout + out.stderr
        assert out.stdout.startswith("ok")


@pytest.mark.gpu
@pytest.mark.parametrize("d,heads,windows,n,kw", [
    (384, 6, 2, 30, {}), (384, 6, 33, 128, {}), (640, 10, 3, 33, {}), (1024, 16, 2, 70, {}), (1088, 17, 2, 40, {}),
    (2048, 32, 1, 21, {}), (384, 6, 3, 50, {"wide": True}), (768, 12, 2, 65, {"wide": True}),
    (768, 12, 2, 65, {"residual_target": 1 << 26}), (384, 6, 33, 128, {"residual_target": 1 << 26})])
def test_passes_equal_the_cpu(d, heads, windows, n, kw):
    from taco_amd import hip, synth
    dev = hip.HipDevice.open(0)
    V = 600
    mb = synth.build_model(synth.Dims(2, heads, d, 2 * d, vocab=V, n_ctx=256), seed=0x17A + d, **kw)
    hm, om = hip.HipModel.load(dev, mb), O.Model(mb)
    batch = hip.HipBatch(hm, windows, windows * n)
    blocks = [np.array(splitmix_tokens(70 + w, n, V - 1), np.uint32) for w in range(windows)]
    inputs, queries = [], []
    for w, blk in enumerate(blocks):
        inputs += [(w, V - 1)] + [(w, int(t)) for t in blk[:-1]]
        queries += [(0, int(t)) for t in blk]
    raw = batch.run_coded_raw(inputs, queries, 32).reshape(windows, n, 3)
    for w in sorted({0, windows // 2, windows - 1}):
        want = O.fast_window_intervals(om, blocks[w], chunk=32)
        assert np.array_equal(raw[w], want), w

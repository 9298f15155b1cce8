"""Version-2 products at the row counts that select their tiles (planes of 16 rows in turn: counts on,
below and above a multiple of 16; register-streamed, 64 x 64, 128 x 192 and 256-row tiles), for the
narrow rescale and the general one (a residual shift below the bound), compact and i64 logits, against
the CPU fast path."""

import numpy as np
import pytest

from oracle import oracle as O
from tests.conftest import splitmix_tokens

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kw", [{}, {"residual_target": 1 << 22}, {"table_len": 20000}])
@pytest.mark.parametrize("windows,n", [(1, 5), (2, 16), (3, 65), (5, 125), (8, 250), (24, 255)])
def test_wide_passes_equal_the_cpu(windows, n, kw):
    from taco_amd import hip, synth
    dev = hip.HipDevice.open(0)
    V = 1500
    mb = synth.build_model(synth.Dims(1, 9, 576, 2112, vocab=V, n_ctx=256), seed=0x71DE, wide=True, **kw)
    hm, om = hip.HipModel.load(dev, mb), O.Model(mb)
    batch = hip.HipBatch(hm, windows, windows * n)
    blocks = [np.array(splitmix_tokens(30 + w, n, V - 1), np.uint32) for w in range(windows)]
    inputs, queries = [], []
    for w, blk in enumerate(blocks):
        inputs += [(w, V - 1)] + [(w, int(t)) for t in blk[:-1]]
        queries += [(0, int(t)) for t in blk]
    raw = batch.run_coded_raw(inputs, queries, 32).reshape(windows, n, 3)
    for w in sorted({0, windows - 1}):
        want = O.fast_window_intervals(om, blocks[w], chunk=32)
        assert np.array_equal(raw[w], want), w

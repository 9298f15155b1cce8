"""The LM head of few rows (k_head_rows): row counts at the edges of its 16-row tiles and at its line
against the tiles (64 and 65 rows), its 8- and 16-wave workgroups for 16, 32 and 64 rows (their LDS line at
64 KiB: widths of 1,088, 2,112 and 4,160 cross it, the last past the LDS for 64 rows; K past the steps in
flight), vocabularies that end inside a 4-column group and inside a 64-column tile, and
both rescales (a logits shift of 31 or more, and below), against the CPU fast path."""

import numpy as np
import pytest

from oracle import oracle as O
from tests.conftest import splitmix_tokens

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,vocab,general", [(1, 1502, False), (1, 1502, True), (12, 131, False), (17, 1001, False),
                                                 (33, 500, False), (33, 500, True), (65, 333, False), (65, 333, True)])
def test_few_rows_of_logits(monkeypatch, heads, vocab, general):
    from taco_amd import hip, synth
    d, plain = 64 * heads, synth.shift_for
    if general:  # the logits' shift alone, 64-bit distances within and past the table
        monkeypatch.setattr(synth, "shift_for",
                            lambda s2, t: 30 if (s2, t) == (synth.SIGMA_ACT_SQ * d, 768) else plain(s2, t))
    mb = synth.build_model(synth.Dims(1, heads, d, 128, vocab=vocab, n_ctx=128), seed=0x4EAD)
    dev = hip.HipDevice.open(0)
    hm, om = hip.HipModel.load(dev, mb), O.Model(mb)
    batch = hip.HipBatch(hm, 1, 65)
    for n in (1, 15, 16, 17, 32, 33, 64, 65):
        blk = np.array(splitmix_tokens(40 + n, n, vocab - 1), np.uint32)
        raw = batch.run_coded_raw([(0, vocab - 1)] + [(0, int(t)) for t in blk[:-1]], [(0, int(t)) for t in blk], 32)
        assert np.array_equal(np.asarray(raw).reshape(n, 3), O.fast_window_intervals(om, blk, chunk=32)), n
        batch.reset(0)

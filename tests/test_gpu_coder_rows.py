"""The coder op over compact logits at the lines of its forms, against the oracle's table: launches of
at most 256 rows (1,024 threads a row) and more (256 threads), Decode targets at the first and last value
of a symbol's interval, vocabularies whose Decode segments hold 64, 128 and 256 symbols, and, on both sides
of the line, nearly flat rows (many ties for the largest) and a table that does not end in zeros."""

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    from taco_amd import hip
    return hip.HipDevice.open(0)


@pytest.mark.parametrize("vocab,rows,bits,kind", [
    (1, 2, 8, ""), (65, 3, 7, ""), (50257, 3, 32, ""), (65536, 2, 32, ""), (70000, 3, 32, ""), (131073, 3, 32, ""),
    (1000, 256, 24, "flat"), (1000, 257, 24, "flat"), (1000, 256, 32, "no zero tail"), (1000, 257, 32, "no zero tail"),
    (70000, 3, 32, "no zero tail"), (1000, 512, 24, "flat"), (1000, 513, 32, "no zero tail")])
def test_decode_finds_the_interval(dev, vocab, rows, bits, kind):
    from taco_amd import hip, synth
    r = np.random.default_rng(vocab + rows)
    table = synth.exp_tables()[1]
    if kind == "no zero tail":
        table = np.ascontiguousarray(table[:300])  # symbols past it weigh the last entry
    spread = 3 if kind == "flat" else 4000
    logits = np.rint(r.standard_normal((rows, vocab)) * spread).astype(np.int64)
    tables = [O.freq_from_weights(O.logits_to_weights(x, table), bits) for x in logits]
    ends = [np.cumsum(np.asarray(f, dtype=object)) for f in tables]
    pick = r.integers(0, vocab, rows)
    pick[0], pick[-1] = vocab - 1, 0
    for first in (True, False):  # the first and the last target of the picked symbol's interval
        targets = [int(e[s]) - (int(f[s]) if first else 1) for f, e, s in zip(tables, ends, pick)]
        got = hip.coder(dev, logits, table, [(1, t) for t in targets], bits)
        enc = hip.coder(dev, logits, table, [(0, int(s)) for s in pick], bits)
        for i, s in enumerate(pick):
            want = (int(s), int(ends[i][s]) - int(tables[i][s]), int(tables[i][s]))
            assert tuple(int(x) for x in got[i]) == want, (i, first)
            assert tuple(int(x) for x in enc[i]) == want, i

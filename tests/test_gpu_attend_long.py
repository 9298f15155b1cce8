"""Prefill attention over more than 512 keys at head_dim 64 (k_attend_long): windows of whole and
partial key stages, appended passes whose groups start inside a window, negative score multipliers,
a table without a zero tail, output shifts outside attn_out_planes, and several tasks per workgroup (the
ring and the loads carried over from one into the next, rounds in both directions), against the CPU fast path."""

import numpy as np
import pytest

from oracle import oracle as O
from tests.conftest import splitmix_tokens

pytestmark = pytest.mark.gpu


def check(dims, lens, kw, cuts):
    from taco_amd import hip, synth
    dev = hip.HipDevice.open(0)
    V = dims["vocab"]
    mb = synth.build_model(synth.Dims(**dims), seed=0xA77E, **kw)
    hm, om = hip.HipModel.load(dev, mb), O.Model(mb)
    blocks = [np.array(splitmix_tokens(90 + w, n, V - 1), np.uint32) for w, n in enumerate(lens)]
    want = [O.fast_window_intervals(om, b, chunk=32) for b in blocks]
    # one pass, or the windows in two passes (groups that start at position `cut` and on)
    for cut in cuts:
        batch = hip.HipBatch(hm, len(lens), sum(lens))
        got = [[] for _ in lens]
        for a, b in ([(0, None)] if cut is None else [(0, cut), (cut, None)]):
            inputs, queries, owner = [], [], []
            for w, blk in enumerate(blocks):
                toks = [V - 1] + [int(t) for t in blk[:-1]]
                for t, q in list(zip(toks, blk))[a:b]:
                    inputs.append((w, t))
                    queries.append((0, int(q)))
                    owner.append(w)
            for w, iv in zip(owner, batch.run_coded_raw(inputs, queries, 32)):
                got[w].append(iv)
        for w in range(len(lens)):
            assert np.array_equal(np.array(got[w]), want[w]), (w, cut)


@pytest.mark.parametrize("lens,kw", [
    ([1024, 513, 640, 641, 577], {}), ([900], {}), ([700, 1000], {"score_mult": -(1 << 31)}),
    ([530, 1024], {"table_len": 700}), ([1024], {"score_target": 1 << 22})])
def test_long_windows_equal_the_cpu(lens, kw):
    check(dict(n_layer=1, n_head=3, d_model=192, d_ff=384, vocab=500, n_ctx=1024), lens, kw, (None, 200))


@pytest.mark.parametrize("lens", [[1024] * 11, [1000, 1024, 513, 600, 128, 65, 64, 1, 900] * 2 + [1024] * 3])
def test_several_tasks_per_workgroup_equal_the_cpu(lens):
    """At most three workgroups a CU are resident, 768 in all: 12 heads over 150 and more groups of 64 rows give
    each two tasks and more, and the round that ends the last ones is partial. In the second pass the
    groups start at position 200 and on."""
    check(dict(n_layer=2, n_head=12, d_model=768, d_ff=256, vocab=300, n_ctx=1024), lens, {}, (None, 200))

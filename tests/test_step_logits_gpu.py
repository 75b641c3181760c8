"""Logits on the host are those on the device, for vocabularies with and without padding rows and sizes around the pinned
halves they travel through."""
import json

import numpy as np
import pytest

import nezavik_models as nm

pytestmark = pytest.mark.gpu


# rows of 4 KB without padding, with padding that divides a half and with some that does not; a row of 200 KB; one of 9 MB
@pytest.mark.parametrize("vocab,sequences", [(1024, 700), (1000, 700), (1100, 500), (1100, 3), (50257, 40), (2300000, 2)])
def test_logits_on_the_host_are_those_on_the_device(ops, tmp_path, vocab, sequences):
    cfg = nm.config([nm.delta(dim=64, vdim=64, kv=2, ff=None)], vocab=vocab, width=64, max_positions=16)
    (tmp_path / "config.json").write_text(json.dumps(cfg))
    e = ops.Engine.open(tmp_path, max_batch=sequences, max_seq=16, synthetic=True)
    slots = np.arange(sequences, dtype=np.int32)
    tokens = (7 * slots + 1) % vocab
    for position, want in ((0, slots), (1, slots[::3]), (2, slots[-1:])):
        got = e.step_logits(tokens, slots, np.full(sequences, position, np.int32), want)
        there = e.last_logits(len(want))
        assert got.shape == (len(want), vocab) and np.isfinite(got).all() and np.ptp(got) > 0
        assert np.array_equal(got, there)
    e.close()

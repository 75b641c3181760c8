"""Logits on the host are those on the device, for vocabularies with and without padding rows and sizes around the pinned
halves they travel through."""
import json

import numpy as np
import pytest

import netinex_models as xm
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


# less than a chunk of 16 KB, one, one and 256 bytes, and three halves with a ragged end
@pytest.mark.parametrize("vocab,sequences", [(90, 3), (4096, 1), (4160, 1), (1100, 1100)])
def test_soft_capped_logits_on_the_way_to_the_host(ops, tmp_path, vocab, sequences):
    """Against the same model without the cap.  Its logits are the same numbers; quotient, tanh (two units in the last place)
    and product round by at most four units of float32 together."""
    cap, got = 4.0, []
    for softcap in (None, cap):
        cfg = xm.config([xm.retention()], vocab=vocab, width=64, softcap=softcap)
        (tmp_path / "config.json").write_text(json.dumps(cfg))
        e = ops.Engine.open(tmp_path, max_batch=sequences, max_seq=16, synthetic=True, seed=3)
        slots = np.arange(sequences, dtype=np.int32)
        for position in range(2):
            got.append(e.step_logits((5 * slots + position) % vocab, slots, np.full(sequences, position, np.int32), slots))
            assert np.array_equal(got[-1], e.last_logits(sequences))
        e.close()
    for plain, capped in zip(got[:2], got[2:]):
        want = cap * np.tanh(plain.astype(np.float64) / cap)
        assert np.ptp(capped) > 0 and (np.abs(capped - want) <= 4 * np.spacing(np.abs(want).astype(np.float32))).all()

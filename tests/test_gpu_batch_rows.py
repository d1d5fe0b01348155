"""Passes at the edges of their 16-row groups: a row's bits do not depend on
how many rows share its pass, in a decode step, over rows of many sequences
and over one sequence's rows (whose conv window crosses the groups)."""

import importlib

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

VOCAB = 4096


@pytest.fixture(scope="module")
def decoder(lab, gpu):
    batch = importlib.import_module("ryzenai-npu-lab_amd.batch")
    return batch.BatchDecoder(64, 80, weights=lab.weights.synthetic_checkpoint(0, VOCAB))


@pytest.mark.parametrize("rows", [15, 16, 17, 33, 48, 49, 63, 64])
def test_rows_do_not_depend_on_their_groups(lab, decoder, rows):
    ids = [int(t) for t in lab.rng.uniform_ints(0, f"rows{rows}", 2 * rows, 12)]
    for seq, pos in ((lambda i: i, lambda i: 0), (lambda i: 0, lambda i: i)):
        table = [(ids[i], seq(i), pos(i)) for i in range(rows)]
        decoder.reset()
        tokens, hidden = decoder.run_rows(table, select=True, hidden=True)
        state = decoder.conv_states.clone()
        decoder.reset()
        for a in range(0, rows, 13):
            t, h = decoder.run_rows(table[a:a + 13], select=True, hidden=True)
            assert np.array_equal(h, hidden[a:a + 13]) and t == tokens[a:a + 13]
        assert bool((decoder.conv_states == state).all())


@pytest.mark.parametrize("sequences", [17, 33, 49, 64])
def test_decode_step_equals_rows(lab, gpu, decoder, sequences):
    batch = importlib.import_module("ryzenai-npu-lab_amd.batch")
    d = batch.BatchDecoder(sequences, 80, share=decoder)
    ids = [int(t) for t in lab.rng.uniform_ints(0, f"step{sequences}", sequences, 12)]
    got = d.decode(ids, 4)
    state, keys, values = d.conv_states.clone(), d.keys.clone(), d.values.clone()
    d.reset()
    step = ids
    for pos in range(4):
        rows = [(step[s], s, pos) for s in range(sequences)]
        step = sum((d.run_rows(rows[a:a + 13], select=True)[0] for a in range(0, sequences, 13)), [])
        assert step == got[pos].tolist()
    for mine, want in ((d.conv_states, state), (d.keys, keys), (d.values, values)):
        assert bool((mine == want).all())

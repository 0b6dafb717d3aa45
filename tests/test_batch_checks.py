"""A batch's tokens are looked at all at once: the same arrays, and the same
batches refused, as run by run."""
import numpy as np
import pytest
import torch

import dibelix_util as U
from llmlb_amd.backend.engine import (_in_order, _token_array, _token_arrays)
from llmlb_amd.backend.ragged import RaggedBatch

VOCAB, CAP = 50, 20


class Sequence:
    def __init__(self, length):
        self.length = length


@pytest.mark.parametrize("runs", [
    [[3], [4], [0]], [[3]], [], [[3], [4, 5]], [[1.7], [2]], [[2 ** 40], [1]],
    [np.array([3], np.uint8), [4]], [torch.tensor([7]), [1]], [[True], [2]],
    [[np.int64(5)], [6]], [(3,), (4,)]])
def test_token_arrays(runs):
    got = _token_arrays(runs)
    assert len(got) == len(runs)
    for a, toks in zip(got, runs):
        want = _token_array(toks)
        assert a.dtype == want.dtype == np.int64
        assert a.shape == want.shape and (a == want).all()


@pytest.mark.parametrize("work, fine", [
    ([(0, [1], [0]), (19, [49], [])], True), ([], True),
    ([(0, [1, 2, 3], [0, 2]), (0, [0], [0])], True),
    ([(0, [1], []), (0, [], [])], False), ([(0, [-1], [])], False),
    ([(0, [1], []), (0, [50], [])], False), ([(20, [1], [])], False),
    ([(18, [1, 2, 3], [])], False), ([(0, [1], [1])], False),
    ([(0, [1], [-1])], False)])
def test_in_order(work, fine):
    work = [(Sequence(n), _token_array(toks), want) for n, toks, want in work]
    assert _in_order(work, VOCAB, CAP) == fine


def test_pack():
    runs = [(4, 9, np.array([7])), (0, 0, [5]), (2, 3, np.array([1, 2, 3]))]
    flat = RaggedBatch.pack(runs)
    assert flat.dtype == np.int32
    assert flat.tolist() == [
        7, 5, 1, 2, 3, 9, 0, 3, 4, 5, 4, 0, 2, 2, 2, 0, 1, 2, 2, 2,
        1, 2, 5, 5, 5, 0, 1, 2, 1, 1, 3, 9, 0, 3, 4, 0, 2]


def test_batches_that_can_be_read_once(tmp_path):
    """A batch and its wanted places may be any iterables."""
    cfg = U.PLAIN
    eng = U.engine(U.write_model(tmp_path / "m", cfg, U.weights(cfg)),
                   blocks=20, rows=4)
    a, b, c, d = (eng.open_sequence() for _ in range(4))
    want = eng.run_batch([(a, [1, 2, 3], [0, 2]), (b, [4], [0])])
    got = eng.run_batch(iter([(c, [1, 2, 3], iter([0, 2])),
                              (d, [4], iter([0]))]))
    assert got.shape == (3, cfg["vocab"]) and torch.equal(got, want)
    assert c.length == 3 and d.length == 1
    for bad, why in (((a, [5], iter([1])), "wanted place"),
                     ((a, [cfg["vocab"]], iter([0])), "vocab")):
        with pytest.raises(ValueError, match=why):
            eng.run_batch(iter([bad]))
    assert a.length == 3

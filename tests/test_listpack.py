"""The request-list packer behind prepare_model_inputs (CPU): the same arrays
as numpy builds from the lists, and the errors the reference's own list walk
(worker.py:596-646) would hit as Python exceptions."""
import numpy as np
import pytest

from aegaeon_amd import _listpack


def test_tables_pack_like_numpy():
    rng = np.random.default_rng(7)
    tables = [rng.integers(0, 2 ** 31 - 1, int(n)).tolist() for n in rng.integers(0, 40, 200)]
    tables[3] = []
    ids, off = _listpack.pack_tables(tables)
    ids = np.frombuffer(ids, dtype=np.int32)
    off = np.frombuffer(off, dtype=np.int64)
    assert off[0] == 0 and np.array_equal(np.diff(off), [len(t) for t in tables])
    assert np.array_equal(ids, np.concatenate([np.asarray(t, dtype=np.int64) for t in tables]))
    # tuples, and an empty batch
    ids2, off2 = _listpack.pack_tables(tuple(tuple(t) for t in tables))
    assert ids2 == ids.tobytes() and off2 == off.tobytes()
    ids3, off3 = _listpack.pack_tables([])
    assert len(ids3) == 0 and np.frombuffer(off3, dtype=np.int64).tolist() == [0]


def test_requests_pack_like_numpy():
    reqs = [(0, [5, 6, 7], 3, 0), (1, [9], 11, 10), (2, [], 4, 4), (3, (1, 2), 2, 0)]
    seq, ctx, tok = _listpack.pack_requests(reqs)
    assert np.frombuffer(seq, dtype=np.int32).tolist() == [3, 11, 4, 2]
    assert np.frombuffer(ctx, dtype=np.int32).tolist() == [0, 10, 4, 0]
    assert np.frombuffer(tok, dtype=np.int64).tolist() == [5, 6, 7, 9, 1, 2]
    big = [(0, [2 ** 40], 1, 0)]
    assert np.frombuffer(_listpack.pack_requests(big)[2], dtype=np.int64).tolist() == [2 ** 40]


def test_errors():
    with pytest.raises(ValueError):  # two tokens for one new position
        _listpack.pack_requests([(0, [1, 2], 5, 4)])
    with pytest.raises(TypeError):
        _listpack.pack_requests([(0, [1])])
    with pytest.raises(TypeError):
        _listpack.pack_tables([[1, "2"]])
    with pytest.raises(TypeError):
        _listpack.pack_tables([3])
    with pytest.raises(OverflowError):
        _listpack.pack_tables([[2 ** 31]])
    with pytest.raises(OverflowError):
        _listpack.pack_requests([(0, [], 2 ** 31, 2 ** 31)])


def _counts(offsets, seq, ctx):
    """step_counts by numpy over int64."""
    qlen = seq.astype(np.int64) - ctx
    prompt = ctx == 0
    top = lambda x: int(x.max()) if x.size else 0
    return (seq.tolist(), int(qlen.sum()), top(np.diff(offsets)[~prompt]), int(prompt.sum()),
            int(qlen[prompt].sum()), int(qlen.max()), top(seq[prompt]), top(seq[~prompt]))


@pytest.mark.parametrize("n,prompts", [(1, 0.0), (1, 1.0), (7, 0.5), (300, 0.0), (300, 1.0),
                                       (513, 0.3)])
def test_step_counts_like_numpy(n, prompts):
    rng = np.random.default_rng(n)
    ctx = rng.integers(1, 5000, n).astype(np.int32)
    ctx[rng.random(n) < prompts] = 0
    seq = (ctx + rng.integers(0, 400, n)).astype(np.int32)
    offsets = np.concatenate([[0], np.cumsum(rng.integers(0, 40, n))]).astype(np.int64)
    want = _counts(offsets, seq, ctx)
    assert _listpack.step_counts(offsets, seq, ctx) == want
    assert _listpack.step_counts(bytearray(offsets), bytearray(seq), bytearray(ctx)) == want


def test_step_counts_errors_and_address():
    seq = np.ones(3, dtype=np.int32)
    with pytest.raises(ValueError):
        _listpack.step_counts(np.zeros(3, dtype=np.int64), seq, seq)
    with pytest.raises(ValueError):
        _listpack.step_counts(np.zeros(4, dtype=np.int64), seq, seq[:2])
    with pytest.raises(ValueError):
        _listpack.step_counts(np.zeros(1, dtype=np.int64), seq[:0], seq[:0])
    assert _listpack.address(seq) == seq.ctypes.data
    assert _listpack.address(bytearray()) is None
    with pytest.raises((TypeError, BufferError, ValueError)):
        _listpack.address(np.ones((4, 4))[:, 1])

"""The table of a step whose long prompts come as arrays, against the same step from lists; which token ids pass."""

import numpy as np
import pytest
import torch


@pytest.mark.parametrize("entries", [
    [(0, 0, list(range(100)))], [(3, 0, list(range(70))), (1, 12, [5]), (0, 7, list(range(200, 300)))],
    [(2, 5, [9]), (5, 0, list(range(65)))]])
def test_table_from_arrays(entries):
    from lit_gpt.mixers import StepBatch

    dev = torch.device("cpu")
    a = StepBatch.build(entries, dev)
    b = StepBatch.build([(s, p, np.array(t) if len(t) > 64 else t) for s, p, t in entries], dev)
    for name in ("tokens", "slot", "pos", "seq_start", "seq_slot", "seq_pos0"):
        x, y = getattr(a, name), getattr(b, name)
        assert x.dtype == y.dtype == torch.int32 and x.tolist() == y.tolist(), name
    assert (a.T, a.B, a.max_len, a.fresh) == (b.T, b.B, b.max_len, b.fresh)
    assert type(b.max_len) is int and type(b.T) is int and type(b.fresh) is bool


def test_checked_ids():
    from generate.batch import _checked

    long = list(range(100))
    assert isinstance(_checked(long, 100), np.ndarray) and _checked(long, 100).tolist() == long
    assert _checked(torch.arange(100), 100).tolist() == long
    short = [1, 2]
    assert _checked(short, 100) is short
    for bad in ([100], [-1], long + [100], [-1] + long, long + [2 ** 70]):
        with pytest.raises(ValueError, match="outside the vocabulary"):
            _checked(bad, 100)
    floats = [float(t) for t in long]
    assert _checked(floats, 100) is floats
    with pytest.raises(TypeError):
        _checked([[1, 2]] * 70, 100)

"""The rows whose logits a step is asked for travel with its table, through pinned memory where the table goes to a GPU: the rows
themselves from lists and arrays, the way the table takes, and steps queued one behind the other without a wait."""

import numpy as np
import pytest
import torch


@pytest.mark.parametrize("n", [3, 70])
@pytest.mark.parametrize("rows", [[], [2], [0, 2, 1]])
def test_rows_beside_the_table(n, rows):
    from lit_gpt.mixers import StepBatch

    dev, toks = torch.device("cpu"), list(range(n))
    for t in (toks, np.array(toks)):
        a, b = StepBatch.build([(1, 4, t), (0, 0, [9])], dev), StepBatch.build([(1, 4, t), (0, 0, [9])], "cpu", rows)
        assert a.rows is None and (b.rows is None if not rows else b.rows.dtype == torch.int32 and b.rows.tolist() == rows)
        for name in ("tokens", "slot", "pos", "seq_start", "seq_slot", "seq_pos0"):
            assert getattr(a, name).tolist() == getattr(b, name).tolist(), name
        with pytest.raises(RuntimeError, match="overflow"):
            StepBatch.build([(1, 4, t)], dev, [2 ** 31])


def test_the_way_of_the_table(monkeypatch):
    from lit_gpt.mixers import _table

    class Host:
        def __init__(self, way=(), n=5):
            self.way, self.n = way, n

        def numel(self):
            return self.n

        def __getitem__(self, part):
            return Host(self.way, len(range(self.n)[part]))

        def copy_(self, host):
            assert self.n == host.n
            return self

        def to(self, device, non_blocking=False):
            return self.way + ("queued" if non_blocking else "waited",)

    monkeypatch.setattr(torch, "empty", lambda n, dtype, pin_memory: Host(("pinned",) * pin_memory, n))
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    for n in (1, 4096, 5000):
        assert _table(Host(n=n), "cuda:0") == _table(Host(n=n), torch.device("cuda")) == ("pinned", "queued")
    assert _table(Host(), "cpu") == ("waited",)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    assert _table(Host(), "cuda:0") == ("waited",)  # a replay would read the pinned memory again


@pytest.mark.gpu
@pytest.mark.parametrize("side", [False, True])
def test_steps_queued_behind_each_other(side):
    """On the default stream and on one of the caller's own: a table's host memory is free for the next one only when it is copied."""
    from generate.batch import BatchEngine
    from lit_gpt.mixers import StepBatch
    from test_gpu_hooks import layered

    m = layered("Fazolorn")
    g = torch.Generator().manual_seed(3)
    prompts = [torch.randint(0, 50, (n,), generator=g).tolist() for n in (40, 3, 64, 1, 17, 64, 30, 9) * 4]
    stream = torch.cuda.Stream() if side else torch.cuda.current_stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.inference_mode(), torch.cuda.stream(stream):
        eng = BatchEngine(m, max_seq_length=64, slots=1)
        torch.cuda._sleep(20_000_000)  # (some ten milliseconds: the host is steps ahead)
        got = [eng.step([("r", p, [0, len(p) - 1])], end=["r"]) for p in prompts]
        for p, y in zip(prompts, got):
            torch.cuda.synchronize()
            x = m.forward_step(StepBatch.build([(0, 0, p)], m.device))
            assert torch.equal(y, m.logits(x[[0, len(p) - 1]].contiguous()))

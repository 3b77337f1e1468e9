"""The head's live-row count, without a GPU: the event that says when its copy has landed is recorded
on the stream that the copy runs on, the current one of the tensors' own device."""

import torch

from solution.head import op


def test_event_is_recorded_on_the_tensors_device(monkeypatch):
    streams, recorded = {}, []

    class Event:
        def record(self, stream="the current device's"):
            recorded.append(stream)

        def synchronize(self):
            assert recorded == [streams["cpu"]]

    empty = torch.empty

    def stream_of(device=None):
        return streams.setdefault(str(device), object())

    monkeypatch.setattr(torch.cuda, "Event", Event)
    monkeypatch.setattr(torch.cuda, "current_stream", stream_of)
    monkeypatch.setattr(torch, "empty", lambda *a, pin_memory=False, **kw: empty(*a, **kw))
    monkeypatch.setattr(op._hip, "head_partition",
                        lambda target, cew, V: (None, None, torch.tensor([3], dtype=torch.int32)))
    order = op._RowOrder(torch.tensor([1, 2, 3, -100]), torch.ones(4), 10, True)
    assert recorded == [streams.get("cpu")], recorded
    assert order.n_live() == 3 and order.n_live() == 3

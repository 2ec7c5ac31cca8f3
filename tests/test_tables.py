"""Tables shared between forwards: complete before they are kept, recorded on every stream that uses them."""

import copy

import pytest
import torch

from vllm_omni_amd.blocks import tables
from vllm_omni_amd.blocks.qwen_image import QwenEmbedRope
from vllm_omni_amd.blocks.wan import WanRotaryPosEmbed


class _Stream:
    def __init__(self, number):
        self.cuda_stream = number


class _OnGpu:
    """Stands for a tensor on a GPU."""

    device = torch.device("cuda", 0)

    def __init__(self):
        self.used_on = []

    def record_stream(self, stream):
        self.used_on.append(stream.cuda_stream)


def test_entries_are_complete_and_recorded(monkeypatch):
    log, now, capturing = [], [_Stream(1)], [False]

    class Event:
        def record(self, stream):
            log.append(("record", stream.cuda_stream))

        def synchronize(self):
            log.append("wait")

    monkeypatch.setattr(torch.cuda, "Event", Event)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: now[0])
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: capturing[0])

    def build(key):
        log.append(("build", key))
        return (_OnGpu(),)

    cache = tables.TableCache(build, 2)
    first = cache("a")
    assert log == [("build", "a"), ("record", 1), "wait"] and first[0].used_on == []
    now[0] = _Stream(2)
    assert cache("a") is first and first[0].used_on == [2] and len(log) == 3
    capturing[0] = True
    captured = cache("b")
    assert log[3:] == [("build", "b")] and cache("b") is not captured   # a capture's own tables are not kept
    assert cache("a") is first
    capturing[0] = False
    cache("b"), cache("c")
    assert cache("a") is not first                                      # two entries are kept, the oldest went


def test_a_copied_module_has_its_own_cache():
    rope = QwenEmbedRope(10000, [8, 28, 28])
    before = rope.tables([(1, 2, 3)], [4], "cpu")
    other = copy.deepcopy(rope)
    other.theta = 1
    assert other._tables._build.__self__ is other and rope.tables([(1, 2, 3)], [4], "cpu") is before
    assert torch.equal(other.tables([(1, 2, 3)], [4], "cpu").img_cos, before.img_cos)


@pytest.mark.gpu
def test_tables_first_made_on_a_busy_stream_are_whole_on_another(gpu):
    qwen, wan = QwenEmbedRope(10000, [16, 56, 56]), WanRotaryPosEmbed(128, (1, 2, 2), 64)
    video = torch.empty(1, 16, 3, 10, 14)
    want_q, want_w = qwen.tables([(1, 9, 11)], [33], "cpu"), wan(video)
    wan, video = wan.to(gpu), video.to(gpu)
    one, two = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(one):
        torch.cuda._sleep(200_000_000)   # the tables are made behind this
        qwen.tables([(1, 9, 11)], [33], gpu), wan(video)
    with torch.cuda.stream(two):
        got = [t.clone() for t in (*qwen.tables([(1, 9, 11)], [33], gpu).tensors(), *wan(video).tensors())]
    torch.cuda.synchronize()
    for g, w in zip(got, (*want_q.tensors(), *want_w.tensors())):
        assert torch.equal(g.cpu(), w)

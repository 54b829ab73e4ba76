"""Which device sources upload, accumulate_grad and accumulate_grads return before reading: those
whose memory torch's caching allocator keeps for the shared stream (record_stream).  Memory that
torch only wraps is waited for, as its owner may reuse it.  CPU: the tensors pass for device
tensors, and the library and the streams are stand-ins that note what was called."""
import types

import numpy as np
import pytest
import torch

import ttperf
from ttperf import store as S

N = 64


class _Device(torch.Tensor):
    """A host tensor that passes for one of cuda:0 (and for a type of torch's)."""

    __module__ = "torch"

    is_cuda = property(lambda self: True)
    device = property(lambda self: torch.device("cuda", 0))


def _tensor(memory):
    if memory == "torch":
        return torch.zeros(N)
    if memory == "a torch slice":
        return torch.zeros(4 * N)[N:2 * N]
    if memory == "an array":  # as from an array interface: wrapped, not allocated
        return torch.from_numpy(np.zeros(N, np.float32))
    return torch.utils.dlpack.from_dlpack(torch.utils.dlpack.to_dlpack(torch.zeros(N)))


def _call(store, entry, sources):
    if entry == "upload":
        store.upload(ttperf.BUF_GRAD, 0, sources[0])
    elif entry == "accumulate":
        store.accumulate_grad(0, sources[0])
    else:
        store.accumulate_grads(list(range(len(sources))), sources)


@pytest.fixture
def bench(monkeypatch):
    log = []

    def entry(name):
        return lambda *a: log.append(name) or 0

    names = ("ttp_download", "ttp_upload", "ttp_accumulate_grad", "ttp_accumulate_grad_multi", "ttp_sync",
             "ttp_destroy")
    lib = types.SimpleNamespace(**{n: entry(n) for n in names})

    def get_stream(h, out):
        asked.append("ttp_get_stream")
        out._obj.value = st.moved_to
        return 0

    lib.ttp_get_stream = get_stream
    asked = []
    monkeypatch.setattr(S.L, "lib", lib)
    stream = types.SimpleNamespace(synchronize=lambda: log.append("torch waits"),
                                   device_index=0, cuda_stream=0)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: stream)
    monkeypatch.setattr(torch.Tensor, "record_stream",
                        lambda self, s: log.append(("kept", self.untyped_storage().data_ptr())))
    st = S.ParamStore.__new__(S.ParamStore)
    st._h, st.mode, st.device, st._in_capture = None, S.L.MODE_FP32, 0, False
    st.tensors = [S.Tensor(st, i, (N,)) for i in range(3)]
    st.total = 3 * N
    st.asked, st.moved_to = asked, 0
    st._stream_handle = 0  # adopted: the store's stream and torch's are both the default one
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    return st, log


@pytest.mark.parametrize("entry", ["upload", "accumulate", "bucket"])
@pytest.mark.parametrize("memory", ["torch", "a torch slice", "an array", "dlpack"])
def test_only_torchs_own_memory_is_left_unread(bench, entry, memory):
    st, log = bench
    src = _tensor(memory).as_subclass(_Device)
    _call(st, entry, [src])
    if memory.startswith(("torch", "a torch")):
        assert len(log) == 2 and log[0].startswith("ttp_")  # queued, nothing waited for
        assert log[1] == ("kept", src.untyped_storage().data_ptr())
    else:
        assert log[-1] == "ttp_sync" and log[-2] in ("ttp_upload", "ttp_accumulate_grad",
                                                     "ttp_accumulate_grad_multi")


def test_a_bucket_with_one_wrapped_source_is_waited_for(bench):
    st, log = bench
    _call(st, "bucket", [_tensor(m).as_subclass(_Device) for m in ("torch", "dlpack", "torch")])
    assert log[-2:] == ["ttp_accumulate_grad_multi", "ttp_sync"]


def test_each_storage_is_kept_once(bench):
    st, log = bench
    base, alone = torch.zeros(2 * N), torch.zeros(N)
    _call(st, "bucket", [t.as_subclass(_Device) for t in (base[:N], alone, base[N:])])
    assert log[0] == "ttp_accumulate_grad_multi" and \
        sorted(log[1:]) == sorted(("kept", t.data_ptr()) for t in (base, alone))


def test_a_pluggable_allocator_is_not_relied_on(bench, monkeypatch):
    st, log = bench
    monkeypatch.setattr(torch.cuda, "get_allocator_backend", lambda: "pluggable")
    _call(st, "accumulate", [_tensor("torch").as_subclass(_Device)])
    assert log[-1] == "ttp_sync"


@pytest.mark.parametrize("entry", ["upload", "accumulate", "bucket", "download"])
def test_a_store_on_its_own_stream_asks_nothing(bench, entry):
    """Its calls are torch's wait, the work and the store's wait, with no question to the library
    or about captures between them."""
    st, log = bench
    st._stream_handle = None
    src = _tensor("torch").as_subclass(_Device)
    if entry == "download":
        st.download(ttperf.BUF_GRAD, 0, out=src)
    else:
        _call(st, entry, [src])
    assert log[0] == "torch waits" and log[2:] == ["ttp_sync"] and not st.asked


def test_a_stream_set_behind_the_stores_back_is_not_taken_for_torchs(bench):
    """ttp_set_stream called on the store's handle: the library's answer counts."""
    st, log = bench
    st.moved_to = 8
    _call(st, "accumulate", [_tensor("torch").as_subclass(_Device)])
    assert log == ["torch waits", "ttp_accumulate_grad", "ttp_sync"] and st.asked


def test_nothing_is_left_unread_while_torch_captures(bench, monkeypatch):
    """The store's call waits, which a capture refuses."""
    st, log = bench
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    _call(st, "upload", [_tensor("torch").as_subclass(_Device)])
    assert log == ["torch waits", "ttp_upload", "ttp_sync"]

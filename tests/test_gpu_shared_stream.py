"""GPU test of device tensors handed to the store without a synchronisation: on torch's current
stream when the store shares it, and (with one) when it does not.  The streams are kept busy, so
that work queued in the wrong order, or memory given away too early, shows."""
import pytest

from gpu_util import torch_mod

pytestmark = pytest.mark.gpu

N = 3 << 20


def _hand_over(store, entry, src):
    import ttperf
    if entry == "upload":
        store.upload(ttperf.BUF_GRAD, 0, src)
    elif entry == "accumulate":
        store.zero_grad()
        store.accumulate_grad(0, src)
    else:
        store.zero_grad()
        store.accumulate_grads([0], [src])


@pytest.mark.parametrize("stream", ["default", "side", "own"])
@pytest.mark.parametrize("entry", ["upload", "accumulate", "bucket"])
def test_order_and_lifetime(entry, stream):
    import ttperf
    torch = torch_mod()
    a = torch.randn(4096, 4096, device="cuda")
    store = ttperf.ParamStore([(N,)], mode="fp32")
    main = torch.cuda.Stream() if stream == "side" else torch.cuda.current_stream()
    if stream != "own":
        store.set_stream(main)
    other = torch.cuda.Stream()
    torch.cuda.synchronize()

    def busy():
        for _ in range(20):
            a @ a

    with torch.cuda.stream(main):
        for k in range(3):
            # a source that its own stream overwrites right after the call
            src = torch.empty(N, device="cuda")
            busy()
            src.fill_(k + 1.0)
            _hand_over(store, entry, src)
            src.fill_(-1.0)
            assert (store.download(ttperf.BUF_GRAD, 0) == k + 1.0).all()
            # one of another stream's memory, freed right after the call and taken again there
            with torch.cuda.stream(other):
                src = torch.full((N,), k + 10.0, device="cuda")
                ptr = src.data_ptr()
            main.wait_stream(other)
            busy()
            _hand_over(store, entry, src)
            del src
            with torch.cuda.stream(other):
                again = torch.full((N,), -2.0, device="cuda")
            assert (store.download(ttperf.BUF_GRAD, 0) == k + 10.0).all(), ptr == again.data_ptr()
            # results handed out are there for any stream
            busy()
            store.upload(ttperf.BUF_MASTER, 0, torch.full((N,), k + 0.5, device="cuda"))
            out = torch.empty(N, device="cuda")
            store.download(ttperf.BUF_MASTER, 0, out=out)
            with torch.cuda.stream(other):
                assert bool((out == k + 0.5).all())
    torch.cuda.synchronize()
    store.close()


def test_an_edited_parameter_list_is_grouped_again():
    import ttperf
    store = ttperf.ParamStore([(8,), (8,), (8,)], mode="fp32")
    opt = ttperf.SGD(store.parameters()[:2], lr=1.0)
    one = store.torch_view(ttperf.BUF_GRAD)

    def step():
        one.fill_(1.0)
        torch_mod().cuda.synchronize()
        store.mark_grads()
        before = [t.numpy()[0] for t in store.tensors]
        opt.step()
        opt.zero_grad()
        return [b - t.numpy()[0] for b, t in zip(before, store.tensors)], \
            [t.grad is None for t in store.tensors]

    assert step() == ([1.0, 1.0, 0.0], [True, True, False])
    opt.params.append(store.tensors[2])
    assert step() == ([1.0, 1.0, 1.0], [True, True, True])
    opt.params[:] = store.tensors[1:2]
    assert step() == ([0.0, 1.0, 0.0], [False, True, False])
    opt.params.append("not a tensor")
    with pytest.raises(ValueError):
        opt.step()
    opt.zero_grad()
    store.close()


@pytest.mark.parametrize("entry", ["upload", "accumulate", "bucket"])
def test_sources_that_torch_only_wraps(entry):
    """Read before the call returns, so that their owner may write to them or take them back:
    another store's view, which that store overwrites on its own stream, and an array interface
    over memory that goes back to another stream's pool."""
    import ttperf
    from ttperf.store import _torch_storages
    torch = torch_mod()
    a = torch.randn(4096, 4096, device="cuda")
    store = ttperf.ParamStore([(N,)], mode="fp32")
    store.set_stream(torch.cuda.current_stream())
    second = ttperf.ParamStore([(N,)], mode="fp32")  # on its own stream
    view = second.torch_view(ttperf.BUF_GRAD, 0)
    other = torch.cuda.Stream()
    assert _torch_storages([view]) is None and _torch_storages([a[:2], view]) is None
    assert [t.data_ptr() for t in _torch_storages([a[1:], a[:1]])] == [a[:1].data_ptr()]

    def busy():
        for _ in range(20):
            a @ a

    for k in range(3):
        second.upload(ttperf.BUF_GRAD, 0, torch.full((N,), k + 1.0, device="cuda"))
        busy()
        _hand_over(store, entry, view)
        second.zero_grad()
        assert (store.download(ttperf.BUF_GRAD, 0) == k + 1.0).all()
        with torch.cuda.stream(other):
            owner = torch.full((N,), k + 10.0, device="cuda")

            class Wrapped:
                __cuda_array_interface__ = dict(owner.__cuda_array_interface__)

            src = torch.as_tensor(Wrapped(), device="cuda")
            ptr = owner.data_ptr()
            assert src.data_ptr() == ptr
        torch.cuda.current_stream().wait_stream(other)
        busy()
        _hand_over(store, entry, src)
        del src, owner
        with torch.cuda.stream(other):
            again = torch.full((N,), -2.0, device="cuda")
        assert (store.download(ttperf.BUF_GRAD, 0) == k + 10.0).all(), ptr == again.data_ptr()
    torch.cuda.synchronize()
    store.close()
    second.close()

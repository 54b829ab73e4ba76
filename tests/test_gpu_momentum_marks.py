"""GPU test of which momentum steps are a tensor's first (its buffer takes the gradient itself;
later ones take momentum * buffer + (1 - dampening) * gradient), over the ways the marks are set:
by the step's decisions, by a launch of their own (more tensors than those set, or no decisions on
the device) and by the one-launch step; with skipped steps, subsets, changes of loss scaling,
checkpoints and replayed graphs between.  Momentum is exact: small integers and powers of two."""
import numpy as np
import pytest

from gpu_util import torch_mod

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [[40000, 5, 64, 7], [9] * 5000, [100, 5, 64, 7]],
                         ids=["decisions", "own launch", "one launch"])
@pytest.mark.parametrize("mode,layout", [("mixed", "default"), ("mixed", "sgd"),
                                         ("fp32", "default")])
def test_first_steps(mode, layout, sizes, tmp_path):
    import ttperf
    torch = torch_mod()
    store = ttperf.ParamStore([(n,) for n in sizes], mode=mode, layout=layout)
    side = torch.cuda.Stream()
    store.set_stream(side)
    count = len(sizes)
    lo = np.array(store.offsets)
    want, seen = np.zeros(store.total, np.float32), np.zeros(count, bool)
    scaled = False

    def expect(value, which):
        for i in which:
            b = slice(lo[i], lo[i] + sizes[i])
            want[b] = 0.5 * want[b] + 0.25 * value if seen[i] else value
            seen[i] = True

    def write(value):
        with torch.cuda.stream(side):
            store.torch_view(ttperf.BUF_GRAD).fill_(value * (4.0 if scaled else 1.0))
        store.mark_grads()

    def step(value, which=None, clip=None):
        write(value)
        store.sgd_step(2.0 ** -10, momentum=0.5, dampening=0.75, indices=which,
                       max_grad_norm=clip)
        if np.isfinite(value):
            expect(np.float32(value), range(count) if which is None else which)
        got = store.download(ttperf.BUF_MOMENTUM)
        for i in {0, 1, count // 2, count - 1}:
            b = slice(lo[i], lo[i] + sizes[i])
            assert np.array_equal(got[b], want[b]), (i, value)
        assert np.array_equal(got, want)

    step(16.0, [1])                      # no decisions on the device
    step(32.0, [1, 2], clip=1e30)        # decisions, without loss scaling
    store.configure_scaler(True, init_scale=4.0, backoff_factor=0.5, growth_interval=1000)
    scaled = True
    step(float("inf"))                   # skipped: no tensor's first
    store.set_scaler_state(4.0, 0)
    step(16.0, [0, 1])
    step(64.0)
    step(float("nan"))
    store.set_scaler_state(4.0, 0)
    step(-32.0)
    store.save_state(tmp_path / "s")
    store.load_state(tmp_path / "s")
    step(128.0)
    store.configure_scaler(False)
    scaled = False
    step(8.0, [0])
    step(8.0)
    store.begin_capture()
    store.sgd_step(2.0 ** -10, momentum=0.5, dampening=0.75)
    graph = store.end_capture()
    for value in (4.0, 2.0):
        write(value)
        graph.replay()
        expect(np.float32(value), range(count))
        assert np.array_equal(store.download(ttperf.BUF_MOMENTUM), want)
    graph.close()
    store.close()

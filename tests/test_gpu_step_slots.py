"""GPU test of the step count's hand-over between optimizers of one store: each keeps its own
count through changes between host and device counting, skipped steps, optimizers that go away
(their slots are taken again) and more optimizers than slots."""
import random

import pytest

from gpu_util import torch_mod

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("live", [2, 5, 70])
def test_counts_of_many_optimizers(live, tmp_path):
    import ttperf
    torch = torch_mod()
    store = ttperf.ParamStore([(64,)] * 4, mode="mixed")
    store.set_stream(torch.cuda.current_stream())
    view = store.torch_view(ttperf.BUF_GRAD)
    r = random.Random(live)
    opts, want, scaler = [], {}, False
    for k in range(12 * live):
        if len(opts) < live or r.random() < 0.05:
            if len(opts) >= live:
                # (not the owner: a store whose owner is gone keeps its count for the next one)
                gone = opts.pop(0) if opts[0] is not last else opts.pop(1)
                del want[id(gone)], gone
            opts.append(ttperf.AdamW(store.parameters()[len(opts) % 4::4], lr=1e-3))
            want[id(opts[-1])] = 0
        if k % 11 == 5:
            scaler = not scaler
            store.configure_scaler(scaler, init_scale=8.0)
        if k % 29 == 28:
            store.save_state(tmp_path / "s")
            store.load_state(tmp_path / "s")
        last = opts[-1] if want[id(opts[-1])] == 0 else r.choice(opts)
        skip = scaler and r.random() < 0.3
        view.fill_(float("inf") if skip else 1.0)
        store.mark_grads()
        last.step()
        want[id(last)] += 0 if skip else 1
        assert store.step_count == want[id(last)], k
    store.close()


def test_slots_out_of_range_are_refused():
    import ttperf
    from ttperf import _lib as L
    store = ttperf.ParamStore([(4,)], mode="fp32")
    for save, load in ((64, -1), (-2, 0), (0, 64), (0, -2)):
        with pytest.raises(ttperf.TTPValueError):
            L.check(L.lib.ttp_swap_step(store.handle, save, load))
    store.begin_capture()
    with pytest.raises(ttperf.TTPError):
        L.check(L.lib.ttp_swap_step(store.handle, 0, 1))
    store.end_capture(discard=True)
    store.close()


@pytest.mark.filterwarnings("ignore:The CUDA Graph is empty")
@pytest.mark.parametrize("scaler", [False, True])
def test_a_capture_of_the_callers_refuses_the_hand_over(scaler):
    """A capture that is torch's, not the store's, would replay a hand-over that happened once.
    Refused, it leaves both counts as they were."""
    import ttperf
    torch = torch_mod()
    store = ttperf.ParamStore([(64,)] * 2, mode="mixed")
    side = torch.cuda.Stream()
    store.set_stream(side)
    if scaler:
        store.configure_scaler(True, init_scale=8.0)
    store.upload(ttperf.BUF_GRAD, ttperf.ALL_TENSORS,
                 torch.ones(store.total, device="cuda", dtype=torch.bfloat16))
    a, b = (ttperf.AdamW([t], lr=1e-3) for t in store.parameters())
    for opt in (a, a, b):
        opt.step()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        with pytest.raises(ttperf.TTPError):
            a.step()
    assert store.step_count == 1  # b's
    a.step()
    assert store.step_count == 3
    b.step()
    assert store.step_count == 2
    store.close()

"""GPU test of the one-launch step of small tensor sets against the general step (norm pass, then
update), which per-kernel timing selects: the same stores, gradients and options give the same
bits in every buffer, the step state and the report.  Tables end inside a lane's vector, a wave's
part, a tile and a chunk, and sit at and beyond the one-launch step's limits (64 tiles, 32,768
elements)."""
import pytest

from gpu_util import captured_launches, torch_mod

pytestmark = pytest.mark.gpu

TABLES = {
    "one": [1],
    "edges": [1, 3, 4, 5, 7, 8, 9, 63, 64, 65, 255, 256, 257, 511, 513, 1023, 1024, 1025],
    "tiles": [4095, 4096, 4097, 8191, 8192, 1],
    "limit": [8192, 8192, 16384],
    "beyond": [8192, 8192, 16385],
    "64 tensors": [17 * k % 97 + 1 for k in range(64)],
    "65 tensors": [17 * k % 97 + 1 for k in range(65)],
}
OPTS = {
    "adamw": ("adam_step", dict(lr=1e-2, weight_decay=0.1)),
    "adam l2": ("adam_step", dict(lr=1e-2, weight_decay=0.1, decoupled=False)),
    "sgd": ("sgd_step", dict(lr=1e-2)),
    "nesterov": ("sgd_step", dict(lr=1e-2, momentum=0.9, nesterov=True, weight_decay=0.1)),
}


def _state(store, opt):
    import ttperf
    bufs = [ttperf.BUF_PARAM, ttperf.BUF_GRAD]
    if store.mode != ttperf._lib.MODE_BF16:
        bufs.append(ttperf.BUF_MASTER)
        if opt.startswith("adam"):
            bufs += [ttperf.BUF_EXP_AVG, ttperf.BUF_EXP_AVG_SQ]
        elif opt == "nesterov":
            bufs.append(ttperf.BUF_MOMENTUM)
    return [store.download(b).tobytes() for b in bufs] + [store.step_count, store.scaler_state()]


@pytest.mark.parametrize("table", list(TABLES))
@pytest.mark.parametrize("opt", list(OPTS))
@pytest.mark.parametrize("mode,layout", [("fp32", "default"), ("mixed", "default"),
                                         ("mixed", "sgd"), ("bf16", "default")])
def test_same_bits_as_the_general_step(mode, layout, opt, table):
    import ttperf
    if (mode == "bf16" and opt != "sgd") or (layout == "sgd" and opt.startswith("adam")):
        pytest.skip("not a step of this store")
    torch = torch_mod()
    call, hp = OPTS[opt]
    sizes = TABLES[table]
    pair = []
    for general in (False, True):
        store = ttperf.ParamStore([(n,) for n in sizes], mode=mode, layout=layout,
                                  decay=[k % 2 == 0 for k in range(len(sizes))])
        store.set_stream(torch.cuda.current_stream())
        store.timing(general)
        gen = torch.Generator(device="cuda").manual_seed(len(sizes))
        w = torch.randn(store.total, device="cuda", generator=gen)
        if mode == "bf16":
            store.upload(ttperf.BUF_PARAM, ttperf.ALL_TENSORS, w.bfloat16())
        else:
            store.upload(ttperf.BUF_MASTER, ttperf.ALL_TENSORS, w)
        # the padding is written too: no step may read it
        view = store.torch_view(ttperf.BUF_GRAD)
        log = []
        for step in range(9):
            view.normal_(0, 2.0 if step % 2 else 1e-3, generator=gen)
            store.mark_grads()
            if step == 3:
                store.configure_scaler(True, init_scale=8.0, growth_interval=2)
            if step == 5:
                view[store.offsets[-1]] = float("inf")  # skipped, and the scale backs off
            kw = dict(hp, max_grad_norm=None if step == 8 else 1.0, report=True)
            if step == 6:
                kw["update_scale"] = False
            if step == 7 and len(sizes) > 1:
                kw["indices"] = list(range(0, len(sizes), 2))
            log.append(getattr(store, call)(**kw))
        side = torch.cuda.Stream()  # (the legacy default stream cannot be captured)
        torch.cuda.synchronize()
        store.set_stream(side)
        store.begin_capture()
        getattr(store, call)(**dict(hp, max_grad_norm=1.0))
        graph = store.end_capture()
        for _ in range(3):
            with torch.cuda.stream(side):
                view.normal_(0, 1.0, generator=gen)
            graph.replay()
            log.append(store.scaler_state())
        pair.append((log, _state(store, opt)))
        graph.close()
        store.close()
    assert repr(pair[0][0]) == repr(pair[1][0])
    assert pair[0][1] == pair[1][1]


@pytest.mark.parametrize("opt", list(OPTS))
@pytest.mark.parametrize("mode,layout", [("fp32", "default"), ("mixed", "default"),
                                         ("mixed", "sgd"), ("bf16", "default")])
def test_which_steps_are_one_launch(mode, layout, opt):
    """At the limits one launch, just beyond them a norm pass and an update; so with per-kernel
    timing and with the norm from per-tensor sums."""
    import ttperf
    if (mode == "bf16" and opt != "sgd") or (layout == "sgd" and opt.startswith("adam")):
        pytest.skip("not a step of this store")
    torch = torch_mod()
    call, hp = OPTS[opt]
    for table, sizes in TABLES.items():
        store = ttperf.ParamStore([(n,) for n in sizes], mode=mode, layout=layout)
        store.torch_view(ttperf.BUF_GRAD).normal_(0, 1.0)
        torch.cuda.synchronize()
        store.mark_grads()
        getattr(store, call)(**dict(hp, max_grad_norm=1.0))  # state and tables are there

        def launches(**kw):
            return captured_launches(store, lambda: getattr(store, call)(**dict(hp, **kw)))

        general = 2 if table in ("beyond", "65 tensors") else 1
        assert launches(max_grad_norm=1.0) == general, table
        store.timing(True)
        assert launches(max_grad_norm=1.0) == 2, table
        store.timing(False)
        store.grad_sumsq_tensors()
        assert launches(max_grad_norm=1.0, tensor_sums=True) == 2, table
        store.close()

"""GPU test of the decisions taken by the norm pass's (or the pending sums' combination's) last
block, at the grids where its tickets can go wrong: one block, one ticket group less, exactly
and more than full, and more tiles than blocks; several calls in a row, since every launch has
to leave the tickets as it found them."""
import numpy as np
import pytest

from gpu_util import torch_mod

pytestmark = pytest.mark.gpu

TILE = {"fp32": 4096, "mixed": 8192}


@pytest.mark.parametrize("mode", ["fp32", "mixed"])
@pytest.mark.parametrize("tiles", [1, 2, 31, 32, 33, 63, 64, 65, 1000, 2047, 2048, 2049, 2500])
def test_norm_over_ticket_grids(mode, tiles):
    import ttperf
    torch = torch_mod()
    n = (tiles - 1) * TILE[mode] + 1 + tiles % 7  # the last tile is nearly empty
    store = ttperf.ParamStore([(n,)], mode=mode)
    store.set_stream(torch.cuda.current_stream())
    view = store.torch_view(ttperf.BUF_GRAD)
    gen = torch.Generator(device="cuda").manual_seed(tiles)
    for k in range(4):
        view[:n].copy_(torch.randn(n, device="cuda", generator=gen))
        store.mark_grads()
        want = float(view[:n].double().square().sum().sqrt())
        # fp64 sums in two orders: n roundings of 2^-53 at most
        assert abs(store.grad_norm() - want) <= n * 2.0 ** -53 * want + 1e-300
        rep = store.sgd_step(1e-3, max_grad_norm=1.0, report=True)
        assert abs(rep["grad_norm"] - want) <= n * 2.0 ** -53 * want + 1e-300
        assert rep["clip_coef"] == np.float32(min(1.0, 1.0 / (rep["grad_norm"] + 1e-6)))
    store.close()


@pytest.mark.parametrize("tensors", [1, 2, 31, 32, 33, 64, 65, 300])
def test_norm_from_pending_sums(tensors):
    """The same over the blocks that combine pending per-tensor sums (one block a tensor)."""
    import ttperf
    torch = torch_mod()
    sizes = [5000 + 37 * k for k in range(tensors)]
    store = ttperf.ParamStore([(n,) for n in sizes], mode="mixed")
    store.set_stream(torch.cuda.current_stream())
    gen = torch.Generator(device="cuda").manual_seed(tensors)
    for k in range(3):
        grads = [torch.randn(n, device="cuda", generator=gen).bfloat16() for n in sizes]
        store.zero_grad()
        for b in range(0, tensors, 64):
            store.accumulate_grads(range(b, min(b + 64, tensors)), grads[b:b + 64], sums=True)
        want = float(sum(g.double().square().sum() for g in grads)) ** 0.5
        rep = store.adam_step(1e-3, max_grad_norm=1.0, report=True, tensor_sums=True)
        assert abs(rep["grad_norm"] - want) <= sum(sizes) * 2.0 ** -53 * want
        assert rep["clip_coef"] == np.float32(min(1.0, 1.0 / (rep["grad_norm"] + 1e-6)))
    store.close()

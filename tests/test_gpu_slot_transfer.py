"""GPU test of the state transfers' lane kernels at their edges: a contiguous device array to and
from the records of 64-element slots, four elements per lane when the array is 16-byte aligned
and one per lane otherwise.  Sizes end inside a lane's word, a record and a 256-element block.
Every slot is read through ttp_buffer_layout's addressing, which neither kernel takes part in.
"""
import numpy as np
import pytest

import oracle as O
from gpu_util import torch_mod

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 3, 4, 5, 63, 64, 65, 66, 255, 256, 257, 259, 1021, 70_003]


def _slots(store, which):
    """A strided torch view of a record-stored buffer's flat elements."""
    torch = torch_mod()
    base, group, stride = store.layout(which)

    class _Device:
        __cuda_array_interface__ = {"data": (base, False), "typestr": "<f4", "version": 3,
                                    "shape": (store.total // group, group),
                                    "strides": (stride * 4, 4)}

    return torch.as_tensor(_Device(), device="cuda:0")


@pytest.mark.parametrize("mode", ["mixed", "fp32"])
@pytest.mark.parametrize("shift", [0, 1, 2, 3])
def test_device_transfer_edges(mode, shift):
    import ttperf
    torch = torch_mod()
    store = ttperf.ParamStore([(n,) for n in SIZES], mode=mode)
    rng = np.random.default_rng(shift)
    bufs = [ttperf.BUF_EXP_AVG, ttperf.BUF_EXP_AVG_SQ]
    bufs += [ttperf.BUF_MASTER] if mode == "mixed" else []
    for which in bufs:
        want = np.zeros(store.total, np.float32)
        for k, n in enumerate(SIZES):
            vals = rng.normal(size=n).astype(np.float32)
            src = torch.zeros(n + shift, device="cuda")[shift:]  # 4 * shift bytes off 16
            src.copy_(torch.from_numpy(vals))
            store.upload(which, k, src)
            want[store.offsets[k]:store.offsets[k] + n] = vals
        got = _slots(store, which).reshape(-1).cpu().numpy()
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32))  # the padding too
        for k, n in enumerate(SIZES):
            out = torch.full((n + shift + 8,), 7.0, device="cuda")
            store.download(which, k, out=out[shift:shift + n])
            out = out.cpu().numpy()
            o = store.offsets[k]
            assert np.array_equal(out[shift:shift + n].view(np.uint32),
                                  want[o:o + n].view(np.uint32))
            assert (out[:shift] == 7.0).all() and (out[shift + n:] == 7.0).all()
        if which == ttperf.BUF_MASTER:
            assert np.array_equal(store.download(ttperf.BUF_PARAM), O.bf16_rne(want))
    store.close()

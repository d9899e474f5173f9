"""What one-call step 0 checks and takes: output buffers of the wrong shape and a single output
(f16 queries over a packed prefix, which read an f16 copy)."""

import pytest
import torch

from maskahead_amd.kernels import Step0Buffers, gather_packed_kv, step0_select

from _util import gpu_prefix, layer_inputs, packed_cpu

pytestmark = pytest.mark.gpu

N, T, D, K = 320, 16, 64, 48


def _layer(dev, seed, dtype=torch.float16):
    q, k, v, kc, vc = layer_inputs(hq=8, hkv=2, d=D, n=N, t=T, seed=seed, dtype=torch.bfloat16)
    store, nq = packed_cpu(k, v)
    return tuple(x.to(dtype).to(dev) for x in (q, kc, vc)) + (gpu_prefix(store, nq, dev),)


def _step0(bufs, layer, rows=range(T), **kw):
    q, kc, vc, p = layer
    return step0_select(bufs, q, p, kc, vc, rows if isinstance(rows, torch.Tensor) else list(rows), K, value=True, **kw)


def test_output_of_the_wrong_shape(gpu):
    layer = _layer(gpu, 1)
    good = torch.empty((1, 2, K, D), dtype=torch.float16, device=gpu)
    for shape in ((1, 2, K - 1, D), (1, 1, K, D), (1, 2, K, D // 2), (1, 2, K + 1, D)):
        bad = torch.empty(shape, dtype=torch.float16, device=gpu)
        for kw in (dict(out_key=bad, out_value=good), dict(out_key=good, out_value=bad), dict(out_key=bad)):
            with pytest.raises(ValueError):
                _step0(Step0Buffers(), layer, **kw)


@pytest.mark.parametrize("name", ["out_key", "out_value"])
def test_one_output_alone(gpu, name):
    layer = _layer(gpu, 2)
    bufs = Step0Buffers()
    for dtype in (torch.float16, torch.float16, torch.bfloat16):     # the second call repeats the first
        got = torch.full((1, 2, K, D), float("nan"), dtype=dtype, device=gpu)
        _, stats, _, _, idx = _step0(bufs, layer, **{name: got})
        both = gather_packed_kv(stats[3], idx, dtype=dtype)
        assert torch.equal(got, both[name == "out_value"])

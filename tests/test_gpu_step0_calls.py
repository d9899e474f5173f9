"""What one-call step 0 checks: output buffers of the wrong shape (f16 queries over a packed
prefix, which read an f16 copy)."""

import pytest
import torch

from maskahead_amd.kernels import Step0Buffers, step0_select

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

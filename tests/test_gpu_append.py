"""The one-launch packed append and quantizers at the edges of their work split (128-token
workgroups, 64-row residual passes, rows that allow no 16-byte loads), bit-exact against
the oracle's quantizers and the tokens themselves."""

import pytest
import torch

from maskahead_amd.cache import PackedKVCache
from maskahead_amd.config import QuantizationConfig
from maskahead_amd.kernels import quantize_key_groups_into, quantize_values_into
from oracle import attention as OA

pytestmark = pytest.mark.gpu


def _tokens(shape, dtype, seed, odd=False):
    g = torch.Generator().manual_seed(seed)
    x = (torch.randn(shape, generator=g) * 3).to(dtype)
    if not odd:
        return x, lambda dev: x.to(dev)
    # the same values behind a row stride and a base that are not multiples of 16 bytes
    b, h, t, d = shape

    def make(dev):
        buf = torch.zeros((b, h, t, d + 3), dtype=dtype, device=dev)
        buf[..., 1:d + 1] = x.to(dev)
        return buf[..., 1:d + 1]

    return x, make


@pytest.mark.parametrize("d,dtype,t,odd", [(128, torch.bfloat16, 32, False), (128, torch.float16, 160, True),
                                           (64, torch.bfloat16, 416, False), (64, torch.float32, 96, True),
                                           (32, torch.bfloat16, 128, False), (256, torch.bfloat16, 288, False),
                                           (96, torch.bfloat16, 64, False)])
def test_quantizers_at_the_splits_edges(gpu, d, dtype, t, odd):
    x, make = _tokens((2, 3, t, d), dtype, 11, odd)
    kq, ks, kz = OA.quantize_keys(x)
    tv = t - 5      # values: any token count
    vq, vs, vz = OA.quantize_values(x[:, :, :tv].contiguous())
    xg = make(gpu)
    out = [torch.zeros(r.shape, dtype=r.dtype, device=gpu) for r in (kq, ks, kz, vq, vs, vz)]
    quantize_key_groups_into(xg, *out[:3], bits=4, token_group=32)
    quantize_values_into(xg[:, :, :tv], *out[3:], bits=4, channel_group=32)
    for got, want in zip(out, (kq, ks, kz, vq, vs, vz)):
        assert torch.equal(got.cpu(), want)


@pytest.mark.parametrize("d,residual,appends,odd", [(128, 32, (70, 32, 32, 5, 200), False),
                                                    (64, 160, (300, 32, 64, 32, 33), False),
                                                    (128, 96, (40, 90, 32, 32), True), (64, 0, (33, 31, 64), False)])
def test_append_equals_the_oracle(gpu, d, residual, appends, odd):
    h = 3
    cache = PackedKVCache(num_layers=1, batch_size=1, num_kv_heads=h, head_dim=d, max_tokens=1024,
                          quant=QuantizationConfig(residual_tokens=residual), device=gpu)
    ks, vs = [], []
    for i, n in enumerate(appends):
        k, kg = _tokens((1, h, n, d), torch.bfloat16, 20 + i, odd)
        v, vg = _tokens((1, h, n, d), torch.bfloat16, 40 + i, odd)
        cache.begin_append(n)
        cache.stage_layer(0, kg(gpu), vg(gpu))
        cache.commit_append()
        ks.append(k)
        vs.append(v)
        k_all, v_all = torch.cat(ks, 2), torch.cat(vs, 2)
        q, r = cache.quantized_length, cache.residual_length
        assert q + r == k_all.shape[2] == cache.length
        view = cache.layer_view(0)
        want = ((*OA.quantize_keys(k_all[:, :, :q].contiguous()), *OA.quantize_values(v_all[:, :, :q].contiguous()))
                if q else ())
        for got, ref in zip((view.k_q, view.k_scale, view.k_zero, view.v_q, view.v_scale, view.v_zero), want):
            assert torch.equal(got.cpu(), ref)
        assert torch.equal(view.k_residual.cpu(), k_all[:, :, q:]) and torch.equal(view.v_residual.cpu(), v_all[:, :, q:])

"""The packed append that quantizes a long 16-bit residual (blocks staged unquantized, or a
long residual_tokens): the same bytes as the oracle's quantizers and the tokens themselves
where its groups are shared between the workgroup that moves the residual and the others,
and no longer than the same tokens take as a prompt."""

import pytest
import torch

from maskahead_amd.cache import PackedKVCache
from maskahead_amd.config import QuantizationConfig
from oracle import attention as OA

pytestmark = pytest.mark.gpu


def _cache(h, d, residual, dev, max_tokens=16384):
    return PackedKVCache(num_layers=1, batch_size=1, num_kv_heads=h, head_dim=d, max_tokens=max_tokens,
                         quant=QuantizationConfig(residual_tokens=residual), device=dev)


def _append(cache, k, v, stage):
    cache.stage = stage
    cache.begin_append(k.shape[2])
    cache.stage_layer(0, k, v)
    cache.commit_append()


@pytest.mark.parametrize("d,residual,staged,new", [
    (128, 32, 33, 31),        # one group, all of it replaced
    (128, 32, 200, 32),       # the kept rows end inside the second group
    (128, 32, 300, 1),
    (64, 0, 256, 32),         # nothing is kept
    (64, 5, 1000, 500),
    (128, 160, 700, 90),      # more rows kept than one pass moves
    (128, 600, 601, 128),     # nearly all rows kept
    (32, 32, 2048, 64),
])
def test_staged_rows_quantized(gpu, d, residual, staged, new):
    h = 3
    g = torch.Generator().manual_seed(staged + new)
    k, v = ((torch.randn((1, h, staged + new, d), generator=g) * 3).to(torch.bfloat16) for _ in "kv")
    cache = _cache(h, d, residual, gpu, 4096)
    _append(cache, k[:, :, :staged].to(gpu), v[:, :, :staged].to(gpu), True)
    assert cache.residual_length == staged
    _append(cache, k[:, :, staged:].to(gpu), v[:, :, staged:].to(gpu), False)
    q = cache.quantized_length
    assert q + cache.residual_length == staged + new and cache.residual_length < residual + 32
    view = cache.layer_view(0)
    want = (*OA.quantize_keys(k[:, :, :q].contiguous()), *OA.quantize_values(v[:, :, :q].contiguous()))
    for got, ref in zip((view.k_q, view.k_scale, view.k_zero, view.v_q, view.v_scale, view.v_zero), want):
        assert torch.equal(got.cpu(), ref)
    assert torch.equal(view.k_residual.cpu(), k[:, :, q:]) and torch.equal(view.v_residual.cpu(), v[:, :, q:])


def test_staged_rows_take_no_longer_than_a_prompt(gpu):
    """8 192 staged rows are the work of an 8 192-token prompt: 12 us.  Quantized by one
    workgroup a lane they took 20 times that; the bound is 5 times, of the fastest of several."""
    h, d, n = 4, 128, 8192
    x = torch.randn((1, h, n, d), device=gpu).to(torch.bfloat16)

    def fastest(staged):
        cache = _cache(h, d, 32, gpu)
        best = float("inf")
        for _ in range(8):
            cache.reset()
            if staged:
                _append(cache, x, x, True)
            tail = x[:, :, :32] if staged else x
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            torch.cuda._sleep(200000)       # the launch is enqueued before its turn comes
            start.record()
            _append(cache, tail, tail, False)
            end.record()
            torch.cuda.synchronize()
            best = min(best, start.elapsed_time(end))
        return best

    assert fastest(True) < 5 * fastest(False)

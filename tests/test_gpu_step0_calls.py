"""What one-call step 0 keeps and checks between calls: output buffers of the wrong shape and
a single output (f16 queries over a packed prefix, which read an f16 copy), the copy that the
statistics name, and selection rows changed in place."""

import pytest
import torch

from maskahead_amd.kernels import Step0Buffers, gather_packed_kv, prefix_scores, splitk_attention, step0_select

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


def test_statistics_keep_their_copy(gpu):
    """Scores taken from one call's statistics after another layer's call, and after the same
    layer's, over one shared workspace."""
    ws = Step0Buffers()
    layers = [_layer(gpu, s) for s in (3, 4)]
    bufs = [Step0Buffers(), Step0Buffers()]
    for call in range(2):                                            # planned, then repeated
        kept = []
        for b, layer in zip(bufs, layers):
            _, stats, mass, score, _ = _step0(b, layer, workspace=ws)
            kept.append((layer, stats[3], stats[3].kf.clone(), tuple(x.clone() for x in stats[:3]), mass.clone(), score.clone()))
        again = _step0(bufs[0], layers[0], workspace=ws)
        for layer, used, key, (mp, lp, op), mass, score in kept:
            assert again[1][3] is not used and torch.equal(used.kf, key)
            m, s = prefix_scores(layer[0], layer[3], (mp, lp, op, used), list(range(T)), value=True)
            assert torch.equal(m, mass) and torch.equal(s, score)
            want = splitk_attention(*layer[:1], layer[3], *layer[1:3], want_prefix=True)[1]
            assert torch.equal(want[3].kf, used.kf) and torch.equal(want[3].vf, used.vf)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rows", [torch.tensor([3, 7], dtype=torch.int64), torch.tensor([3, 7], dtype=torch.int32)])
@pytest.mark.parametrize("where", ["cpu", "gpu"])
def test_rows_changed_in_place(gpu, dtype, rows, where):
    layer = _layer(gpu, 5, dtype)
    rows = rows.clone() if where == "cpu" else rows.to(gpu)
    bufs = Step0Buffers()
    for values in ((3, 7), (3, 7), (0, 15), (2, 2)):
        rows.copy_(torch.tensor(values))
        got = _step0(bufs, layer, rows)
        want = _step0(Step0Buffers(), layer, list(values))
        assert torch.equal(got[2], want[2]) and torch.equal(got[3], want[3]) and torch.equal(got[4], want[4])


def test_captured_f16_step0(gpu):
    """A captured f16 step 0 owns its copy: replays over new queries, with eager calls of the same
    prefix between them, equal the eager results."""
    q, kc, vc, p = _layer(gpu, 6)
    static = [x.clone() for x in (q, kc, vc)]
    bufs, ws, eager = Step0Buffers(), Step0Buffers(), Step0Buffers()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        _step0(bufs, (*static, p), workspace=ws)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        out, stats, mass, score, idx = _step0(bufs, (*static, p), workspace=ws)
    for scale in (1.0, 0.5, -0.75, 1.25):
        for s, x in zip(static, (q, kc, vc)):
            s.copy_(x * scale)
        graph.replay()
        torch.cuda.synchronize()
        want = _step0(eager, (*static, p))
        assert torch.equal(out, want[0]) and torch.equal(mass, want[2]) and torch.equal(score, want[3])
        assert torch.equal(idx, want[4]) and torch.equal(stats[3].kf, want[1][3].kf)

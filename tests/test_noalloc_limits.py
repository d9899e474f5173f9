"""Which calls ma_splitk_attention_noalloc takes: every one whose partials fit 32 MiB with a
partial per split -- a packed prefix's tail (an odd key group of 32 tokens, a 16-bit residual)
needs one more, which must not refuse it.  The limit is checked on the host before anything
else, so it is tested without a GPU; two calls past 32 MiB by their tail run on one."""

import ctypes
import random

import pytest
import torch

from maskahead_amd import _native as N

from _util import gpu_prefix, layer_inputs, packed_cpu, same_bits

LIMIT = 32 << 20
CUS = 256


def _status(b, h, g, t, d, nq, nf, split=0):
    """Of a call without operands: refused by the size check, or by a later one."""
    p = N.MaPrefix()
    p.nq, p.nf = nq, nf
    none = N.MaTensor4()
    return N.load().ma_splitk_attention_noalloc(none, b, h * g, t, d, ctypes.byref(p), h, none, none, t, 0, 0, 0, 1.0,
                                                none, None, None, None, split, None)


def _bytes_without_tail(b, h, g, t, d, nq, nf, split=0):
    """Partials (f16 row, three f32) of the current block and of splits of about one workgroup
    a CU, 7 row tiles each, packed and 16-bit tokens split apart."""
    units = b * h * -(-(-(-g * t // 32)) // 7)
    n = nq + nf
    sn = split or -(-(-(-n // max(1, CUS // units - 1))) // 64) * 64
    return b * h * (-(-nq // sn) + -(-nf // sn) + 1) * g * t * (2 * d + 12) + 256


SIZES = [  # batch, KV heads, heads each, block, head_dim, packed tokens, 16-bit tokens
    (2, 8, 7, 512, 128, 65632, 0),
    (1, 4, 7, 2048, 128, 80800, 0),
    (1, 8, 8, 512, 128, 4064, 300),
    (2, 8, 7, 512, 128, 96, 0),
    (1, 8, 8, 896, 128, 32, 0),       # a tail alone takes the one split's place
    (1, 8, 8, 512, 128, 32, 700),
]


@pytest.mark.parametrize("size", SIZES)
def test_a_tail_does_not_refuse_a_call(size):
    assert _bytes_without_tail(*size) <= LIMIT
    assert _status(*size) != N.MA_EWORKSPACE


def test_calls_within_the_limit_over_many_sizes():
    rng = random.Random(7)
    taken = 0
    for _ in range(4000):
        h, g, d = rng.choice([(4, 7), (8, 4), (8, 8), (2, 7), (4, 4)]) + (rng.choice([64, 128]),)
        size = (rng.choice([1, 1, 2, 4]), h, g, rng.choice([8, 32, 96, 256, 512, 1024]), d,
                rng.choice([0, 32, 96, 32 * rng.randrange(4000)]), rng.choice([0, 17, 32, 200, 300, rng.randrange(5000)]),
                rng.choice([0, 0, 0, 64, 512, 4096]))
        if size[5] + size[6] and _bytes_without_tail(*size) <= LIMIT:
            taken += 1
            assert _status(*size) != N.MA_EWORKSPACE, size
    assert taken > 1000


def test_calls_beyond_the_limit_stay_refused():
    for size in [(8, 8, 4, 256, 128, 0, 64), (8, 8, 4, 256, 128, 64, 0), (8, 8, 4, 256, 128, 96, 0),
                 (8, 8, 4, 256, 128, 32, 0)]:
        assert _bytes_without_tail(*size) > LIMIT and _status(*size) == N.MA_EWORKSPACE


@pytest.mark.gpu
@pytest.mark.parametrize("b,h,g,t,d,nq,nf", [(1, 8, 8, 512, 128, 4064, 300), (2, 8, 7, 512, 128, 96, 0)])
def test_calls_past_the_limit_by_their_tail(gpu, b, h, g, t, d, nq, nf):
    q, k, v, kc, vc = (x.to(gpu) for x in layer_inputs(b=b, hq=h * g, hkv=h, d=d, n=nq + nf, t=t, seed=nq,
                                                       dtype=torch.bfloat16))
    store, _ = packed_cpu(k[:, :, :nq].cpu(), v[:, :, :nq].cpu())
    p = gpu_prefix(store, nq, gpu, kf=k[:, :, nq:].cpu() if nf else None, vf=v[:, :, nq:].cpu() if nf else None)
    lib = N.load()
    need = int(lib.ma_splitk_workspace_bytes(b, h, h * g, t, d, nq, nf, 0))
    assert LIMIT < need <= LIMIT * 3 // 2
    ws = torch.empty((need,), dtype=torch.uint8, device=gpu)
    got = []
    for name, extra in (("ma_splitk_attention", [ws.data_ptr(), need]), ("ma_splitk_attention_noalloc", [])):
        out = torch.empty_like(q)
        mp = torch.empty((b, h, g * t), dtype=torch.float32, device=gpu)
        lp = torch.empty_like(mp)
        op = torch.empty((b, h, g * t, d), dtype=q.dtype, device=gpu)
        N.call(name, N.t4(q), b, h * g, t, d, ctypes.byref(p.native()), h, N.t4(kc), N.t4(vc), t, 0, 0, 0, d ** -0.5,
               N.t4(out), N.ptr(mp), N.ptr(lp), N.ptr(op), 0, *extra, N.stream_of(q))
        got.append((out, mp, lp, op))
    for x, y in zip(*got):
        assert torch.isfinite(x.float()).all() and same_bits(x, y)

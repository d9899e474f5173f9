"""Pass 1's row groups of up to 8 row tiles: one group of 7 and of 8, groups of equal size, a
shorter last one, a last tile of few rows, and prefill chunks where groups of 8 are chosen and
where groups of 7 are, over packed and 16-bit prefixes, against the oracle."""

import pytest
import torch

from maskahead_amd.kernels.splitk import Prefix, splitk_attention
from oracle import attention as OA

from _util import assert_attention_close, dequant_cpu, gpu_prefix, layer_inputs, packed_cpu, rel_err

pytestmark = pytest.mark.gpu

CASES = [  # heads, head_dim, block, tokens, split_tokens
    ((7, 1), 128, 32, 640, 0),
    ((8, 1), 128, 32, 640, 0),       # 8 row tiles: two groups of 4
    ((8, 1), 128, 32, 640, 128),     # the same, splits given
    ((9, 1), 64, 32, 320, 0),        # 9: 5 and 4
    ((15, 1), 128, 31, 1000, 0),     # 465 rows: 15 tiles, the last of 17 rows
    ((32, 8), 64, 256, 4512, 0),     # 32 tiles a head: groups of 8
    ((28, 4), 128, 512, 4096, 0),    # 112 tiles
    ((14, 2), 64, 512, 2016, 0),
    ((14, 2), 64, 512, 2016, 512),
]


@pytest.mark.parametrize("heads,d,t,n,split", CASES)
@pytest.mark.parametrize("packed", [False, True])
def test_row_groups_against_the_oracle(gpu, heads, d, t, n, split, packed):
    hq, hkv = heads
    q, k, v, kc, vc = layer_inputs(hq=hq, hkv=hkv, d=d, n=n, t=t, seed=n + t, dtype=torch.bfloat16)
    if packed:
        nq = (n - 32) // 32 * 32     # and a 16-bit residual of 32 tokens or a few more
        store, nq = packed_cpu(k[:, :, :nq], v[:, :, :nq])
        kd, vd = dequant_cpu(store, nq)
        p = gpu_prefix(store, nq, gpu, kf=k[:, :, nq:], vf=v[:, :, nq:])
        k, v = torch.cat([kd, k[:, :, nq:].float()], 2), torch.cat([vd, v[:, :, nq:].float()], 2)
    else:
        p = Prefix.dense(k.to(gpu), v.to(gpu))
    out, stats = splitk_attention(q.to(gpu), p, kc.to(gpu), vc.to(gpu), want_prefix=True, split_tokens=split)
    want = OA.splitk_attention(q, k, v, kc, vc)
    assert_attention_close(out, want[0])
    mp, lp, op = (x.cpu() for x in stats[:3])
    assert rel_err(mp, want[1]) < 1e-5 and rel_err(lp, want[2]) < 1e-4
    assert_attention_close(op, want[3], atol=1e-2, rtol=1e-2)

"""What a packed prefix leaves behind its whole 64-token tiles -- an odd key group of 32
tokens, a 16-bit residual, or both -- in split-K attention (a segment of the packed launch,
or a launch of its own when long) and in the score pass (a tile staged by items), against
the oracle; dead slots hold NaN."""

import pytest
import torch

from maskahead_amd.kernels.splitk import prefix_scores, splitk_attention
from oracle import attention as OA

from _util import assert_attention_close, dequant_cpu, gpu_prefix, layer_inputs, packed_cpu, rel_err

pytestmark = pytest.mark.gpu

CASES = [  # packed tokens, residual, heads, head_dim, block, mask, split_tokens
    (32, 0, (4, 2), 128, 8, False, 0),
    (32, 1, (4, 2), 64, 8, True, 0),
    (64, 33, (4, 2), 128, 16, False, 0),
    (96, 63, (28, 4), 128, 32, True, 0),
    (352, 0, (28, 4), 128, 32, True, 64),
    (352, 31, (8, 2), 64, 32, False, 128),
    (992, 45, (16, 4), 64, 96, True, 0),
    (1024, 192, (28, 4), 128, 32, False, 0),    # the longest tail of the packed launch
    (1056, 225, (28, 4), 128, 32, True, 0),     # one token more than it takes: two launches
    (1056, 700, (8, 2), 128, 32, True, 256),
]


@pytest.mark.parametrize("nq,tail,heads,d,t,masked,split", CASES)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_tail_against_the_oracle(gpu, nq, tail, heads, d, t, masked, split, dtype):
    hq, hkv = heads
    n = nq + tail
    q, k, v, kc, vc = layer_inputs(hq=hq, hkv=hkv, d=d, n=n, t=t, seed=nq + tail, dtype=torch.bfloat16)
    store, nq = packed_cpu(k[:, :, :nq], v[:, :, :nq], pad_groups=1, pad_tokens=7)
    kd, vd = dequant_cpu(store, nq)
    kt, vt = k[:, :, nq:].to(dtype), v[:, :, nq:].to(dtype)
    k_all, v_all = torch.cat([kd, kt.float()], 2), torch.cat([vd, vt.float()], 2)
    mask = None
    if masked:
        g = torch.Generator().manual_seed(n)
        mask = (torch.rand((1, hkv, n), generator=g) > 0.3).to(torch.uint8)
        mask[:, :, 0] = 1
        dead = mask[:, :, nq:, None] == 0
        kt, vt = (x.masked_fill(dead, float("nan")) for x in (kt, vt))
        store["vs"][:, :, :nq].masked_fill_(mask[:, :, :nq, None] == 0, float("nan"))
    p = gpu_prefix(store, nq, gpu, kf=kt if tail else None, vf=vt if tail else None, mask=mask)
    qg = q.to(gpu)
    out, stats = splitk_attention(qg, p, kc.to(gpu), vc.to(gpu), want_prefix=True, split_tokens=split)
    want = OA.splitk_attention(q, k_all, v_all, kc, vc, mask=mask)
    mp, lp, op = (x.cpu() for x in stats[:3])
    assert_attention_close(out, want[0])
    assert rel_err(mp, want[1]) < 1e-5 and rel_err(lp, want[2]) < 1e-4
    assert_attention_close(op, want[3], atol=1e-2, rtol=1e-2)
    # scores from the same statistics: the value distance reads packed V rounded to bf16 where
    # the reference reads an unpacked copy
    rows = list(range(t))
    v_dist = torch.cat([vd.to(torch.bfloat16).float() if stats[3].vround else vd, vt.float()], 2)
    if masked:
        v_dist = torch.where(mask[..., None] != 0, v_dist, torch.zeros(()))
    mass, score = prefix_scores(qg, p, stats, rows, value=True)
    m_only, _ = prefix_scores(qg, p, stats, rows, value=False)
    wmass, wscore = OA.prefix_scores(q, k_all, v_dist, mp, lp, op, rows, mask=mask, value_aware=True)
    assert rel_err(mass, wmass) < 2e-5 and rel_err(score, wscore) < 2e-5
    assert torch.equal(m_only, mass)
    if masked:
        assert torch.all(mass.cpu()[mask == 0] == 0) and torch.all(score.cpu()[mask == 0] == 0)

"""Prefix mass of more selection rows than one pass of the score kernel holds (above 512 per
KV head), and the merge of few splits: odd row and token counts, chosen rows, dead slots,
every prefix kind, against the oracle from the same statistics."""

import pytest
import torch

from maskahead_amd.kernels import prefix_scores_topk, topk_ascending
from maskahead_amd.kernels.splitk import Prefix, prefix_scores, splitk_attention
from oracle import attention as OA

from _util import assert_attention_close, dequant_cpu, gpu_prefix, layer_inputs, packed_cpu, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,n,heads,d,t,rows,masked", [
    ("packed", 64, (8, 2), 128, 129, None, False),          # 516 rows: 9 pairs of row tiles, one of them padding
    ("packed", 32 + 17, (28, 4), 128, 96, None, True),      # an odd group and a residual, one ragged tile
    ("packed", 992 + 40, (16, 4), 64, 160, "some", True),
    ("bf16", 1, (8, 2), 128, 144, None, False),
    ("bf16", 517, (28, 4), 128, 128, "some", True),
    ("f16", 450, (16, 4), 64, 140, None, False),
    ("f32", 130, (8, 2), 128, 150, None, True),              # element-wise staging
])
def test_mass_of_many_rows(gpu, kind, n, heads, d, t, rows, masked):
    hq, hkv = heads
    q, k, v, kc, vc = layer_inputs(hq=hq, hkv=hkv, d=d, n=n, t=t, seed=n + t, dtype=torch.bfloat16)
    mask = None
    if masked:
        g = torch.Generator().manual_seed(n)
        mask = (torch.rand((1, hkv, n), generator=g) > 0.3).to(torch.uint8)
        mask[:, :, 0] = 1
    if kind == "packed":
        nq = n // 32 * 32
        store, nq = packed_cpu(k[:, :, :nq], v[:, :, :nq], pad_groups=1)
        kd, vd = dequant_cpu(store, nq)
        p = gpu_prefix(store, nq, gpu, kf=k[:, :, nq:] if n > nq else None, vf=v[:, :, nq:] if n > nq else None, mask=mask)
        k_used, v_used = torch.cat([kd, k[:, :, nq:].float()], 2), torch.cat([vd, v[:, :, nq:].float()], 2)
    else:
        dt = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}[kind]
        k_used, v_used = k.to(dt).float(), v.to(dt).float()
        p = Prefix.dense(k.to(dt).to(gpu), v.to(dt).to(gpu), mask=None if mask is None else mask.to(gpu))
    qg = q.to(gpu)
    out, stats = splitk_attention(qg, p, kc.to(gpu), vc.to(gpu), causal_block=32, want_prefix=True)
    want = OA.splitk_attention(q, k_used, v_used, kc, vc, mask=mask, causal_block=32)
    assert_attention_close(out, want[0])
    mp, lp, op = (x.cpu() for x in stats[:3])
    # a logit is an f32 sum of d products: off by at most d 2^-24 sum |q_i k_i| (one may be ~0, so
    # no relative bound holds for it)
    qa = q.float().abs().reshape(hkv, -1, d)
    bound = d * 2.0 ** -24 * d ** -0.5 * torch.matmul(qa, k_used[0].abs().transpose(-1, -2)).amax(-1)
    assert torch.all((mp[0].double() - want[1][0].double()).abs() <= bound) and rel_err(lp, want[2]) < 1e-4
    assert_attention_close(op, want[3], atol=1e-2, rtol=1e-2)
    sel = list(range(t)) if rows is None else list(range(t - 1, 0, -1))[: t - 9]
    mass, _ = prefix_scores(qg, p, stats, sel, value=False)
    wmass, _ = OA.prefix_scores(q, k_used, v_used, mp, lp, op, sel, mask=mask, value_aware=False)
    assert rel_err(mass, wmass) < 2e-5
    if masked:
        assert torch.all(mass.cpu()[mask == 0] == 0)


@pytest.mark.parametrize("kind,rows", [("packed", None), ("packed", "some"), ("bf16", None)])
def test_mass_of_many_rows_in_two_passes(gpu, kind, rows):
    """516 to 524 selection rows over 8 x 16 500 tokens, at least 8 tiles a CU: two passes, the
    second adding to the first's mass; the select's histogram is of the sum."""
    hq, hkv, d, n, t = 32, 8, 128, 16500, 131
    q, k, v, kc, vc = layer_inputs(hq=hq, hkv=hkv, d=d, n=n, t=t, seed=n, dtype=torch.bfloat16)
    g = torch.Generator().manual_seed(n)
    mask = (torch.rand((1, hkv, n), generator=g) > 0.3).to(torch.uint8)
    mask[:, :, 0] = 1
    if kind == "packed":
        nq = (n - 32) // 32 * 32
        store, nq = packed_cpu(k[:, :, :nq], v[:, :, :nq])
        kd, _ = dequant_cpu(store, nq)
        p = gpu_prefix(store, nq, gpu, kf=k[:, :, nq:], vf=v[:, :, nq:], mask=mask)
        k_used = torch.cat([kd, k[:, :, nq:].float()], 2)
    else:
        k_used = k.float()
        p = Prefix.dense(k.to(gpu), v.to(gpu), mask=mask.to(gpu))
    qg = q.to(gpu)
    _, stats = splitk_attention(qg, p, kc.to(gpu), vc.to(gpu), want_prefix=True)
    mp, lp, op = (x.cpu() for x in stats[:3])
    sel = list(range(t)) if rows is None else list(range(t - 1, 1, -1))
    mass, _ = prefix_scores(qg, p, stats, sel, value=False)
    want, _ = OA.prefix_scores(q, k_used, None, mp, lp, None, sel, mask=mask, value_aware=False)
    assert rel_err(mass, want) < 2e-5 and torch.all(mass.cpu()[mask == 0] == 0)
    m2, _, idx = prefix_scores_topk(qg, p, stats, sel, 500, value=False, rank="mass")
    assert torch.equal(m2, mass) and torch.equal(idx, topk_ascending(mass, 500, p.mask))

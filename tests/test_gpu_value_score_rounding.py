"""The bf16 value score where its f32 sum decides the rounding and where it must not: many
random entries, roots exactly between two bf16 values, sums beyond the f32 range, entries
equal to the centre, NaN -- bit for bit the oracle's float64 result, rows and slot form."""

import pytest
import torch

from maskahead_amd.kernels.keep import value_score, value_score_slots
from maskahead_amd.kernels.splitk import Prefix
from oracle import attention as OA

from _util import same_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,n", [(128, 30011), (64, 20003), (32, 97), (128, 15)])
def test_random_entries(gpu, d, n):
    g = torch.Generator().manual_seed(n)
    a = torch.rand((1, 2, n), generator=g)
    v = (torch.randn((1, 2, n, d), generator=g) * torch.exp(torch.randn((1, 2, n, 1), generator=g))).to(torch.bfloat16)
    want = OA.value_score_bf16(a, v)
    assert same_bits(value_score(a.to(gpu), v.to(gpu), fp32=False), want)
    if d >= 64:
        slots = torch.stack([torch.randperm(n, generator=g) for _ in range(2)]).to(torch.int32)[None]
        rows = torch.gather(v, 2, slots.long().unsqueeze(-1).expand(-1, -1, -1, d))
        got = value_score_slots(a.to(gpu), Prefix.dense(v.to(gpu), v.to(gpu)), slots.to(gpu), fp32=False)
        assert same_bits(got, OA.value_score_bf16(a, rows))


def test_ties_and_extremes(gpu):
    # norm^2 = 1 + 2^-7 + 2^-16 = (1 + 2^-8)^2: the root is the middle of bf16 1 and 1 + 2^-7
    tie = torch.zeros(128)
    tie[0], tie[1], tie[2], tie[3] = 1.0, 2.0 ** -4, 2.0 ** -4, 2.0 ** -8
    # above it by less than an f32 ulp (the rounding through f32 makes it a tie again), and by 4
    above, over = tie.clone(), tie.clone()
    above[4], over[4] = 2.0 ** -20, 2.0 ** -10
    rows = [tie, above, over, torch.zeros(128), torch.full((128,), 2.0 ** 70), torch.full((128,), 2.0 ** -80),
            tie * 2.0 ** -60, tie * 2.0 ** 40]
    # every row with its negative at the same weight: the centre is exactly 0
    v = torch.stack([s * r for r in rows for s in (1.0, -1.0)]).to(torch.bfloat16)[None, None]
    a = torch.full((1, 1, v.shape[2]), 0.5)
    want = OA.value_score_bf16(a, v)
    assert want[0, 0, 0] == 0.5 and want[0, 0, 2] == 0.5 and want[0, 0, 4] == 0.5 * (1 + 2.0 ** -7)
    assert same_bits(value_score(a.to(gpu), v.to(gpu), fp32=False), want)
    v[0, 0, 3, 5] = float("nan")
    got = value_score(a.to(gpu), v.to(gpu), fp32=False).cpu()
    assert torch.isnan(got).all() and torch.isnan(OA.value_score_bf16(a, v)).all()

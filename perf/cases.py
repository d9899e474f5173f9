"""The work a decoding session gives the KV read/keep path, as measured cases.

Every case is one pass of a kind of call that a block-diffusion session makes, over the
layers it makes it for:

  step0      step 0 of a block (FastLayerPath.step0): attention over [prefix | block], the
             prefix mass, the read set and its gather into the compact buffer
  substep    a later denoising sub-step (FastLayerPath.compact_attention)
  probe      a lookahead probe (FastLayerPath.probe): several masked blocks, block-causal
  prefill    one prefill chunk that keeps its prefix mass (FastLayerPath.prefill_chunk)
  keep       the keep step of a 16-bit cache: value_score, keep set, compaction, append
  lookahead  the lookahead keep score and keep set of every layer of an int4 cache
  evict      the lazy rebuild of an int4 cache after a keep set (plan and data)
  load       a prompt loaded into an int4 cache and the first blocks committed after it

Prefix keys hold a group of keys that the block attends to, as many as the read budget
(attention sinks among them), well above the rest: the read set is then the same for any
correct rounding of the scores.
"""

import copy
import math

import torch

from maskahead_amd.cache import PackedKVCache
from maskahead_amd.config import QuantizationConfig
from maskahead_amd.eviction import EvictionConfig, EvictionState
from maskahead_amd.kernels.rebuild import rebuild_plan
from maskahead_amd.runtime.fastpath import CompactLayerState, FastLayerPath
from maskahead_amd.runtime.session import lookahead_scores, value_score

GROUP = 32       # tokens of a packed key group, channels of a packed value group
RESIDUAL = 32    # newest tokens an int4 cache keeps at 16 bits
BLOCK = 32       # tokens of a block
SINKS = 4
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16}


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # the first blocks of a generation: a short prompt in an int4 cache, one layer, all latency
        dict(name="step0_first_block", op="step0", kv="int4", dtype="bf16", hq=28, hkv=4, d=128, n=544, t=32, k=256,
             rows="all", dead=0.0, layers=1),
        # the long-context decoding step: int4 cache of 32 768 tokens and its 16-bit residual
        dict(name="step0_int4_32k", op="step0", kv="int4", dtype="bf16", hq=28, hkv=4, d=128, n=32800, t=32, k=2048,
             rows="all", dead=0.0, layers=8),
        # the same without quantization
        dict(name="step0_bf16_32k", op="step0", kv="bf16", dtype="bf16", hq=28, hkv=4, d=128, n=32768, t=32, k=2048,
             rows="all", dead=0.0, layers=4),
        # a block after lazy evictions: a ragged int4 cache whose dead slots are masked
        dict(name="step0_evicted", op="step0", kv="int4", dtype="bf16", hq=28, hkv=4, d=128, n=6997, t=32, k=2048,
             rows="all", dead=0.15, layers=8),
        # a model run in f16 (its packed prefix is read through an f16 copy)
        dict(name="step0_f16_8k", op="step0", kv="int4", dtype="f16", hq=28, hkv=4, d=128, n=8192, t=32, k=2048,
             rows="all", dead=0.0, layers=4),
        # the other denoising steps of a block, every layer of a 28-layer model
        dict(name="substep_2k", op="substep", b=1, hq=28, hkv=4, d=128, k=2048, t=32, layers=28),
        # the lookahead probe of three blocks over a 16-bit cache of 65 536 tokens
        dict(name="probe_bf16_64k", op="probe", kv="bf16", dtype="bf16", hq=32, hkv=8, d=128, n=65536, t=96, layers=2),
        # a 512-token chunk of a long prompt
        dict(name="prefill_int4_16k", op="prefill", kv="int4", dtype="bf16", hq=28, hkv=4, d=128, n=16384, t=512,
             layers=2),
        # the keep step that follows the probe: 8 192 of 65 536 entries per head
        dict(name="keep_bf16_64k", op="keep", hkv=8, d=128, n=65536, keep=8192, window=128, layers=4),
        # the keep score and set of a lookahead eviction, all layers in one call
        dict(name="lookahead_int4_32k", op="lookahead", hkv=4, d=128, n=32800, keep=4096, window=128, layers=28),
        # the rebuild of that eviction
        dict(name="evict_int4_32k", op="evict", hkv=4, d=128, n=32800, keep=4096, window=128, layers=28),
        # a prompt quantized into the cache and two blocks committed
        dict(name="load_int4_8k", op="load", hkv=4, d=128, n=8192, blocks=2, layers=28),
    ]


def _spread(rng, lo, hi):
    """A size between lo and hi, uniform over its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["step0", "step0", "step0", "substep", "probe", "prefill", "keep", "lookahead", "evict", "load"])
    hq, hkv = rng.choice([(28, 4), (32, 8), (16, 4)])
    d = rng.choice([128, 128, 128, 64])
    kv = rng.choice(["int4", "int4", "bf16"])
    if op == "step0":
        n = _spread(rng, 300, 100000)
        if kv == "bf16":
            n = min(n, 32768)
        return dict(op=op, kv=kv, dtype=rng.choice(["bf16", "bf16", "bf16", "f16"]), hq=hq, hkv=min(hkv, 4) if n > 32768 else hkv,
                    d=d, n=n, t=rng.choice([8, 16, 32]), k=_spread(rng, min(64, n // 3), min(2048, n // 2)),
                    rows=rng.choice(["all", "all", "middle"]), dead=rng.choice([0.0, 0.0, 0.1, 0.3]),
                    layers=max(1, min(4, 120000 // n)))
    if op == "substep":
        b = rng.choice([1, 1, 2, 4])
        return dict(op=op, b=b, hq=hq, hkv=hkv, d=d, k=_spread(rng, 64, 2048), t=rng.choice([8, 16, 32]),
                    layers=max(1, 28 // b))
    if op == "probe":
        return dict(op=op, kv=kv, dtype="bf16", hq=hq, hkv=hkv, d=d, n=_spread(rng, 500, 40000),
                    t=BLOCK * rng.choice([2, 3, 4]) if hq < 32 else 2 * BLOCK, layers=2)
    if op == "prefill":
        return dict(op=op, kv=kv, dtype="bf16", hq=hq, hkv=hkv, d=d, n=_spread(rng, 512, 14000),
                    t=rng.choice([96, 256, 384, 512]), layers=2)
    if op == "keep":
        n = _spread(rng, 8000, 65536)
        return dict(op=op, hkv=hkv, d=d, n=n, keep=_spread(rng, 512, n // 3 - 2048 + 512), window=rng.choice([0, 32, 128]),
                    layers=rng.choice([1, 2, 4]))
    if op in ("lookahead", "evict"):
        n = _spread(rng, 3000, 32800)
        return dict(op=op, hkv=4, d=d, n=n, keep=_spread(rng, 400, min(n // 4, 6000)), window=rng.choice([32, 128]),
                    layers=rng.choice([4, 14, 28]))
    return dict(op="load", hkv=4, d=d, n=_spread(rng, 100, 8192), blocks=rng.choice([1, 2, 4]),
                layers=rng.choice([4, 14, 28]))


# ------------------------------------------------------------------ inputs
def _quantized(n):
    """Tokens of an int4 cache of n tokens that are quantized (whole groups past the residual)."""
    over = max(0, n - RESIDUAL)
    return over - over % GROUP


def _rows(case):
    """The selection rows: every block position, or the middle one."""
    return list(range(case["t"])) if case.get("rows", "all") == "all" else [case["t"] // 2]


def _live(case, g):
    """uint8 [1, Hkv, n]: the live slots, or None when all are."""
    if not case.get("dead"):
        return None
    live = torch.rand((1, case["hkv"], case["n"]), generator=g, device="cuda") >= case["dead"]
    live[:, :, :SINKS] = True
    live[:, :, -RESIDUAL:] = True
    return live.to(torch.uint8)


def _layer_inputs(case, g, live):
    """(q, k, v, kc, vc) of one layer.  Keys: N(0, 1) with a LogNormal(0, 0.5) scale per
    channel; the queries share a direction u that only the attended keys carry."""
    hq, hkv, d, n, t = case["hq"], case["hkv"], case["d"], case["n"], case["t"]
    dt = DTYPES[case.get("dtype", "bf16")]

    def normal(*shape):
        return torch.randn(shape, generator=g, device="cuda")

    chan = torch.exp(0.5 * normal(1, hkv, 1, d))
    u = normal(1, hkv, 1, d)
    u = u / u.norm(dim=-1, keepdim=True)
    k = normal(1, hkv, n, d) * chan
    k -= (k * u).sum(-1, keepdim=True) * u
    attended = case.get("k", max(SINKS, n // 16))
    boost = 5.0 if case.get("rows", "all") == "all" else 10.0
    amount = math.sqrt(boost * math.sqrt(d))
    rank = torch.rand((1, hkv, n), generator=g, device="cuda")
    rank[:, :, :SINKS] = 2.0
    if live is not None:
        rank = rank * live
    lift = torch.zeros((1, hkv, n), device="cuda")
    lift.scatter_(-1, rank.topk(min(attended, n), dim=-1).indices, amount)
    lift[:, :, :SINKS] *= 1.4
    k += lift.unsqueeze(-1) * u
    q = normal(1, hq, t, d) + amount * u.repeat_interleave(hq // hkv, dim=1)
    v, kc, vc = normal(1, hkv, n, d), normal(1, hkv, t, d) * chan, normal(1, hkv, t, d)
    return tuple(x.to(dt) for x in (q, k, v, kc, vc))


class _Prompt:
    """A prefill's keys and values per layer, as a model hands them over."""

    def __init__(self, kv):
        self.kv = kv

    def __getitem__(self, layer):
        return self.kv[layer]

    def get_seq_length(self):
        return int(self.kv[0][0].shape[2])


def _cache(case, kv, spare=0):
    """A cache holding the given per-layer keys and values."""
    n = int(kv[0][0].shape[2])
    bits = 4 if case.get("kv", "int4") == "int4" else 16
    cache = PackedKVCache(num_layers=len(kv), batch_size=1, num_kv_heads=case["hkv"], head_dim=case["d"],
                          max_tokens=n + spare + 64, quant=QuantizationConfig(k_bits=bits, v_bits=bits), device="cuda",
                          compute_dtype=DTYPES[case.get("dtype", "bf16")])
    cache.load_dynamic_cache(_Prompt(kv))
    return cache


def _values(case, g, layers):
    """Per-layer (k, v) of the calls that attend to nothing."""
    shape = (1, case["hkv"], case["n"], case["d"])
    out = []
    for _ in range(layers):
        chan = torch.exp(0.5 * torch.randn((1, case["hkv"], 1, case["d"]), generator=g, device="cuda"))
        out.append(((torch.randn(shape, generator=g, device="cuda") * chan).to(torch.bfloat16),
                    torch.randn(shape, generator=g, device="cuda").to(torch.bfloat16)))
    return out


def _mass(case, g):
    """[layers, 1, Hkv, n] masses: a smooth profile over the context times a heavy-tailed
    factor per entry, summing to 1 per head."""
    L, h, n = case["layers"], case["hkv"], case["n"]
    coarse = torch.randn((L * h, 1, n // 64 + 2), generator=g, device="cuda")
    smooth = torch.nn.functional.interpolate(coarse, size=n, mode="linear", align_corners=True)
    return torch.softmax(1.5 * smooth.view(L, 1, h, n) + torch.randn((L, 1, h, n), generator=g, device="cuda"), dim=-1)


def _keep_cfg(case):
    return EvictionConfig(policy="lookahead", recent_window=case["window"], capacity_floor=max(case["keep"], 1))


def _keep_set(case, g):
    """Sorted live indices [L, 1, H, keep] of a keep set: the window, a fifth of the entries
    clustered in key groups that mostly survive (24 of 32), the rest scattered over the
    others (at most 15 of a group, so that the rebuild quantizes them afresh)."""
    L, h, n, keep, window = (case[x] for x in ("layers", "hkv", "n", "keep", "window"))
    groups = (n - window) // GROUP - 2           # the window's own groups aside
    full = keep // (5 * 24)
    order = torch.rand((L * h, groups, GROUP), generator=g, device="cuda").argsort(-1).argsort(-1)
    dense = torch.rand((L * h, groups), generator=g, device="cuda").argsort(-1).argsort(-1) < full
    scattered = torch.rand((L * h, groups, GROUP), generator=g, device="cuda") * (order < 15)
    clustered = 2.0 * (order < 24)
    rank = torch.zeros((L * h, n), device="cuda")
    rank[:, :groups * GROUP] = torch.where(dense.unsqueeze(-1), clustered, scattered).flatten(1)
    rank[:, n - window:] = 3.0
    return rank.topk(keep, dim=-1).indices.sort(dim=-1).values.view(L, 1, h, keep)


def _inputs(case, seed):
    """What prepare and exact both start from: everything drawn from the seed."""
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    op = case["op"]
    if op in ("step0", "probe", "prefill"):
        lives = [_live(case, g) for _ in range(case["layers"])]
        return dict(live=lives, layers=[_layer_inputs(case, g, lv) for lv in lives])
    if op == "substep":
        b, hq, hkv, d, k, t = (case[x] for x in ("b", "hq", "hkv", "d", "k", "t"))
        lay = []
        for _ in range(case["layers"]):
            lay.append(tuple(torch.randn(s, generator=g, device="cuda").to(torch.bfloat16) for s in
                             ((b, hq, t, d), (b, hkv, k, d), (b, hkv, k, d), (b, hkv, t, d), (b, hkv, t, d))))
        return dict(layers=lay)
    kv = _values(case, g, case["layers"])
    if op == "load":
        nb = case["blocks"]
        return dict(kv=kv, blocks=[_values(dict(case, n=BLOCK), g, case["layers"]) for _ in range(nb)])
    if op == "evict":
        return dict(kv=kv, keep=_keep_set(case, g))
    mass = _mass(case, g)
    if op == "keep":
        return dict(kv=kv, mass=mass, block=_values(dict(case, n=BLOCK), g, case["layers"]))
    return dict(kv=kv, mass=mass, probe=_mass(case, g))


def prepare(case, seed):
    x = _inputs(case, seed)
    op = case["op"]
    s = dict(case=case)
    if op in ("step0", "probe", "prefill"):
        cache = _cache(case, [(k, v) for _, k, v, _, _ in x["layers"]], spare=case["t"])
        masks = {i: m for i, m in enumerate(x["live"]) if m is not None}
        s["path"] = FastLayerPath(cache=cache, block_size=case["t"] if op == "step0" else BLOCK,
                                  query_indices=_rows(case), compute_dtype=cache.compute_dtype, slot_masks=masks)
        s["calls"] = [(q, kc, vc) for q, _, _, kc, vc in x["layers"]]
    elif op == "substep":
        cache = PackedKVCache(num_layers=1, batch_size=case["b"], num_kv_heads=case["hkv"], head_dim=case["d"],
                              max_tokens=64, quant=QuantizationConfig(), device="cuda")
        path = FastLayerPath(cache=cache, block_size=case["t"])
        for i, (_, k, v, _, _) in enumerate(x["layers"]):
            room = torch.zeros((case["b"], case["hkv"], case["t"], case["d"]), dtype=k.dtype, device="cuda")
            path.states[i] = CompactLayerState(key=torch.cat([k, room], 2), value=torch.cat([v, room], 2),
                                               selected_k=case["k"])
        s["path"], s["calls"] = path, [(q, kc, vc) for q, _, _, kc, vc in x["layers"]]
    elif op == "load":
        total = case["n"] + BLOCK * case["blocks"]
        s["cache"] = PackedKVCache(num_layers=case["layers"], batch_size=1, num_kv_heads=case["hkv"],
                                   head_dim=case["d"], max_tokens=total + 64, quant=QuantizationConfig(),
                                   device="cuda")
        s["prompt"], s["blocks"] = _Prompt(x["kv"]), x["blocks"]
    else:
        s["cache"] = _cache(dict(case, kv="bf16" if op == "keep" else "int4"), x["kv"], spare=BLOCK)
        if op == "evict":
            live = x["keep"].to(torch.int32).contiguous()
            s["pos"], s["phys"] = live, live.clone()
        else:
            state = EvictionState(num_layers=case["layers"], batch_size=1, num_kv_heads=case["hkv"],
                                  capacity=case["n"] + BLOCK, device="cuda")
            state.append(range(case["n"]))
            s["state"], s["cfg"] = state, _keep_cfg(case)
            s["mass"] = {i: x["mass"][i] for i in range(case["layers"])}
            if op == "keep":
                s["block"] = x["block"]
            else:
                s["probe"] = {i: x["probe"][i] for i in range(case["layers"])}
    return s


# ------------------------------------------------------------------ one pass
def _planes(cache):
    """The stored planes of every layer, the rows in use."""
    v = cache.all_layers_view()
    names = ("k_q", "k_scale", "k_zero", "v_q", "v_scale", "v_zero", "k_residual", "v_residual", "k_fp", "v_fp")
    return {name: getattr(v, name) for name in names if getattr(v, name) is not None}


def run(s):
    case = s["case"]
    op = case["op"]
    if op == "step0":
        path, k = s["path"], case["k"]
        outs = [path.step0(i, q, kc, vc, select=True, topk=k, want_mass=True) for i, (q, kc, vc) in enumerate(s["calls"])]
        return [(o, path.last_mass[i], path.states[i].indices, path.states[i].key[:, :, :k], path.states[i].value[:, :, :k])
                for i, o in enumerate(outs)]
    if op == "substep":
        return [s["path"].compact_attention(i, q, kc, vc) for i, (q, kc, vc) in enumerate(s["calls"])]
    if op == "probe":
        outs = [s["path"].probe(i, q, kc, vc) for i, (q, kc, vc) in enumerate(s["calls"])]
        return [(o, s["path"].probe_mass[i]) for i, o in enumerate(outs)]
    if op == "prefill":
        outs = [s["path"].prefill_chunk(i, q, kc, vc, want_mass=True) for i, (q, kc, vc) in enumerate(s["calls"])]
        return [(o, s["path"].chunk_mass[i]) for i, o in enumerate(outs)]
    if op == "keep":
        n = case["n"]
        score = torch.stack([value_score(s["mass"][i], s["cache"].v_fp[i, :, :, :n]) for i in range(case["layers"])])
        keep = s["state"].survivors(s["cfg"], case["keep"], None, score, check=False)
        cache = copy.copy(s["cache"])        # the compaction writes new planes and leaves these
        cache.compact(keep)
        cache.begin_append(BLOCK)
        for i, (k, v) in enumerate(s["block"]):
            cache.stage_layer(i, k, v)
        cache.commit_append()
        return [score, keep, _planes(cache)]
    if op == "lookahead":
        score = lookahead_scores(s["cache"], s["state"], s["mass"], s["probe"])
        keep = s["state"].survivors(s["cfg"], case["keep"], None, score, check=False)
        return [score, keep]
    if op == "evict":
        cache = copy.copy(s["cache"])        # the rebuild writes new planes and leaves these
        groups, encode, stage = rebuild_plan(s["phys"], s["pos"], case["keep"], quantized_length=cache.quantized_length,
                                             need=GROUP // 2, tail_groups=0, window=case["window"])
        remap = cache.rebuild(groups, encode, groups[..., :0], stage)
        return [remap, _planes(cache)]
    cache = s["cache"]
    cache.reset()
    cache.load_dynamic_cache(s["prompt"])
    for block in s["blocks"]:
        cache.begin_append(BLOCK)
        for i, (k, v) in enumerate(block):
            cache.stage_layer(i, k, v)
        cache.commit_append()
    return _planes(cache)


# ------------------------------------------------------------------ what a pass cannot do without
def _stored(case, n):
    """Bytes of K and V of n stored tokens of one KV head (codes with f16 scale and zero, or 16-bit)."""
    d = case["d"]
    if case.get("kv", "int4") != "int4":
        return 4 * d * n
    nq = _quantized(n)
    return nq * (d + 4 * d // GROUP * 2) + 4 * d * (n - nq)


def work(case):
    op, L, d = case["op"], case["layers"], case["d"]
    if op in ("step0", "substep", "probe", "prefill"):
        hq, hkv, t, b = case["hq"], case["hkv"], case["t"], case.get("b", 1)
        n = case["k"] if op == "substep" else case["n"]
        prefix = 4 * d * n if op == "substep" else _stored(case, n) + (n if case.get("dead") else 0)
        io = b * (2 * 2 * hq * t * d + hkv * (prefix + 2 * 2 * t * d))
        flops = 4.0 * b * hq * t * d * (n + t)
        if op == "step0":
            k, rows = case["k"], len(_rows(case))
            io += hkv * (4 * n + 8 * k + 4 * d * k)
            flops += 2.0 * hq * rows * d * n
        elif op == "probe":
            io += hkv * 4 * n
            flops += 2.0 * hq * (t - BLOCK) * d * n
        elif op == "prefill":
            io += hkv * 4 * n
            flops += 2.0 * hq * t * d * n
        return dict(bytes=L * io, flops=L * flops)
    lanes, n = L * case["hkv"], case["n"]
    if op == "load":
        m = n + BLOCK * case["blocks"]
        return dict(bytes=lanes * (4 * d * m + _stored(case, m)), flops=0)
    c = case["keep"]
    if op == "evict":
        return dict(bytes=lanes * (8 * c + 8 * n + 2 * _stored(case, c)), flops=0)
    if op == "lookahead":
        return dict(bytes=lanes * (n * (8 + 4 + 4) + _quantized(n) * (d // 2 + 4 * d // GROUP) + 2 * d * (n - _quantized(n))
                                   + 8 * c), flops=lanes * n * d * 5.0)
    return dict(bytes=lanes * (n * (4 + 4 + 2 * d) + 8 * c + 2 * 4 * d * c + 2 * 4 * d * BLOCK), flops=lanes * n * d * 5.0)


def tolerance(case):
    # scores, sets and bytes of the keep path follow a fixed rounding chain
    if case["op"] in ("keep", "lookahead", "evict", "load"):
        return "exact"
    # 16-bit outputs of sums over 16-bit products
    return {"rel": 1e-2, "max": 0.1, "differ": 1e-3}


# ------------------------------------------------------------------ the same in 64 bits
def _codec(x):
    """float64 values an int4 store holds for groups x [..., GROUP] (last axis): the affine
    rule in the arithmetic of x's dtype, scale and zero stored as float16."""
    lo, hi = x.amin(-1, keepdim=True), x.amax(-1, keepdim=True)
    step = ((hi - lo) / 15).clamp_min(1e-8)
    code = torch.round((x - lo) / step).clamp(0, 15)
    return code.double() * step.to(torch.float16).double() + lo.to(torch.float16).double()


def _held(case, k, v):
    """float64 keys and values as the cache holds them."""
    if case.get("kv", "int4") != "int4":
        return k.double(), v.double()
    nq = _quantized(k.shape[2])
    b, h, _, d = k.shape
    kq = _codec(k[:, :, :nq].reshape(b, h, nq // GROUP, GROUP, d).transpose(-1, -2)).transpose(-1, -2).reshape(b, h, nq, d)
    vq = _codec(v[:, :, :nq].reshape(b, h, nq, d // GROUP, GROUP)).reshape(b, h, nq, d)
    return torch.cat([kq, k[:, :, nq:].double()], 2), torch.cat([vq, v[:, :, nq:].double()], 2)


def _attend(q, k, v, kc, vc, live=None, causal=0, rows=None):
    """float64 attention over [k | kc] of one sequence; with rows (block positions) also the
    prefix mass of those rows and their mean prefix output: q [Hq, T, D], the rest [H, n, D]."""
    hq, t, d = q.shape
    h = k.shape[0]
    g = hq // h
    out, mass, centre = torch.empty((hq, t, d), dtype=torch.float64, device=q.device), [], []
    seen = None
    if causal:
        pos = torch.arange(t, device=q.device) // causal
        seen = pos[None, :] <= pos[:, None]
    for i in range(h):
        for j in range(g):      # one query head at a time: no large temporary
            qi = q[i * g + j].double()
            s = torch.mm(qi, k[i].t().contiguous()) * d ** -0.5
            if live is not None:
                s.masked_fill_(~live[i].bool()[None, :], -math.inf)
            sc = torch.mm(qi, kc[i].double().t().contiguous()) * d ** -0.5
            if seen is not None:
                sc.masked_fill_(~seen, -math.inf)
            out[i * g + j] = torch.mm(torch.softmax(torch.cat([s, sc], 1), 1), torch.cat([v[i], vc[i].double()]))
            if rows is not None:
                p = torch.softmax(s[rows], 1)
                a, c = p.sum(0), torch.mm(p, v[i]).sum(0)
                if j == 0:
                    mass.append(a)
                    centre.append(c)
                else:
                    mass[i] += a
                    centre[i] += c
    if rows is None:
        return out, None, None
    m = g * len(rows)
    return out, torch.stack(mass) / m, torch.stack(centre) / m


def _distance_score(a, v):
    """a_j * ||v_j - c|| with c the a-weighted mean of v."""
    c = (a.unsqueeze(-1) * v).sum(-2, keepdim=True) / a.sum(-1).clamp_min(1e-12)[..., None, None]
    return a * (v - c).norm(dim=-1)


def exact(case, seed):
    op = case["op"]
    if op in ("evict", "load"):
        return None          # codes, copies and indices: compared as whole values
    x = _inputs(case, seed)
    if op == "substep":
        return [torch.stack([_attend(q[b], k[b].double(), v[b].double(), kc[b], vc[b])[0] for b in range(case["b"])])
                for q, k, v, kc, vc in x["layers"]]
    if op in ("step0", "probe", "prefill"):
        res = []
        for (q, k, v, kc, vc), live in zip(x["layers"], x["live"]):
            kd, vd = _held(case, k, v)
            causal = 0 if op == "step0" else BLOCK
            t = case["t"]
            rows = _rows(case) if op == "step0" else list(range(BLOCK, t)) if op == "probe" else list(range(t))
            out, mass, centre = _attend(q[0], kd[0], vd[0], kc[0], vc[0], None if live is None else live[0], causal, rows)
            if op == "step0":
                rank = mass * (vd[0] - centre[:, None, :]).norm(dim=-1)
                at = rank.topk(case["k"], dim=-1).indices.sort(dim=-1).values[None, :, :, None].expand(-1, -1, -1, case["d"])
                res.append((out[None], mass[None], None, kd.gather(2, at), vd.gather(2, at)))
            else:
                res.append((out[None], mass[None] * ((t - BLOCK) // BLOCK if op == "probe" else 1)))
        return res
    if op == "keep":
        return [torch.stack([_distance_score(x["mass"][i].double(), v.double()) for i, (_, v) in enumerate(x["kv"])]),
                None, None]
    scores = []
    for i, (k, v) in enumerate(x["kv"]):
        a = (x["mass"][i] + x["probe"][i]).double()
        scores.append(_distance_score(a, _held(case, k, v)[1]))
    return [torch.stack(scores), None]

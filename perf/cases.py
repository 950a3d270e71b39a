"""The work that programs give this package, as cases that can be timed and compared.

A case names one call of a public entry point and its sizes. Three kinds of program stand behind them: a serving engine that
runs a routed-expert layer step by step (`moe.forward` with its mailbox and salience, a lone layer call, a lone projection),
a checker or exporter that wants an expert's dense weights (`moe.dense_W`), and a quantiser (`encode`).
"""
import math
import types

import torch

from nestquant_amd import encode, moe, salience

DEV = "cuda"


# ---- the layer's shape in full: 256 experts of 6144 x 2048, 8 picks per token, 26 experts at level 4, 51 at 3 or 4, the rest at 2
FULL = dict(H=6144, I=2048, E=256, topk=8, Bmax=4, levels="mixed")


def listed():
    return [
        # one user generating: a bf16 hidden state, fp32 router weights and int32 ids, as a serving engine hands them over
        dict(name="step_1_token", kind="step", T=1, routing="softmax", x="bf16", w="fp32", ids="int32", **FULL),
        # a few users generating together: the largest step that is one decode call
        dict(name="step_4_tokens", kind="step", T=4, routing="softmax", x="bf16", w="fp32", ids="int32", **FULL),
        # a busy server's generating step, and a short prompt of a ragged length: between the decode call and the long prompts
        dict(name="step_48_tokens", kind="step", T=48, routing="softmax", x="bf16", w="fp32", ids="int32", **FULL),
        dict(name="step_201_tokens", kind="step", T=201, routing="zipf", x="bf16", w="fp16", ids="int64", **FULL),
        # prompts: a ragged one over the mixed levels, and the long one with every expert at level 4 and skewed popularity
        dict(name="prompt_1003_tokens", kind="step", T=1003, routing="softmax", x="bf16", w="fp32", ids="int32", **FULL),
        dict(name="prompt_4096_tokens", kind="step", T=4096, routing="zipf", x="fp16", w="fp16", ids="int64", **dict(FULL, levels="all4")),
        # a small layer, where launches and host work are what counts
        dict(name="small_layer_2_tokens", kind="layer", T=2, H=512, I=256, E=12, topk=4, Bmax=4, levels="mixed", routing="softmax",
             x="fp16", w="fp16", ids="int64"),
        # one expert's gate|up projection for eight tokens
        dict(name="projection_8_tokens", kind="projection", T=8, H=6144, I=2048, level=3, x="fp16"),
        # an expert's dense weights, for an export or a check against another implementation
        dict(name="dense_gate_up", kind="dense", H=6144, I=2048, proj=0, level=4),
        # a quantiser: the base plane of one weight, base plane + both refinement planes, and a fit that knows its inputs
        dict(name="encode_base", kind="encode_level2", N=512, K=256, sign_seed=0),
        dict(name="encode_nested", kind="encode_nested", N=256, K=384, sign_seed=0, var=False, interleave=False),
        dict(name="encode_with_hessian", kind="encode_ldlq", N=128, K=256, sign_seed=0, var=True),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "between", "between", "prompt", "prompt", "layer", "projection", "dense", "encode"])
    big = rng.random() < 0.5
    H, I = (6144, 2048) if big else (128 * rng.randint(4, 48), 128 * rng.randint(2, 16))
    E = 256 if big else _log(rng, 16, 256)
    topk = 8 if big else rng.choice([2, 4, 6, 8])
    dt = dict(x=rng.choice(["bf16", "bf16", "fp16", "fp32"]), w=rng.choice(["fp32", "fp16", "bf16"]), ids=rng.choice(["int32", "int64"]),
              levels=rng.choice(["mixed", "mixed", "all2", "all3", "all4"]), routing=rng.choice(["softmax", "zipf"]))
    if kind == "decode":
        return dict(kind="step", T=rng.randint(1, 8), H=H, I=I, E=E, topk=topk, Bmax=rng.choice([4, 8]), **dt)
    if kind == "between":
        return dict(kind="step", T=_log(rng, 9, 383), H=H, I=I, E=E, topk=topk, Bmax=rng.choice([4, 8]), **dt)
    if kind == "prompt":
        return dict(kind="step", T=_log(rng, 384, 4096), H=H, I=I, E=E, topk=topk, Bmax=4, **dt)
    if kind == "layer":
        return dict(dt, kind="layer", T=rng.randint(1, 4), H=128 * rng.randint(2, 12), I=128 * rng.randint(1, 6), E=rng.randint(8, 32),
                    topk=rng.choice([2, 4, 8]), Bmax=4)
    if kind == "projection":
        return dict(kind="projection", T=rng.randint(1, 8), H=H, I=I, level=rng.choice([2, 3, 4]), x=dt["x"])
    if kind == "dense":
        return dict(kind="dense", H=H, I=I, proj=rng.randint(0, 1), level=rng.choice([2, 3, 4]))
    fn = rng.choice(["encode_level2", "encode_level2", "encode_nested", "encode_ldlq"])
    N, K = 128 * rng.randint(1, 4), 128 * rng.randint(1, 4)
    most = {"encode_level2": 8, "encode_nested": 4, "encode_ldlq": 3}[fn]            # blocks of 128 x 128: the slowest of these stays below a second or two
    while N * K > most * 128 * 128:
        N, K = (N - 128, K) if N >= K else (N, K - 128)
    c = dict(kind=fn, N=N, K=K, sign_seed=rng.randint(0, 1 << 20))
    if fn != "encode_level2":
        c["var"] = rng.random() < 0.5                            # the sign variant of the base plane
    if fn == "encode_nested":
        c["interleave"] = rng.random() < 0.5                     # the second one-bit plane of the nested level 4
    return c


# ---- inputs --------------------------------------------------------------------------------------------------------------
_F = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}
_I = {"int32": torch.int32, "int64": torch.int64}


def _levels(case, g):
    """the experts' levels: a tenth at level 4, two tenths at 3 or 4, the rest at 2 (or all at one level), placed by the seed"""
    E = case["E"]
    if case["levels"] != "mixed":
        return [int(case["levels"][3])] * E
    perm = torch.randperm(E, generator=g).tolist()
    pick = torch.randint(3, 5, (E,), generator=g).tolist()
    n4, nf = round(E * 26 / 256), round(E * 51 / 256)
    lv = [2] * E
    for i, e in enumerate(perm):
        lv[e] = 4 if i < n4 else pick[i] if i < n4 + nf else 2
    return lv


def _experts(H, I, E, seed):
    """E experts with random planes, each plane a view of one allocation per kind, as a loader that fills a pool has them: codes
    uniform, block words as the quantiser finds them (step size N / Mb between 0 and 0.8), signs with the scale of 1 / sqrt(inputs)"""
    g = torch.Generator(device=DEV).manual_seed(seed)
    word = lambda n: torch.randint(-2**31, 2**31 - 1, (E, n), generator=g, dtype=torch.int32, device=DEV)
    sign = lambda n, s: (torch.randint(0, 2, (E, n), generator=g, device=DEV) * 2 - 1).half() * s

    def block_words(n):
        Mb = torch.randint(120, 256, (E, n), generator=g, device=DEV)
        N = torch.minimum((torch.rand(E, n, generator=g, device=DEV) * 0.8 * Mb).round().long(), 257 - Mb)
        return (Mb | (N << 8)).to(torch.int32)
    planes = []
    for N, K in ((2 * I, H), (H, I)):
        units = (N // 16) * (K // 128)
        planes.append((word(units * 128), word(units * 128), block_words(units), block_words(units)))
    signs = torch.cat([sign(H, 1), sign(2 * I, H**-0.5), sign(I, 1), sign(H, I**-0.5), sign(H, 1)], 1).contiguous()
    ex = []
    for e in range(E):
        gu, dn = (types.SimpleNamespace(base=b[e], slot=r[e], d3=d3[e], d4n=d4[e], var=None, flags=None, bk=0, rk=0, nested=True)
                  for b, r, d3, d4 in planes)
        ex.append(types.SimpleNamespace(gu=gu, dn=dn, signs=signs[e], H=H, I=I, nested=True, lr=None))
    return ex


def _routing(case, g):
    """(ids [T, topk] distinct per token, weights summing to 1): a softmax router over N(0, 1) logits, or Zipf(1.1) popularity"""
    T, E, k = case["T"], case["E"], case["topk"]
    u = torch.rand(T, E, generator=g).clamp_(1e-9, 1 - 1e-7)
    if case["routing"] == "zipf":
        pop = -1.1 * torch.log(1.0 + torch.randperm(E, generator=g).float())
        score = pop - torch.log(-torch.log(u))                   # Gumbel top-k: picks without replacement by popularity
    else:
        score = torch.randn(T, E, generator=g)
    top, ids = torch.topk(score, k, dim=-1)
    return ids.to(_I[case["ids"]]).to(DEV), torch.softmax(top, -1).to(_F[case["w"]]).to(DEV)


def prepare(case, seed):
    g = torch.Generator().manual_seed(seed)
    kind = case["kind"]
    if kind.startswith("encode"):
        N, K = case["N"], case["K"]
        st = dict(kind=kind, W=torch.randn(N, K, generator=g).to(DEV), opt=dict(seed=case["sign_seed"]))
        st["opt"].update({k: case[k] for k in ("var", "interleave") if k in case})
        if kind == "encode_ldlq":                                # second moment of correlated inputs with a decaying spectrum
            X = torch.randn(4 * K, K, generator=g) * (1 + torch.arange(K)) ** -0.25
            X = X @ torch.linalg.qr(torch.randn(K, K, generator=g))[0]
            st["Hess"] = (X.T @ X / (4 * K)).to(DEV)
        return st
    H, I = case["H"], case["I"]
    if kind == "dense":
        return dict(kind=kind, ex=_experts(H, I, 1, seed)[0], proj=case["proj"], level=case["level"])
    x = torch.randn(case["T"], H, generator=g).to(DEV).to(_F[case["x"]])
    if kind == "projection":
        L = moe.MoELayer(1, H, I, Bmax=8, topk=1, dev=DEV)
        ex = _experts(H, I, 1, seed)
        L.set(0, ex[0], case["level"])
        return dict(kind=kind, layer=L, ex=ex, x=x)
    L = moe.MoELayer(case["E"], H, I, Bmax=case["Bmax"], topk=case["topk"], dev=DEV)
    ex = _experts(H, I, case["E"], seed)
    for e, lv in enumerate(_levels(case, g)):
        L.set(e, ex[e], lv)
    ids, w = _routing(case, g)
    st = dict(kind=kind, layer=L, ex=ex, x=x, ids=ids, w=w)
    if kind == "step":
        st["mailbox"], st["sal"] = moe.Mailbox(L), salience.Salience(case["E"], dev=DEV)
    return st


_PLANES = ("su", "sv", "base", "var", "p3", "d3", "p4", "d4", "p4n", "d4n", "Q", "Q3", "Q4", "Q4n")


def run(state):
    s, kind = state, state["kind"]
    if kind == "step":
        return moe.forward(s["layer"], s["mailbox"], s["x"], s["w"], s["ids"], sal=s["sal"])
    if kind == "layer":
        return s["layer"](s["x"], s["ids"], s["w"])
    if kind == "projection":
        return moe.proj_gemv(s["layer"], s["x"])
    if kind == "dense":
        return moe.dense_W(s["ex"], s["proj"], s["level"])
    if kind == "encode_level2":
        r = encode.encode_level2(s["W"], **s["opt"])
    elif kind == "encode_nested":
        r = encode.encode_nested(s["W"], **s["opt"])
    else:
        r = encode.encode_ldlq(s["W"], s["Hess"], **s["opt"])
    return {k: r[k] for k in _PLANES if r.get(k) is not None}


# ---- what a pass cannot do without ---------------------------------------------------------------------------------------
_UNIT = {2: 512, 3: 512 + 256 + 4, 4: 512 + 512 + 4}             # bytes of a unit of 16 x 128 weights at each level


def work(case):
    kind = case["kind"]
    if kind.startswith("encode"):
        N, K = case["N"], case["K"]
        fits = {"encode_level2": 1}.get(kind, 3) + int(case.get("var", False))
        # every fit: per 256-weight ring two passes of 256 steps over 65536 states, each a difference, a square, a sum, a minimum
        return {"bytes": N * K * 4 * (1 + fits) + N * K // 4 * (1 if kind == "encode_level2" else 2.5), "flops": fits * (N * K // 256) * 2 * 256 * 65536 * 4}
    H, I = case["H"], case["I"]
    size = {"fp16": 2, "bf16": 2, "fp32": 4}
    if kind == "dense":
        units = (2 * I // 16) * (H // 128) if case["proj"] == 0 else (H // 16) * (I // 128)
        return {"bytes": units * (_UNIT[case["level"]] + 4096), "flops": 0}
    T = case["T"]
    if kind == "projection":
        return {"bytes": (2 * I // 16) * (H // 128) * _UNIT[case["level"]] + T * (H * size[case["x"]] + 2 * I * 4), "flops": 2 * T * 2 * I * H}
    E, k = case["E"], case["topk"]
    if case["routing"] == "zipf":                                # expected number of distinct experts (picks taken as independent)
        p = [(1 + r) ** -1.1 for r in range(E)]
        tot = sum(p)
        distinct = sum(1 - (1 - min(1.0, k * v / tot)) ** T for v in p)
    else:
        distinct = E * (1 - (1 - k / E) ** T)
    unit = _UNIT[int(case["levels"][3])] if case["levels"] != "mixed" else 0.70 * _UNIT[2] + 0.10 * _UNIT[3] + 0.20 * _UNIT[4]
    out = size[case["x"]] if kind == "step" else 4
    return {"bytes": distinct * (3 * H * I // 2048) * unit + T * H * (size[case["x"]] + out), "flops": 2 * T * k * 3 * H * I}


def tolerance(case):
    kind = case["kind"]
    if kind in ("dense", "encode_level2"):
        return "exact"
    if kind.startswith("encode"):
        # sums in another order can tip a block word or, rarely, a ring's path between two of equal cost
        return {"rel": 1e-3, "max": 0.9, "differ": 2e-3}
    if kind == "projection":
        return {"rel": 2e-5}                                     # fp16 products, fp32 sums
    if kind == "step" and case["x"] != "fp32":
        return {"rel": 2e-3, "max": 2e-2}                        # the result is rounded to the activations' 16-bit type
    return {"rel": 2e-4}                                         # fp32 sums around two roundings of the activations to fp16

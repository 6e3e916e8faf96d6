"""The MoE work that this library is measured on: what a user's program calls, at the sizes it calls it with.

Three kinds of pass, each through the public entry points of tinystrata_amd:
  layer  a stack of MoE layers (moe.MoELayer): router top-k, grouping or sort, Q8_1 activations, the expert products,
         the shared expert and the router-weighted combine.  Every layer has weights and hidden rows of its own, so
         that the experts stream from HBM as they do in a model.
  ids    a stack of layers by the id-indexed products (ops.mmvq_ids), the route of models whose experts are Q4_0 or
         Q6_K: router, Q8_1, gate and up rows of the picked experts, SwiGLU, down rows, combine.
  dense  single matrices times a few Q8_1 columns (ops.iq_mmvq): the dense projections beside the experts.
Decode passes and small batches are replayed from a HIP graph, as a serving loop replays its step; prompt chunks are
called eagerly.  Expert weights are N(0, 0.02) rows quantized by the library's host quantizer (Q4_0 and Q6_K, which it
has no quantizer for: random codes with finite scales); every expert takes its rows from a pool of quantized rows in
an order of its own.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

from tinystrata_amd import moe, ops

Q4_0, Q8_0, Q4_K, Q6_K, IQ3_XXS, IQ3_S = 2, 8, 12, 14, 18, 21
BLOCK = {Q4_0: (32, 18), Q8_0: (32, 34), Q4_K: (256, 144), Q6_K: (256, 210), IQ3_XXS: (256, 98), IQ3_S: (256, 110)}
TYPES = {"q4_0": Q4_0, "q8_0": Q8_0, "q4_k": Q4_K, "q6_k": Q6_K, "iq3_xxs": IQ3_XXS, "iq3_s": IQ3_S}
POOL_ROWS = 1024
DEV = "cuda"


def _case(name, kind="layer", gu="iq3_xxs", down="iq3_s", n=2048, ff=512, experts=256, k=8, shared=False, tokens=1,
          layers=1, route="normal", outliers=False, norm=False, graph=False):
    c = dict(kind=kind, gu=gu, down=down, n=n, ff=ff, experts=experts, k=k, shared=shared, tokens=tokens,
             layers=layers, route=route, outliers=outliers, norm=norm, graph=graph)
    return {"name": name, **c} if name else c


def listed():
    iq3 = dict(gu="iq3_xxs", down="iq3_s", ff=512, experts=256, shared=True)
    q4k = dict(gu="q4_k", down="q4_k", ff=768, experts=128)
    q80 = dict(gu="q8_0", down="q8_0", ff=768, experts=128)
    return [
        # one sequence decoding: one token per step through the layers of a 256-expert model with a shared expert
        _case("decode1_iq3", tokens=1, layers=16, graph=True, **iq3),
        # the same on the 128-expert model in 8 bits
        _case("decode1_q8_0", tokens=1, layers=8, graph=True, **q80),
        # speculative decoding: four draft tokens verified at once, their picks correlated
        _case("verify4_iq3", tokens=4, layers=8, route="correlated", graph=True, **iq3),
        # eight sequences decoding together, each layer ending with the next one's norm and its Q8_1 image
        _case("batch8_q4_k", tokens=8, layers=4, norm=True, graph=True, **q4k),
        # a serving batch: 32 sequences decoding together, about one token per expert
        _case("batch32_iq3", tokens=32, layers=4, graph=True, **iq3),
        # a short prompt (or a batch of 60 sequences) on the 8-bit model, a few tokens per expert
        _case("chunk60_q8_0", tokens=60, layers=2, graph=True, **q80),
        # a prompt chunk with skewed routing
        _case("chunk512_q4_k", tokens=512, route="zipf1.1", **q4k),
        # the ragged last chunk of a prompt, its layer ending with the norm
        _case("chunk777_q8_0", tokens=777, route="zipf1.1", norm=True, **q80),
        # a long prompt's chunk with skewed routing and outlier channels
        _case("chunk4096_iq3", tokens=4096, route="zipf1.3", outliers=True, **iq3),
        # a model of few wide experts, two tokens: beyond what the fused decode layer takes
        _case("wide2_q4_k", gu="q4_k", down="q4_k", n=4096, ff=1536, experts=64, k=4, tokens=2, layers=4, graph=True),
        # a model with small-format experts, one token per step, by the id-indexed products
        _case("ids1_q6_k", kind="ids", gu="q4_0", down="q6_k", n=2048, ff=1792, experts=64, k=4, tokens=1, layers=8,
              graph=True),
        # dense projections of a decode step of four tokens: one column block per matrix
        _case("dense4_q6_k", kind="dense", gu="q6_k", down="q6_k", n=2048, ff=6144, experts=1, k=1, tokens=4,
              layers=8, graph=True),
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["layer"] * 6 + ["ids", "dense"])
    n = rng.choice([1024, 1536, 2048, 2048, 2560, 4096])
    if kind == "dense":
        t = rng.choice(["q4_0", "q8_0", "q4_k", "q6_k", "iq3_xxs", "iq3_s"])
        return _case(None, kind, t, t, n=n, ff=log_int(500, 12000), experts=1, k=1, tokens=rng.randint(1, 8), layers=4,
                     graph=True)
    if kind == "ids":
        gu, down = rng.choice([("q4_0", "q4_0"), ("q4_0", "q6_k"), ("q6_k", "q6_k"), ("q4_k", "q6_k")])
        return _case(None, kind, gu, down, n=n, ff=rng.choice([768, 1280, 1792]), experts=64,
                     k=rng.choice([2, 4, 6]), tokens=rng.randint(1, 4), layers=4, graph=True)
    gu, down = rng.choice([("iq3_xxs", "iq3_s"), ("iq3_xxs", "iq3_s"), ("q4_k", "q4_k"), ("q8_0", "q8_0"),
                           ("iq3_s", "iq3_s"), ("q4_k", "q8_0")])
    ff = rng.choice([256, 512, 512, 768, 768, 1024] + ([704] if (gu, down) == ("q8_0", "q8_0") else []))
    # the sizes that the fused decode layer takes: its row chunks have to fit their share of the LDS
    n = min(n, 2048 if gu in ("q8_0", "iq3_s") else 2560 if ff > 512 else n)
    k, shared = rng.choice([4, 6, 8]), rng.random() < 0.5
    # at most 1e11 operations: the 8-bit products then take about as long as the longest listed chunk
    tokens = log_int(1, min(3000, 1e11 / (6.0 * (k + 1) * n * ff)))
    graph = tokens <= 64
    layers = 4 if tokens <= 8 else 2 if graph else 1
    return _case(None, kind, gu, down, n=n, ff=ff, experts=rng.choice([64, 128, 192, 256]), k=k, shared=shared,
                 tokens=tokens, layers=layers,
                 route=rng.choice(["normal", "correlated"] if tokens <= 8 else ["normal", "zipf1.1", "zipf1.3"]),
                 outliers=rng.random() < 0.25, norm=rng.random() < 0.25, graph=graph)


# ---------------------------------------------------------------------------------------------------- inputs
@functools.lru_cache(maxsize=64)
def _pool(type_name: str, cols: int) -> torch.Tensor:
    """POOL_ROWS quantized rows of `cols` weights, uint8 [POOL_ROWS, row bytes] on the device."""
    t = TYPES[type_name]
    qk, nb = BLOCK[t]
    rng = np.random.default_rng(1000 * t + cols)
    if t in (Q4_0, Q6_K):
        b = rng.integers(0, 256, (POOL_ROWS, cols // qk, nb), dtype=np.uint8)
        lo, hi, at = (0.001, 0.006, 0) if t == Q4_0 else (0.0001, 0.0004, 208)
        b[..., at:at + 2] = rng.uniform(lo, hi, (POOL_ROWS, cols // qk)).astype(np.float16)[..., None].view(np.uint8)
        rows = b.reshape(POOL_ROWS, -1)
    else:
        rows = ops.quantize_weights(t, rng.normal(0, 0.02, (POOL_ROWS, cols)).astype(np.float32))
    return torch.from_numpy(np.ascontiguousarray(rows)).to(DEV)


def _take(pool, pick):
    """pool[pick] by the widest words that a row is made of."""
    word = torch.int64 if pool.shape[1] % 8 == 0 else torch.int32 if pool.shape[1] % 4 == 0 else torch.int16
    return pool.view(word).index_select(0, pick).view(torch.uint8)


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _sizes(c):
    qk, nb = BLOCK[TYPES[c["gu"]]]
    dqk, dnb = BLOCK[TYPES[c["down"]]]
    gu_row, d_row = c["n"] // qk * nb, c["ff"] // dqk * dnb
    up = c["ff"] * gu_row
    total = 2 * up + c["n"] * d_row
    return gu_row, d_row, up, 2 * up, total, (total + 255) // 256 * 256


def _blobs(c, count, g):
    """`count` expert blobs [gate rows | up rows | down rows], uint8 [count, stride]."""
    gu_row, d_row, up, down, total, stride = _sizes(c)
    out = torch.zeros((count, stride), dtype=torch.uint8, device=DEV)
    pick = torch.randint(POOL_ROWS, (count * 2 * c["ff"],), generator=g, device=DEV)
    out[:, :down] = _take(_pool(c["gu"], c["n"]), pick).view(count, -1)
    pick = torch.randint(POOL_ROWS, (count * c["n"],), generator=g, device=DEV)
    out[:, down:total] = _take(_pool(c["down"], c["ff"]), pick).view(count, -1)
    return out


def _logits(c, g, layers):
    E, T = c["experts"], c["tokens"]

    def normal(*shape):
        return torch.randn(shape, generator=g, device=DEV)

    if c["route"] == "correlated":
        return normal(layers, 1, E) + 0.5 * normal(layers, T, E)
    z = normal(layers, T, E)
    if c["route"].startswith("zipf"):
        rank = torch.argsort(torch.rand((layers, 1, E), generator=g, device=DEV), dim=-1)
        z = z - float(c["route"][4:]) * torch.log(1.0 + rank)
    return z.contiguous()


def _inputs(c, seed):
    """What run() and exact() start from: weights, hidden rows, router logits, gates and norm weights."""
    g = _gen(seed)
    Ly, T, N, FF, E = c["layers"], c["tokens"], c["n"], c["ff"], c["experts"]
    s = {}
    if c["kind"] == "dense":
        pool = _pool(c["gu"], N)
        s["w"] = [_take(pool, torch.randint(POOL_ROWS, (FF,), generator=g, device=DEV)).reshape(-1) for _ in range(Ly)]
    else:
        s["blobs"] = [_blobs(c, E, g) for _ in range(Ly)]
        s["shared"] = [_blobs(c, 1, g)[0] if c["shared"] else None for _ in range(Ly)]
        s["logits"] = _logits(c, g, Ly)
        s["sgate"] = torch.randn((Ly, T), generator=g, device=DEV) if c["shared"] else None
    s["x"] = torch.randn((Ly, T, N), generator=g, device=DEV)
    if c["outliers"]:
        s["x"][..., torch.randperm(N, generator=g, device=DEV)[:N // 100]] *= 20.0
    s["norm_w"] = 1.0 + 0.1 * torch.randn((Ly, N), generator=g, device=DEV) if c["norm"] else None
    return s


# ---------------------------------------------------------------------------------------------------- the passes
EPS = 1e-6


def prepare(case, seed):
    s = _inputs(case, seed)
    c = s["case"] = case
    Ly, T, N, FF, E, k = c["layers"], c["tokens"], c["n"], c["ff"], c["experts"], c["k"]
    f32, i32, u8 = torch.float32, torch.int32, torch.uint8
    dev = torch.device(DEV, torch.cuda.current_device())
    if c["kind"] == "dense":
        s["xq"] = torch.empty((Ly, T, N // 32 * 36), dtype=u8, device=dev)
        s["y"] = torch.empty((Ly, T, FF), dtype=f32, device=dev)
    else:
        s["y"] = torch.empty((Ly, T, N), dtype=f32, device=dev)
        if c["norm"]:
            s["h"] = torch.empty((Ly, T, N), dtype=f32, device=dev)
            s["hq"] = torch.empty((Ly, T, N // 32 * 36), dtype=u8, device=dev)
    if c["kind"] == "layer":
        L = ops.native_expert_layout(TYPES[c["gu"]], TYPES[c["down"]], N, FF)
        s["layers"] = []
        for l in range(Ly):
            W = moe.MoEWeights(L=L, n_expert=E, stride=s["blobs"][l].shape[1], blobs=s["blobs"][l].view(-1),
                               shared=s["shared"][l])
            s["layers"].append(moe.MoELayer(W, k, T, dev))
    elif c["kind"] == "ids":
        s["table"] = [b.data_ptr() + b.shape[1] * torch.arange(E, dtype=torch.int64, device=dev) for b in s["blobs"]]
        s["ids"] = torch.empty((Ly, T, k), dtype=i32, device=dev)
        s["wts"] = torch.empty((Ly, T, k), dtype=f32, device=dev)
        s["xq"] = torch.empty((T, N // 32 * 36), dtype=u8, device=dev)
        s["gate"], s["up"] = (torch.empty((T * k, FF), dtype=f32, device=dev) for _ in range(2))
        s["hq1"] = torch.empty((T * k, FF // 32 * 36), dtype=u8, device=dev)
        s["parts"] = torch.empty((T * k, N), dtype=f32, device=dev)
    s["graph"] = None
    if c["graph"]:
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            _pass(s)
        torch.cuda.current_stream().wait_stream(side)
        s["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s["graph"]):
            _pass(s)
    return s


def _pass(s):
    c = s["case"]
    T, N, FF, k = c["tokens"], c["n"], c["ff"], c["k"]
    if c["kind"] == "dense":
        for l in range(c["layers"]):
            ops.quantize_q8_1_rows(s["x"][l], s["xq"][l])
            ops.iq_mmvq(TYPES[c["gu"]], s["w"][l], s["xq"][l], N, FF, T, y=s["y"][l])
        return
    s["y"].zero_()
    if c["kind"] == "layer":
        for l, layer in enumerate(s["layers"]):
            sgate = s["sgate"][l] if c["shared"] else None
            if c["norm"]:
                layer(s["x"][l], s["logits"][l], sgate, s["y"][l], norm_w=s["norm_w"][l], eps=EPS, h=s["h"][l],
                      hq=s["hq"][l])
            else:
                layer(s["x"][l], s["logits"][l], sgate, s["y"][l])
        return
    _, _, up, down, _, _ = _sizes(c)
    for l in range(c["layers"]):
        ops.native_router_topk(s["logits"][l], k, s["ids"][l], s["wts"][l])
        ops.quantize_q8_1_rows(s["x"][l], s["xq"])
        for off, out in ((0, s["gate"]), (up, s["up"])):
            ops.mmvq_ids(TYPES[c["gu"]], s["table"][l], s["ids"][l], off, s["xq"], s["xq"].shape[1], k, out, FF, T * k,
                         N, FF)
        ops.native_swiglu_quantize_q8_1(s["gate"], s["up"], s["hq1"])
        ops.mmvq_ids(TYPES[c["down"]], s["table"][l], s["ids"][l], down, s["hq1"], s["hq1"].shape[1], 1, s["parts"], N,
                     T * k, FF, N)
        ops.moe_combine(s["y"][l], s["parts"], s["wts"][l], k)


def run(state):
    if state["graph"] is not None:
        state["graph"].replay()
    else:
        _pass(state)
    c = state["case"]
    out = {"y": state["y"]}
    if c["kind"] == "layer":
        out["ids"] = [layer.ids for layer in state["layers"]]
        out["wts"] = [layer.wts for layer in state["layers"]]
        if c["norm"]:
            out["h"], out["hq"] = state["h"], state["hq"]
    elif c["kind"] == "ids":
        out["ids"], out["wts"] = state["ids"], state["wts"]
    return out


@functools.lru_cache(maxsize=256)
def _distinct(experts, k, tokens, route):
    """Distinct experts that a layer's tokens pick (one routing of a fixed seed)."""
    rng = np.random.default_rng(0)
    z = rng.normal(0, 1, (tokens, experts))
    if route == "correlated":
        z = rng.normal(0, 1, (1, experts)) + 0.5 * z
    elif route.startswith("zipf"):
        z = z - float(route[4:]) * np.log(1.0 + rng.permutation(experts))
    return len(np.unique(np.argpartition(-z, k - 1, axis=1)[:, :k]))


def work(case):
    c = case
    T, N, FF, E, k = c["tokens"], c["n"], c["ff"], c["experts"], c["k"]
    if c["kind"] == "dense":
        qk, nb = BLOCK[TYPES[c["gu"]]]
        by = FF * (N // qk) * nb + 4 * T * (N + FF)
        return {"bytes": c["layers"] * by, "flops": c["layers"] * 2 * T * N * FF}
    total = _sizes(c)[4]
    used = _distinct(E, k, T, c["route"]) + (1 if c["shared"] else 0)
    by = used * total + 4 * T * (N + E + N + 2 * k) + (4 * T if c["shared"] else 0)
    if c["norm"]:
        by += 4 * N + T * (4 * N + N // 32 * 36)
    rows = T * (k + (1 if c["shared"] else 0))
    return {"bytes": c["layers"] * by, "flops": c["layers"] * 2 * rows * 3 * N * FF}


def tolerance(case):
    # A dense product only sums exact integer blocks in another order: 0.8e-7 to 1.5e-7 between two such sums.  Behind
    # the SwiGLU the sums' last bits decide some Q8_1 codes of h that lie on a rounding edge; one such code moves a
    # token's output by up to 1e-3 of its norm (kernel by kernel against the fused layer, and each against 64 bits:
    # 1e-7 without a changed code, up to 5.8e-4 with some).  The norm's Q8_1 image has rounding edges of its own: up
    # to 1.3e-3 of its bytes differed.
    if case["kind"] == "dense":
        return {"rel": 6e-7}
    return {"rel": 2e-3, "differ": 5e-3} if case["norm"] else {"rel": 2e-3}


# ---------------------------------------------------------------------------------------------------- 64 bits
# The codebooks of IQ3_XXS and IQ3_S as the format defines them (ggml, MIT License, LICENSE-ggml): three hexadecimal
# digits per entry, four 3-bit level numbers, the first value's lowest; a level is 8 i + 4 (62 for 7) or 2 i + 1.
_IQ3_XXS_GRID = (
    "00000200400900b00f01001201902203b03d04104304804a05105505805a06106c07808008208408909009209909b09f0a90af0bd0c1"
    "0c70c80ca0d50f810b11f12412f13b13d14114715a16a19d1b41c81cc1ce1e31f120120320820a21121321821a21c227228240242249"
    "25025228128328828a2912982ba2c02c22d02d92e62f63013053283503543663793853d23e040040240940b410412416419422441443"
    "44544844a45145847347747848048248948f49049249f4a04ad4c14c84cc4f84fc51d52b54355756157c5c15c35ce5e560160860a611"
    "61362863563a6406426506596646666816836886956aa6ba6c96db71872773a74074675276d78c79e7b37db7f080480f81d81f82b82f"
    "87c89089f8a08b08b68c78e59049299349559639789c59c89ca9d8a0aa21a38a40a46a56a6da8ca9aabaac2aebb08b13b17b3ab42b59"
    "ba8bd4be2c14c24c26c34c51c71c8fcb4cd8cded24d45d6ad9bdc3dd1e03e05e07e08e1ae2ae56e60e8aea5eaaec0ecdedbef0f11f21"
    "f40f42f54f98"
)
_IQ3_S_GRID = (
    "00000100200500700800900a00c00e01001101501b02002202502702902b03003203903c03f04004104204404804904d050053057059"
    "05d06407107507a08008108508708808b08e09109509809c0a20a50a70a90ab0b80bb0c30c90cd0d00d20d90db0de0e40e80ea0f70f9"
    "0fd10010b10f11111411a12012312913814214415015215615b16116516717617b18618918b1991aa1b91c01c21c41d01d21d61db1e8"
    "1ec20020120220420820920b20d20f21021221921c21e22c22e23123a24024124324624824c25125825b26126826a27827e28028a28d"
    "28f29029429a2a02a32ad2b02ba2c12c42c72c82cb2d12d72d82dc2e12f22f830330530a30c31931b32232632832c34134834b351358"
    "35a3693903943973a43a63c13c33c83ca3d13dd3e13f23f840040140340540740840a40c40e41141341741841a42142342542842a437"
    "43843b43d44044244844b44f45245545945c46246948148448749149349849f4a14ab4af4b94bc4c04c24c54c94d24d44d94db4e24e8"
    "4f650150751051351a51d52153a53d54454955255f56056b5785805825875915ad5b15c55c95d65d85e35e860260960b60d60f612619"
    "61b61d62262462762963363964164364564c65165366067067a67e68068a69069a69c6a86c16c86cc6d16d36d76d86e16e36e76ed6fb"
    "70370970e71271972a73073474174874a75575a76476e77b78e7a17c17c37d07d27dd80080480a81081481781a821828838842847849"
    "84b85285885d86386986d88188388888d89189b8a08af8b28b88c48c98cb8d08d28d98dd90090291491f92093994594795197298b99c"
    "9b09c89cd9d89e39e9a02a08a0ca12a20a24a27a2aa36a3ca41a43a45a4aa51a5aa7aa80a89a93a98a9eaabac2ac7ac8ad7ae4ae9af5"
    "afbb01b04b10b1ab26b4ab56b69b6bba2bc2bc4bd2c09c0bc0dc19c1bc30c40c50c57c74c8ac9cca2cadcb2cb8cc0ccccd1ce0d15d23"
    "d32d40d43d5cd70d85da0dc9dcbe00e04e07e10e12e1ee20e2ce32e42e49e54e63e65e81e84e88e8ee91e98ea9ec2edaeddeebf01f05"
    "f0bf10f28f52f62f82f99fc0"
)


def _grid(text, xxs):
    code = torch.tensor([int(text[i:i + 3], 16) for i in range(0, len(text), 3)], device=DEV)
    lev = torch.stack([(code >> (3 * i)) & 7 for i in range(4)], dim=1)
    return (torch.where(lev == 7, 62, 8 * lev + 4) if xxs else 2 * lev + 1).double()


def _half(b):
    return b.contiguous().view(torch.float16).double()


def _bits(b, count):
    return (b.unsqueeze(-1) >> torch.arange(count, device=b.device)) & 1


def _dequantize(type_name, raw, rows, cols):
    """The rows' values in 64 bits, from the format's definition."""
    t = TYPES[type_name]
    qk, nb = BLOCK[t]
    b = raw.reshape(rows * (cols // qk), nb)
    n = b.shape[0]
    if t == Q8_0:
        v = _half(b[:, :2]) * b[:, 2:].contiguous().view(torch.int8).double()
    elif t == Q4_0:
        q = b[:, 2:].int()
        v = _half(b[:, :2]) * (torch.cat([q & 15, q >> 4], dim=1) - 8)
    elif t == Q6_K:
        ql, qh = b[:, :128].int().view(n, 2, 2, 32), b[:, 128:192].int().view(n, 2, 1, 32)
        low = torch.stack([ql[:, :, 0] & 15, ql[:, :, 1] & 15, ql[:, :, 0] >> 4, ql[:, :, 1] >> 4], dim=2)
        high = torch.cat([(qh >> (2 * i)) & 3 for i in range(4)], dim=2)
        sc = b[:, 192:208].contiguous().view(torch.int8).double().view(n, 2, 4, 2, 1)
        v = sc * ((low | high << 4) - 32).view(n, 2, 4, 2, 16) * _half(b[:, 208:210]).view(n, 1, 1, 1, 1)
    elif t == Q4_K:
        s = b[:, 4:16].int()
        sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | (s[:, 0:4] >> 6) << 4], dim=1).double()
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | (s[:, 4:8] >> 6) << 4], dim=1).double()
        q = b[:, 16:].int().view(n, 4, 32)
        q = torch.stack([q & 15, q >> 4], dim=2).view(n, 8, 32)
        v = (_half(b[:, :2]) * sc).unsqueeze(2) * q - (_half(b[:, 2:4]) * mn).unsqueeze(2)
    elif t == IQ3_XXS:
        aux = b[:, 66:98].contiguous().view(torch.int32).long() & 0xFFFFFFFF
        sg = (aux.unsqueeze(2) >> (7 * torch.arange(4, device=b.device))) & 127
        bit = _bits(sg, 7)
        bit = torch.cat([bit, bit.sum(-1, keepdim=True) & 1], dim=-1)
        v = _grid(_IQ3_XXS_GRID, True)[b[:, 2:66].long()].view(n, 8, 4, 8) * (1 - 2 * bit)
        v = v * (_half(b[:, :2]) * (2 * (aux >> 28) + 1) * 0.25).view(n, 8, 1, 1)
    else:
        idx = b[:, 2:66].long().view(n, 8, 8) | _bits(b[:, 66:74].long(), 8) << 8
        v = _grid(_IQ3_S_GRID, False)[idx].view(n, 8, 4, 8) * (1 - 2 * _bits(b[:, 74:106].long(), 8).view(n, 8, 4, 8))
        sc = torch.stack([b[:, 106:110].long() & 15, b[:, 106:110].long() >> 4], dim=2).view(n, 8)
        v = v * (_half(b[:, :2]) * (2 * sc + 1)).view(n, 8, 1, 1)
    return v.reshape(rows, cols).double()


def _q8_1(v, sums=False):
    """What the products see of v: Q8_1's codes times its scale (and Q4_0's block sums), the rule in v's own type."""
    b = v.reshape(*v.shape[:-1], -1, 32)
    d = b.abs().amax(-1, keepdim=True) / 127
    q = b / torch.where(d > 0, d, torch.ones_like(d))
    q = torch.sign(q) * torch.floor(q.abs() + 0.5)
    d16 = d.half().double()
    out = (q.double() * d16).reshape(v.shape)
    if not sums:
        return out
    return out, b.sum(-1).half().double(), d16[..., 0] * q.double().sum(-1)


def _times(type_name, w, raw, v):
    """The product's contract in 64 bits: w . Q8_1(v); Q4_0's offset of -8 multiplies the block's stored sum."""
    if TYPES[type_name] != Q4_0:
        return _q8_1(v) @ w.T
    a, stored, own = _q8_1(v, sums=True)
    dw = _half(raw.reshape(-1, 18)[:, :2]).view(w.shape[0], -1)
    return a @ w.T - 8.0 * (stored - own) @ dw.T


def _expert(c, blob, v):
    _, _, up, down, total, _ = _sizes(c)
    N, FF = c["n"], c["ff"]
    part = []
    for lo, hi in ((0, up), (up, down)):
        raw = blob[lo:hi]
        part.append(_times(c["gu"], _dequantize(c["gu"], raw, FF, N), raw, v))
    h = part[0] / (1 + torch.exp(-part[0])) * part[1]
    raw = blob[down:total]
    return _times(c["down"], _dequantize(c["down"], raw, N, FF), raw, h)


def exact(case, seed):
    c, s = case, _inputs(case, seed)
    Ly, T, N, k = c["layers"], c["tokens"], c["n"], c["k"]
    if c["kind"] == "dense":
        y = [_times(c["gu"], _dequantize(c["gu"], s["w"][l], c["ff"], N), s["w"][l], s["x"][l]) for l in range(Ly)]
        return {"y": torch.stack(y)}
    ys, wts, hs = [], [], []
    for l in range(Ly):
        p = torch.softmax(s["logits"][l].double(), dim=1)
        top, ids = torch.topk(p, k, dim=1)
        w = top / torch.clamp(top.sum(1, keepdim=True), min=2.0 ** -14)
        y = torch.zeros((T, N), dtype=torch.float64, device=DEV)
        for e in torch.unique(ids).tolist():
            t, j = torch.nonzero(ids == e, as_tuple=True)
            y[t] += w[t, j].unsqueeze(1) * _expert(c, s["blobs"][l][e], s["x"][l][t])
        if c["shared"]:
            y += torch.sigmoid(s["sgate"][l].double()).unsqueeze(1) * _expert(c, s["shared"][l], s["x"][l])
        ys.append(y)
        wts.append(w)
        if c["norm"]:
            hs.append(y / torch.sqrt((y * y).mean(1, keepdim=True) + EPS) * s["norm_w"][l].double())
    out = {"y": torch.stack(ys), "ids": [None] * Ly if c["kind"] == "layer" else None,
           "wts": wts if c["kind"] == "layer" else torch.stack(wts)}
    if c["norm"]:
        out["h"], out["hq"] = torch.stack(hs), None
    return out

"""A whole MoE layer on the GPU (tinystrata_amd.moe.MoELayer: routing, grouping, experts, shared expert, combine)
against the oracle's layer at the benchmark configurations (marked gpu).

Pass/fail: 1e-3 relative L2 against the oracle in Q8_1 mode (the GPU's activation contract).  The gap to the
reference CPU's own activation format (Q8_K for IQ3 / Q4_K, Q8_0 for Q8_0) is printed: ~2e-2 expected for IQ3 and
Q4_K, ~0 for Q8_0.  Full-size prompt chunks are checked on a sample of tokens: a token's output depends only on its
own input and routing, whatever other tokens share its experts.
"""
import numpy as np
import pytest
import torch

import oracle as O
from tinystrata_amd import moe, ops
from tinystrata_amd._lib import IQ3_S, IQ3_XXS, Q4_K, Q8_0

from gpu_util import dev, host, pool, rel_l2

pytestmark = pytest.mark.gpu

CONFIGS = {
    # name: (gu, d, N, FF, E, k, shared, T)
    "c1_decode_q8_0": (Q8_0, Q8_0, 2048, 768, 128, 8, False, 1),
    "c2_decode_iq3": (IQ3_XXS, IQ3_S, 2048, 512, 256, 8, True, 1),
    "c3_verify_iq3": (IQ3_XXS, IQ3_S, 2048, 512, 256, 8, True, 4),
    "c4_prefill_q4_k_32tok": (Q4_K, Q4_K, 2048, 768, 128, 8, False, 32),
    "c5_prefill_iq3_16tok": (IQ3_XXS, IQ3_S, 2048, 512, 256, 8, True, 16),
}


def make_layer(gu, d, N, FF, E, shared, distinct=8, seed=0):
    L = ops.native_expert_layout(gu, d, N, FF)
    p = pool(gu, d, N, FF, distinct, seed)
    order = (np.arange(E) * 5 + 3) % distinct
    W = moe.weights_from_pool(L, dev(p), E, order, (distinct - 1) if shared else None)
    return L, p, order, W


def run_layer(W, k, x, logits, sgate, fused=True):
    T, N = x.shape
    layer = moe.MoELayer(W, k, T, torch.device("cuda"), fused=fused)
    y = torch.zeros((T, N), device="cuda")
    layer(dev(x), dev(logits), None if sgate is None else dev(sgate), y)
    return host(y), host(layer.ids)


def inputs(cfg, T, E, N, seed):
    rng = np.random.default_rng(seed)
    x = rng.normal(0, 1, (T, N)).astype(np.float32)
    if cfg.startswith("c5"):
        x[:, rng.choice(N, N // 100, replace=False)] *= 20.0          # 1% outlier channels
    z = rng.normal(0, 1, E)
    if cfg.startswith("c3"):
        logits = z[None, :] + 0.5 * rng.normal(0, 1, (T, E))
    elif cfg.startswith("c4") or cfg.startswith("c5"):
        s = 1.1 if cfg.startswith("c4") else 1.3
        logits = rng.normal(0, 1, (T, E)) + np.log(1.0 / (1 + rng.permutation(E)) ** s)
    else:
        logits = rng.normal(0, 1, (T, E))
    sgate = rng.normal(0, 1, T).astype(np.float32)
    return x, logits.astype(np.float32), sgate


# the decode configurations run both the two-launch layer and the reference's kernel-by-kernel sequence; prompt chunks
# have one path
LAYER_CASES = [(c, f) for c in CONFIGS for f in ((True, False) if CONFIGS[c][7] <= 8 else (True,))]


@pytest.mark.parametrize("cfg,fused", LAYER_CASES,
                         ids=[f"{c}-{'two_launch' if f else 'kernel_by_kernel'}" for c, f in LAYER_CASES])
def test_layer_against_oracle(cfg, fused):
    gu, d, N, FF, E, k, shared, T = CONFIGS[cfg]
    L, p, order, W = make_layer(gu, d, N, FF, E, shared)
    x, logits, sgate = inputs(cfg, T, E, N, seed=len(cfg))
    got, ids = run_layer(W, k, x, logits, sgate if shared else None, fused=fused)
    Lo = O.layout(gu, d, N, FF)
    blobs = p[order]
    sh = p[len(p) - 1] if shared else None
    y0, eids, _ = O.moe_layer(0, Lo, x, logits, k, blobs, p.shape[1], sh, sgate if shared else None)
    assert (ids == eids).all()
    err = rel_l2(got, y0)
    y1, _, _ = O.moe_layer(1, Lo, x, logits, k, blobs, p.shape[1], sh, sgate if shared else None)
    print(f"{cfg}: rel L2 vs oracle(Q8_1) {err:.2e}; vs reference CPU activations {rel_l2(got, y1):.2e}")
    assert err < 1e-3


def prompt_selection(ids: np.ndarray, n_expert: int, tile: int = 64, most: int = 400, edges: int = 96):
    """Tokens of a prompt chunk chosen from its routing, where the grouped products' tiling has its edges: every token
    of the most-loaded expert's last two token tiles, every token of each expert with fewer than 16 rows, and the
    tokens on both sides of tile boundaries (sorted rows tile*i - 1 and tile*i of each expert; at least `edges` of them,
    thinned evenly when there are more than the room left under `most`).  Sorted rows are
    the prompt path's order: by expert, entries in entry order.  Returns (sorted token list, description)."""
    T, k = ids.shape
    flat = ids.ravel()
    order = np.argsort(flat * (T * k) + np.arange(T * k), kind="stable")  # (expert, entry) order
    counts = np.bincount(flat, minlength=n_expert)
    starts = np.concatenate([[0], np.cumsum(counts)])
    heavy = int(np.argmax(counts))
    nh = int(counts[heavy])
    last = max(0, (nh - 1) // tile * tile - tile)  # the heavy expert's last two tiles
    pick_heavy = {int(order[starts[heavy] + r]) // k for r in range(last, nh)}
    small = [e for e in range(n_expert) if 0 < counts[e] < 16]
    pick_small = {int(order[starts[e] + r]) // k for e in small for r in range(int(counts[e]))}
    pick_edge = set()
    for e in range(n_expert):
        for b in range(tile, int(counts[e]), tile):
            pick_edge.add(int(order[starts[e] + b - 1]) // k)
            pick_edge.add(int(order[starts[e] + b]) // k)
    chosen = pick_heavy | pick_small
    rest = sorted(pick_edge - chosen)
    room = max(edges, most - len(chosen))
    if len(rest) > room:  # the boundary tokens are thinned evenly when there are too many
        rest = [rest[i] for i in np.linspace(0, len(rest) - 1, room).astype(int)]
    sel = sorted(chosen | set(rest))
    desc = (f"heaviest expert {heavy} ({nh} rows): {len(pick_heavy)} tokens of its last two {tile}-row tiles; "
            f"{len(small)} experts under 16 rows: {len(pick_small)} tokens; tile-boundary tokens {len(rest)} of "
            f"{len(pick_edge)}; {len(sel)} tokens in all; rows per expert min {int(counts[counts > 0].min())} "
            f"max {nh}")
    return np.asarray(sel, np.int64), desc


@pytest.mark.parametrize("cfg,T,E,k,shared,gu,d,FF", [
    ("c4_prefill_q4_k", 512, 128, 8, False, Q4_K, Q4_K, 768),
    ("c5_prefill_iq3", 4096, 256, 8, True, IQ3_XXS, IQ3_S, 512),
])
def test_full_prefill_selected_tokens(cfg, T, E, k, shared, gu, d, FF):
    """A full-size prompt chunk against the oracle on the tokens where the tiling has its edges (prompt_selection).
    A token's output depends only on its own input and routing, whatever other tokens share its experts (the
    reference's token-independence invariant), so checking those tokens checks the tiles they sit in."""
    N = 2048
    L, p, order, W = make_layer(gu, d, N, FF, E, shared)
    x, logits, sgate = inputs(cfg, T, E, N, seed=T)
    got, ids = run_layer(W, k, x, logits, sgate if shared else None)
    assert np.isfinite(got).all()
    eids_all, _ = O.router_topk(logits, k)
    assert (ids == eids_all).all()
    sel, desc = prompt_selection(ids, E)
    print(f"{cfg}: {desc}")
    assert len(sel) >= 64
    Lo = O.layout(gu, d, N, FF)
    y0, eids, _ = O.moe_layer(0, Lo, x[sel], logits[sel], k, p[order], p.shape[1],
                              p[len(p) - 1] if shared else None, sgate[sel] if shared else None)
    assert (ids[sel] == eids).all()
    err = rel_l2(got[sel], y0)
    worst = max(rel_l2(got[t], y0[i]) for i, t in enumerate(sel))
    print(f"{cfg}: {T} tokens, {len(sel)} selected: rel L2 {err:.2e}, worst token {worst:.2e}")
    assert err < 1e-3


DECODE_CASES = [
    # (gu, d, N, FF, E, k, shared, T): the edges of the two-launch decode layer
    (IQ3_XXS, IQ3_S, 2048, 512, 256, 8, True, 8),     # 64 entries, the most one call takes
    (Q4_K, Q4_K, 2048, 768, 128, 8, True, 2),         # 16-row chunks of gate/up rows
    (Q8_0, Q8_0, 2048, 768, 64, 4, True, 3),          # 8-row chunks
    (IQ3_S, IQ3_XXS, 4096, 256, 512, 2, False, 5),    # widest rows, 512 experts
    (IQ3_XXS, Q8_0, 2048, 1024, 64, 1, True, 1),      # top-1, widest FF
    # two to four tokens on the slot-by-slot launch A: shared expert items of 2 and 1 rows, no shared expert, rows of
    # one and of two 16-byte pieces per lane, 2 rows of a slot per block
    (IQ3_XXS, IQ3_S, 2048, 512, 256, 8, True, 2),
    (Q4_K, Q4_K, 2048, 512, 128, 8, False, 3),
    (IQ3_S, IQ3_S, 2048, 256, 128, 6, True, 4),
    # one token on the run-per-block launch A (the slot-by-slot one has no wave mapping for these): 17 slots, and
    # 9 slots of 4 pairs per block
    (IQ3_XXS, IQ3_S, 2048, 512, 128, 16, True, 1),
    (IQ3_XXS, IQ3_S, 2048, 1024, 256, 8, True, 1),
]


@pytest.mark.parametrize("case", DECODE_CASES, ids=lambda c: f"{c[0]}-{c[1]}-N{c[2]}-FF{c[3]}-E{c[4]}-k{c[5]}-T{c[7]}")
def test_decode_layer_edges(case):
    gu, d, N, FF, E, k, shared, T = case
    L, p, order, W = make_layer(gu, d, N, FF, E, shared, distinct=5, seed=3)
    x, logits, sgate = inputs("edge", T, E, N, seed=N + FF + E + T)
    got, ids = run_layer(W, k, x, logits, sgate if shared else None)
    Lo = O.layout(gu, d, N, FF)
    sh = p[len(p) - 1] if shared else None
    y0, eids, _ = O.moe_layer(0, Lo, x, logits, k, p[order], p.shape[1], sh, sgate if shared else None)
    assert (ids == eids).all()
    err = rel_l2(got, y0)
    print(f"{case}: rel L2 {err:.2e}")
    assert err < 1e-3


@pytest.mark.parametrize("T", [1, 3, 6])
@pytest.mark.parametrize("FF", [128, 384])
def test_decode_layer_q8_0_odd_row_pieces(FF, T):
    """Q8_0 down rows of an odd number of 8-byte pieces (136 and 408 bytes): rows and units start at every even offset of
    a 16-byte piece in the LDS slabs."""
    gu, d, N, E, k, shared = Q8_0, Q8_0, 512, 64, 4, True
    L, p, order, W = make_layer(gu, d, N, FF, E, shared, distinct=5, seed=4)
    x, logits, sgate = inputs("edge", T, E, N, seed=FF + T)
    got, ids = run_layer(W, k, x, logits, sgate)
    y0, eids, _ = O.moe_layer(0, O.layout(gu, d, N, FF), x, logits, k, p[order], p.shape[1], p[len(p) - 1], sgate)
    assert (ids == eids).all()
    assert rel_l2(got, y0) < 1e-3


def test_decode_layer_residual_alias_and_replay():
    """y may alias x (x <- x + moe(x)); a captured graph replays to the same bits as the eager call, every time."""
    gu, d, N, FF, E, k, shared, T = CONFIGS["c3_verify_iq3"]
    L, p, order, W = make_layer(gu, d, N, FF, E, shared)
    x, logits, sgate = inputs("c3", T, E, N, seed=11)
    ref, _, _ = O.moe_layer(0, O.layout(gu, d, N, FF), x, logits, k, p[order], p.shape[1], p[len(p) - 1], sgate)
    layer = moe.MoELayer(W, k, T, torch.device("cuda"))
    xd, ld, sd = dev(x), dev(logits), dev(sgate)
    buf = xd.clone()
    layer(buf, ld, sd, buf)
    eager = host(buf)
    assert rel_l2(eager.astype(np.float64) - x, ref) < 1e-3
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        buf.copy_(xd)
        layer(buf, ld, sd, buf)
    torch.cuda.current_stream().wait_stream(s)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        buf.copy_(xd)
        layer(buf, ld, sd, buf)
    for _ in range(3):
        g.replay()
        assert (host(buf) == eager).all()
        buf.zero_()
        torch.cuda.synchronize()


@pytest.mark.parametrize("k,ties", [(8, False), (8, True), (12, False), (12, True), (3, True)])
def test_one_token_routing_matches_router(k, ties):
    """At one token every launch A block routes the token itself, as far as its last pick (k 3 to 12): the layer's ids
    and weights are the router kernel's bit for bit, also when probabilities tie (logits drawn from a few values, so
    equal probabilities must go to the lower expert id)."""
    gu, d, N, FF, E, _, shared, T = CONFIGS["c2_decode_iq3"]
    L, p, order, W = make_layer(gu, d, N, FF, E, shared)
    for seed in range(4):
        rng = np.random.default_rng(100 + seed)
        x = rng.normal(0, 1, (1, N)).astype(np.float32)
        logits = (rng.integers(0, 6, (1, E)) * 0.5 if ties else rng.normal(0, 2, (1, E))).astype(np.float32)
        sgate = rng.normal(0, 1, 1).astype(np.float32)
        layer = moe.MoELayer(W, k, 1, torch.device("cuda"), fused=True)
        y = torch.zeros((1, N), device="cuda")
        layer(dev(x), dev(logits), dev(sgate), y)
        ids_r = torch.empty((1, k), dtype=torch.int32, device="cuda")
        wts_r = torch.empty((1, k), dtype=torch.float32, device="cuda")
        ops.native_router_topk(dev(logits), k, ids_r, wts_r)
        torch.cuda.synchronize()
        assert (host(layer.ids) == host(ids_r)).all(), (seed, host(layer.ids), host(ids_r))
        assert (host(layer.wts).view(np.uint32) == host(wts_r).view(np.uint32)).all(), seed


def test_decode_layer_matches_kernel_by_kernel():
    """The two launches and the reference's kernel-by-kernel sequence route identically and agree to float order."""
    gu, d, N, FF, E, k, shared, T = CONFIGS["c3_verify_iq3"]
    L, p, order, W = make_layer(gu, d, N, FF, E, shared)
    x, logits, sgate = inputs("c3", T, E, N, seed=5)
    a, ia = run_layer(W, k, x, logits, sgate, fused=True)
    b, ib = run_layer(W, k, x, logits, sgate, fused=False)
    assert (ia == ib).all()
    assert rel_l2(a, b) < 1e-5


NORM_CASES = [("c2_decode_iq3", True), ("c3_verify_iq3", True), ("c2_decode_iq3", False), ("c1_decode_q8_0", True),
              ("c5_prefill_iq3_16tok", True)]


@pytest.mark.parametrize("cfg,fused", NORM_CASES,
                         ids=[f"{c}-{'two_launch' if f else 'kernel_by_kernel'}" for c, f in NORM_CASES])
def test_moe_block_norm(cfg, fused):
    """The MoE block's end (k_moe_out_small with the norm): y is bit for bit the layer's y without the norm; h is the
    closed-form norm of that y (float64 oracle, within float32 rounding); hq is the Q8_1 image of h byte for byte.
    Three calls in a row give the same bits (the second launch's completion count starts from zero every call)."""
    gu, d, N, FF, E, k, shared, T = CONFIGS[cfg]
    L, p, order, W = make_layer(gu, d, N, FF, E, shared)
    x, logits, sgate = inputs(cfg, T, E, N, seed=len(cfg) + 5)
    rng = np.random.default_rng(9)
    wn = (1.0 + 0.1 * rng.normal(0, 1, N)).astype(np.float32)
    eps = 1e-6
    layer = moe.MoELayer(W, k, T, torch.device("cuda"), fused=fused)
    xd, ld, sd, wd = dev(x), dev(logits), dev(sgate) if shared else None, dev(wn)
    y_plain = torch.zeros((T, N), device="cuda")
    layer(xd, ld, sd, y_plain)
    outs = []
    for _ in range(3):
        y = torch.zeros((T, N), device="cuda")
        h = torch.full((T, N), float("nan"), device="cuda")
        hq = torch.zeros((T, N // 32 * 36), dtype=torch.uint8, device="cuda")
        layer(xd, ld, sd, y, norm_w=wd, eps=eps, h=h, hq=hq)
        outs.append((host(y), host(h), host(hq)))
    yp = host(y_plain)
    for yv, hv, hqv in outs:
        assert (yv == yp).all() and (hv == outs[0][1]).all() and (hqv == outs[0][2]).all()
    yv, hv, hqv = outs[0]
    ref = O.rms_norm(yv, wn, eps)
    err = np.abs(hv - ref).max() / np.abs(ref).max()
    print(f"{cfg}: h against the closed-form norm: max error {err:.2e} of max |h|")
    assert err < 2e-6
    assert (hqv == O.quantize_q8_1(hv)).all()


def test_prompt_layer_graph_replay():
    """A prompt chunk's layer (the shared expert's products on a second stream) captured in a graph replays to the
    eager call's bits, every time, with eager work and synchronisations between the replays."""
    gu, d, N, FF, E, k, shared, T = CONFIGS["c5_prefill_iq3_16tok"]
    T = 300
    L, p, order, W = make_layer(gu, d, N, FF, E, shared)
    x, logits, sgate = inputs("c5", T, E, N, seed=17)
    layer = moe.MoELayer(W, k, T, torch.device("cuda"))
    xd, ld, sd = dev(x), dev(logits), dev(sgate)
    y = torch.zeros((T, N), device="cuda")
    layer(xd, ld, sd, y)
    eager = host(y)
    ref, _, _ = O.moe_layer(0, O.layout(gu, d, N, FF), x[:8], logits[:8], k, p[order], p.shape[1], p[len(p) - 1],
                            sgate[:8])
    assert rel_l2(eager[:8], ref) < 1e-3
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        y.zero_()
        layer(xd, ld, sd, y)
    torch.cuda.current_stream().wait_stream(s)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        y.zero_()
        layer(xd, ld, sd, y)
    for _ in range(3):
        g.replay()
        assert (host(y) == eager).all()
        y.fill_(7.0)
        torch.cuda.synchronize()

"""The single-matrix product on Q4_0 and Q6_K, and several matrices per launch: picked on the device through a table
(tsx_moe_mmvq_ids, reference lfm_native_mmvq_ids) or given by the host (tsx_moe_mmvq_slots, lfm_native_mmvq_slots),
against the CPU oracle (marked gpu).

Bars: the integer sub-block sums bit-exact; float outputs within 1e-5 relative of the oracle (the same integer sums,
another float order); each matrix of a many-matrix launch bit-identical to the same matrix through tsx_moe_mmvq."""
import numpy as np
import pytest
import torch

import oracle as O
from tinystrata_amd import ops
from tinystrata_amd._lib import IQ3_S, IQ3_XXS, Q4_0, Q4_K, Q6_K, Q8_0

from gpu_util import dev, host

pytestmark = pytest.mark.gpu
ALL = (IQ3_XXS, IQ3_S, Q4_K, Q8_0, Q4_0, Q6_K)


def weights(t, rows, n, seed):
    """rows x n of type t: quantized N(0, 0.02) for the expert formats, random blocks with finite scales for Q4_0 and
    Q6_K (no ggml quantizer offline; every byte pattern is a valid code)."""
    rng = np.random.default_rng(seed)
    if t in (IQ3_XXS, IQ3_S, Q4_K, Q8_0):
        return ops.quantize_weights(t, rng.normal(0, 0.02, (rows, n)).astype(np.float32))
    if t == Q4_0:
        b = rng.integers(0, 256, (rows, n // 32, 18), dtype=np.uint8)
        b[..., 0:2] = rng.uniform(0.001, 0.05, (rows, n // 32)).astype(np.float16)[..., None].view(np.uint8)
    else:
        b = rng.integers(0, 256, (rows, n // 256, 210), dtype=np.uint8)
        b[..., 208:210] = rng.uniform(0.0001, 0.002, (rows, n // 256)).astype(np.float16)[..., None].view(np.uint8)
    return b.reshape(rows, -1)


@pytest.mark.parametrize("t", (Q4_0, Q6_K))
@pytest.mark.parametrize("n_in,n_out,ncols", [(2048, 96, 1), (512, 300, 4), (768, 64, 8)])
def test_small_formats(t, n_in, n_out, ncols):
    print(f"small format t={t} {n_out}x{n_in} ncols={ncols}", flush=True)
    w = weights(t, n_out, n_in, n_in + n_out)
    xq = O.quantize_q8_1(np.random.default_rng(t).normal(0, 1, (ncols, n_in)).astype(np.float32))
    got = host(ops.iq_mmvq(t, dev(w), dev(xq), n_in, n_out, ncols))
    exp = O.mmvq_q8_1(t, w, n_in, n_out, xq, ncols)
    np.testing.assert_allclose(got, exp, rtol=1e-5, atol=1e-5 * np.abs(exp).max())
    s, q = ops.subblock_sums(t, dev(w), n_in, n_out, dev(xq), ncols)
    es, eq = O.subblock_sums(t, w, n_in, n_out, xq, ncols)
    assert (host(s) == es).all() and (host(q) == eq).all()


@pytest.mark.parametrize("t", ALL)
@pytest.mark.parametrize("shift", [4, 8, 12])
def test_mmvq_matrix_on_a_4_byte_boundary(t, shift):
    """The products read a row's fields as the aligned words around them: a matrix that starts 4, 8 or 12 bytes behind a
    16-byte boundary, with rows of an odd number of blocks (every block start that the format's size allows), gives the
    bits of the same matrix on a 256-byte boundary and the exact integer sums."""
    n_in, n_out = 768, 21
    print(f"4-byte boundary t={t} shift={shift}", flush=True)
    w = weights(t, n_out, n_in, 300 + t)
    xq = O.quantize_q8_1(np.random.default_rng(t).normal(0, 1, (2, n_in)).astype(np.float32))
    buf = torch.zeros(w.size + shift + 16, dtype=torch.uint8, device="cuda")
    buf[shift:shift + w.size] = dev(w.ravel())
    got = host(ops.iq_mmvq(t, buf[shift:], dev(xq), n_in, n_out, 2))
    assert np.array_equal(got, host(ops.iq_mmvq(t, dev(w), dev(xq), n_in, n_out, 2)))
    s, q = ops.subblock_sums(t, buf[shift:], n_in, n_out, dev(xq), 2)
    es, eq = O.subblock_sums(t, w, n_in, n_out, xq, 2)
    assert (host(s) == es).all() and (host(q) == eq).all()


@pytest.mark.parametrize("t", ALL)
@pytest.mark.parametrize("shift", [1, 2, 3, 7])
def test_products_on_any_byte_address(t, shift):
    """Weights that start off a 4-byte boundary - a matrix, an id-indexed offset, a group's blob, experts an odd number of
    bytes apart - give the bits of the same weights on a 256-byte boundary."""
    n_in, n_out = 768, 21
    print(f"byte address t={t} shift={shift}", flush=True)
    w = weights(t, n_out, n_in, 400 + t)
    xq = O.quantize_q8_1(np.random.default_rng(t).normal(0, 1, (3, n_in)).astype(np.float32))
    buf = torch.zeros(w.size + shift + 16, dtype=torch.uint8, device="cuda")
    buf[shift:shift + w.size] = dev(w.ravel())
    exp = host(ops.iq_mmvq(t, dev(w), dev(xq), n_in, n_out, 3))
    assert np.array_equal(host(ops.iq_mmvq(t, buf[shift:], dev(xq), n_in, n_out, 3)), exp)
    table = torch.tensor([buf.data_ptr()], dtype=torch.int64, device="cuda")
    y = torch.full((3, n_out), 7.0, device="cuda")
    ops.mmvq_ids(t, table, torch.zeros(3, dtype=torch.int32, device="cuda"), shift, dev(xq), n_in // 32 * 36, 1, y, n_out, 3,
                 n_in, n_out)
    assert np.array_equal(host(y), exp)
    if t in (Q4_0, Q6_K):
        return
    # two experts of the prompt's row-dot product, w.size + shift bytes apart
    blob = torch.zeros(2 * w.size + 2 * shift + 16, dtype=torch.uint8, device="cuda")
    blob[:w.size] = dev(w.ravel())
    blob[w.size + shift:2 * w.size + shift] = dev(w[::-1].copy().ravel())
    x = torch.randn((4, n_in), generator=torch.Generator(device="cuda").manual_seed(t), device="cuda")
    xm = ops.mmq_quantize(x, None, t, n_in, n_in, 4)
    bounds = torch.tensor([0, 2, 4], dtype=torch.int32, device="cuda")
    got = torch.empty((4, n_out), device="cuda")
    ops.mmq_run(blob, t, n_out, n_in, w.size + shift, 2, xm, bounds, None, 4, got, n_out)
    one = host(ops.iq_mmvq(t, dev(w), ops.quantize_q8_1_rows(x), n_in, n_out, 4))
    np.testing.assert_allclose(host(got)[:2], one[:2], rtol=1e-5, atol=1e-5 * np.abs(one).max())
    np.testing.assert_allclose(host(got)[2:, ::-1], one[2:], rtol=1e-5, atol=1e-5 * np.abs(one).max())
    # a group whose blob lies off a 4-byte boundary
    L = ops.native_expert_layout(t, t, 256, 256)
    e = np.concatenate([weights(t, 512, 256, 1).ravel(), weights(t, 256, 256, 2).ravel()])
    assert e.size == L.down_off + 256 * L.d_row
    eb = torch.zeros(e.size + shift + 16, dtype=torch.uint8, device="cuda")
    eb[shift:shift + e.size] = dev(e)
    xe = ops.quantize_q8_1_rows(x[:2, :256].contiguous())
    i32 = lambda *v: torch.tensor(v, dtype=torch.int32, device="cuda")
    scratch = torch.empty(ops.native_expert_scratch_bytes(2, 256), dtype=torch.uint8, device="cuda")
    outs = []
    for base in (dev(e), eb[shift:]):
        out = torch.full((2, 256), float("nan"), device="cuda")
        ops.native_expert_grouped(L, torch.tensor([base.data_ptr()], dtype=torch.int64, device="cuda"), i32(0, 2), i32(1),
                                  i32(0, 1), i32(0, 1), 1, 2, xe, scratch, out)
        outs.append(host(out))
    assert np.array_equal(outs[0], outs[1])


@pytest.mark.parametrize("t", ALL)
@pytest.mark.parametrize("x_every", [1, 3])
def test_mmvq_ids(t, x_every):
    n_in, n_out, n_mat, count = 512, 80, 6, 11
    print(f"mmvq_ids t={t} x_every={x_every}", flush=True)
    rb = ops.iq_row_bytes(t, n_in)
    stride = (n_out * rb + 255) // 256 * 256 + 64        # matrices apart in one buffer, behind a 64-byte offset
    host_w = np.zeros((n_mat, stride), np.uint8)
    mats = []
    for m in range(n_mat):
        w = weights(t, n_out, n_in, 100 + m)
        host_w[m, 64:64 + w.size] = w.ravel()
        mats.append(w)
    buf = dev(host_w.ravel())
    table = torch.tensor([buf.data_ptr() + m * stride for m in range(n_mat)], dtype=torch.int64, device="cuda")
    ids = np.array([3, 0, 5, -1, 2, 2, 9, 1, 4, 0, 5], np.int32)  # -1 and 9 are outside the table: zeros
    nx = (count + x_every - 1) // x_every
    xq = O.quantize_q8_1(np.random.default_rng(7).normal(0, 1, (nx, n_in)).astype(np.float32)).reshape(-1)
    xs = n_in // 32 * 36
    y_stride = n_out + 5
    y = torch.full((count * y_stride,), 7.0, device="cuda")
    ops.mmvq_ids(t, table, dev(ids), 64, dev(xq), xs, x_every, y, y_stride, count, n_in, n_out)
    got = host(y).reshape(count, y_stride)
    for j in range(count):
        assert (got[j, n_out:] == 7.0).all()              # nothing past the matrix's rows
        if not 0 <= ids[j] < n_mat:
            assert (got[j, :n_out] == 0.0).all()
            continue
        xj = xq[(j // x_every) * xs:(j // x_every + 1) * xs]
        exp = O.mmvq_q8_1(t, mats[ids[j]], n_in, n_out, xj, 1)[0]
        np.testing.assert_allclose(got[j, :n_out], exp, rtol=1e-5, atol=1e-5 * np.abs(exp).max())
        one = host(ops.iq_mmvq(t, dev(mats[ids[j]]), dev(xj), n_in, n_out, 1))[0]
        assert np.array_equal(got[j, :n_out], one)


def tiled(t, rows, n, seed, distinct=37):
    """rows x n of type t that repeat `distinct` rows, and the repeating oracle result of a Q8_1 column block."""
    w = weights(t, distinct, n, seed)
    rep = np.tile(w, (rows // distinct + 1, 1))[:rows]
    return rep, lambda xq, ncols: np.tile(O.mmvq_q8_1(t, w, n, distinct, xq, ncols), (1, rows // distinct + 1))[:, :rows]


@pytest.mark.parametrize("t", ALL)
@pytest.mark.parametrize("n_in,n_out,ncols", [(2048, 4097, 5), (2048, 8195, 1), (256, 32771, 8), (256, 65541, 3)])
def test_mmvq_several_rows_per_lane_group(t, n_in, n_out, ncols):
    """Every format with two and with four rows of each lane group (from 4096 and 8192 waves), 64 and 8 lanes a row, a last
    block of few rows, one to eight columns: every output, against the oracle."""
    print(f"several rows per lane group t={t} {n_out}x{n_in} ncols={ncols}", flush=True)
    w, oracle = tiled(t, n_out, n_in, n_out + t)
    xq = O.quantize_q8_1(np.random.default_rng(t).normal(0, 1, (ncols, n_in)).astype(np.float32))
    exp = oracle(xq, ncols)
    y = torch.full((ncols * n_out + 8,), 7.0, device="cuda")
    ops.iq_mmvq(t, dev(w), dev(xq), n_in, n_out, ncols, y=y)
    got = host(y)
    assert (got[ncols * n_out:] == 7.0).all()
    np.testing.assert_allclose(got[:ncols * n_out].reshape(ncols, n_out), exp, rtol=1e-5, atol=1e-5 * np.abs(exp).max())


@pytest.mark.parametrize("t", ALL)
@pytest.mark.parametrize("n_in,n_out,count", [(2048, 1031, 4), (2048, 1031, 8), (256, 4099, 9)])
def test_mmvq_ids_several_rows_per_lane_group(t, n_in, n_out, count):
    """The id-indexed product with two and four rows of each lane group: a last block of few rows, ids outside the table
    among the others (zeros), and outputs apart with a sentinel between them."""
    print(f"ids, several rows per lane group t={t} {n_out}x{n_in} count={count}", flush=True)
    mats = [tiled(t, n_out, n_in, 500 + t + m) for m in range(2)]
    buf = dev(np.concatenate([m[0].ravel() for m in mats]))
    table = torch.tensor([buf.data_ptr() + m * mats[0][0].size for m in range(2)], dtype=torch.int64, device="cuda")
    ids = np.array([1, 0, -1, 1, 2, 0, 0, 1, 1][:count], np.int32)
    xq = O.quantize_q8_1(np.random.default_rng(t).normal(0, 1, (count, n_in)).astype(np.float32))
    y_stride = n_out + 3
    y = torch.full((count * y_stride,), 7.0, device="cuda")
    ops.mmvq_ids(t, table, dev(ids), 0, dev(xq), n_in // 32 * 36, 1, y, y_stride, count, n_in, n_out)
    got = host(y).reshape(count, y_stride)
    assert (got[:, n_out:] == 7.0).all()
    for j, i in enumerate(ids):
        exp = mats[i][1](xq.reshape(count, -1)[j], 1)[0] if 0 <= i < 2 else np.zeros(n_out)
        np.testing.assert_allclose(got[j, :n_out], exp, rtol=1e-5, atol=1e-5 * np.abs(exp).max())


@pytest.mark.parametrize("t", (IQ3_XXS, Q4_0, Q6_K))
def test_mmvq_slots(t):
    n_in, n_out, count = 768, 48, 5
    ws = [dev(weights(t, n_out, n_in, 200 + j)) for j in range(count)]
    xqs = [O.quantize_q8_1(np.random.default_rng(j).normal(0, 1, (1, n_in)).astype(np.float32)) for j in range(count)]
    xs = [dev(x) for x in xqs]
    ys = [torch.zeros(n_out, device="cuda") for _ in range(count)]
    ops.mmvq_slots(t, ws, xs, ys, n_in, n_out)
    for j in range(count):
        one = host(ops.iq_mmvq(t, ws[j], xs[j], n_in, n_out, 1))[0]
        assert np.array_equal(host(ys[j]), one)
        exp = O.mmvq_q8_1(t, host(ws[j]), n_in, n_out, xqs[j], 1)[0]
        np.testing.assert_allclose(host(ys[j]), exp, rtol=1e-5, atol=1e-5 * np.abs(exp).max())

"""The kernels that form f32 products from three bf16 parts per operand
(csrc/kernels/split.h): every wave shape of the forward against a float64
reference, at tile edges and remainders, operands too large for the split
(infinities, magnitudes of 2^40 and more), which take f32 products instead, and
operands near the bottom of f32's range, which keep all their bits.

Gate: an output is a convex combination of V rows (|V| up to about 5 here), so
an error of 2^-22 in a weight's exponent and 2^-22 in its product are below
5e-6 in it; the score error is a few 2^-24 of a sum of d products of order
sqrt(d) before the 1/sqrt(d) scale.  2e-5 covers the sum of both at d = 256.
"""
import numpy as np
import pytest

from gpuhelp import SEED_DO, SEED_K, SEED_Q, SEED_V, dev_normal, host
from npref import attention_backward_f64, attention_f64

pytestmark = pytest.mark.gpu


def _product(gpu, zt, op, a, b):
    """a @ b through zt_matmul ("nn"), zt_weight_grad ("tn": a stored K x M) or zt_input_grad ("nt": b stored N x K)."""
    (M, K), N = a.shape, b.shape[1]
    out = gpu.zeros(M * N, device="cuda")
    aa = (a.t() if op == "tn" else a).contiguous().view(-1)
    bb = (b.t() if op == "nt" else b).contiguous().view(-1)
    if op == "nn":
        zt.matmul(aa, bb, out, M, K, N)
    elif op == "tn":
        zt.weight_grad(out, aa, bb, K, M, N)
    else:
        zt.input_grad(out, aa, bb, M, K, N)
    gpu.cuda.synchronize()
    return out.view(M, N)


@pytest.mark.parametrize("op", ["nn", "tn", "nt"])
@pytest.mark.parametrize("tile", [64, 128])
@pytest.mark.parametrize("M,K,N", [(128, 32, 128), (256, 96, 128), (129, 33, 127), (1, 65, 130), (200, 257, 68)])
def test_split_products(gpu, zt, tune, op, tile, M, K, N):
    """Whole tiles and every kind of remainder.  Per element the six products
    drop at most 2^-23 of a product and K / 32 + 32 roundings of 2^-24 follow:
    (2 + K / 32 + 32) 2^-24 of the sum of the products' magnitudes."""
    tune({"ZT_GEMM_TILE": tile})
    gen = gpu.Generator(device="cuda").manual_seed(M * 1009 + K)
    a, b = (gpu.randn(s, device="cuda", generator=gen) for s in ((M, K), (K, N)))
    want = a.double().cpu() @ b.double().cpu()
    bound = (a.double().abs().cpu() @ b.double().abs().cpu()) * ((34 + K / 32) * 2.0 ** -24)
    assert gpu.all((_product(gpu, zt, op, a, b).double().cpu() - want).abs() <= bound)


@pytest.mark.parametrize("op", ["nn", "tn", "nt"])
@pytest.mark.parametrize("which", ["a", "b", "ab"])
def test_split_products_with_infinities(gpu, zt, tune, op, which):
    """An infinity in A, B or both gives what f32 arithmetic gives: the same
    infinities and NaN as float64, and the rest unchanged."""
    tune({"ZT_GEMM_TILE": 128})
    M, K, N = 150, 70, 140
    gen = gpu.Generator(device="cuda").manual_seed(5)
    a, b = (gpu.randn(s, device="cuda", generator=gen) for s in ((M, K), (K, N)))
    if "a" in which:
        a[7, 40] = float("inf")
        a[140, 2] = -2.0 ** 80
    if "b" in which:
        b[41, 133] = float("-inf")
    want = (a.double().cpu() @ b.double().cpu())
    got = _product(gpu, zt, op, a, b).double().cpu()
    fin = gpu.isfinite(want)
    assert gpu.equal(gpu.isnan(got), gpu.isnan(want)) and gpu.equal(got[~fin & ~gpu.isnan(want)], want[~fin & ~gpu.isnan(want)])
    assert gpu.all((got[fin] - want[fin]).abs() <= 1e-5 * gpu.clamp(want[fin].abs(), min=1.0))

TOL = 2e-5


def _forward(gpu, zt, q, k, v, T, H, Hkv, D):
    out = gpu.full((T * H * D,), float("nan"), device="cuda")
    zt.forward(q, k, v, out, T, H, Hkv, D)
    gpu.cuda.synchronize()
    return host(out)


def _inputs(gpu, zt, T, H, Hkv, D):
    return (dev_normal(gpu, zt, T * H * D, SEED_Q), dev_normal(gpu, zt, T * Hkv * D, SEED_K),
            dev_normal(gpu, zt, T * Hkv * D, SEED_V))


@pytest.mark.parametrize("shape", [11, 12, 14, 21, 22])
@pytest.mark.parametrize("T,H,Hkv,D", [(2, 4, 2, 32), (33, 4, 2, 32), (129, 4, 1, 64), (257, 3, 1, 64), (63, 2, 2, 36),
                                       (65, 4, 1, 96), (100, 4, 4, 128), (161, 8, 2, 128), (97, 2, 1, 192),
                                       (70, 4, 1, 256), (31, 2, 2, 256)])
def test_every_wave_shape(gpu, zt, tune, shape, T, H, Hkv, D):
    """(A shape a width does not have falls back to one it has.)"""
    tune({"ZT_ATTN_FSHAPE": shape})
    q, k, v = _inputs(gpu, zt, T, H, Hkv, D)
    want = attention_f64(host(q), host(k), host(v), T, H, Hkv, D).ravel()
    assert np.max(np.abs(_forward(gpu, zt, q, k, v, T, H, Hkv, D) - want)) <= TOL


@pytest.mark.parametrize("shape", [12, 21])
@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("where", ["k", "v", "q", "kq"])
def test_large_finite_operands_take_the_f32_products(gpu, zt, tune, shape, D, where):
    """An entry of 2^70 in one row of K, V or Q (and in both K and Q, at
    different columns, so no product of two of them): its own products are
    formed in f32, and rows and columns it does not reach keep their bits."""
    tune({"ZT_ATTN_FSHAPE": shape})
    T, H, Hkv, S = 150, 4, 2, 70
    q, k, v = _inputs(gpu, zt, T, H, Hkv, D)
    good = _forward(gpu, zt, q, k, v, T, H, Hkv, D).reshape(T, H, D)
    big = 2.0 ** 70
    if "k" in where:
        k = k.clone()
        k.view(T, Hkv, D)[S, 1, 3] = -big
    if "q" in where:
        q = q.clone()
        q.view(T, H, D)[S, 2, 5] = big
    if "v" in where:
        v = v.clone()
        v.view(T, Hkv, D)[S, 1, 3] = big
    got = _forward(gpu, zt, q, k, v, T, H, Hkv, D).reshape(T, H, D)
    want = attention_f64(host(q), host(k), host(v), T, H, Hkv, D).reshape(T, H, D)
    scale = np.maximum(1.0, np.abs(want))
    assert np.max(np.abs(got - want) / scale) <= TOL
    assert np.array_equal(got[:, :2].view(np.uint32), good[:, :2].view(np.uint32))      # the other kv head
    if where != "kq":  # (a tile with both is formed in f32 throughout)
        assert np.array_equal(got[:S].view(np.uint32), good[:S].view(np.uint32))        # earlier rows
    if where == "v":
        keep = [c for c in range(D) if c != 3]
        assert np.array_equal(got[..., keep].view(np.uint32), good[..., keep].view(np.uint32))


def _train(gpu, zt, q, k, v, do, T, H, Hkv, D):
    out, lse = gpu.empty_like(q), gpu.empty(T * H, device="cuda")
    dq, dk, dv = (gpu.full_like(x, float("nan")) for x in (q, k, v))
    ws = gpu.full((zt.backward_train_workspace_bytes(1, T, H, Hkv, D) // 4,), float("nan"), device="cuda")
    zt.forward_train_ws(q, k, v, out, lse, ws, T, H, Hkv, D)
    zt.backward_train_ws(q, k, v, out, do, lse, dq, dk, dv, ws, T, H, Hkv, D, stage=3 | zt.ZT_WS_SCORES)
    gpu.cuda.synchronize()
    return [host(x) for x in (dq, dk, dv)]


@pytest.mark.parametrize("blocks", [1, 2, 4])
@pytest.mark.parametrize("T,H,Hkv,D", [(2, 4, 2, 32), (33, 4, 2, 32), (161, 4, 1, 32), (65, 4, 2, 64), (97, 3, 1, 64),
                                       (47, 2, 1, 80), (100, 4, 1, 96), (130, 3, 3, 128), (257, 8, 2, 128)])
def test_every_dkdv_shape(gpu, zt, tune, blocks, T, H, Hkv, D):
    """The score-reading dk/dv kernel's shapes (groups that halve, MHA, a group
    of three).  dk and dv sum up to T H / Hkv terms with 32-term f32 steps, each
    of a difference of two sums of D products: a few 2^-22 of the gradient's
    scale; 1e-5 of the largest value leaves a factor of ten."""
    tune({"ZT_ATTN_BSHAPE": blocks})
    q, k, v = _inputs(gpu, zt, T, H, Hkv, D)
    do = dev_normal(gpu, zt, T * H * D, SEED_DO)
    want = attention_backward_f64(*(host(x) for x in (q, k, v, do)), T, H, Hkv, D)
    for got, w in zip(_train(gpu, zt, q, k, v, do, T, H, Hkv, D), want):
        w = np.asarray(w).ravel()
        assert np.max(np.abs(got - w)) <= 1e-5 * max(1.0, np.abs(w).max())


@pytest.mark.parametrize("where", ["q", "do", "v"])
def test_dkdv_with_large_operands(gpu, zt, where):
    """Rows of 2^70 in dO (dv and dk of its keys), or in V or Q where the result
    stays finite: the gradients follow float64, the other kv head keeps its bits."""
    T, H, Hkv, D, S = 90, 4, 2, 64, 50
    q, k, v = _inputs(gpu, zt, T, H, Hkv, D)
    do = dev_normal(gpu, zt, T * H * D, SEED_DO)
    good = _train(gpu, zt, q, k, v, do, T, H, Hkv, D)
    x = {"q": q, "do": do, "v": v}[where].clone()
    x.view(T, -1, D)[S, -1, 3] = 2.0 ** 70
    args = {"q": q, "k": k, "v": v, "do": do, where: x}
    got = _train(gpu, zt, args["q"], args["k"], args["v"], args["do"], T, H, Hkv, D)
    want = attention_backward_f64(*(host(args[n]) for n in ("q", "k", "v", "do")), T, H, Hkv, D)
    for n, g, w, o, heads in zip(("dq", "dk", "dv"), got, want, good, (H, Hkv, Hkv)):
        g, w, o = (np.asarray(y).reshape(T, heads, D) for y in (g, w, o))
        assert np.all(np.isfinite(g))
        err, tol = np.abs(g - w), np.full(D, 1e-5 * np.abs(w).max())
        if where == "q" and n == "dk":
            # Row S's softmax is one-hot, so its dS = dP - delta is exactly 0, as the
            # difference of two f32 sums of the same D products dO V, each off by up to
            # D 2^-24 of the sum of their magnitudes; column 3 of dk takes it times 2^70.
            mags = np.abs(host(do).reshape(T, H, D)[S, -1] * host(v).reshape(T, Hkv, D)[:, -1]).sum(1).max()
            tol[3] += 2 * D * 2.0 ** -24 * mags * 2.0 ** 70 / np.sqrt(D)
        assert np.all(err <= tol)
        assert np.array_equal(g[:, :heads // 2].view(np.uint32), o[:, :heads // 2].astype(np.float32).view(np.uint32))


@pytest.mark.parametrize("where", ["", "do", "k"])
@pytest.mark.parametrize("T,H,Hkv,D", [(2, 2, 1, 128), (33, 4, 2, 96), (129, 2, 1, 36), (161, 4, 4, 128),
                                       (300, 4, 2, 192)])
def test_dq_product_on_split_operands(gpu, zt, tune, T, H, Hkv, D, where):
    """The 128-tile dq = dS K product: edges of tiles, slabs and columns, a row
    of dO with an entry of 2^70 (its dS is past the split's range) and a column of
    K with one (Q holds 0 there, so the scores do not).  Same gate as the shapes
    of dk/dv above, over the entries the large value reaches and over the rest."""
    tune({"ZT_DQDS_TILE": 128, "ZT_DQDS_K": 1})
    q, k, v = _inputs(gpu, zt, T, H, Hkv, D)
    do = dev_normal(gpu, zt, T * H * D, SEED_DO)
    S, reached = T // 2, np.zeros((T, H, D), bool)
    if where == "do":
        do.view(T, H, D)[S, -1, 3] = 2.0 ** 70
        reached[S, -1] = True
    if where == "k":
        q.view(T, H, D)[:, :, 3] = 0.0
        k.view(T, Hkv, D)[S, -1, 3] = 2.0 ** 70
        reached[S:, H - H // Hkv:, 3] = True
    want = np.asarray(attention_backward_f64(*(host(x) for x in (q, k, v, do)), T, H, Hkv, D)[0]).reshape(T, H, D)
    got = _train(gpu, zt, q, k, v, do, T, H, Hkv, D)[0].reshape(T, H, D)
    for part in (reached, ~reached):
        if part.any():
            assert np.max(np.abs(got[part] - want[part])) <= 1e-5 * max(1.0, np.abs(want[part]).max())


def _scaled(gpu, x, e):
    """x 2^e, rounded once to f32 (denormal values kept)."""
    return (x.double().cpu() * 2.0 ** e).float().cuda()


@pytest.mark.parametrize("op", ["nn", "tn", "nt"])
@pytest.mark.parametrize("e", [-116, -124, -135])
@pytest.mark.parametrize("which", ["a", "b"])
def test_small_operands_keep_their_bits_in_products(gpu, zt, tune, op, e, which):
    """One operand near or in f32's denormal range: test_split_products' bound
    (relative to the sum of the products' magnitudes), plus the results' own
    denormal rounding, 2^-150 an addition."""
    tune({"ZT_GEMM_TILE": 128})
    M, K, N = 130, 96, 128
    gen = gpu.Generator(device="cuda").manual_seed(11)
    a, b = (gpu.randn(s, device="cuda", generator=gen) for s in ((M, K), (K, N)))
    a, b = (_scaled(gpu, a, e), b) if which == "a" else (a, _scaled(gpu, b, e))
    want = a.double().cpu() @ b.double().cpu()
    n = 34 + K / 32
    bound = (a.double().abs().cpu() @ b.double().abs().cpu()) * (n * 2.0 ** -24) + n * 2.0 ** -150
    assert gpu.all((_product(gpu, zt, op, a, b).double().cpu() - want).abs() <= bound)


@pytest.mark.parametrize("shape", [12, 21])
@pytest.mark.parametrize("D", [64, 128, 256])
def test_small_values_keep_their_bits_in_the_forward(gpu, zt, tune, shape, D):
    """V scaled by 2^-124: the output is the same combination, to the same relative gate."""
    tune({"ZT_ATTN_FSHAPE": shape})
    T, H, Hkv = 100, 4, 2
    q, k, v = _inputs(gpu, zt, T, H, Hkv, D)
    v = _scaled(gpu, v, -124)
    want = attention_f64(host(q), host(k), host(v), T, H, Hkv, D).ravel()
    assert np.max(np.abs(_forward(gpu, zt, q, k, v, T, H, Hkv, D) - want)) <= TOL * 2.0 ** -124


@pytest.mark.parametrize("D", [32, 64, 128])
def test_small_gradients_keep_their_bits(gpu, zt, tune, D):
    """dO scaled by 2^-124 scales every gradient by it: test_every_dkdv_shape's
    gate relative to the gradient (with the dq product on split operands too)."""
    tune({"ZT_DQDS_TILE": 128, "ZT_DQDS_K": 1})
    T, H, Hkv = 161, 4, 2
    q, k, v = _inputs(gpu, zt, T, H, Hkv, D)
    do = _scaled(gpu, dev_normal(gpu, zt, T * H * D, SEED_DO), -124)
    want = attention_backward_f64(*(host(x) for x in (q, k, v, do)), T, H, Hkv, D)
    for got, w in zip(_train(gpu, zt, q, k, v, do, T, H, Hkv, D), want):
        w = np.asarray(w).ravel()
        assert np.max(np.abs(got - w)) <= 1e-5 * np.abs(w).max()


@pytest.mark.parametrize("op,tile", [("nn", 128), ("tn", 128), ("nt", 128), ("tn", 64), ("nt", 64)])
@pytest.mark.parametrize("which", ["a", "b", "ab", "ab apart"])
def test_whole_tiles_with_large_values(gpu, zt, tune, op, tile, which):
    """Infinities and magnitudes past the split's range in whole tiles, in one
    operand, in both in the same slab, and in both in different slabs: the result is
    what f32 arithmetic gives, with test_split_products' bound where it is finite."""
    tune({"ZT_GEMM_TILE": tile})
    M, K, N = 256, 96, 128
    gen = gpu.Generator(device="cuda").manual_seed(tile)
    a, b = (gpu.randn(s, device="cuda", generator=gen) for s in ((M, K), (K, N)))
    if "a" in which:
        a[7, 40], a[140, 41], a[255, 2] = float("inf"), -2.0 ** 45, 2.0 ** 80
    if "b" in which:
        k = 90 if "apart" in which else 43
        b[k, 100], b[k + 1, 3] = float("-inf"), 2.0 ** 41
    want = a.double().cpu() @ b.double().cpu()
    got = _product(gpu, zt, op, a, b).double().cpu()
    fin = gpu.isfinite(want)
    assert gpu.equal(gpu.isnan(got), gpu.isnan(want))
    assert gpu.equal(got[~fin & ~gpu.isnan(want)], want[~fin & ~gpu.isnan(want)])
    bound = (a.double().abs().cpu() @ b.double().abs().cpu()) * ((34 + K / 32) * 2.0 ** -24)
    assert gpu.all((got - want).abs()[fin] <= bound[fin])


def _close_by_part(got, want, parts):
    """1e-5 of the largest value (test_every_dkdv_shape's gate) within each part of the entries."""
    for part in parts:
        assert np.all(np.isfinite(got[part]))
        assert np.max(np.abs(got[part] - want[part])) <= 1e-5 * max(1.0, np.abs(want[part]).max())


@pytest.mark.parametrize("T,H,Hkv,D", [(90, 4, 2, 64), (90, 4, 4, 128), (161, 4, 2, 32)])
def test_gradients_with_both_operands_large(gpu, zt, tune, T, H, Hkv, D):
    """2^70 in both operands of a product, where the two do not meet, so that the
    tile's whole product is formed in f32 and stays in its ordinary range."""
    tune({"ZT_DQDS_TILE": 128, "ZT_DQDS_K": 1})
    big, g = 2.0 ** 70, H // Hkv

    def run(q, k, v, do):
        want = attention_backward_f64(*(host(x) for x in (q, k, v, do)), T, H, Hkv, D)
        got = _train(gpu, zt, q, k, v, do, T, H, Hkv, D)
        return [(x.reshape(T, -1, D), np.asarray(w).reshape(T, -1, D)) for x, w in zip(got, want)]

    def inputs():
        q, k, v = _inputs(gpu, zt, T, H, Hkv, D)
        return q, k, v, dev_normal(gpu, zt, T * H * D, SEED_DO)

    # dP = dO V^T: column 3 of dO large and of V zero, column 5 the other way round.
    q, k, v, do = inputs()
    v.view(T, Hkv, D)[:, :, 3], do.view(T, H, D)[:, :, 5] = 0.0, 0.0
    do.view(T, H, D)[50, -1, 3], v.view(T, Hkv, D)[40, -1, 5] = big, big
    dq, dk, dv = run(q, k, v, do)
    col = np.zeros((T, Hkv, D), bool)
    col[:, -1, 3] = True  # dv of the large column
    _close_by_part(*dq, [np.ones((T, H, D), bool)])
    _close_by_part(*dk, [np.ones((T, Hkv, D), bool)])
    _close_by_part(*dv, [col, ~col])

    # dK = dS^T Q: row 50's dS large, row 52's Q large in a column where K is zero.
    q, k, v, do = inputs()
    k.view(T, Hkv, D)[:, :, 7] = 0.0
    do.view(T, H, D)[50, -1, 3], q.view(T, H, D)[52, -1, 7] = big, big
    dk = run(q, k, v, do)[1]
    head = np.zeros((T, Hkv, D), bool)
    head[:, -1] = True
    _close_by_part(*dk, [head, ~head])

    # dQ = dS K: row 50's dS large, key 52's K large (hidden from row 50) in a column where Q is zero.
    q, k, v, do = inputs()
    q.view(T, H, D)[:, :, 7] = 0.0
    do.view(T, H, D)[50, -1, 3], k.view(T, Hkv, D)[52, -1, 7] = big, big
    dq = run(q, k, v, do)[0]
    row, col = np.zeros((T, H, D), bool), np.zeros((T, H, D), bool)
    row[50, -1], col[52:, H - g:, 7] = True, True
    _close_by_part(*dq, [row, col, ~(row | col)])

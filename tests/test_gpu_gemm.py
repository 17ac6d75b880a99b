"""GPU parity of the grouped expert GEMMs with the dequantisation fused in, against the CPU oracle's
P = s*digit -> fp32 GEMM on the same seeded inputs. Tolerance: 1e-3 relative L2 (the reference's
relerr, cudalm.cu:9842) for the bf16-MFMA kernels, 1e-5 for the fp32 kernels."""
import numpy as np
import pytest

from __graft_entry__ import load_package
from oracle.binding import make_spans

pkg = load_package()
f32 = np.float32
pytestmark = pytest.mark.gpu
TOL_MFMA = 1e-3
TOL_F32 = 1e-5


@pytest.fixture(scope="module")
def q():
    return pkg.load()


def dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def to_bf16_bits(t):
    """fp32 torch tensor holding bf16-representable values -> uint16 bit pattern tensor"""
    import torch
    return (t.view(torch.int32) >> 16).to(torch.int16)


def make_weights(orc, seed, E, rows, cols, group=128):
    """E expert matrices [rows, cols] encoded by the oracle; returns (d, s, rendered fp32 view)"""
    n = E * rows * cols
    tab, nq, ng = make_spans([n], group)
    P = orc.normal(n, seed, 1, 0.02)
    d = np.zeros(n // 2, np.int8); r = np.zeros(n, np.int8); s = np.zeros(ng, f32)
    orc.encode(P, d, r, s, tab, group, 7, 1, ng)
    orc.render(P, d, s, tab, group, 1, 0, ng)
    return d, s, P


def zipf_rows(total, E, seed):
    rng = np.random.default_rng(seed)
    p = (np.arange(E) + 1.0) ** -1.1
    p /= p.sum()
    cnt = rng.multinomial(total, p)
    return [int(c) for c in cnt]


def run_case(q, orc, mode, E, rowsM, K, N, act, math, seed=0, beta=0.0, group=128, nt_beta=1.0):
    """One grouped call over E experts with the given row counts. Returns (got list, want list)."""
    import torch
    tot = sum(rowsM)
    off = np.concatenate([[0], np.cumsum(rowsM)]).astype(int)
    bf = act == pkg.ACT_BF16
    if mode == "nt":
        A = orc.normal(tot * K, seed, 10); B = orc.normal(tot * N, seed, 11)
        if bf:
            A = orc.bf16_round(A); B = orc.bf16_round(B)
        C0 = orc.normal(E * K * N, seed, 12, 0.1)
        dA, dB, dC = dev(A), dev(B), dev(C0.copy())
        pa = to_bf16_bits(dA) if bf else dA
        pb = to_bf16_bits(dB) if bf else dB
        esz = 2 if bf else 4
        items = [(pa.data_ptr() + off[e] * K * esz, pb.data_ptr() + off[e] * N * esz, dC.data_ptr() + e * K * N * 4, 0, 0, rowsM[e], nt_beta)
                 for e in range(E)]
        pr = q.problems(items)
        q.gemm_nt(pr, E, K, N, act, math)
        torch.cuda.synchronize()
        want = C0.copy()
        for e in range(E):
            if rowsM[e]:
                if nt_beta == 0.0:
                    want[e * K * N:(e + 1) * K * N] = 0.0
                orc.gemm_nt(A[off[e] * K:], B[off[e] * N:], want[e * K * N:(e + 1) * K * N], rowsM[e], K, N)
        return dC.cpu().numpy(), want
    wr, wc = (K, N) if mode == "nn" else (N, K)
    d, s, P = make_weights(orc, seed, E, wr, wc, group)
    A = orc.normal(tot * K, seed, 10)
    if bf:
        A = orc.bf16_round(A)
    C0 = orc.normal(tot * N, seed, 12)
    dA, dC, dd, ds = dev(A), dev(C0.copy()), dev(d), dev(s)
    pa = to_bf16_bits(dA) if bf else dA
    esz = 2 if bf else 4
    items = [(pa.data_ptr() + off[e] * K * esz, None, dC.data_ptr() + off[e] * N * 4, e * wr * wc, e * wr * wc // group,
              rowsM[e], beta) for e in range(E)]
    pr = q.problems(items)
    (q.gemm_nn if mode == "nn" else q.gemm_tn)(dd, ds, group, pr, E, K, N, act, math)
    torch.cuda.synchronize()
    want = C0.copy()
    for e in range(E):
        if not rowsM[e]:
            continue
        w = P[e * wr * wc:(e + 1) * wr * wc]
        if mode == "nn":
            orc.gemm_nn(A[off[e] * K:], w, want[off[e] * N:off[e + 1] * N], rowsM[e], K, N)
        else:
            orc.gemm_tn(A[off[e] * K:], w, want[off[e] * N:off[e + 1] * N], rowsM[e], K, N, beta)
    return dC.cpu().numpy(), want


# ------------------------------------------------------------------ fp32 kernels
@pytest.mark.parametrize("mode", ["nn", "tn", "nt"])
def test_f32_ragged_small(q, orc, mode):
    """Ragged shapes incl. an empty expert and rows not a multiple of any tile (cudalm.cu:9919-9946 style)."""
    K, N = (128, 256) if mode != "tn" else (256, 128)
    got, want = run_case(q, orc, mode, 4, [67, 0, 5, 130], K, N, pkg.ACT_F32, pkg.MATH_F32, seed=3,
                         beta=1.0 if mode == "tn" else 0.0)
    assert orc.relerr(got, want) < TOL_F32


def test_f32_c1_single_expert(q, orc):
    """X fp32 [1024,512], 512->1536 up and 1536->512 down; forward, dgrad, wgrad."""
    for (K, N) in [(512, 1536), (1536, 512)]:
        for mode in ["nn", "tn", "nt"]:
            kk, nn = (K, N) if mode != "tn" else (N, K)
            got, want = run_case(q, orc, mode, 1, [1024], kk, nn, pkg.ACT_F32, pkg.MATH_F32, seed=0)
            assert orc.relerr(got, want) < TOL_F32, (mode, K, N)


def test_f32_c1_whole_chain_into_the_integer_step(q, orc):
    """BASELINE config 1 as one chain on its own two matrices: X fp32 [1024,512] ~ N(0,1), W_up [512,1536] and W_down
    [1536,512] from 0.02 N(0,1) through encode; H = X.W_up, Y = H.W_down; dH = dY.W_down^T, dX = dH.W_up^T;
    dW_down = H^T.dY, dW_up = X^T.dH with dY ~ N(0,1) (the configuration as the reference's test states it: no activation between the two);
    then one Integer AdamW step, t = 1, from fresh state (m8 = v8 = 0, moment scales 0) on both matrices with the weight
    gradients scaled to the config's 1e-3 (the device clip scalar: gsp). Every GEMM against the oracle's at 1e-5; the
    step byte for byte against the oracle's step fed the same gradient bits (the step's parity is defined on equal
    gradients: it rounds stochastically on every bit of them)."""
    import torch
    M, D, F, group, dmax = 1024, 512, 1536, 128, 7
    n_up, n_dn = D * F, F * D
    tab, nq, ng = make_spans([n_up, n_dn], group)
    P = orc.normal(nq, 0, 1, 0.02)
    hd = np.zeros(nq // 2, np.int8); hr = np.zeros(nq, np.int8); hs = np.zeros(ng, f32)
    orc.encode(P, hd, hr, hs, tab, group, dmax, 1, ng)
    orc.span_sref(tab, hs)
    orc.render(P, hd, hs, tab, group, 1, 0, ng)
    X = orc.normal(M * D, 0, 2); dY = orc.normal(M * D, 0, 3)
    dd, ds, dX_, ddY = dev(hd), dev(hs), dev(X), dev(dY)
    z = lambda k: torch.zeros(k, device="cuda")
    H, Y, dH, dXo, G = z(M * F), z(M * D), z(M * F), z(M * D), z(nq)
    one = lambda A, B, C, wq, beta=0.0: q.problems([(A, B, C, wq, wq // group, M, beta)])
    f = (pkg.ACT_F32, pkg.MATH_F32)
    q.gemm_nn(dd, ds, group, one(dX_, None, H, 0), 1, D, F, *f)
    q.gemm_nn(dd, ds, group, one(H, None, Y, n_up), 1, F, D, *f)
    q.gemm_tn(dd, ds, group, one(ddY, None, dH, n_up), 1, D, F, *f)
    q.gemm_tn(dd, ds, group, one(dH, None, dXo, 0), 1, F, D, *f)
    q.gemm_nt(q.problems([(H.data_ptr(), ddY.data_ptr(), G.data_ptr() + n_up * 4, 0, 0, M, 1.0)]), 1, F, D, *f)
    q.gemm_nt(q.problems([(dX_.data_ptr(), dH.data_ptr(), G.data_ptr(), 0, 0, M, 1.0)]), 1, D, F, *f)
    torch.cuda.synchronize()
    w_up, w_dn = P[:n_up], P[n_up:]
    hH = np.zeros(M * F, f32); orc.gemm_nn(X, w_up, hH, M, D, F)
    hY = np.zeros(M * D, f32); orc.gemm_nn(hH, w_dn, hY, M, F, D)
    hdH = np.zeros(M * F, f32); orc.gemm_tn(dY, w_dn, hdH, M, D, F, 0.0)
    hdX = np.zeros(M * D, f32); orc.gemm_tn(hdH, w_up, hdX, M, F, D, 0.0)
    hG = np.zeros(nq, f32); orc.gemm_nt(hH, dY, hG[n_up:], M, F, D); orc.gemm_nt(X, hdH, hG[:n_up], M, D, F)
    for name, got, want in [("H", H, hH), ("Y", Y, hY), ("dH", dH, hdH), ("dX", dXo, hdX), ("dW", G, hG)]:
        assert orc.relerr(got.cpu().numpy(), want) < TOL_F32, name
    # the step on the device's own gradient bits, scaled to ~1e-3 by the clip scalar
    gG = G.cpu().numpy()
    scale = np.array([1e-3 / float(np.sqrt(np.mean(gG.astype(np.float64) ** 2))), 0.0], f32)
    r, m8, v8 = dev(hr), torch.zeros(nq, dtype=torch.int8, device="cuda"), torch.zeros(nq, dtype=torch.uint8, device="cuda")
    m8s, v8s = z(ng), z(ng)
    hm8, hv8, hm8s, hv8s = np.zeros(nq, np.int8), np.zeros(nq, np.uint8), np.zeros(ng, f32), np.zeros(ng, f32)
    bc1, bc2 = f32(1) - f32(0.9), f32(1) - f32(0.95)
    span_bytes = tab.view(np.uint8)
    hp = (3e-4, 0.9, 0.95, 0.1, 1.0)
    tail = (float(f32(1) / bc1), float(f32(1) / np.sqrt(bc2)), 0, 1, 1, None, 1, 0, ng)
    q.step(None, G, dd, r, ds, m8, m8s, v8, v8s, dev(span_bytes), 2, group, dmax, *hp, dev(scale), *tail)
    orc.step(None, gG, hd, hr, hs, hm8, hm8s, hv8, hv8s, tab, group, dmax, *hp, scale, *tail)
    torch.cuda.synchronize()
    assert int((hm8 != 0).sum()) > nq // 2 and int((hv8 != 0).sum()) > nq // 2        # the step did something
    for name, got, want in [("d", dd, hd), ("r", r, hr), ("m8", m8, hm8), ("v8", v8, hv8), ("m8s", m8s, hm8s), ("v8s", v8s, hv8s)]:
        assert np.array_equal(got.cpu().numpy().view(np.uint8), want.view(np.uint8)), name


def test_f32_bf16_acts_and_group64(q, orc):
    got, want = run_case(q, orc, "nn", 3, [40, 1, 77], 192, 128, pkg.ACT_BF16, pkg.MATH_F32, seed=5, group=64)
    assert orc.relerr(got, want) < TOL_F32
    got, want = run_case(q, orc, "tn", 3, [40, 1, 77], 128, 192, pkg.ACT_BF16, pkg.MATH_F32, seed=6, group=64)
    assert orc.relerr(got, want) < TOL_F32


@pytest.mark.parametrize("mode,K,N,rows,act", [
    ("nn", 40, 3072, [2049], "f32"), ("tn", 128, 3080, [2047], "f32"), ("nt", 2048, 3072, [33], "f32"),      # 64x64 outputs per workgroup
    ("nn", 136, 512, [1, 513, 31], "f32"), ("tn", 128, 264, [577], "bf16"), ("nt", 520, 512, [0, 129], "bf16"),  # 32x32, four along the contraction
    ("nn", 392, 128, [9, 1, 33], "f32"), ("tn", 640, 72, [5], "f32"), ("nt", 40, 72, [300, 7], "f32"),        # 32x32, sixteen
    ("nn", 37, 128, [50, 6], "f32"), ("tn", 128, 45, [66], "bf16"), ("nt", 45, 37, [101], "f32")])            # units put together element by element
def test_f32_shapes_of_a_workgroup(q, orc, mode, K, N, rows, act):
    got, want = run_case(q, orc, mode, len(rows), rows, K, N, pkg.ACT_F32 if act == "f32" else pkg.ACT_BF16, pkg.MATH_F32, seed=11,
                         beta=1.0 if mode == "tn" else 0.0)
    assert orc.relerr(got, want) < TOL_F32


@pytest.mark.parametrize("mode", ["nn", "tn"])
@pytest.mark.parametrize("lo,hi,x", [(120, 127.9, -40), (-149, -127, 60), (-60, -40, -86)])
def test_f32_scales_and_inputs_at_the_ends_of_the_range(q, mode, lo, hi, x):
    """A weight is the product s * digit, finite where that is: scales above 2^124, whose sixteenfold is not; subnormal scales;
    subnormal products."""
    import torch
    M, K, N, group = 40, 64, 64, 32
    rng = np.random.default_rng(5)
    d = rng.integers(-1, 2, K * N)
    s = (2.0 ** rng.uniform(lo, hi, K * N // group)).astype(f32)
    W = (np.repeat(s, group) * d.astype(f32)).astype(np.float64).reshape((K, N) if mode == "nn" else (N, K))
    A = (rng.standard_normal((M, K)) * 2.0 ** x).astype(f32)
    want = A.astype(np.float64) @ (W if mode == "nn" else W.T)
    C = torch.zeros(M, N, device="cuda")
    packed = (d[0::2] & 15 | (d[1::2] & 15) << 4).astype(np.uint8)
    (q.gemm_nn if mode == "nn" else q.gemm_tn)(dev(packed), dev(s), group, q.problems([(dev(A), None, C, 0, 0, M, 0.0)]), 1, K, N, pkg.ACT_F32, pkg.MATH_F32)
    got = C.cpu().numpy().astype(np.float64)
    assert np.isfinite(got).all()
    assert np.linalg.norm(got - want) < TOL_F32 * np.linalg.norm(want)


def f32_call(q, mode, A, X, digits, s, group, rows, K, N, beta=0.0):
    """One fp32 call over the problems of `rows`; A [rows, K] and X the old output or, for nt, dY [rows, N]. Returns the output and what
    64 bits give for it, the weight the fp32 product s * digit."""
    import torch
    E, off = len(rows), np.concatenate([[0], np.cumsum(rows)])
    if mode == "nt":
        C = torch.zeros(E * K * N, device="cuda")
        a, b = dev(A), dev(X)
        probs = [(a.data_ptr() + off[e] * K * 4, b.data_ptr() + off[e] * N * 4, C.data_ptr() + e * K * N * 4, 0, 0, rows[e], 0.0) for e in range(E)]
        q.gemm_nt(q.problems(probs), E, K, N, pkg.ACT_F32, pkg.MATH_F32)
        with np.errstate(all="ignore"):
            want = np.concatenate([(A[off[e]:off[e + 1]].astype(np.float64).T @ X[off[e]:off[e + 1]].astype(np.float64)).ravel() for e in range(E)])
        return C.cpu().numpy().astype(np.float64), want
    with np.errstate(all="ignore"):
        W = (np.repeat(s, group) * digits.astype(f32)).astype(np.float64).reshape((E, K, N) if mode == "nn" else (E, N, K))
        want = np.concatenate([A[off[e]:off[e + 1]].astype(np.float64) @ (W[e] if mode == "nn" else W[e].T) for e in range(E)]) + beta * X
    C, a = dev(X), dev(A)
    packed = (digits[0::2] & 15 | (digits[1::2] & 15) << 4).astype(np.uint8)
    probs = [(a.data_ptr() + off[e] * K * 4, None, C.data_ptr() + off[e] * N * 4, e * K * N, e * K * N // group, rows[e], beta) for e in range(E)]
    (q.gemm_nn if mode == "nn" else q.gemm_tn)(dev(packed), dev(s), group, q.problems(probs), E, K, N, pkg.ACT_F32, pkg.MATH_F32)
    return C.cpu().numpy().astype(np.float64), want


def f32_inputs(seed, mode, rows, K, N, group):
    rng = np.random.default_rng(seed)
    n = len(rows) * K * N
    digits = rng.integers(-7, 8, n) if mode != "nt" else None
    s = (rng.uniform(0.5, 1.5, n // group) * 0.0086).astype(f32) if mode != "nt" else None
    return rng.standard_normal((sum(rows), K)).astype(f32), rng.standard_normal((sum(rows), N)).astype(f32), digits, s


@pytest.mark.parametrize("mode,K,N,group,rows", [
    ("nn", 64, 64, 64, [1, 33]), ("nn", 320, 192, 64, [31, 2, 65]), ("nn", 768, 256, 128, [4]), ("nn", 1536, 256, 256, [100]),
    ("tn", 64, 64, 64, [1, 33]), ("tn", 320, 45, 64, [31, 0, 65]), ("tn", 1536, 72, 128, [4]), ("tn", 512, 66, 256, [100]),
    ("nt", 1024, 1028, 0, [1]), ("nt", 1156, 1028, 0, [2, 31, 33]), ("nt", 68, 132, 0, [127, 40]), ("nt", 64, 64, 0, [128]), ("nt", 132, 260, 0, [300, 0, 97]),
    ("nt", 1028, 964, 0, [192, 1]), ("nt", 64, 132, 0, [191, 63]), ("nt", 68, 64, 0, [193, 224, 256, 289]), ("nt", 4, 4, 0, [1000])])
def test_f32_in_three_parts(q, mode, K, N, group, rows):
    """The fp32 products as products of bf16 parts, at the edges of their tiles and steps. Against 64 bits: one rounding of the weight or
    of activation times scale, and at most three (nt: six) roundings per sixteen of the contraction, each half a unit (2^-24) of a running sum
    that is, root mean square, within the size of the result."""
    A, X, digits, s = f32_inputs(41, mode, rows, K, N, group)
    got, want = f32_call(q, mode, A, X, digits, s, group, rows, K, N, beta=1.0 if mode == "tn" else 0.0)
    depth = max(rows) if mode == "nt" else K
    assert np.linalg.norm(got - want) < 2.0 ** -24 * (1 + np.sqrt((6 if mode == "nt" else 3) * (depth / 16 + 1))) * np.linalg.norm(want)


@pytest.mark.parametrize("mode", ["nn", "tn", "nt"])
@pytest.mark.parametrize("where,value", [("row", np.inf), ("row", np.nan), ("one", np.inf), ("one", 3.4e38), ("all", 2.0 ** 61), ("all", 2.0 ** -111),
                                         ("all", 2.0 ** -104), ("one", 2.0 ** -140), ("scale", 2.0 ** 51), ("scale", 2.0 ** -130)])
def test_f32_parts_leave_what_they_do_not_hold(q, mode, where, value):
    """Infinities, values and scales at the ends of the range, and NaN: what 64 bits give, rounded to fp32, the same elements infinite or not a
    number; finite sums to the relative error of fp32 sums."""
    if mode == "nt" and where == "scale":
        pytest.skip("no scales")
    K, N, group, rows = 192, 128, 64, [40, 130]
    A, X, digits, s = f32_inputs(42, mode, rows, K, N, group)
    if mode == "nt" and where == "all" and value < 1:
        X *= f32(2.0 ** 20)                              # products stay above the subnormals, whose last place is a fixed size
    if where == "row": A[7, 3::5] = value
    elif where == "one": A[50, 9] = value
    elif where == "all": A *= f32(value)
    else: s *= f32(value / 0.0086)
    old = np.zeros_like(X)
    got, want = f32_call(q, mode, A, X if mode == "nt" else old, digits, s, group, rows, K, N)
    with np.errstate(all="ignore"):
        want = want.astype(f32).astype(np.float64)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want))
    ok = np.isfinite(want)
    assert np.array_equal(np.sign(got[np.isinf(got)]), np.sign(want[np.isinf(want)]))
    scale = np.abs(want[ok]).max()
    assert np.linalg.norm((got[ok] - want[ok]) / scale) < TOL_F32 * np.linalg.norm(want[ok] / scale)


@pytest.mark.parametrize("mode", ["nn", "tn", "nt"])
@pytest.mark.parametrize("rows", [[40], [130]])
@pytest.mark.parametrize("n,big", [(104, 0), (109, 0), (112, 0), (118, 0), (121, 0), (125, 0), (130, 0), (138, 0), (145, 0), (121, 60), (130, 110)])
def test_f32_small_values_beside_large_ones(q, mode, n, big, rows):
    """Values of some 2^-n beside others, of some 2^big, whose products vanish -- the digit is 0, the gradient is 0 -- so that the small values are the
    result, column by column: the sums of K products to the roundings of up to K/16 + 24 additions (2^-24 of the terms' magnitudes each) and,
    where the numbers end, half the last place (2^-150) per product and addition."""
    K, N, group = 256, 128, 64
    rng = np.random.default_rng(43)
    A, X, digits, s = f32_inputs(43, mode, rows, K, N, group)
    small = f32(2.0) ** f32(-n)
    if mode == "nt":                                     # a token every eight is ordinary in A and 0 in X
        lift = f32(2.0 ** 40)
        keep = np.arange(rows[0]) % 8 == 0
        A[~keep] *= small; A[keep] *= f32(2.0 ** big); X[keep] = 0.0; X *= lift
        terms = np.abs(A.astype(np.float64)).T @ np.abs(X.astype(np.float64))
        grid, depth = 0.0, rows[0]
    else:                                                # one of the contraction every eight is ordinary in A and has digits 0
        keep = np.arange(K) % 8 == 0
        A[:, ~keep] *= small; A[:, keep] *= f32(2.0 ** big)
        W = digits.reshape((K, N) if mode == "nn" else (N, K))
        if mode == "nn": W[keep] = 0
        else: W[:, keep] = 0
        digits = np.ascontiguousarray(W).reshape(-1)
        s[:] = rng.uniform(0.5, 1.5, s.shape).astype(f32)
        w = np.repeat(s, group).astype(np.float64) * np.abs(digits)
        terms = np.abs(A.astype(np.float64)) @ (w.reshape(K, N) if mode == "nn" else w.reshape(N, K).T)
        grid, depth = 1.0, K
    got, want = f32_call(q, mode, A, X if mode == "nt" else np.zeros_like(X), digits, s, group, rows, K, N)
    bound = (depth / 16 + 24) * 2.0 ** -24 * terms.reshape(want.shape) + 8 * (1 + depth * grid) * 2.0 ** -150
    assert (np.abs(got - want) <= bound).all(), (np.abs(got - want) / bound).max()


@pytest.mark.parametrize("mode,M,K,N", [("nt", 1, 512, 256), ("nt", 2, 512, 256), ("nt", 31, 512, 256), ("nt", 32, 512, 256), ("nt", 64, 512, 260),
                                        ("nt", 1024, 64, 128), ("nt", 1024, 512, 512), ("nt", 4096, 256, 512), ("nt", 16384, 64, 64),
                                        ("nn", 1, 8192, 512), ("nn", 40, 8192, 128), ("nn", 64, 16384, 128), ("nn", 300, 512, 512),
                                        ("tn", 1, 8192, 512), ("tn", 40, 8192, 64), ("tn", 64, 16384, 128)])
def test_f32_parts_are_no_further_off_than_the_fp32_core(q, mode, M, K, N):
    """Relative error against 64 bits of a call whose operands lie on 16 bytes (bf16 parts) and of the same call on operands a float further (fp32
    matrix core), many additions of few outputs among them. Nothing is added to the core's error but 2 % for chance in the last bits."""
    import torch
    g = torch.Generator(device="cuda").manual_seed(7)
    rnd = lambda n: torch.randn(n + 4, generator=g, device="cuda")
    err = []
    a, b, group = rnd(M * K), rnd(M * N), 64
    digits = torch.randint(-7, 8, (K * N,), generator=g, device="cuda")
    packed = ((digits[0::2] & 15) | (digits[1::2] & 15) << 4).to(torch.uint8)
    s = torch.rand(K * N // group, generator=g, device="cuda") * 0.0086 + 0.001
    if mode != "nt":
        W = (s.double().repeat_interleave(group) * digits.double()).view((K, N) if mode == "nn" else (N, K))
    for off in (0, 1):
        A, B = a[off:off + M * K], b[off:off + M * N]
        C = torch.zeros(K * N if mode == "nt" else M * N, device="cuda")
        if mode == "nt":
            q.gemm_nt(q.problems([(A.data_ptr(), B.data_ptr(), C.data_ptr(), 0, 0, M, 0.0)]), 1, K, N, pkg.ACT_F32, pkg.MATH_F32)
            want = A.view(M, K).double().t() @ B.view(M, N).double()
        else:
            (q.gemm_nn if mode == "nn" else q.gemm_tn)(packed, s, group, q.problems([(A.data_ptr(), None, C.data_ptr(), 0, 0, M, 0.0)]), 1, K, N,
                                                       pkg.ACT_F32, pkg.MATH_F32)
            want = A.view(M, K).double() @ (W if mode == "nn" else W.t())
        err.append(float((C.view(want.shape).double() - want).norm() / want.norm()))
    assert err[0] <= 1.02 * err[1], err


@pytest.mark.parametrize("mode,K,N,math,company", [("nn", 768, 2048, "f16", [600]), ("tn", 768, 2048, "mfma", [3000]), ("nn", 768, 512, "f32", [3000]),
                                                   ("nn", 768, 512, "f32", [13000]), ("tn", 768, 512, "f32", [3000])])
@pytest.mark.parametrize("M", [3, 16])
def test_rows_alone_and_in_company(q, orc, mode, K, N, math, company, M):
    """The kernel, and with it the order of the sums, is chosen by the sizes of the whole call: a problem's rows come out with the
    same bits in every call of the same sizes, and beside other problems within what two orders of K fp32 additions differ by
    (each within sqrt(K) * 2^-24 of the exact sum: 3.3e-6 for both)."""
    act, m = (pkg.ACT_F32, pkg.MATH_F32) if math == "f32" else (pkg.ACT_BF16, pkg.MATH_MFMA_F16 if math == "f16" else pkg.MATH_MFMA)
    alone, _ = run_case(q, orc, mode, 1, [M], K, N, act, m, seed=31)
    again, _ = run_case(q, orc, mode, 1, [M], K, N, act, m, seed=31)
    beside, _ = run_case(q, orc, mode, 2, [M] + company, K, N, act, m, seed=31)
    assert np.array_equal(alone.view(np.uint32), again.view(np.uint32))
    assert orc.relerr(beside[:M * N], alone) < 3.3e-6


# ------------------------------------------------------------------ bf16 MFMA kernels
@pytest.mark.parametrize("mode", ["nn", "tn", "nt"])
def test_mfma_grouped_zipf_small(q, orc, mode):
    """8 experts, Zipf row counts incl. tiny and empty experts, D=256 F=384."""
    rows = zipf_rows(1500, 8, 1)
    rows[5] = 0
    rows[6] = 1
    K, N = {"nn": (256, 384), "tn": (384, 256), "nt": (256, 384)}[mode]
    got, want = run_case(q, orc, mode, 8, rows, K, N, pkg.ACT_BF16, pkg.MATH_MFMA, seed=2,
                         beta=1.0 if mode == "tn" else 0.0)
    err = orc.relerr(got, want)
    assert err < TOL_MFMA, err


@pytest.mark.parametrize("mode,K,N,group", [("nn", 768, 256, 128), ("nn", 32, 128, 64), ("nn", 96, 384, 64), ("nn", 2048, 512, 256),
                                            ("tn", 768, 256, 128), ("tn", 64, 128, 64), ("tn", 192, 384, 64), ("tn", 2048, 128, 256)])
@pytest.mark.parametrize("rows", [[1], [16, 0, 9], [17, 32, 3, 31], [33, 64, 48]])
def test_mfma_few_rows(q, orc, mode, K, N, group, rows):
    """The kernels for experts of few rows: every row tile, contractions shorter than a step per wavefront, scale groups
    that split a lane group's columns, both load widths of the input gradient; beta 0 and 1."""
    for beta in ((0.0,) if mode == "nn" else (0.0, 1.0)):
        got, want = run_case(q, orc, mode, len(rows), rows, K, N, pkg.ACT_BF16, pkg.MATH_MFMA_F16 if mode == "nn" else pkg.MATH_MFMA,
                             seed=21, beta=beta, group=group)
        assert orc.relerr(got, want) < (4e-4 if mode == "nn" else 3e-6)


@pytest.mark.parametrize("K,N,rows,group", [(32, 2048, [1, 16, 0, 9] * 7, 128), (64, 1152, [20, 0] * 35, 128),          # strips of 128 columns; fewer steps than wavefronts
                                            (32, 2048, [1, 16, 0, 9] * 17, 128),                                          # the plain call on strips of 256: 408 of them, from three of 128 to a CU
                                            (512, 2048, [1, 16, 0, 9] * 8, 128), (512, 2048, [1, 16, 0, 9] * 8, 256),     # 192 of 256, gate|up too
                                            (384, 2048, [7] * 20, 128), (384, 2048, [7] * 19, 128),                       # 160, gate|up only, and fewer
                                            (512, 1408, [16, 3] * 16, 128), (512, 1408, [7] * 43, 128),                   # half a strip at the end; 258 of 256 and 473 of 128
                                            (512, 2048, [7] * 32, 128), (512, 2048, [7] * 33, 256),                       # a full round, and 264: the plain call
                                            (512, 2048, [5] * 48, 128), (768, 4096, [7] * 22, 128),                       # beyond: three of 128 to a CU; 352, a large matrix
                                            (768, 2048, [17, 32, 1, 16] * 6, 256), (640, 2048, [17, 32, 1, 16] * 6, 128),      # more than 16 rows, one scale for both halves; gate|up on 128
                                            (768, 3968, [31, 5, 16, 17, 2] * 2 + [3], 128), (768, 3840, [31, 5, 16] * 4, 128),      # either side of 3 M weights; half a strip at the end
                                            (2048, 384, [16, 1, 0, 7], 128), (2048, 512, [32, 17, 9], 256), (2080, 128, [5], 128),     # eight wavefronts along the contraction
                                            (2048, 256, [3, 17] * 33, 128), (2048, 256, [16, 3] * 33, 256),                    # 132 strips: gate|up on 128 columns, up to there on 64
                                            (2048, 1152, [32, 17, 9], 128),                                               # four
                                            (160, 384, [70, 5, 0, 33, 9, 9, 2], 128), (576, 384, [129, 64, 1], 64),               # larger problems on 32 rows, gate|up on 64
                                            (96, 256, [70, 3] + [5] * 70, 128), (544, 1152, [97, 34, 0, 31] * 4, 64),    # both on 32
                                            (1056, 896, [64, 40, 34] * 16, 128)])                                        # both on 64
def test_f16_forward_of_few_rows_in_every_form(q, K, N, rows, group):
    """The shapes of the forward of few rows, at most 32 per problem and more: products with the weights rounded once to fp16, within what K fp32 additions
    in some order differ from 64 bits by (sqrt(K) * 2^-24 relative to the sums, four times that for their cancelling), and the same bits with the row moves and the SwiGLU
    folded in."""
    import torch
    E, R = len(rows), sum(rows)
    g = torch.Generator(device="cuda"); g.manual_seed(K + N + E)
    digit = torch.randint(-8, 8, (2, E, K, N), generator=g, device="cuda", dtype=torch.int8)
    scale = (torch.rand(2, E, K, N // group, generator=g, device="cuda") + 0.5) * 0.01
    nib = digit.reshape(-1).to(torch.uint8) & 15
    d, s = (nib[0::2] | nib[1::2] << 4).view(torch.int8), scale.reshape(-1)
    w = (scale.repeat_interleave(group, 3) * digit * 256).half().double() / 256
    x = torch.randn(R + 5, K, generator=g, device="cuda").bfloat16()
    idx = torch.randperm(R + 5, generator=g, device="cuda")[:R].int()
    A = x[idx.long()].contiguous()
    at = np.concatenate([[0], np.cumsum(rows)]).astype(int)
    n = E * K * N
    out = {k: torch.full((R, N), 3.0, device="cuda") for k in ("g", "u", "gg", "gp", "up")}
    act = torch.zeros(R, N, device="cuda", dtype=torch.bfloat16)
    spread = torch.zeros(R + 5, N, device="cuda")

    def lists(C, first, src=None, B=None):
        return q.problems([((src.data_ptr() + int(at[e]) * 4) if src is not None else A.data_ptr() + int(at[e]) * K * 2, None if B is None else B.data_ptr() + int(at[e]) * N * 2,
                            C.data_ptr() + int(at[e]) * (4 if C is idx else N * 4), first * n + e * K * N, (first * n + e * K * N) // group, rows[e], 0.0) for e in range(E)])
    bf = pkg.ACT_BF16, pkg.MATH_MFMA_F16
    q.gemm_nn(d, s, group, lists(out["g"], 0), E, K, N, *bf)
    q.gemm_nn(d, s, group, lists(out["u"], 1), E, K, N, *bf)
    q.gemm_nn_gather(d, s, group, lists(out["gg"], 0, idx), E, K, N, x)
    q.gemm_nn_scatter(d, s, group, lists(idx, 0), E, K, N, spread, None)
    q.gemm_nn_gather_swiglu(d, s, group, lists(out["gp"], 0, idx), lists(out["up"], 1, None, act), E, K, N, x)
    torch.cuda.synchronize()
    tol = 4 * K ** 0.5 * 2.0 ** -24
    for m, k in enumerate("gu"):
        for e in range(E):
            if rows[e]:
                want = A[at[e]:at[e + 1]].double().cpu() @ w[m, e].cpu()
                got = out[k][at[e]:at[e + 1]].double().cpu()
                assert float((got - want).norm() / want.norm()) < tol, (k, e)
    assert torch.equal(out["gg"], out["g"]) and torch.equal(out["gp"], out["g"]) and torch.equal(out["up"], out["u"])
    assert torch.equal(spread[idx.long()], out["g"])
    fused = (out["g"] * torch.sigmoid(out["g"]) * out["u"]).bfloat16().float()
    assert float((act.float() - fused).abs().max()) <= float(fused.abs().max()) * 2.0 ** -7


@pytest.mark.parametrize("mode,math", [("nn", "f16"), ("tn", "mfma"), ("nn", "f32"), ("tn", "f32")])
@pytest.mark.parametrize("M", [5, 40, 100])
def test_few_rows_outputs_at_any_float(q, orc, mode, math, M):
    """An output that begins four bytes behind a 16-byte boundary, as a view into a larger buffer may: the same bits as on the
    boundary, and nothing written before or behind."""
    import torch
    K, N = 256, 128
    act, m = (pkg.ACT_F32, pkg.MATH_F32) if math == "f32" else (pkg.ACT_BF16, pkg.MATH_MFMA_F16 if math == "f16" else pkg.MATH_MFMA)
    d, s, _ = make_weights(orc, 41, 1, *((K, N) if mode == "nn" else (N, K)))
    A = dev(orc.bf16_round(orc.normal(M * K, 41, 1))); a = A if math == "f32" else to_bf16_bits(A)
    dd, ds = dev(d), dev(s)
    outs = []
    for at in (4, 5):
        buf = torch.full((M * N + 9,), 3.0, device="cuda")
        (q.gemm_nn if mode == "nn" else q.gemm_tn)(dd, ds, 128, q.problems([(a, None, buf.data_ptr() + 4 * at, 0, 0, M, 1.0 if mode == "tn" else 0.0)]),
                                                   1, K, N, act, m)
        outs.append(buf[at:at + M * N].clone())
        assert bool((buf[:at] == 3.0).all()) and bool((buf[at + M * N:] == 3.0).all())
    assert torch.equal(outs[0], outs[1])


@pytest.mark.parametrize("K,N,group", [(768, 256, 128), (128, 128, 64), (2048, 256, 256)])
@pytest.mark.parametrize("rows", [[65, 1, 130, 34], [257]])
def test_mfma_few_tiles(q, orc, K, N, group, rows):
    """Calls with too few tiles for the tiled kernels take the kernels for few rows with 64-row tiles: last tiles of every
    height behind whole ones, alone, paired and with the SwiGLU behind."""
    for mode, tol in (("nn", 4e-4), ("tn", 3e-6)):
        got, want = run_case(q, orc, mode, len(rows), rows, K, N, pkg.ACT_BF16, pkg.MATH_MFMA_F16 if mode == "nn" else pkg.MATH_MFMA, seed=23,
                             beta=1.0 if mode == "tn" else 0.0, group=group)
        assert orc.relerr(got, want) < tol
    if group == 128:
        got, want = _pair_case(q, orc, rows, K, N, pkg.ACT_BF16, pkg.MATH_MFMA, 1.0, seed=24)
        assert orc.relerr(got, want) < 3e-6
        (f, sep), want = _swiglu_case(q, orc, rows, K, N, pkg.ACT_BF16, pkg.MATH_MFMA_F16, seed=25)
        assert orc.relerr(f[0], want) < 4e-4
        for a, b in zip(f[:2], sep[:2]):
            assert np.array_equal(a.view(np.uint32), b.view(np.uint32))


@pytest.mark.parametrize("K,N,rows", [(576, 1024, [100, 896]), (576, 1024, [129, 896]), (512, 1024, [100, 896]),     # 128 strips of 64 x 128, and over
                                      (1152, 1152, [33] + [20] * 40), (1152, 1152, [65] + [40] * 40),        # 41 of 9: few rows to a problem, and more
                                      (1152, 1280, [50] + [23] * 40), (1152, 1280, [65] + [23] * 40),
                                      (1024, 256, [1000] * 11), (1024, 256, [1000] * 17),                    # four times the width, up to 512 strips
                                      (544, 1024, [33] * 16), (544, 1024, [33] * 17), (512, 1024, [33] * 16),                 # 32 rows x 128: 256 of them, and over
                                      (96, 1408, [97] + [7] * 27), (96, 1408, [97] + [7] * 28), (64, 2816, [65, 33] + [32] * 13),     # to 352 and over, more or less of them than taller ones
                                      (64, 1408, [300, 0, 64] + [1, 31, 33] * 11), (64, 1408, [33] * 64),
                                      (96, 128, [33] + [5] * 40), (96, 256, [70] + [5] * 61), (96, 256, [70] + [5] * 62)])     # gate|up on 64 rows, up to 128 of 32; on 32
def test_f16_forward_on_both_sides_of_the_lines(q, orc, K, N, rows):
    """The sizes of a call choose between the kernels for few rows and the tiled ones; on either side of each line the SwiGLU call
    gives the bits of the separate ones, and both the oracle's values."""
    (f, sep), want = _swiglu_case(q, orc, rows, K, N, pkg.ACT_BF16, pkg.MATH_MFMA_F16, seed=26)
    assert orc.relerr(f[0], want) < 4e-4            # one rounding of the weights to 11 bits
    for a, b in zip(f[:2], sep[:2]):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))


@pytest.mark.parametrize("mode,K,N", [("nn", 768, 2048), ("nn", 2048, 768), ("tn", 768, 2048), ("tn", 2048, 768),
                                      ("nt", 768, 2048), ("nt", 2048, 768)])
def test_mfma_layer_shapes(q, orc, mode, K, N):
    """The 32-expert D=768 F=2048 layer's GEMM shapes on a 4-expert slice with Zipf rows (the CPU
    oracle finishes these in seconds)."""
    rows = zipf_rows(1100, 4, 7)
    got, want = run_case(q, orc, mode, 4, rows, K, N, pkg.ACT_BF16, pkg.MATH_MFMA, seed=4)
    err = orc.relerr(got, want)
    assert err < TOL_MFMA, err


# ------------------------------------------------------------------ forward on the fp16 matrix core
@pytest.mark.parametrize("K,N,rows", [(768, 2048, None), (2048, 768, None), (256, 384, [300, 0, 64, 1, 129, 517, 193, 255]),
                                      (32, 128, [5, 700]), (64, 256, [1, 65, 130, 200, 256, 257])])
def test_mfma_f16_forward_vs_oracle(q, orc, K, N, rows):
    """QLMX_MATH_MFMA_F16: bf16 activations converted exactly, weights rounded once to fp16, one MFMA per product.
    Tolerance 1e-3 relative L2 against the oracle's fp32 GEMM on the rendered weights; the rounding of s*digit to
    11 bits predicts about 2e-4. Every last-tile height, empty experts, single-step contractions."""
    rows = rows or zipf_rows(1100, 4, 7)
    got, want = run_case(q, orc, "nn", len(rows), rows, K, N, pkg.ACT_BF16, pkg.MATH_MFMA_F16, seed=4)
    err = orc.relerr(got, want)
    print("fp16 forward K=%d N=%d: relative L2 %.2e" % (K, N, err))
    assert err < 1e-3, err
    assert err < 4e-4, err          # observed 1.5e-4 .. 2.5e-4
    # rows of empty experts and everything outside the written tiles stay as they were
    off = np.concatenate([[0], np.cumsum(rows)]).astype(int)
    assert got.size == off[-1] * N


@pytest.mark.parametrize("E,M,K,N,group", [(16, 1000, 32, 640, 64), (12, 530, 96, 1152, 128), (16, 700, 96, 384, 64), (20, 700, 160, 384, 128),
                                           (5, 300, 32, 384, 64), (40, 128, 224, 128, 32)])
def test_mfma_f16_forward_tile_shapes(q, E, M, K, N, group):
    """The five tile shapes of the fp16 forward, with and without half a step at the end and a narrow tile at a row's end, plain, behind a gather with
    the SwiGLU and in front of a scatter. A weight is rounded once, by at most 2^-11 of it over 1 to 2, uniformly: 2^-11 / sqrt(3) of the
    result bounds the root mean square. The fused forms see the same products: the same bits."""
    import torch
    rng = np.random.default_rng(77)
    rows = [M] * (E - 3) + [M + 1, 0, M - 1]
    off = np.concatenate([[0], np.cumsum(rows)]).astype(int)
    R, n = int(off[-1]), E * K * N
    digits = rng.integers(-7, 8, 2 * n).astype(np.int8)
    s = (rng.uniform(0.5, 1.5, 2 * n // group) * 0.0086).astype(f32)
    dd, ds = dev((digits[0::2] & 15 | (digits[1::2] & 15) << 4).astype(np.uint8)), dev(s)
    x = dev(rng.standard_normal((R, K)).astype(f32)).bfloat16()
    tok = torch.from_numpy(rng.permutation(R).astype(np.int32)).cuda()
    xs = x[tok.long()].contiguous()
    sep = [torch.full((R, N), 7.0, device="cuda") for _ in range(2)]
    for m in range(2):
        q.gemm_nn(dd, ds, group, q.problems([(xs.data_ptr() + off[e] * K * 2, None, sep[m].data_ptr() + off[e] * N * 4, m * n + e * K * N, (m * n + e * K * N) // group,
                                              rows[e], 0.0) for e in range(E)]), E, K, N, pkg.ACT_BF16, pkg.MATH_MFMA_F16)
    W = (np.repeat(s[:n // group], group).astype(np.float64) * digits[:n]).reshape(E, K, N)
    xh = xs.float().cpu().numpy().astype(np.float64)
    want = np.concatenate([xh[off[e]:off[e + 1]] @ W[e] for e in range(E)])
    got = sep[0].cpu().numpy()
    assert np.linalg.norm(got - want) < 2.0 ** -11 / np.sqrt(3) * np.linalg.norm(want)
    if group >= 64:
        gp, up, act = torch.full((R, N), 7.0, device="cuda"), torch.full((R, N), 7.0, device="cuda"), torch.zeros(R, N, device="cuda", dtype=torch.bfloat16)
        q.gemm_nn_gather_swiglu(dd, ds, group, q.problems([(tok.data_ptr() + off[e] * 4, None, gp.data_ptr() + off[e] * N * 4, e * K * N, e * K * N // group, rows[e], 0.0)
                                                           for e in range(E)]),
                                q.problems([(0, act.data_ptr() + off[e] * N * 2, up.data_ptr() + off[e] * N * 4, n + e * K * N, (n + e * K * N) // group, rows[e], 0.0)
                                            for e in range(E)]), E, K, N, x)
        assert torch.equal(gp, sep[0]) and torch.equal(up, sep[1])
        z = sep[0].double()
        assert torch.allclose(act.double(), z * torch.sigmoid(z) * sep[1].double(), rtol=2.0 ** -8, atol=1e-6)      # one rounding to bf16
    gate, out = dev(rng.uniform(0.1, 1.0, R).astype(f32)), dev(rng.standard_normal((R, N)).astype(f32))
    ref = out.clone()
    ref[tok.long()] += gate[tok.long()].unsqueeze(1) * sep[0]
    q.gemm_nn_scatter(dd, ds, group, q.problems([(xs.data_ptr() + off[e] * K * 2, None, tok.data_ptr() + off[e] * 4, e * K * N, e * K * N // group, rows[e], 0.0)
                                                 for e in range(E)]), E, K, N, out, gate)
    assert torch.equal(out, ref)


@pytest.mark.parametrize("rows,K,N", [([700] * 14 + [701, 699, 0], 96, 192), ([300, 65, 129, 193, 255], 160, 320), ([130] * 40, 64, 704), ([1000, 1, 257], 96, 64),
                                      ([530] * 12, 608, 448), ([190] * 64, 224, 192)])
@pytest.mark.parametrize("gathered", [False, True])
def test_swiglu_forward_of_odd_halves(q, rows, K, N, gathered):
    """gate | up with SwiGLU where the columns are an odd multiple of 64, so that a launch of wide tiles ends in narrow ones: pre-activations against 64
    bits (bound as above), the activation from them, and nothing behind the last row."""
    import torch
    group, E, rng = 64, len(rows), np.random.default_rng(79)
    off = np.concatenate([[0], np.cumsum(rows)]).astype(int)
    R, n = int(off[-1]), E * K * N
    digits = rng.integers(-7, 8, 2 * n).astype(np.int8)
    s = (rng.uniform(0.5, 1.5, 2 * n // group) * 0.0086).astype(f32)
    dd, ds = dev((digits[0::2] & 15 | (digits[1::2] & 15) << 4).astype(np.uint8)), dev(s)
    x = dev(rng.standard_normal((R, K)).astype(f32)).bfloat16()
    tok = torch.from_numpy((rng.permutation(R) if gathered else np.arange(R)).astype(np.int32)).cuda()
    xs = x[tok.long()]
    pre, act = [torch.full((R + 1, N), 7.0, device="cuda") for _ in range(2)], torch.full((R + 1, N), 7.0, device="cuda", dtype=torch.bfloat16)
    rows_of = (lambda e: tok.data_ptr() + off[e] * 4) if gathered else (lambda e: x.data_ptr() + off[e] * K * 2)
    gate = q.problems([(rows_of(e), None, pre[0].data_ptr() + off[e] * N * 4, e * K * N, e * K * N // group, rows[e], 0.0) for e in range(E)])
    up = q.problems([(0, act.data_ptr() + off[e] * N * 2, pre[1].data_ptr() + off[e] * N * 4, n + e * K * N, (n + e * K * N) // group, rows[e], 0.0) for e in range(E)])
    if gathered:
        q.gemm_nn_gather_swiglu(dd, ds, group, gate, up, E, K, N, x)
    else:
        q.gemm_nn_swiglu(dd, ds, group, gate, up, E, K, N, pkg.ACT_BF16, pkg.MATH_MFMA_F16)
    for m in range(2):
        W = (np.repeat(s[m * n // group:(m + 1) * n // group], group).astype(np.float64) * digits[m * n:(m + 1) * n]).reshape(E, K, N)
        xh = xs.float().cpu().numpy().astype(np.float64)
        got = pre[m][:R].cpu().numpy()
        for e in range(E):
            want = xh[off[e]:off[e + 1]] @ W[e]
            for c in range(0, N, 64):
                d = np.linalg.norm(got[off[e]:off[e + 1], c:c + 64] - want[:, c:c + 64])
                assert d <= 2.0 ** -11 / np.sqrt(3) * np.linalg.norm(want[:, c:c + 64]), (m, e, c)
    z = pre[0][:R].double()
    assert torch.allclose(act[:R].double(), z * torch.sigmoid(z) * pre[1][:R].double(), rtol=2.0 ** -8, atol=1e-6)
    assert (pre[0][R] == 7.0).all() and (pre[1][R] == 7.0).all() and (act[R] == 7.0).all()


@pytest.mark.parametrize("rows", [[700, 1, 333, 257], [1024], [63, 640, 97]])
def test_swiglu_epilogues_at_any_word(q, rows):
    """The SwiGLU epilogues read and write four columns at a time: outputs and pre-activations that are aligned to a pair of elements only give the
    bits of aligned ones, and nothing around them is touched."""
    import torch
    K, N, group, E = 128, 2048, 128, len(rows)
    rng = np.random.default_rng(78)
    off = np.concatenate([[0], np.cumsum(rows)]).astype(int)
    R, n = int(off[-1]), E * K * N
    digits = rng.integers(-7, 8, 2 * n).astype(np.int8)
    dd = dev((digits[0::2] & 15 | (digits[1::2] & 15) << 4).astype(np.uint8))
    ds = dev((rng.uniform(0.5, 1.5, 2 * n // group) * 0.0086).astype(f32))
    x = dev(rng.standard_normal((R, K)).astype(f32)).bfloat16()
    tok = torch.from_numpy(rng.permutation(R).astype(np.int32)).cuda()
    z, u = dev(rng.standard_normal((R, N)).astype(f32)), dev(rng.standard_normal((R, N)).astype(f32))

    def at(o, dtype, src=None):
        t = torch.full((R * N + 16,), 3.0, device="cuda", dtype=dtype)
        if src is not None:
            t[o:o + R * N] = src.reshape(-1)
        return t

    def run(o):
        gp, up, act = at(o, torch.float32), at(o, torch.float32), at(o, torch.bfloat16)
        q.gemm_nn_gather_swiglu(dd, ds, group, q.problems([(tok.data_ptr() + off[e] * 4, None, gp.data_ptr() + (o + off[e] * N) * 4, e * K * N, e * K * N // group,
                                                            rows[e], 0.0) for e in range(E)]),
                                q.problems([(0, act.data_ptr() + (o + off[e] * N) * 2, up.data_ptr() + (o + off[e] * N) * 4, n + e * K * N, (n + e * K * N) // group,
                                             rows[e], 0.0) for e in range(E)]), E, K, N, x)
        zz, uu, dg, du = at(o, torch.float32, z), at(o, torch.float32, u), at(o, torch.bfloat16), at(o, torch.bfloat16)
        cut = [t[o:] for t in (zz, uu, dg, du)]
        q.gemm_tn_swiglu_bwd(dd, ds, group, q.problems([(x.data_ptr() + off[e] * K * 2, None, cut[0].data_ptr() + off[e] * N * 4, e * K * N, e * K * N // group, rows[e], 0.0)
                                                        for e in range(E)]), E, K, N, *cut)
        out = [gp, up, act, dg, du]
        for t in out:
            assert (t[:o] == 3.0).all() and (t[o + R * N:] == 3.0).all()
        return [t[o:o + R * N] for t in out]

    for a, b in zip(run(0), run(2)):
        assert torch.equal(a, b)


def test_mfma_f16_forward_range_edges(q, orc):
    """Where fp16 would lose bits the kernel's 2^8 range shift keeps them: weights scaled down to 1e-6 (below fp16's
    normal range unshifted) still meet the bar; activations far below fp16's normal range change nothing measurable;
    other orientations given QLMX_MATH_MFMA_F16 run their bf16 kernels unchanged."""
    import torch
    E, K, N, rows = 2, 256, 256, [200, 90]
    n = E * K * N
    tab, nq, ng = make_spans([n], 128)
    for wscale, ascale in ((1e-6, 1.0), (0.02, 1e-3), (30.0, 100.0)):
        P = orc.normal(n, 31, 1, wscale)
        d = np.zeros(n // 2, np.int8); r = np.zeros(n, np.int8); s = np.zeros(ng, f32)
        orc.encode(P, d, r, s, tab, 128, 7, 1, ng)
        orc.render(P, d, s, tab, 128, 1, 0, ng)
        off = np.concatenate([[0], np.cumsum(rows)]).astype(int)
        A = orc.bf16_round(orc.normal(int(off[-1]) * K, 31, 2, ascale))
        A[:64] = orc.bf16_round(orc.normal(64, 31, 3, 1e-7))          # a few values that become fp16 subnormals
        dA, dC = dev(A), torch.zeros(int(off[-1]) * N, device="cuda")
        pa = to_bf16_bits(dA)
        items = [(pa.data_ptr() + int(off[e]) * K * 2, None, dC.data_ptr() + int(off[e]) * N * 4, e * K * N, e * K * N // 128, rows[e], 0.0)
                 for e in range(E)]
        q.gemm_nn(dev(d), dev(s), 128, q.problems(items), E, K, N, pkg.ACT_BF16, pkg.MATH_MFMA_F16)
        torch.cuda.synchronize()
        want = np.zeros(int(off[-1]) * N, f32)
        for e in range(E):
            orc.gemm_nn(A[off[e] * K:], P[e * K * N:(e + 1) * K * N], want[off[e] * N:off[e + 1] * N], rows[e], K, N)
        err = orc.relerr(dC.cpu().numpy(), want)
        assert err < 1e-3, (wscale, ascale, err)
    got, want = run_case(q, orc, "tn", 3, [70, 0, 132], 256, 128, pkg.ACT_BF16, pkg.MATH_MFMA_F16, seed=14)
    got2, _ = run_case(q, orc, "tn", 3, [70, 0, 132], 256, 128, pkg.ACT_BF16, pkg.MATH_MFMA, seed=14)
    assert np.array_equal(got, got2)


def test_mfma_f32_acts_are_rounded_once(q, orc):
    """fp32 activations on the MFMA path are rounded to bf16 on load: equal to feeding pre-rounded ones."""
    import torch
    got32, _ = run_case(q, orc, "tn", 2, [100, 200], 256, 128, pkg.ACT_F32, pkg.MATH_MFMA, seed=9)
    # same inputs, rounded on the host first
    E, K, N = 2, 256, 128
    d, s, P = make_weights(orc, 9, E, N, K)
    A = orc.bf16_round(orc.normal(300 * K, 9, 10))
    want = np.zeros(300 * N, f32)
    off = [0, 100, 300]
    for e in range(E):
        orc.gemm_tn(A[off[e] * K:], P[e * N * K:(e + 1) * N * K], want[off[e] * N:off[e + 1] * N], off[e + 1] - off[e], K, N, 0.0)
    assert orc.relerr(got32, want) < TOL_MFMA


@pytest.mark.parametrize("math", ["f32", "mfma"])
def test_attention_projection_spans_are_one_expert(q, orc, math):
    """wq/wk/wv/wo are QLM spans too (qlm.cuh:480-483): a dense [D,D] or [D,KD] projection is the
    grouped GEMM with a single problem. D=768, KD=256, 1536 rows; forward, dgrad and wgrad."""
    act, mth, tol = (pkg.ACT_BF16, pkg.MATH_MFMA, TOL_MFMA) if math == "mfma" else (pkg.ACT_F32, pkg.MATH_F32, TOL_F32)
    for (K, N) in [(768, 768), (768, 256)]:
        for mode in ["nn", "tn", "nt"]:
            kk, nn = (K, N) if mode != "tn" else (N, K)
            got, want = run_case(q, orc, mode, 1, [1536], kk, nn, act, mth, seed=9)
            assert orc.relerr(got, want) < tol, (mode, K, N)


@pytest.mark.parametrize("beta", [0.0, 1.0])
def test_mfma_tn_many_rows_per_expert(q, orc, beta):
    """Experts with well over a thousand rows on average take the input-gradient kernel whose
    activation tiles go straight to LDS; a ragged tail expert and an empty one ride along."""
    got, want = run_case(q, orc, "tn", 4, [2100, 1500, 0, 1311], 384, 256, pkg.ACT_BF16, pkg.MATH_MFMA, seed=4, beta=beta)
    assert orc.relerr(got, want) < TOL_MFMA


def _pair_case(q, orc, rowsM, K, N, act, math, beta, seed=7, swap=False):
    """C = A1 . W1^T + A2 . W2^T (+ C) per expert through qlmx_moe_gemm_tn_pair; W1 and W2 are the two halves
    of one digit array (`swap`: the second operand pair lies before the first in memory)."""
    import torch
    E = len(rowsM); tot = sum(rowsM)
    off = np.concatenate([[0], np.cumsum(rowsM)]).astype(int)
    bf = act == pkg.ACT_BF16
    d, s, P = make_weights(orc, seed, 2 * E, N, K)
    A = [orc.normal(tot * K, seed, 20 + i) for i in range(2)]
    if bf:
        A = [orc.bf16_round(a) for a in A]
    C0 = orc.normal(tot * N, seed, 12)
    both = dev(np.concatenate(A))
    pb = to_bf16_bits(both) if bf else both
    esz = 2 if bf else 4
    dC, dd, ds = dev(C0.copy()), dev(d), dev(s)
    wsel = [1, 0] if swap else [0, 1]
    def items(i, b):
        w0 = wsel[i] * E
        return [(pb.data_ptr() + (wsel[i] * tot + off[e]) * K * esz, None, dC.data_ptr() + off[e] * N * 4 if i == 0 else None,
                 (w0 + e) * N * K, (w0 + e) * N * K // 128, rowsM[e], b) for e in range(E)]
    q.gemm_tn_pair(dd, ds, 128, q.problems(items(0, beta)), q.problems(items(1, 0.0)), E, K, N, act, math)
    torch.cuda.synchronize()
    want = C0.copy()
    for e in range(E):
        if not rowsM[e]:
            continue
        for i in range(2):
            w = P[(wsel[i] * E + e) * N * K:(wsel[i] * E + e + 1) * N * K]
            orc.gemm_tn(A[wsel[i]][off[e] * K:], w, want[off[e] * N:off[e + 1] * N], rowsM[e], K, N, beta if i == 0 else 1.0)
    return dC.cpu().numpy(), want


@pytest.mark.parametrize("beta", [0.0, 1.0])
@pytest.mark.parametrize("swap", [False, True])
def test_mfma_tn_pair_one_launch(q, orc, beta, swap):
    """The two input-gradient GEMMs that share an output, as one continued contraction: ragged experts,
    an empty one, last tiles of 1..128 rows, either order of the operand pairs in memory."""
    got, want = _pair_case(q, orc, [300, 0, 64, 1, 129, 517], 256, 384, pkg.ACT_BF16, pkg.MATH_MFMA, beta, swap=swap)
    assert orc.relerr(got, want) < TOL_MFMA


def test_mfma_tn_pair_layer_shape(q, orc):
    got, want = _pair_case(q, orc, [700, 40, 333], 2048, 768, pkg.ACT_BF16, pkg.MATH_MFMA, 0.0, seed=8)
    assert orc.relerr(got, want) < TOL_MFMA


@pytest.mark.parametrize("act,math", [("f32", "f32"), ("bf16", "f32"), ("f32", "mfma")])
def test_tn_pair_other_paths_take_two_launches(q, orc, act, math):
    a = pkg.ACT_BF16 if act == "bf16" else pkg.ACT_F32
    m = pkg.MATH_MFMA if math == "mfma" else pkg.MATH_F32
    got, want = _pair_case(q, orc, [70, 0, 130], 256, 128, a, m, 1.0, seed=9)
    assert orc.relerr(got, want) < (TOL_MFMA if math == "mfma" else TOL_F32)


def test_tn_pair_rejects_mismatched_rows(q):
    import torch
    z = torch.zeros(1 << 16, device="cuda")
    zb = torch.zeros(1 << 16, dtype=torch.int8, device="cuda")
    a = q.problems([(z, None, z, 0, 0, 64, 0.0)]); b = q.problems([(z, None, None, 0, 0, 32, 0.0)])
    with pytest.raises(pkg.QlmxError, match="rows"):
        q.gemm_tn_pair(zb, z, 128, a, b, 1, 128, 128, pkg.ACT_BF16, pkg.MATH_MFMA)
    # a pair needs two table entries: half as many problems as a plain call
    many = q.problems([(z, None, z, 0, 0, 1, 0.0)] * 513)
    with pytest.raises(pkg.QlmxError, match="limit"):
        q.gemm_tn_pair(zb, z, 128, many, many, 513, 128, 128, pkg.ACT_BF16, pkg.MATH_MFMA)
    q.gemm_tn_pair(zb, z, 128, a, a, 0, 128, 128, pkg.ACT_BF16, pkg.MATH_MFMA)       # no problems: nothing to do


def _swiglu_case(q, orc, rowsM, K, N, act, math, seed=13):
    """gate | up | SwiGLU through qlmx_moe_gemm_nn_swiglu against the library's separate calls: returns
    (gp, up, ap as fp32) of both ways plus the oracle's gp."""
    import torch
    E = len(rowsM); tot = sum(rowsM)
    off = np.concatenate([[0], np.cumsum(rowsM)]).astype(int)
    bf = act == pkg.ACT_BF16
    d, s, P = make_weights(orc, seed, 2 * E, K, N)
    A = orc.normal(tot * K, seed, 10)
    if bf or math == pkg.MATH_MFMA:
        A = orc.bf16_round(A)                       # the matrix cores see bf16 activations either way
    dA, dd, ds = dev(A), dev(d), dev(s)
    pa = to_bf16_bits(dA) if bf else dA
    esz = 2 if bf else 4
    out = []
    for fused in (True, False):
        gp = torch.full((tot * N,), 7.0, device="cuda"); up = torch.full((tot * N,), 7.0, device="cuda")
        ap = torch.zeros(tot * N, dtype=torch.bfloat16, device="cuda")
        gate = q.problems([(pa.data_ptr() + off[e] * K * esz, None, gp.data_ptr() + off[e] * N * 4, e * K * N, e * K * N // 128, rowsM[e], 0.0) for e in range(E)])
        upp = q.problems([(None, ap.data_ptr() + off[e] * N * 2, up.data_ptr() + off[e] * N * 4, (E + e) * K * N, (E + e) * K * N // 128, rowsM[e], 0.0) for e in range(E)])
        if fused:
            q.gemm_nn_swiglu(dd, ds, 128, gate, upp, E, K, N, act, math)
        else:
            up2 = q.problems([(pa.data_ptr() + off[e] * K * esz, None, up.data_ptr() + off[e] * N * 4, (E + e) * K * N, (E + e) * K * N // 128, rowsM[e], 0.0) for e in range(E)])
            q.gemm_nn(dd, ds, 128, gate, E, K, N, act, math)
            q.gemm_nn(dd, ds, 128, up2, E, K, N, act, math)
            q.swiglu(gp, up, ap, tot * N, pkg.ACT_BF16)
        torch.cuda.synchronize()
        out.append((gp.cpu().numpy(), up.cpu().numpy(), ap.float().cpu().numpy()))
    want = np.zeros(tot * N, f32)
    for e in range(E):
        if rowsM[e]:
            orc.gemm_nn(A[off[e] * K:], P[e * K * N:(e + 1) * K * N], want[off[e] * N:off[e + 1] * N], rowsM[e], K, N)
    return out, want


@pytest.mark.parametrize("rowsM,K,N", [([300, 0, 64, 1, 129, 517], 256, 384), ([700, 40, 333], 768, 2048)])
def test_mfma_nn_swiglu_one_launch(q, orc, rowsM, K, N):
    """Gate and up columns share a tile and the SwiGLU runs on the accumulators: gp and up bit-identical to the
    two separate GEMM calls (same MFMA sequence per element), ap bit-identical to the SwiGLU kernel on them;
    ragged experts, an empty one, last tiles of every height."""
    (f, sep), want = _swiglu_case(q, orc, rowsM, K, N, pkg.ACT_BF16, pkg.MATH_MFMA)
    assert orc.relerr(f[0], want) < TOL_MFMA
    for a, b in zip(f, sep):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))


@pytest.mark.parametrize("act,math", [("f32", "f32"), ("bf16", "f32"), ("f32", "mfma")])
def test_nn_swiglu_other_paths(q, orc, act, math):
    a = pkg.ACT_BF16 if act == "bf16" else pkg.ACT_F32
    m = pkg.MATH_MFMA if math == "mfma" else pkg.MATH_F32
    (f, sep), want = _swiglu_case(q, orc, [70, 0, 132], 256, 128, a, m, seed=14)
    assert orc.relerr(f[0], want) < (TOL_MFMA if math == "mfma" else TOL_F32)
    for x, y in zip(f, sep):
        assert np.array_equal(x.view(np.uint32), y.view(np.uint32))


@pytest.mark.parametrize("beta", [0.0, 1.0])
def test_mfma_nt_split_contraction(q, orc, beta):
    """One expert with far more rows than the others: its contraction is cut into slices that add up
    in turn. Overwriting and accumulating, next to a small, an empty and a ragged expert; untouched
    experts keep their gradient."""
    got, want = run_case(q, orc, "nt", 4, [1700, 40, 0, 333], 256, 256, pkg.ACT_BF16, pkg.MATH_MFMA, seed=6, nt_beta=beta)
    assert orc.relerr(got, want) < TOL_MFMA
    K = N = 256
    assert np.array_equal(got[2 * K * N:3 * K * N], want[2 * K * N:3 * K * N])
    # twice in a row: the flags of the first launch must not satisfy the second
    got2, want2 = run_case(q, orc, "nt", 4, [1700, 40, 0, 333], 256, 256, pkg.ACT_BF16, pkg.MATH_MFMA, seed=7, nt_beta=beta)
    assert orc.relerr(got2, want2) < TOL_MFMA
    # as many slices as a chain holds (15), of a length that rounding up to whole steps changes
    got3, want3 = run_case(q, orc, "nt", 2, [3841, 10], 64, 128, pkg.ACT_BF16, pkg.MATH_MFMA, seed=8, nt_beta=beta)
    assert orc.relerr(got3, want3) < TOL_MFMA


def test_mfma_nt_split_contraction_timeout_is_reported_once(q, orc):
    """A slice's wait for its predecessor is bounded. Forced from the host (qlmx_test_force_wait_timeout: the next
    launch waits for one poll for a tag nobody publishes) every wait gives up, every workgroup still finishes, and
    the NEXT nt call reports QLMX_E_HIP -- once; the call after it is a normal, correct launch."""
    import torch
    q.call("qlmx_test_force_wait_timeout", 2)
    run_case(q, orc, "nt", 4, [1700, 40, 0, 333], 256, 256, pkg.ACT_BF16, pkg.MATH_MFMA, seed=16)     # completes; output not checked
    torch.cuda.synchronize()
    with pytest.raises(pkg.QlmxError, match="gave up waiting"):
        run_case(q, orc, "nt", 4, [1700, 40, 0, 333], 256, 256, pkg.ACT_BF16, pkg.MATH_MFMA, seed=16)
    got, want = run_case(q, orc, "nt", 4, [1700, 40, 0, 333], 256, 256, pkg.ACT_BF16, pkg.MATH_MFMA, seed=16)
    assert orc.relerr(got, want) < TOL_MFMA


@pytest.mark.parametrize("mode", ["nn", "tn"])
def test_mfma_last_tile_heights(q, orc, mode):
    """The last row tile of a problem runs at the smallest height (in steps of 64 rows) that holds it:
    row counts on both sides of every step, for the forward (256-row tiles) and the input gradient (128)."""
    rows = [1, 64, 65, 128, 129, 192, 193, 256, 257, 449]
    K, N = (64, 128) if mode == "nn" else (128, 128)
    for beta in ([0.0] if mode == "nn" else [0.0, 1.0]):
        got, want = run_case(q, orc, mode, len(rows), rows, K, N, pkg.ACT_BF16, pkg.MATH_MFMA, seed=11, beta=beta)
        assert orc.relerr(got, want) < TOL_MFMA, (mode, beta)


@pytest.mark.parametrize("mode", ["nn", "tn", "nt"])
def test_mfma_more_problems_than_lanes(q, orc, mode):
    """70 experts, some empty: the problem table is longer than one wavefront's lookup pass."""
    rng = np.random.default_rng(3)
    rows = [int(r) for r in rng.integers(0, 40, 70)]
    rows[0] = 0; rows[69] = 37
    K, N = {"nn": (64, 128), "tn": (128, 128), "nt": (64, 128)}[mode]
    got, want = run_case(q, orc, mode, 70, rows, K, N, pkg.ACT_BF16, pkg.MATH_MFMA, seed=12)
    assert orc.relerr(got, want) < TOL_MFMA


def test_paired_calls_with_more_table_entries_than_lanes(q, orc):
    """70 experts with a second half each: 140 table entries, every other one owning no tile, looked up in
    three passes of a wavefront."""
    rng = np.random.default_rng(5)
    rows = [int(r) for r in rng.integers(0, 40, 70)]
    rows[0] = 0; rows[69] = 37
    got, want = _pair_case(q, orc, rows, 128, 128, pkg.ACT_BF16, pkg.MATH_MFMA, 1.0, seed=15)
    assert orc.relerr(got, want) < TOL_MFMA
    (f, sep), want = _swiglu_case(q, orc, rows, 64, 128, pkg.ACT_BF16, pkg.MATH_MFMA, seed=16)
    assert orc.relerr(f[0], want) < TOL_MFMA
    for a, b in zip(f, sep):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))


def test_mfma_table_ring_wraps(q, orc):
    """150 grouped launches without a synchronisation between them go more than twice round the ring of
    problem tables (and four times round the unit-table ring of the weight gradient); a launch whose
    table had been overwritten too early would compute on the wrong pointers. Calls that take a slot without
    launching (nothing but empty problems; an error found while the table is written) are mixed in."""
    import torch
    E, rows, K, N = 3, [70, 0, 33], 64, 128
    tot = sum(rows)
    off = np.concatenate([[0], np.cumsum(rows)]).astype(int)
    d, s, P = make_weights(orc, 21, E, K, N)
    A = orc.bf16_round(orc.normal(tot * K, 21, 10)); B = orc.bf16_round(orc.normal(tot * N, 21, 11))
    dA, dB, dd, ds = dev(A), dev(B), dev(d), dev(s)
    pa, pb = to_bf16_bits(dA), to_bf16_bits(dB)
    want_nn = np.zeros(tot * N, f32); want_nt = np.zeros(E * K * N, f32)
    for e in range(E):
        if rows[e]:
            orc.gemm_nn(A[off[e] * K:], P[e * K * N:(e + 1) * K * N], want_nn[off[e] * N:off[e + 1] * N], rows[e], K, N)
            orc.gemm_nt(A[off[e] * K:], B[off[e] * N:], want_nt[e * K * N:(e + 1) * K * N], rows[e], K, N)
    outs = []
    for it in range(75):
        c1 = torch.zeros(tot * N, device="cuda"); c2 = torch.zeros(E * K * N, device="cuda")
        q.gemm_nn(dd, ds, 128, q.problems([(pa.data_ptr() + off[e] * K * 2, None, c1.data_ptr() + off[e] * N * 4, e * K * N, e * K * N // 128,
                                            rows[e], 0.0) for e in range(E)]), E, K, N, pkg.ACT_BF16, pkg.MATH_MFMA)
        q.gemm_nt(q.problems([(pa.data_ptr() + off[e] * K * 2, pb.data_ptr() + off[e] * N * 2, c2.data_ptr() + e * K * N * 4, 0, 0,
                               rows[e], 0.0) for e in range(E)]), E, K, N, pkg.ACT_BF16, pkg.MATH_MFMA)
        outs.append((c1, c2))
        if it % 5 == 4:
            # calls that take a table slot and launch nothing: only empty problems, and an error found after
            # the slot was taken (a pair whose halves differ in rows is caught earlier, so a NULL input is used)
            q.gemm_nn(dd, ds, 128, q.problems([(pa, None, c1, 0, 0, 0, 0.0)]), 1, K, N, pkg.ACT_BF16, pkg.MATH_MFMA)
            with pytest.raises(pkg.QlmxError):
                q.gemm_nn(dd, ds, 128, q.problems([(pa, None, c1, 0, 0, 8, 0.0), (None, None, c1, 0, 0, 8, 0.0)]), 2, K, N, pkg.ACT_BF16, pkg.MATH_MFMA)
    torch.cuda.synchronize()
    for c1, c2 in outs:
        assert orc.relerr(c1.cpu().numpy(), want_nn) < TOL_MFMA and orc.relerr(c2.cpu().numpy(), want_nt) < TOL_MFMA


def test_mfma_rejects_unsupported_shapes(q):
    import torch
    x = torch.zeros(4096, device="cuda")
    pr = q.problems([(x, None, x, 0, 0, 4, 0.0)])
    with pytest.raises(pkg.QlmxError, match="multiple"):
        q.gemm_nn(x, x, 128, pr, 1, 32, 100, pkg.ACT_F32, pkg.MATH_MFMA)


def test_mfma_nt_wide_tile(q, orc):
    """The opt-in 256 x 256 weight-gradient tile (qlmx_nt_tile): overwriting and accumulating, ragged, empty and
    sliced experts, a K that is not a multiple of the tile; bit-equal to the 256 x 128 tile where no contraction
    is sliced (same products, same order of additions)."""
    q.call("qlmx_nt_tile", 256)
    try:
        for beta in (0.0, 1.0):
            for (E, rows, K, N, seed) in [(4, [1700, 40, 0, 333], 256, 256, 6), (3, [300, 77, 512], 320, 512, 9), (2, [3841, 10], 64, 256, 8)]:
                got, want = run_case(q, orc, "nt", E, rows, K, N, pkg.ACT_BF16, pkg.MATH_MFMA, seed=seed, nt_beta=beta)
                assert orc.relerr(got, want) < TOL_MFMA
        wide, _ = run_case(q, orc, "nt", 3, [64, 200, 96], 256, 512, pkg.ACT_BF16, pkg.MATH_MFMA, seed=10, nt_beta=0.0)
    finally:
        q.call("qlmx_nt_tile", 128)
    narrow, _ = run_case(q, orc, "nt", 3, [64, 200, 96], 256, 512, pkg.ACT_BF16, pkg.MATH_MFMA, seed=10, nt_beta=0.0)
    assert np.array_equal(wide.view(np.uint32), narrow.view(np.uint32))
    with pytest.raises(pkg.QlmxError, match="128 or 256"):
        q.call("qlmx_nt_tile", 64)


def test_side_stream_fork_join(q, orc):
    """qlmx_side_fork / qlmx_side_join: work queued on the side stream starts after what the caller's stream held
    at the fork, the caller's stream continues after it at the join; a backward flush with its weight gradient on
    the side stream beside its input gradient gives the bits of the two launches one after the other."""
    import torch
    cur = torch.cuda.current_stream().cuda_stream
    # ordering: a long fill on the caller's stream, a copy of its last bytes on the side stream, a read after the join
    n = 1 << 28
    src = torch.zeros(n, dtype=torch.uint8, device="cuda"); dst = torch.zeros(4096, dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    for rep in range(3):
        src.fill_(rep + 1)
        side = q.side_fork(cur)
        assert side and side != cur
        q.call("qlmx_memcpy_d2d", dst, src[n - 4096:], 4096, side)
        q.side_join(cur)
        got = dst.clone()                                  # on the caller's stream, after the join
        torch.cuda.synchronize()
        assert int(got.min()) == rep + 1 and int(got.max()) == rep + 1
    # a flush both ways
    E, rows, K, N = 6, [700, 33, 0, 1290, 256, 64], 256, 512
    tot = sum(rows); off = np.concatenate([[0], np.cumsum(rows)]).astype(int)
    d, s, P = make_weights(orc, 17, E, K, N, 128)          # forward weights [K, N] per expert; dX[rows, K] = dY[rows, N] . W^T
    dY = orc.bf16_round(orc.normal(tot * N, 17, 10)); X = orc.bf16_round(orc.normal(tot * K, 17, 11))
    dYb, Xb = to_bf16_bits(dev(dY)), to_bf16_bits(dev(X))
    dd, ds = dev(d), dev(s)
    outs = []
    for beside in (False, True):
        G = dev(orc.normal(E * K * N, 17, 12, 0.1)); dX = torch.zeros(tot * K, device="cuda")
        nt = q.problems([(Xb.data_ptr() + off[e] * K * 2, dYb.data_ptr() + off[e] * N * 2, G.data_ptr() + e * K * N * 4, 0, 0, rows[e], 1.0) for e in range(E)])
        tn = q.problems([(dYb.data_ptr() + off[e] * N * 2, None, dX.data_ptr() + off[e] * K * 4, e * N * K, e * N * K // 128, rows[e], 0.0) for e in range(E)])
        st = q.side_fork(cur) if beside else cur
        q.gemm_nt(nt, E, K, N, pkg.ACT_BF16, pkg.MATH_MFMA, st)
        q.gemm_tn(dd, ds, 128, tn, E, N, K, pkg.ACT_BF16, pkg.MATH_MFMA, cur)
        if beside:
            q.side_join(cur)
        outs.append((G.clone(), dX.clone()))
        torch.cuda.synchronize()
    assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1])
    assert float(outs[0][1].abs().max()) > 0.0


@pytest.mark.parametrize("form", ["plain", "added", "continued", "swiglu", "scatter"])
@pytest.mark.parametrize("rows,K,N,tall", [([9, 16, 0, 1], 256, 512, False), ([40, 33, 64, 17, 1], 128, 1024, False), ([125, 131, 97], 512, 384, True), ([1200, 3], 256, 256, True)])
def test_backward_pair_of_few_rows(q, form, rows, K, N, tall):
    """The kernels for few rows in one grid with the weight gradient: the bits of the two launches, for every form of the input gradient, row tiles of
    one and two sixteens, a sliced weight gradient behind it, no weight gradient at all, and a second one of each kind. Before the end nothing of a pair has run; an
    input gradient whose tiles are of 64 rows on its own has, where no weight gradient was there before it."""
    import torch
    cur = torch.cuda.current_stream().cuda_stream
    E, R, bf = len(rows), sum(rows), (pkg.ACT_BF16, pkg.MATH_MFMA)
    at = np.concatenate([[0], np.cumsum(rows)]).astype(int)
    g = torch.Generator(device="cuda"); g.manual_seed(R + K)
    rnd = lambda *shape: torch.randn(*shape, generator=g, device="cuda")
    digit = torch.randint(-7, 8, (2 * E * K * N // 2, 2), generator=g, device="cuda")
    d = ((digit[:, 0] & 15) | (digit[:, 1] & 15) << 4).to(torch.uint8).view(torch.int8)
    s = torch.rand(2 * E * K * N // 128, generator=g, device="cuda") * 0.01 + 0.005
    dY, dY2, X = rnd(R, N).bfloat16(), rnd(R, N).bfloat16(), rnd(R, K).bfloat16()
    gp, up = rnd(R, K), rnd(R, K)
    idx = torch.randperm(R + 3, generator=g, device="cuda")[:R].int()
    wgrad = lambda G, src, beta: q.problems([(X.data_ptr() + int(at[e]) * K * 2, src.data_ptr() + int(at[e]) * N * 2, G.data_ptr() + e * K * N * 4, 0, 0, rows[e], beta) for e in range(E)])

    def igrad(C, src, first, beta=0.0, size=4):
        width = 1 if C is idx else K
        return q.problems([(src.data_ptr() + int(at[e]) * N * 2, None, C.data_ptr() + int(at[e]) * width * 4, (first + e) * N * K, (first + e) * N * K // 128, rows[e], beta) for e in range(E)])

    def one(pair, partner):
        """The outputs, and what has run before the pair's end (a launch that opens a segment of the table ring issues what is held, once in several launches)."""
        G, dX, spread = torch.ones(E * K * N, device="cuda"), torch.ones(R, K, device="cuda"), torch.ones(R + 3, K, device="cuda")
        dg, du = torch.zeros(R, K, device="cuda", dtype=torch.bfloat16), torch.zeros(R, K, device="cuda", dtype=torch.bfloat16)

        def weights(beta=0.0, src=dY): q.gemm_nt(wgrad(G, src, beta), E, K, N, *bf, cur)

        def inputs():
            if form == "plain": q.gemm_tn(d, s, 128, igrad(dX, dY, 0), E, N, K, *bf, cur)
            elif form == "added": q.gemm_tn(d, s, 128, igrad(dX, dY, 0, 1.0), E, N, K, *bf, cur)
            elif form == "continued": q.gemm_tn_pair(d, s, 128, igrad(dX, dY, 0), igrad(dX, dY2, E, 1.0), E, N, K, *bf, cur)
            elif form == "swiglu": q.gemm_tn_swiglu_bwd(d, s, 128, igrad(gp, dY, 0), E, N, K, gp, up, dg, du, cur)
            else: q.gemm_tn_pair_scatter(d, s, 128, igrad(idx, dY, 0), igrad(idx, dY2, E), E, N, K, spread, cur)
        if pair:
            q.pair_begin(cur)
        if partner in ("before", "twice"): weights()
        inputs()
        if partner == "twice":
            weights(1.0, dY2)
            inputs()
        if partner == "after": weights()
        ran = None
        if pair:
            torch.cuda.synchronize()
            ran = [bool((G != 1).any()), bool((dX != 1).any() or (spread != 1).any() or dg.any() or du.any())]
            q.pair_end(cur)
        torch.cuda.synchronize()
        return (G, dX, spread, dg, du), ran
    outs = []
    for pair in (False, True):
        for partner in ("after", "before", "none", "twice"):
            for _ in range(3):
                out, ran = one(pair, partner)
                if not pair or partner == "twice" or ran == [False, tall and partner != "before"]:
                    break
            else:
                raise AssertionError((partner, ran))
            outs.append(out)
    for a, b in zip(outs[:4], outs[4:]):
        for x, y in zip(a, b):
            assert torch.equal(x, y)
    changed = {"plain": 1, "added": 1, "continued": 1, "swiglu": 3, "scatter": 2}[form]
    assert float((outs[4][changed].float() - 1).abs().max()) > 0.0 and float((outs[4][0] - 1).abs().max()) > 0.0


def test_backward_pair_is_one_launch_with_the_same_bits(q, orc):
    """qlmx_pair_begin / qlmx_pair_end: the input gradient and the weight gradient of a flush held back and issued as
    one grid give the bits of the two launches one after the other -- plain, with a sliced weight-gradient contraction
    (chain flags inside the combined grid), with the continued input gradient -- and everything else keeps its order
    on the stream: a second launch of a held kind, a copy queued between the two, the end without a partner."""
    import torch
    cur = torch.cuda.current_stream().cuda_stream
    for (E, rows, K, N, seed, paired) in [(6, [700, 33, 0, 1290, 256, 64], 256, 512, 17, False),
                                         (5, [9000, 12, 300, 0, 129], 256, 384, 18, False),
                                         (4, [513, 64, 1, 2000], 384, 256, 19, True)]:
        tot = sum(rows); off = np.concatenate([[0], np.cumsum(rows)]).astype(int)
        d, s, P = make_weights(orc, seed, 2 * E, K, N, 128)      # forward weights [K, N] per expert; dX[rows, K] = dY[rows, N] . W^T
        dY = orc.bf16_round(orc.normal(tot * N, seed, 10)); dY2 = orc.bf16_round(orc.normal(tot * N, seed, 13)); X = orc.bf16_round(orc.normal(tot * K, seed, 11))
        dYb, dY2b, Xb = to_bf16_bits(dev(dY)), to_bf16_bits(dev(dY2)), to_bf16_bits(dev(X))
        dd, ds = dev(d), dev(s)
        outs = []
        for pair in (False, True):
            G = dev(orc.normal(E * K * N, seed, 12, 0.1)); dX = torch.zeros(tot * K, device="cuda")
            nt = q.problems([(Xb.data_ptr() + off[e] * K * 2, dYb.data_ptr() + off[e] * N * 2, G.data_ptr() + e * K * N * 4, 0, 0, rows[e], 1.0) for e in range(E)])
            tn = q.problems([(dYb.data_ptr() + off[e] * N * 2, None, dX.data_ptr() + off[e] * K * 4, e * N * K, e * N * K // 128, rows[e], 0.0) for e in range(E)])
            tn2 = q.problems([(dY2b.data_ptr() + off[e] * N * 2, None, dX.data_ptr() + off[e] * K * 4, (E + e) * N * K, (E + e) * N * K // 128, rows[e], 0.0) for e in range(E)])
            if pair:
                q.pair_begin(cur)
            q.gemm_nt(nt, E, K, N, pkg.ACT_BF16, pkg.MATH_MFMA, cur)
            if paired:
                q.gemm_tn_pair(dd, ds, 128, tn, tn2, E, N, K, pkg.ACT_BF16, pkg.MATH_MFMA, cur)
            else:
                q.gemm_tn(dd, ds, 128, tn, E, N, K, pkg.ACT_BF16, pkg.MATH_MFMA, cur)
            if pair:
                q.pair_end(cur)
            outs.append((G.clone(), dX.clone()))
            torch.cuda.synchronize()
        assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1]), (E, rows)
        assert float(outs[0][1].abs().max()) > 0.0 and float((outs[0][0] - dev(orc.normal(E * K * N, seed, 12, 0.1))).abs().max()) > 0.0
    # order: dX = dY . W1^T, then dX += dY2 . W2^T (second launch of the held kind), a copy of dX queued before the end,
    # and a weight gradient that finds no partner at the end
    E, rows, K, N, seed = 3, [300, 70, 1025], 256, 256, 23
    tot = sum(rows); off = np.concatenate([[0], np.cumsum(rows)]).astype(int)
    d, s, P = make_weights(orc, seed, 2 * E, K, N, 128)
    dYb = to_bf16_bits(dev(orc.bf16_round(orc.normal(tot * N, seed, 10)))); dY2b = to_bf16_bits(dev(orc.bf16_round(orc.normal(tot * N, seed, 13))))
    Xb = to_bf16_bits(dev(orc.bf16_round(orc.normal(tot * K, seed, 11))))
    dd, ds = dev(d), dev(s)
    res = []
    for pair in (False, True):
        G = torch.zeros(E * K * N, device="cuda"); dX = torch.zeros(tot * K, device="cuda"); snap = torch.zeros(tot * K, device="cuda")
        nt = q.problems([(Xb.data_ptr() + off[e] * K * 2, dYb.data_ptr() + off[e] * N * 2, G.data_ptr() + e * K * N * 4, 0, 0, rows[e], 0.0) for e in range(E)])
        t1 = q.problems([(dYb.data_ptr() + off[e] * N * 2, None, dX.data_ptr() + off[e] * K * 4, e * N * K, e * N * K // 128, rows[e], 0.0) for e in range(E)])
        t2 = q.problems([(dY2b.data_ptr() + off[e] * N * 2, None, dX.data_ptr() + off[e] * K * 4, (E + e) * N * K, (E + e) * N * K // 128, rows[e], 1.0) for e in range(E)])
        if pair:
            q.pair_begin(cur)
        q.gemm_tn(dd, ds, 128, t1, E, N, K, pkg.ACT_BF16, pkg.MATH_MFMA, cur)
        q.gemm_tn(dd, ds, 128, t2, E, N, K, pkg.ACT_BF16, pkg.MATH_MFMA, cur)          # issues t1, is held itself
        q.call("qlmx_memcpy_d2d", snap, dX, tot * K * 4, cur)                           # issues t2
        q.gemm_nt(nt, E, K, N, pkg.ACT_BF16, pkg.MATH_MFMA, cur)                        # held, no partner
        if pair:
            q.pair_end(cur)
        torch.cuda.synchronize()
        res.append((G.clone(), dX.clone(), snap.clone()))
    for a, b in zip(res[0], res[1]):
        assert torch.equal(a, b)
    assert torch.equal(res[1][1], res[1][2]) and float(res[1][0].abs().max()) > 0.0
    # a weight gradient on the wide tile is never held: it goes behind a held one (it accumulates into the same output)
    res = []
    for pair in (False, True):
        G = torch.zeros(E * K * N, device="cuda")
        n0 = q.problems([(Xb.data_ptr() + off[e] * K * 2, dYb.data_ptr() + off[e] * N * 2, G.data_ptr() + e * K * N * 4, 0, 0, rows[e], 0.0) for e in range(E)])
        n1 = q.problems([(Xb.data_ptr() + off[e] * K * 2, dY2b.data_ptr() + off[e] * N * 2, G.data_ptr() + e * K * N * 4, 0, 0, rows[e], 1.0) for e in range(E)])
        if pair:
            q.pair_begin(cur)
        q.gemm_nt(n0, E, K, N, pkg.ACT_BF16, pkg.MATH_MFMA, cur)
        q.call("qlmx_nt_tile", 256)
        try:
            q.gemm_nt(n1, E, K, N, pkg.ACT_BF16, pkg.MATH_MFMA, cur)
        finally:
            q.call("qlmx_nt_tile", 128)
        if pair:
            q.pair_end(cur)
        torch.cuda.synchronize()
        res.append(G.clone())
    assert torch.equal(res[0], res[1]) and float(res[0].abs().max()) > 0.0
    # misuse
    with pytest.raises(pkg.QlmxError, match="no pair is open"):
        q.pair_end(cur)
    q.pair_begin(cur)
    try:
        with pytest.raises(pkg.QlmxError, match="already open"):
            q.pair_begin(cur)
    finally:
        q.pair_end(cur)

"""GPU parity of the decode-shaped (few-token) expert path: the streaming GEMV behind
qlmx_moe_gemm_nn and the fused qlmx_moe_decode_forward, against the CPU oracle's rendered-weights
fp32 layer (moe_forward call order, cudalm.cu:4193-4228). Tolerance 1e-3 relative L2 as stated for
matmul outputs. The fused layer has two multiply loops and every layer test runs with both: the default
one (exact digits, inputs of 31 bits under a common power of two, or fp32 multiply-adds) is as close to the oracle as two
orders of fp32 sums and the libm exp are (observed 4e-7, held to 2e-5; against 64 bits further down, held to 6e-7),
the other (qlmx_decode_math(1)) takes its inputs as fp16 pairs (11 significant bits; observed 2.4e-4 ..
4.9e-4 on a layer's output, held to 7e-4 here). Routing indices come from the oracle's router and are consumed as
given."""
import numpy as np
import pytest

from __graft_entry__ import load_package
from oracle.binding import make_spans

pkg = load_package()
f32 = np.float32
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def q():
    return pkg.load()


@pytest.fixture(params=[0, 1], ids=["fp32", "fp16-inputs"])
def tol(request, q):
    """Selects the decode layer's multiply loop for one test and returns the bound its output is held to."""
    q.call("qlmx_decode_math", request.param)
    yield 7e-4 if request.param else 2e-5
    q.call("qlmx_decode_math", 0)


def dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def encode_layer(orc, seed, E, D, F, group=128):
    """w1 | w3 | w2 back to back in one digit array (three consecutive spans)."""
    n = E * D * F
    tab, nq, ng = make_spans([n, n, n], group)
    P = orc.normal(nq, seed, 1, 0.02)
    d = np.zeros(nq // 2, np.int8); r = np.zeros(nq, np.int8); s = np.zeros(ng, f32)
    orc.encode(P, d, r, s, tab, group, 7, 1, ng)
    orc.render(P, d, s, tab, group, 1, 0, ng)
    return d, s, P, n


@pytest.mark.parametrize("K,N", [(768, 2048), (2048, 768), (512, 1536)])
def test_gemv_small_rows_vs_oracle(q, orc, K, N):
    """qlmx_moe_gemm_nn with 1..4 rows per expert takes the streaming path; an empty expert is skipped."""
    import torch
    E = 5
    rows = [1, 4, 0, 2, 3]
    n = E * K * N
    tab, nq, ng = make_spans([n], 128)
    P = orc.normal(n, 3, 1, 0.02)
    d = np.zeros(n // 2, np.int8); r = np.zeros(n, np.int8); s = np.zeros(ng, f32)
    orc.encode(P, d, r, s, tab, 128, 7, 1, ng)
    orc.render(P, d, s, tab, 128, 1, 0, ng)
    off = np.concatenate([[0], np.cumsum(rows)])
    A = orc.normal(int(off[-1]) * K, 3, 2)
    dA, dC, dd, ds = dev(A), torch.full((int(off[-1]) * N,), 7.0, device="cuda"), dev(d), dev(s)
    items = [(dA.data_ptr() + int(off[e]) * K * 4, None, dC.data_ptr() + int(off[e]) * N * 4, e * K * N, e * K * N // 128, rows[e], 0.0)
             for e in range(E)]
    q.gemm_nn(dd, ds, 128, q.problems(items), E, K, N, pkg.ACT_F32, pkg.MATH_F32)
    torch.cuda.synchronize()
    want = np.zeros(int(off[-1]) * N, f32)
    for e in range(E):
        if rows[e]:
            orc.gemm_nn(A[off[e] * K:], P[e * K * N:(e + 1) * K * N], want[off[e] * N:off[e + 1] * N], rows[e], K, N)
    err = orc.relerr(dC.cpu().numpy(), want)
    assert err < 1e-5, err
    # a second call reuses the tickets and scratch: same answer
    dC.fill_(0)
    q.gemm_nn(dd, ds, 128, q.problems(items), E, K, N, pkg.ACT_F32, pkg.MATH_F32)
    torch.cuda.synchronize()
    assert orc.relerr(dC.cpu().numpy(), want) < 1e-5
    # forty calls without a synchronisation between them go twice round the ring of problem tables,
    # each call with its own output (and a different problem order): every one must come out right
    outs = [torch.zeros(int(off[-1]) * N, device="cuda") for _ in range(40)]
    for it, o in enumerate(outs):
        its = [(dA.data_ptr() + int(off[e]) * K * 4, None, o.data_ptr() + int(off[e]) * N * 4, e * K * N, e * K * N // 128, rows[e], 0.0)
               for e in range(E)]
        if it & 1:
            its.reverse()
        q.gemm_nn(dd, ds, 128, q.problems(its), E, K, N, pkg.ACT_F32, pkg.MATH_F32)
    torch.cuda.synchronize()
    for o in outs:
        assert orc.relerr(o.cpu().numpy(), want) < 1e-5


def run_few_rows(q, K, N, rows, floats_off):
    """qlmx_moe_gemm_nn in fp32 on rows that start so many floats behind 16 bytes, against 64 bits"""
    import torch
    E, group, rng = len(rows), 64, np.random.default_rng(K + N)
    digits = rng.integers(-7, 8, (E, K, N))
    s = (0.0086 * rng.uniform(0.5, 1.5, (E, K, N // group))).astype(f32)
    A = rng.standard_normal((sum(rows), K), dtype=f32)
    off = np.concatenate([[0], np.cumsum(rows)])
    flat = digits.reshape(-1) & 15
    dA, dC = dev(np.concatenate([np.zeros(floats_off, f32), A.reshape(-1)])), torch.full((sum(rows), N), 7.0, device="cuda")
    dd, ds = dev((flat[0::2] | flat[1::2] << 4).astype(np.uint8)), dev(s)
    items = [(dA.data_ptr() + (floats_off + int(off[e]) * K) * 4, None, dC.data_ptr() + int(off[e]) * N * 4, e * K * N, e * K * N // group, rows[e], 0.0)
             for e in range(E)]
    q.gemm_nn(dd, ds, group, q.problems(items), E, K, N, pkg.ACT_F32, pkg.MATH_F32)
    got = dC.cpu().numpy()
    for e in range(E):
        if rows[e]:
            want = A[off[e]:off[e + 1]].astype(np.float64) @ (digits[e] * np.repeat(s[e].astype(np.float64), group, axis=1))
            assert np.linalg.norm(got[off[e]:off[e + 1]] - want) < np.sqrt(K / 4) * 2.0 ** -24 * np.linalg.norm(want), e


@pytest.mark.parametrize("K,N,rows", [(768, 2048, [1, 4]), (8000, 320, [2]), (8192, 320, [3, 4]), (8192, 128, [1, 0, 2]), (8224, 64, [4]), (16384, 64, [1] * 8), (20000, 512, [1, 4]),
                                      (96, 8256, [2]), (130, 16384, [4, 1]), (8704, 8256, [1])])
def test_gemv_of_long_contractions(q, K, N, rows):
    """The streaming path (which rows a float off 16 bytes take) at contractions of more slices than are added up in one go, and rows wider than a workgroup, against 64 bits: K
    additions spread over at least four partial sums, each a random walk of at most sqrt(K / 4) roundings of 2^-24."""
    run_few_rows(q, K, N, rows, 1)


@pytest.mark.parametrize("K,N,rows", [(4224, 128, [1]), (4288, 128, [1, 0, 1]), (4288, 192, [1]), (6656, 64, [1, 3]), (5888, 64, [2, 2]), (7040, 64, [4]), (7104, 64, [4]),
                                      (10112, 320, [3, 4]), (10176, 320, [3, 4]), (16384, 64, [1] * 8), (16384, 64, [1] * 9), (16384, 640, [1])])
def test_few_rows_of_long_and_narrow_matrices(q, K, N, rows):
    """Both sides of the lines between the streaming path and the kernels in parts for few rows and a long contraction; bound as above."""
    run_few_rows(q, K, N, rows, 0)


@pytest.mark.parametrize("T,E,D,F,K", [(1, 32, 768, 2048, 2), (4, 32, 768, 2048, 2), (16, 32, 768, 2048, 2), (4, 8, 768, 2048, 2), (16, 8, 768, 2048, 2),
                                       (16, 4, 256, 384, 4), (5, 3, 128, 256, 1), (7, 6, 1024, 640, 3), (3, 4, 2048, 256, 2)])
def test_decode_forward_vs_oracle_layer(q, orc, tol, T, E, D, F, K):
    import torch
    d, s, P, n = encode_layer(orc, 11 + T, E, D, F)
    x = orc.normal(T * D, 11, 2)
    rt = orc.normal(T * E, 11, 3)
    pr = np.zeros(T * E, f32); asn = np.zeros(K * T, np.int32); gate = np.zeros(K * T, f32)
    orc.router_topk(rt, pr, asn, gate, T, E, K)
    res = orc.normal(T * D, 11, 4)                      # residual the layer accumulates into
    want = res.copy()
    rc, ws = orc.moe_forward(x, P[:n], P[n:2 * n], P[2 * n:], asn, gate, want, T, D, F, E, K)
    orc.moe_ws_free(ws)
    assert rc == 0
    out = dev(res)
    dd, ds = dev(d), dev(s)
    q.decode_forward(dev(x), dev(asn), dev(gate), out, dd, ds, 128, 0, n, 2 * n, T, K, E, D, F)
    torch.cuda.synchronize()
    err = orc.relerr(out.cpu().numpy() - res, want - res)
    assert err < 1e-3, err
    assert err < tol, err
    # run-to-run determinism: slice order, not arrival order, fixes the sums
    out2 = dev(res)
    q.decode_forward(dev(x), dev(asn), dev(gate), out2, dd, ds, 128, 0, n, 2 * n, T, K, E, D, F)
    torch.cuda.synchronize()
    assert torch.equal(out, out2)


@pytest.mark.parametrize("T", [2, 3, 5, 6, 7, 9, 11, 13, 24, 32])
def test_decode_token_counts_cover_leftover_groups(q, orc, tol, T):
    """Token counts whose numbers of problems leave every remainder modulo the 8 XCDs (the groups left over after
    a full round are cut into pieces over the XCDs), up to the 64 (pass, token) pairs a call may carry."""
    import torch
    E, D, F, K = 16, 256, 512, 2
    d, s, P, n = encode_layer(orc, 70 + T, E, D, F)
    x = orc.normal(T * D, 70 + T, 2)
    rt = orc.normal(T * E, 70 + T, 3)
    pr = np.zeros(T * E, f32); asn = np.zeros(K * T, np.int32); gate = np.zeros(K * T, f32)
    orc.router_topk(rt, pr, asn, gate, T, E, K)
    want = np.zeros(T * D, f32)
    rc, ws = orc.moe_forward(x, P[:n], P[n:2 * n], P[2 * n:], asn, gate, want, T, D, F, E, K)
    orc.moe_ws_free(ws)
    assert rc == 0
    out = torch.zeros(T * D, device="cuda")
    q.decode_forward(dev(x), dev(asn), dev(gate), out, dev(d), dev(s), 128, 0, n, 2 * n, T, K, E, D, F)
    torch.cuda.synchronize()
    assert orc.relerr(out.cpu().numpy(), want) < tol


@pytest.mark.parametrize("T,E,D,F,K", [(1, 8, 128, 128, 8), (64, 5, 128, 384, 1), (8, 16, 384, 640, 8), (1, 4, 1152, 2816, 2)]
                         + [(T, 16, 512, 2048, 2) for T in (7, 8, 9, 10, 11, 12, 13, 14, 15, 16)])
def test_decode_few_pairs_and_many(q, orc, tol, T, E, D, F, K):
    """Both sides of the line between the kernel of few pairs and the one with a problem table -- the smallest shapes, chunks that end in the
    middle, the most pairs, an expert that is none, every remainder of problems modulo 8 -- by either entry point, to the same bits."""
    import torch
    d, s, P, n = encode_layer(orc, 90 + T, E, D, F)
    x = orc.normal(T * D, 90 + T, 2)
    rt = orc.normal(T * E, 90 + T, 3)
    pr = np.zeros(T * E, f32); asn = np.zeros(K * T, np.int32); gate = np.zeros(K * T, f32)
    orc.router_topk(rt, pr, asn, gate, T, E, K)
    ref_gate = gate.copy(); ref_gate[K * T - 1] = 0.0
    want = np.zeros(T * D, f32)
    rc, ws = orc.moe_forward(x, P[:n], P[n:2 * n], P[2 * n:], asn, ref_gate, want, T, D, F, E, K)
    orc.moe_ws_free(ws)
    assert rc == 0
    bad = asn.copy(); bad[K * T - 1] = E
    outs = [torch.zeros(T * D, device="cuda") for _ in range(3)]
    for o, f in zip(outs, (q.decode_forward, q.decode_forward, q.decode_forward_noalloc)):
        f(dev(x), dev(bad), dev(gate), o, dev(d), dev(s), 128, 0, n, 2 * n, T, K, E, D, F)
    torch.cuda.synchronize()
    assert orc.relerr(outs[0].cpu().numpy(), want) < tol
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])


def test_decode_all_tokens_one_expert(q, orc, tol):
    """Collision case: 16 tokens on the same two experts -> problems are cut into row pairs."""
    import torch
    T, E, D, F, K = 16, 4, 256, 512, 2
    d, s, P, n = encode_layer(orc, 5, E, D, F)
    x = orc.normal(T * D, 5, 2)
    asn = np.concatenate([np.full(T, 2), np.full(T, 0)]).astype(np.int32)
    gate = orc.uniform(K * T, 5, 3, 0.1, 0.6)
    want = np.zeros(T * D, f32)
    rc, ws = orc.moe_forward(x, P[:n], P[n:2 * n], P[2 * n:], asn, gate, want, T, D, F, E, K)
    orc.moe_ws_free(ws)
    out = torch.zeros(T * D, device="cuda")
    q.decode_forward(dev(x), dev(asn), dev(gate), out, dev(d), dev(s), 128, 0, n, 2 * n, T, K, E, D, F)
    torch.cuda.synchronize()
    assert orc.relerr(out.cpu().numpy(), want) < tol


def test_decode_group_256_and_rejected_groups(q, orc, tol):
    """Scale groups of 256 (one per task row) go through the same kernel; 64 and 96 are refused."""
    import torch
    T, E, D, F, K = 4, 4, 512, 768, 2
    d, s, P, n = encode_layer(orc, 21, E, D, F, group=256)
    x = orc.normal(T * D, 21, 2)
    rt = orc.normal(T * E, 21, 3)
    pr = np.zeros(T * E, f32); asn = np.zeros(K * T, np.int32); gate = np.zeros(K * T, f32)
    orc.router_topk(rt, pr, asn, gate, T, E, K)
    want = np.zeros(T * D, f32)
    rc, ws = orc.moe_forward(x, P[:n], P[n:2 * n], P[2 * n:], asn, gate, want, T, D, F, E, K)
    orc.moe_ws_free(ws)
    out = torch.zeros(T * D, device="cuda")
    q.decode_forward(dev(x), dev(asn), dev(gate), out, dev(d), dev(s), 256, 0, n, 2 * n, T, K, E, D, F)
    torch.cuda.synchronize()
    assert orc.relerr(out.cpu().numpy(), want) < tol
    for g in (64, 96):
        with pytest.raises(pkg.QlmxError, match="group"):
            q.decode_forward(dev(x), dev(asn), dev(gate), out, dev(d), dev(s), g, 0, n, 2 * n, T, K, E, D, F)


def test_decode_invalid_expert_is_skipped(q, orc, tol):
    """A pair with an out-of-range expert adds nothing; the other pairs are unaffected."""
    import torch
    T, E, D, F, K = 3, 4, 256, 512, 2
    d, s, P, n = encode_layer(orc, 9, E, D, F)
    x = orc.normal(T * D, 9, 2)
    asn = np.array([1, 3, 0, 2, 1, 3], np.int32)          # [k][t]
    gate = orc.uniform(K * T, 9, 3, 0.1, 0.6)
    bad = asn.copy(); bad[4] = 7                          # pass 1, token 1 -> expert 7 of 4
    gate_ref = gate.copy(); gate_ref[4] = 0.0             # the reference result with that pair's weight zeroed
    want = np.zeros(T * D, f32)
    rc, ws = orc.moe_forward(x, P[:n], P[n:2 * n], P[2 * n:], asn, gate_ref, want, T, D, F, E, K)
    orc.moe_ws_free(ws)
    out = torch.zeros(T * D, device="cuda")
    q.decode_forward(dev(x), dev(bad), dev(gate), out, dev(d), dev(s), 128, 0, n, 2 * n, T, K, E, D, F)
    torch.cuda.synchronize()
    assert orc.relerr(out.cpu().numpy(), want) < tol
    allbad = np.full(K * T, -1, np.int32)
    out.zero_()
    q.decode_forward(dev(x), dev(allbad), dev(gate), out, dev(d), dev(s), 128, 0, n, 2 * n, T, K, E, D, F)
    torch.cuda.synchronize()
    assert float(out.abs().max()) == 0.0


def test_decode_repeated_calls_alternating_shapes(q, orc, tol):
    """The hand-over words carry the call's epoch: stale partial sums of earlier calls, of other
    shapes and token counts, must never be taken for current ones."""
    import torch
    cases = []
    for (T, E, D, F, K, seed) in [(16, 8, 256, 512, 2, 31), (1, 8, 256, 512, 2, 32), (5, 4, 512, 256, 3, 33)]:
        d, s, P, n = encode_layer(orc, seed, E, D, F)
        x = orc.normal(T * D, seed, 2)
        rt = orc.normal(T * E, seed, 3)
        pr = np.zeros(T * E, f32); asn = np.zeros(K * T, np.int32); gate = np.zeros(K * T, f32)
        orc.router_topk(rt, pr, asn, gate, T, E, K)
        want = np.zeros(T * D, f32)
        rc, ws = orc.moe_forward(x, P[:n], P[n:2 * n], P[2 * n:], asn, gate, want, T, D, F, E, K)
        orc.moe_ws_free(ws)
        cases.append((T, E, D, F, K, n, dev(x), dev(asn), dev(gate), dev(d), dev(s), want))
    outs = []
    for rep in range(12):
        T, E, D, F, K, n, x, asn, gate, d, s, want = cases[rep % 3]
        out = torch.zeros(T * D, device="cuda")
        q.decode_forward(x, asn, gate, out, d, s, 128, 0, n, 2 * n, T, K, E, D, F)
        outs.append((out, want))
    torch.cuda.synchronize()
    for out, want in outs:
        assert orc.relerr(out.cpu().numpy(), want) < tol


def test_decode_wait_timeout_is_reported_once(q, orc, tol):
    """The waits between the three task lists are bounded. Forced from the host (qlmx_test_force_wait_timeout: for
    one launch every wait looks, for one poll, for a tag nobody writes) all of them give up, the kernel still ends
    normally, the NEXT call returns QLMX_E_HIP once, and the call after that is correct again."""
    import torch
    T, E, D, F, K = 8, 8, 256, 512, 2
    d, s, P, n = encode_layer(orc, 51, E, D, F)
    x = orc.normal(T * D, 51, 2)
    rt = orc.normal(T * E, 51, 3)
    pr = np.zeros(T * E, f32); asn = np.zeros(K * T, np.int32); gate = np.zeros(K * T, f32)
    orc.router_topk(rt, pr, asn, gate, T, E, K)
    want = np.zeros(T * D, f32)
    rc, ws = orc.moe_forward(x, P[:n], P[n:2 * n], P[2 * n:], asn, gate, want, T, D, F, E, K)
    orc.moe_ws_free(ws)
    args = (dev(x), dev(asn), dev(gate))
    dd, ds = dev(d), dev(s)
    out = torch.zeros(T * D, device="cuda")
    q.call("qlmx_test_force_wait_timeout", 1)
    q.decode_forward(*args, out, dd, ds, 128, 0, n, 2 * n, T, K, E, D, F)      # gives up everywhere, ends normally
    torch.cuda.synchronize()
    with pytest.raises(pkg.QlmxError, match="gave up waiting"):
        q.decode_forward(*args, out, dd, ds, 128, 0, n, 2 * n, T, K, E, D, F)
    out.zero_()
    q.decode_forward(*args, out, dd, ds, 128, 0, n, 2 * n, T, K, E, D, F)
    torch.cuda.synchronize()
    assert orc.relerr(out.cpu().numpy(), want) < tol


def test_decode_on_two_streams_in_turn(q, orc):
    """Calls of both kernels that follow each other on two streams, one event apart, over the one workspace: every call finds the tag
    of the call before it, whichever stream that was on. Behind a workspace that has just grown, too: its new memory is
    cleared before a stream that does not wait for the null stream uses it."""
    import torch
    q.call("qlmx_decode_math", 0)
    calls = []
    for seed, (T, E, D, F, K) in enumerate([(1, 4, 256, 512, 2), (16, 8, 768, 1024, 2), (2, 4, 512, 256, 3), (12, 8, 768, 1024, 2)]):
        d, s, P, n = encode_layer(orc, 60 + seed, E, D, F)
        x = orc.normal(T * D, 60 + seed, 2); rt = orc.normal(T * E, 60 + seed, 3)
        pr = np.zeros(T * E, f32); asn = np.zeros(K * T, np.int32); gate = np.zeros(K * T, f32)
        orc.router_topk(rt, pr, asn, gate, T, E, K)
        want = np.zeros(T * D, f32)
        rc, ws = orc.moe_forward(x, P[:n], P[n:2 * n], P[2 * n:], asn, gate, want, T, D, F, E, K)
        orc.moe_ws_free(ws)
        assert rc == 0
        calls.append((dev(x), dev(asn), dev(gate), dev(d), dev(s), n, (T, K, E, D, F), want))
    # 64 pairs of a wide layer: more partial sums than any other call of these tests
    T, E, D, F, K = 64, 1, 1024, 8192, 1
    g = torch.Generator(device="cuda").manual_seed(1)
    big = (torch.randn(T * D, generator=g, device="cuda"), torch.zeros(T, dtype=torch.int32, device="cuda"), torch.ones(T, device="cuda"),
           torch.randint(0, 256, (3 * D * F // 2,), generator=g, dtype=torch.uint8, device="cuda"), torch.full((3 * D * F // 128,), 0.01, device="cuda"))
    grown = [torch.zeros(T * D, device="cuda") for _ in range(2)]
    outs = [[torch.zeros(c[6][0] * c[6][3], device="cuda") for c in calls] for _ in range(20)]
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    turn = 0

    def run(x, asn, gate, out, d, s, n, shape):
        nonlocal turn
        here, other = streams[turn & 1], streams[1 - (turn & 1)]
        here.wait_stream(other)
        q.decode_forward(x, asn, gate, out, d, s, 128, 0, n, 2 * n, *shape, stream=here.cuda_stream)
        turn += 1

    run(*big[:3], grown[0], *big[3:], D * F, (T, K, E, D, F))
    for row in outs:
        for out, (x, asn, gate, d, s, n, shape, _) in zip(row, calls):
            run(x, asn, gate, out, d, s, n, shape)
    run(*big[:3], grown[1], *big[3:], D * F, (T, K, E, D, F))
    torch.cuda.synchronize()
    q.call("qlmx_decode_status")
    assert torch.isfinite(grown[0]).all() and torch.equal(*grown)
    for row in outs:
        for out, first, c in zip(row, outs[0], calls):
            assert torch.equal(out, first) and orc.relerr(out.cpu().numpy(), c[7]) < 2e-5


def test_decode_limits(q):
    import torch
    z = torch.zeros(65536, device="cuda")
    zi = torch.zeros(256, dtype=torch.int32, device="cuda")
    with pytest.raises(pkg.QlmxError, match="pairs"):
        q.decode_forward(z, zi, z, z, z, z, 128, 0, 0, 0, 64, 2, 4, 128, 128)
    with pytest.raises(pkg.QlmxError, match="multiples of 32"):
        q.decode_forward(z, zi, z, z, z, z, 128, 0, 0, 0, 2, 2, 4, 100, 128)


@pytest.mark.parametrize("D,F,group", [(128, 128, 128), (384, 640, 128), (256, 768, 256), (896, 512, 128)])
def test_decode_inputs_of_very_different_size(q, orc, D, F, group):
    """The default loop brings the inputs of a wavefront's rows to a common fixed point: tokens that are tiny or huge, one value far above the
    rest, all zeros, or not a number share experts (and problems of two) with ordinary ones, and each is held to the bound by
    itself; widths that end inside a task's rows and columns."""
    import torch
    q.call("qlmx_decode_math", 0)
    T, E, K = 7, 2, 2
    d, s, P, n = encode_layer(orc, 31, E, D, F, group)
    x = orc.normal(T * D, 31, 2).reshape(T, D)
    x[1] *= f32(1e-18); x[2] *= f32(1e12); x[3, D // 3] = 3e4; x[4] = 0.0
    asn = np.array([0, 0, 0, 1, 1, 1, 0] + [1, 1, 1, 0, 0, 0, 1], np.int32)
    gate = np.full(K * T, 0.5, f32)
    want = np.zeros(T * D, f32)
    rc, ws = orc.moe_forward(x.reshape(-1), P[:n], P[n:2 * n], P[2 * n:], asn, gate, want, T, D, F, E, K)
    orc.moe_ws_free(ws)
    want = want.reshape(T, D)
    x[6, 5] = np.nan
    out = torch.zeros(T, D, device="cuda")
    q.decode_forward(dev(x), dev(asn), dev(gate), out, dev(d), dev(s), group, 0, n, 2 * n, T, K, E, D, F)
    got = out.cpu().numpy()
    for t in (0, 1, 2, 3, 5):
        assert orc.relerr(got[t], want[t]) < 2e-5, t
    assert not got[4].any() and np.isnan(got[6]).all()


class Layer64:
    """A decode layer whose digits and scales a test changes before it runs: d1, d3 [E, D, F], d2 [E, F, D], s1, s3
    [E, D, F / group], s2 [E, F, D / group], and the layer's output in 64 bits from those digits and scales."""
    T, E, K = 3, 2, 2

    def __init__(self, orc, seed, D=384, F=640, group=128):
        self.D, self.F, self.group = D, F, group
        T, E, K, D, F = self.T, self.E, self.K, self.D, self.F
        rng = np.random.default_rng(seed)
        self.d1, self.d3 = (rng.integers(-7, 8, (E, D, F)) for _ in range(2))
        self.d2 = rng.integers(-7, 8, (E, F, D))
        self.s1, self.s3 = (f32(0.01) * (f32(0.5) + rng.random((E, D, F // self.group), dtype=f32)) for _ in range(2))
        self.s2 = f32(0.01) * (f32(0.5) + rng.random((E, F, D // self.group), dtype=f32))
        self.x = rng.standard_normal((T, D), dtype=f32)
        self.asn = np.array([0, 0, 0, 1, 1, 1], np.int32)             # an expert's three tokens: a problem of two rows, one of one
        self.gate = (f32(0.2) + rng.random(K * T, dtype=f32)).astype(f32)

    def want(self):
        y = np.zeros((self.T, self.D))
        w = lambda d, s: d * np.repeat(s.astype(np.float64), self.group, axis=2)
        w1, w3, w2 = w(self.d1, self.s1), w(self.d3, self.s3), w(self.d2, self.s2)
        for j, e in enumerate(self.asn):
            x = self.x[j % self.T].astype(np.float64)
            g, u = x @ w1[e], x @ w3[e]
            with np.errstate(over="ignore"):
                y[j % self.T] += self.gate[j].astype(np.float64) * ((g / (1.0 + np.exp(-g)) * u) @ w2[e])
        return y

    def run(self, q):
        import torch
        q.call("qlmx_decode_math", 0)
        digits = np.concatenate([m.reshape(-1) for m in (self.d1, self.d3, self.d2)]).astype(np.int64) & 15
        scales = np.concatenate([m.reshape(-1) for m in (self.s1, self.s3, self.s2)]).astype(f32)
        out = torch.zeros(self.T, self.D, device="cuda")
        n = self.E * self.D * self.F
        q.decode_forward(dev(self.x), dev(self.asn), dev(self.gate), out, dev((digits[0::2] | digits[1::2] << 4).astype(np.uint8)), dev(scales),
                         self.group, 0, n, 2 * n, self.T, self.K, self.E, self.D, self.F)
        return out.cpu().numpy()


# A value of the output passes some ten fp32 roundings after the products: staging, the four wavefronts' and the slices' sums, SwiGLU,
# the gated sum over the passes, 2^-24 each: 6e-7 if all of them added up. 1.7e-7 at most is what the cases below show.
REL64 = 6e-7


def rel64(got, want):
    return float(np.linalg.norm(got - want) / np.linalg.norm(want))


@pytest.mark.parametrize("n", [0, 10, 14, 22, 30, 40])
def test_decode_neighbouring_scale_groups_of_different_size(q, orc, n):
    """A column's sum holds nothing of the scale group beside it, so the size of that group's scales must not show in it: every
    second group of the down projection 2^-n of its neighbours, and every second group of gate and up with the down
    projection's rows behind them as much larger, so that the output shows those columns' own error."""
    a = Layer64(orc, 100 + n)
    a.s2[:, :, 1::2] *= f32(2.0 ** -n)
    got, want = a.run(q), a.want()
    for c in range(0, a.D, a.group):
        assert rel64(got[:, c:c + a.group], want[:, c:c + a.group]) < REL64, c
    b = Layer64(orc, 200 + n)
    b.s1[:, :, 1::2] *= f32(2.0 ** -n); b.s3[:, :, 1::2] *= f32(2.0 ** -n)
    for f in range(b.group, b.F, 2 * b.group):
        b.s2[:, f:f + b.group] *= f32(2.0 ** min(2 * n, 100))
    got, want = b.run(q), b.want()
    assert rel64(got, want) < REL64


@pytest.mark.parametrize("D,F,group", [(384, 640, 128), (128, 128, 128), (512, 768, 256)])
@pytest.mark.parametrize("n", [4, 9, 12, 20, 30])
def test_decode_columns_that_take_nothing_of_the_largest_input(q, orc, n, D, F, group):
    """One input 2^n times the others, whose digits are zero in most columns: those columns are sums of the small inputs alone.
    The few columns that do hold it have down rows of zeros, so the output is of the small ones alone too."""
    a = Layer64(orc, 300 + n, D, F, group)
    a.x[:, 5] *= f32(2.0 ** n); a.x[1, D // 2] *= f32(2.0 ** n)
    for d in (a.d1, a.d3):
        d[:, (5, D // 2), 8:] = 0
    a.d2[:, :8] = 0
    got, want = a.run(q), a.want()
    for t in range(a.T):
        assert rel64(got[t], want[t]) < REL64, t


@pytest.mark.parametrize("D,F,group", [(384, 640, 128), (512, 768, 256)])
@pytest.mark.parametrize("v", [np.nan, np.inf])
def test_decode_nan_and_infinite_scales_stay_in_their_columns(q, orc, v, D, F, group):
    """A scale of the down projection that is no finite number reaches the columns of its group as fp32 multiply-adds take it
    there (an infinity times the digit 0 is NaN), and no others."""
    a = Layer64(orc, 400, D, F, group)
    want = a.want()
    a.s2[1, 77, 1] = v
    got = a.run(q)
    there = slice(a.group, 2 * a.group)
    nan = np.isnan(v) | (a.d2[1, 77, there] == 0)
    assert np.array_equal(np.isnan(got[:, there]), np.broadcast_to(nan, (a.T, a.group)))
    assert np.array_equal(np.isinf(got[:, there]), np.broadcast_to(~nan, (a.T, a.group)))
    for c in [c for c in range(0, D, group) if c != group]:
        assert rel64(got[:, c:c + a.group], want[:, c:c + a.group]) < REL64, c

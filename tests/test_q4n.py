"""q4n wire format (quantize_params / dequantize_params qtype 3, cudalm.cu:638-656, 688-696): the
oracle's restatement and the library's host functions against the bytes the compiled reference wrote
(tests/golden/q4n.npz). Host code only, so these run without a GPU; byte-exact both ways."""
import os
import subprocess
import sys

import numpy as np
import pytest

from __graft_entry__ import load_package

pkg = load_package()
f32 = np.float32
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def lib():
    return pkg.Qlmx(init=False)


def test_oracle_matches_reference_bytes(orc, golden):
    g = golden("q4n")
    n, group = (int(v) for v in g["dims"])
    buf, nraw = orc.q4n_quantize(g["P"], group)
    assert nraw == 1
    assert np.array_equal(buf, g["buf"])
    ok, back = orc.q4n_dequantize(g["buf"], n, group)
    assert ok == 1 and np.array_equal(back.view(np.uint32), g["back"].view(np.uint32))
    assert np.array_equal(back.view(np.uint32), g["P"].view(np.uint32))       # the format is lossless here
    b64, _ = orc.q4n_quantize(g["P"][:300], 64)
    assert np.array_equal(b64, g["buf64"])


def test_library_matches_reference_bytes(lib, golden):
    g = golden("q4n")
    n, group = (int(v) for v in g["dims"])
    buf, nraw = lib.q4n_quantize(g["P"], group)
    assert nraw == 1 and np.array_equal(buf, g["buf"])
    back, used = lib.q4n_dequantize(g["buf"], n, group)
    assert used == g["buf"].size
    assert np.array_equal(back.view(np.uint32), g["back"].view(np.uint32))
    b64, _ = lib.q4n_quantize(g["P"][:300], 64)
    assert np.array_equal(b64, g["buf64"])


def test_layout_closed_form(lib):
    """One group written by hand: scale 0.25, digits -7..7 cycling -> 4 + 64 bytes, nibble rule
    ((b & 15) ^ 8) - 8 with the even element in the low nibble."""
    d = (np.arange(128) % 15 - 7).astype(f32)
    P = (d * f32(0.25)).astype(f32)
    buf, nraw = lib.q4n_quantize(P, 128)
    assert nraw == 0 and buf.size == 4 + 64
    assert buf[:4].view(f32)[0] == f32(0.25)          # amax/7 = 0.25 exactly
    lo = ((buf[4:] & 15).astype(int) ^ 8) - 8
    hi = ((buf[4:] >> 4).astype(int) ^ 8) - 8
    assert np.array_equal(lo, d[0::2]) and np.array_equal(hi, d[1::2])


def test_rendered_qlm_view_round_trips_without_raw_groups(lib, orc):
    from oracle.binding import make_spans
    n, group = 128 * 40, 128
    tab, nq, ng = make_spans([n], group)
    P = orc.normal(n, 5, 1, 0.02)
    d = np.zeros(nq // 2, np.int8); r = np.zeros(nq, np.int8); s = np.zeros(ng, f32)
    orc.encode(P, d, r, s, tab, group, 7, 1, ng)
    orc.render(P, d, s, tab, group, 1, 0, ng)
    buf, nraw = lib.q4n_quantize(P, group)
    assert nraw == 0 and buf.size == ng * (4 + 64)
    back, _ = lib.q4n_dequantize(buf, n, group)
    assert np.array_equal(back.view(np.uint32), P.view(np.uint32))
    ob, oraw = orc.q4n_quantize(P, group)
    assert oraw == 0 and np.array_equal(ob, buf)


@pytest.mark.parametrize("n,group", [(1, 2), (15, 16), (17, 34), (8 * 128 + 9, 128), (262143, 64), (262145, 128), (700001, 96), (2300000, 128)])
def test_sizes_around_the_vector_and_thread_shares(lib, orc, n, group):
    """Tails of a vector and of a group, and value counts that are one, two and many threads' shares; groups that are
    raw, zero, hold infinities and NaN, or take a later candidate."""
    rng = np.random.default_rng(n)
    P = (rng.integers(-7, 8, n) * f32(0.0173)).astype(f32)
    ng = -(-n // group)
    for k, q in enumerate(rng.permutation(ng)[:max(1, ng // 5)]):
        v = P[q * group:(q + 1) * group]
        if k % 5 == 0: v[:] = rng.normal(size=v.size)
        elif k % 5 == 1: v[:] = 0.0
        elif k % 5 == 2: v[-1] = np.inf
        elif k % 5 == 3: v[0] = np.nan
        else: v[:] = (rng.integers(-3, 4, v.size) * f32(3e-41)).astype(f32)
    want, wraw = orc.q4n_quantize(P, group)
    got, raw = lib.q4n_quantize(P, group)
    assert raw == wraw and np.array_equal(got, want)
    back, used = lib.q4n_dequantize(got, n, group)
    ok, wback = orc.q4n_dequantize(want, n, group)
    assert ok == 1 and used == want.size and np.array_equal(back.view(np.uint32), wback.view(np.uint32))


@pytest.mark.parametrize("exponent", [-126, -100, -93, -91, -90, -89, 0, 86, 87, 88, 89, 90, 91, 120])
@pytest.mark.parametrize("group", [128, 64, 34])
def test_groups_that_fit_and_groups_that_nearly_do(lib, orc, exponent, group):
    """Scales of any mantissa at both ends of the range in which a reciprocal stands for the division: digits up to 7 down to 1, values one unit in the last
    place off at the front and at the back, negative zeros, one value between the digits."""
    rng = np.random.default_rng((exponent + 200) * 1000 + group)
    groups = []
    for i in range(420):
        most = 7 - i % 7
        d = rng.integers(-most, most + 1, group).astype(f32)
        d[rng.integers(group)] = most if i % 2 else -most
        scale = np.ldexp(f32(1 + rng.random()), exponent).astype(f32)
        v = (d * scale).astype(f32)
        at = (0, group - 1, int(rng.integers(group)))[i % 3]
        if i % 5 == 1: v[at] = np.nextafter(v[at], f32(np.inf))
        elif i % 5 == 2: v[v == 0] = f32(-0.0)
        elif i % 5 == 3: v[at] = f32(0.5) * scale
        groups.append(v)
    P = np.concatenate(groups)
    want, wraw = orc.q4n_quantize(P, group)
    got, raw = lib.q4n_quantize(P, group)
    assert raw == wraw and np.array_equal(got, want)
    back, used = lib.q4n_dequantize(got, P.size, group)
    assert used == got.size and np.array_equal(back + f32(0), P + f32(0))       # a zero comes back positive


@pytest.mark.parametrize("tail", [0, 1, 6, 7, 8, 9, 15, 31, 33, 39])
def test_every_even_group_up_to_eighty(lib, orc, tail):
    """Groups and last groups of every remainder of 8 and of 32: ones that fit, with the digits of the last eight looked at twice, and ones that a value at
    the back keeps raw."""
    rng = np.random.default_rng(tail)
    for group in range(2, 82, 2):
        n = 36 * group + min(tail, group - 1)
        P = rng.integers(-7, 8, n).astype(f32) * f32(0.0173)
        P[group * np.arange(36)] = f32(7) * f32(0.0173)
        for q in range(0, 37, 3):
            v = P[q * group:(q + 1) * group]
            if v.size: v[-1 - q % min(9, v.size)] += f32(0.003)
        want, wraw = orc.q4n_quantize(P, group)
        got, raw = lib.q4n_quantize(P, group)
        assert raw == wraw and np.array_equal(got, want), group
        back, used = lib.q4n_dequantize(got, n, group)
        assert used == got.size and np.array_equal(back + f32(0), P + f32(0)), group


def test_callers_share_the_threads(lib):
    """Calls from several threads at once, and calls after the threads have gone for want of work."""
    import threading
    import time
    rng = np.random.default_rng(9)
    data = [(rng.integers(-7, 8, n) * f32(0.031)).astype(f32) for n in (900001, 60000, 400000, 1300000)]
    alone = [lib.q4n_quantize(P, 128)[0] for P in data]
    ok = [0] * len(data)

    def caller(i):
        for _ in range(20):
            buf, raw = lib.q4n_quantize(data[i], 128)
            back, _ = lib.q4n_dequantize(buf, data[i].size, 128)
            ok[i] += raw == 0 and np.array_equal(buf, alone[i]) and np.array_equal(back, data[i])
    for pause in (0.0, 1.3):
        time.sleep(pause)
        ts = [threading.Thread(target=caller, args=(i,)) for i in range(len(data))]
        [t.start() for t in ts]
        [t.join() for t in ts]
    assert ok == [40] * len(data)


def test_a_child_of_fork_has_threads_of_its_own():
    """Children made while threads of the library sleep, and while other threads are in calls: each writes the same bytes on threads of its own, and ends in time."""
    code = CREW_CODE + """
import signal
want = lib.q4n_quantize(P, 128)[0]
def child():
    pid = os.fork()
    if pid: return pid
    try:
        signal.alarm(20)                  # a child that waits for what only its parent has
        own.update(os.listdir("/proc/self/task"))
        ok = np.array_equal(lib.q4n_quantize(P, 128)[0], want)
        os._exit(0 if ok and (crew() or os.cpu_count() == 1) else 1)
    finally:
        os._exit(2)
def finish(pid): assert os.waitstatus_to_exitcode(os.waitpid(pid, 0)[1]) == 0
assert crew() or os.cpu_count() == 1
finish(child())
stop = []
def busy():
    while not stop: call()
busy_ones = [threading.Thread(target=busy) for _ in range(3)]
[t.start() for t in busy_ones]
pids = []
for i in range(8):
    time.sleep(0.01)
    pids.append(child())
stop.append(1)
[t.join() for t in busy_ones]
for pid in pids: finish(pid)
"""
    r = subprocess.run([sys.executable, "-c", code], cwd=ROOT, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr[-2000:]


MODES = ("default", "flush", "up", "down", "zero")
MODE_CODE = """
import ctypes, threading
libm = ctypes.CDLL("libm.so.6")
def mode(name):            # of the calling thread: flush-to-zero with denormals-are-zero, or a direction of rounding
    env = (ctypes.c_uint32 * 8)()
    libm.fegetenv(env)
    env[7] = env[7] & ~0xE040 | {"default": 0, "flush": 0x8040, "up": 0x4000, "down": 0x2000, "zero": 0x6000}[name]
    libm.fesetenv(env)
def threaded(f, *args):
    t = threading.Thread(target=f, args=args); t.start(); t.join()
"""


@pytest.mark.parametrize("first", MODES)
def test_a_caller_has_its_own_floating_point_mode_and_no_other(first):
    """A caller that rounds otherwise or flushes small values to zero, and right behind it callers in every mode: each gets what one thread in its mode gives, on the
    threads that the first has left too. In the default mode that is every value, bit for bit, subnormal ones among them."""
    code = MODE_CODE + """
import numpy as np
from __graft_entry__ import load_package
from oracle.binding import Oracle
lib, orc, f32 = load_package().Qlmx(init=False), Oracle(), np.float32
rng = np.random.default_rng(3)
P = rng.integers(-7, 8, 1200000).astype(f32).reshape(-1, 100)
P[:, 0] = 7
P *= (0.01 + 0.01 * rng.random((len(P), 1))).astype(f32)
P[1::5] = rng.integers(-7, 8, P[1::5].shape) * f32(2.0 ** -140)
P[2::5] = rng.normal(size=P[2::5].shape)
P[3::5] *= f32(2.0 ** -100)
P[4::5, ::9] = f32(2.0 ** -145)          # beside values that are not small
P = np.ascontiguousarray(P.reshape(-1))
def check(name):
    mode(name)
    got, raw = lib.q4n_quantize(P, 100)
    want, wraw = orc.q4n_quantize(P, 100)
    back, used = lib.q4n_dequantize(want, P.size, 100)
    ok, wback = orc.q4n_dequantize(want, P.size, 100)
    mode("default")
    assert ok == 1 and used == want.size and raw == wraw and np.array_equal(got, want), name
    assert np.array_equal(back.view(np.uint32), wback.view(np.uint32)), name
    if name == "default":
        assert np.array_equal(back + f32(0), P + f32(0))
    done.append(name)
done = []
for name in (%r,) + %r:
    threaded(check, name)
assert len(done) == 6, done
""" % (first, MODES)
    r = subprocess.run([sys.executable, "-c", code], cwd=ROOT, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr[-2000:]


CREW_CODE = MODE_CODE + """
import numpy as np, os, time
from __graft_entry__ import load_package
lib, f32 = load_package().Qlmx(init=False), np.float32
P = (np.arange(1200000) % 15 - 7).astype(f32) * f32(0.25)
wire = lib.q4n_quantize(P[:1280], 128)[0]
own = set(os.listdir("/proc/self/task"))        # before any thread of the library
def call(): assert lib.q4n_quantize(P, 128)[1] == 0
def crew(): return sorted(int(t) for t in set(os.listdir("/proc/self/task")) - own)
def ran(t): return int(open("/proc/self/task/%d/schedstat" % t).read().split()[0])
"""


@pytest.mark.skipif(len(os.sched_getaffinity(0)) < 4, reason="needs four CPUs")
def test_kept_threads_run_where_their_caller_may():
    """A caller bound to two CPUs starts the threads; those that work for the next caller, which is not bound, are not bound either, and the bound caller's are again."""
    code = CREW_CODE + """
everywhere = os.sched_getaffinity(0)
two = set(sorted(everywhere)[:2])
def bound():
    os.sched_setaffinity(0, two)
    for i in range(5): call()
    own.add(str(threading.get_native_id()))
threaded(bound)
for want, many in ((everywhere, 20), (two, 20)):
    os.sched_setaffinity(0, want)
    worked, wrong = set(), set()
    for i in range(many):
        before = {t: ran(t) for t in crew()}
        call()
        for t in crew():
            if ran(t) - before.get(t, 0) > 100000:          # more than to wake and find nothing left
                worked.add(t)
                if os.sched_getaffinity(t) != want: wrong.add(t)
    assert worked and not wrong, (want, worked, wrong)
"""
    r = subprocess.run([sys.executable, "-c", code], cwd=ROOT, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr[-2000:]


@pytest.mark.skipif(os.getpriority(os.PRIO_PROCESS, 0) >= 19, reason="needs a priority below its own")
def test_kept_threads_serve_callers_of_their_own_priority():
    """Threads started by a caller of low priority do nothing for one of ordinary priority, which has threads of its own as long as they are there, and the other
    way round; once they have gone the next caller's are kept."""
    code = CREW_CODE + """
def low():
    os.setpriority(os.PRIO_PROCESS, 0, 19)
    for i in range(5): call()
    own.add(str(threading.get_native_id()))
def worked(): return [t for t in kept if ran(t) - before[t] > 100000]
threaded(low)
kept = crew()
assert kept and all(os.getpriority(os.PRIO_PROCESS, t) == 19 for t in kept)
for i in range(10):
    before = {t: ran(t) for t in kept}
    call()
    assert not worked()
time.sleep(2.5)
assert not crew()
call()
kept = crew()
assert kept and all(os.getpriority(os.PRIO_PROCESS, t) == os.getpriority(os.PRIO_PROCESS, 0) for t in kept)
before = {t: ran(t) for t in kept}
threaded(low)
assert not worked()
"""
    r = subprocess.run([sys.executable, "-c", code], cwd=ROOT, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr[-2000:]


def test_kept_threads_leave_faults_to_the_programs_handlers():
    """A program may answer a fault on its buffers in a handler (pages mapped or unprotected on first use), and has to be asked on the library's threads as on its own;
    signals sent to the process are for the program's threads."""
    code = CREW_CODE + """
import signal
call()
time.sleep(0.2)          # a thread starts with all signals blocked
assert crew()
for t in crew():
    status = dict(line.split(":", 1) for line in open("/proc/self/task/%d/status" % t))
    blocked = int(status["SigBlk"], 16)
    for name in ("SIGSEGV", "SIGBUS", "SIGFPE", "SIGILL", "SIGTRAP", "SIGSYS"):
        assert not blocked >> (getattr(signal, name) - 1) & 1, name
    for name in ("SIGINT", "SIGTERM", "SIGALRM", "SIGUSR1"):
        assert blocked >> (getattr(signal, name) - 1) & 1, name
"""
    r = subprocess.run([sys.executable, "-c", code], cwd=ROOT, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr[-2000:]


def test_truncated_buffer_is_refused(lib, orc, golden):
    g = golden("q4n")
    n, group = (int(v) for v in g["dims"])
    for cut in (3, 40, g["buf"].size - 1):
        with pytest.raises(pkg.QlmxError, match="buffer ends"):
            lib.q4n_dequantize(g["buf"][:cut].copy(), n, group)
        ok, _ = orc.q4n_dequantize(g["buf"][:cut].copy(), n, group)
        assert ok == 0


@pytest.mark.parametrize("n", [2 ** 31, 2 ** 50, 2 ** 64 - 1, 2 ** 64 - 200])
def test_count_larger_than_the_buffer_is_refused(lib, n):
    """A count that the buffer cannot hold (a damaged file names any) ends at the group where the buffer does, whatever the
    scratch for that many groups would have been."""
    import ctypes
    group = 128
    whole, _ = lib.q4n_quantize(np.zeros(3 * group, f32), group)
    for buf, at in ((whole[:8].copy(), 0), (whole, 3)):
        P, used = np.zeros(4 * group, f32), ctypes.c_size_t(0)
        with pytest.raises(pkg.QlmxError, match="buffer ends inside group %d$" % at):
            lib.call("qlmx_q4n_dequantize", buf, buf.size, P, n, group, ctypes.addressof(used))


def limited(code, spare):
    """Runs `code` in a process that may take `spare` bytes of memory more than it holds when the library is loaded."""
    head = ("import resource, numpy as np\nfrom __graft_entry__ import load_package\n"
            "pkg = load_package(); lib = pkg.Qlmx(init=False); f32 = np.float32\n"
            "def limit():\n"
            "    now = int(open('/proc/self/statm').read().split()[0]) * resource.getpagesize()\n"
            "    resource.setrlimit(resource.RLIMIT_AS, (now + %d, now + %d))\n" % (spare, spare))
    return subprocess.run([sys.executable, "-c", head + code], cwd=ROOT, capture_output=True, text=True, timeout=100)


def test_scratch_is_bounded_by_the_values():
    """A group far longer than the values is one group of all of them: no scratch for what is not there."""
    r = limited("P = (np.arange(300000) %% 15 - 7).astype(f32) * f32(0.25)\n"
                "want, _ = lib.q4n_quantize(P, 300000)\nlimit()\n"
                "for group in (300002, 2 ** 31 - 2):\n"
                "    got, raw = lib.q4n_quantize(P, group)\n"
                "    assert raw == 0 and np.array_equal(got, want)\n"
                "    back, used = lib.q4n_dequantize(got, P.size, group)\n"
                "    assert used == got.size and np.array_equal(back, P)\n".replace("%%", "%"), 256 << 20)
    assert r.returncode == 0, r.stderr[-2000:]


def test_allocation_failure_is_an_error_code():
    """Scratch that cannot be had is reported as an error of the call; the process goes on and a smaller call works."""
    r = limited("n = 24 << 20\nbuf = np.zeros(5 * n, np.uint8); P = np.zeros(n, f32); out = np.zeros(8 * n, np.uint8)\nlimit()\n"
                "import ctypes; u = ctypes.c_size_t(0)\n"
                "for name, args in (('qlmx_q4n_dequantize', (buf, buf.size, P, n, 1, ctypes.addressof(u))),\n"
                "                   ('qlmx_q4n_quantize', (P, n, 2, out, out.size, ctypes.addressof(u), None))):\n"
                "    try:\n        lib.call(name, *args)\n"
                "    except pkg.QlmxError as e:\n        assert 'memory' in str(e), e\n"
                "    else:\n        raise AssertionError(name)\n"
                "back, used = lib.q4n_dequantize(buf[:50], 10, 1)\nassert used == 50 and not back.any()\n", 40 << 20)
    assert r.returncode == 0, r.stderr[-2000:]


def test_against_reference_library_when_present(lib, orc, ref):
    rng = np.random.default_rng(7)
    for group in (128, 64, 32):
        n = group * 9 + 10
        s = f32(0.0173)
        P = (rng.integers(-7, 8, n).astype(f32) * s).astype(f32)
        P[group:2 * group] = rng.normal(size=group).astype(f32)
        want = ref.q4n_quantize(P, group)
        got, _ = lib.q4n_quantize(P, group)
        ob, _ = orc.q4n_quantize(P, group)
        assert np.array_equal(got, want) and np.array_equal(ob, want)

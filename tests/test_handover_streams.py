"""Which stream the self-referential kernels in one launch and the counters they share go to: the library's own entry points
against a runtime that only writes down what it is asked for, so no GPU is needed."""
import os
import subprocess
import sys

import pytest

from nl_hecate_amd import ffi

# A runtime in front of the real one: device memory is host memory that nobody reads, kernels are names.
RUNTIME = r"""
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <thread>
#include <utility>
struct dim3 { unsigned x, y, z; };
static std::map<const void *, std::string> names;
static std::string said;
static struct { dim3 grid, block; size_t lds; void *stream; } pushed;
static const char *moment = nullptr;   // the next call of this name is followed by then(with)
static void (*then)(void *) = nullptr;
static void *with = nullptr;
static void say(const char *what, const char *which, const void *stream) {
    char line[1024];
    snprintf(line, sizeof line, "%s %s %zu\n", what, which, (size_t)stream);
    said += line;
}
static std::thread other;
static const char *failing = nullptr;   // the next call of this name fails
static int answer(const char *call) {
    if (failing && !strcmp(failing, call)) { failing = nullptr; return 1; }
    if (!moment || strcmp(moment, call)) return 0;
    moment = nullptr;
    other = std::thread(then, with);
    std::this_thread::sleep_for(std::chrono::milliseconds(200));   // it is done by then, or waits for this thread
    return 0;
}
extern "C" {
const char *what_was_said() { return said.c_str(); }
void say_nothing() { said.clear(); }
// Another thread calls f(stream) right behind the next call of that name; join_other() waits for its end.
void fail_next(const char *call) { failing = strdup(call); }
void join_other() { if (other.joinable()) other.join(); }
void behind_next(const char *call, void (*f)(void *), void *stream) { moment = strdup(call); then = f; with = stream; }

void **__hipRegisterFatBinary(const void *) { static void *m; return &m; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *f, char *, const char *name, unsigned, void *, void *, void *, void *, int *) { names[f] = name; }
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
int __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, void *s) { pushed = {g, b, lds, s}; return 0; }
int __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *lds, void **s) { *g = pushed.grid; *b = pushed.block; *lds = pushed.lds; *s = pushed.stream; return 0; }
int hipLaunchKernel(const void *f, dim3, dim3, void **, size_t, void *s) { say("launch", names[f].c_str(), s); return 0; }
int hipGetDevice(int *d) { *d = 0; return 0; }
int hipGetLastError() { return answer("hipGetLastError"); }
const char *hipGetErrorString(int) { return "failed on purpose"; }
int hipFuncSetAttribute(const void *, int, int) { return answer("hipFuncSetAttribute"); }
int hipThreadExchangeStreamCaptureMode(int *mode) {   // 0 global, 2 relaxed
    static int now = 0;
    std::swap(now, *mode);
    say("mode", now == 2 ? "relaxed" : "global", nullptr);
    return 0;
}
int hipMalloc(void **p, size_t n) { *p = malloc(n); say("alloc", "", nullptr); return 0; }
int hipFree(void *p) { free(p); say("free", "", nullptr); return 0; }
int hipStreamSynchronize(void *s) { say("synchronize", "", s); return 0; }
int hipDeviceSynchronize() { say("synchronize", "device", nullptr); return 0; }
int hipEventCreateWithFlags(void **e, unsigned) { static size_t n = 0; *e = (void *)(++n << 16); return 0; }
int hipEventDestroy(void *) { return 0; }
int hipEventSynchronize(void *) { say("synchronize", "event", nullptr); return 0; }
int hipEventRecord(void *e, void *s) { say("record", std::to_string((size_t)e).c_str(), s); return 0; }
int hipStreamWaitEvent(void *s, void *e, unsigned) { say("wait", std::to_string((size_t)e).c_str(), s); return answer("hipStreamWaitEvent"); }
int hipStreamIsCapturing(void *s, int *status) { *status = 0; say("query", "", s); return answer("hipStreamIsCapturing"); }
}
"""

DRIVER = r"""
import ctypes, sys
fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
fake.what_was_said.restype = ctypes.c_char_p
fake.behind_next.argtypes = [ctypes.c_char_p, ctypes.c_void_p, ctypes.c_void_p]
from nl_hecate_amd.ffi import lib
lib.load()
some = 4096   # a device address that nobody reads
forward = lambda B, s, C, d=64: lib.selfref_chunkwise_forward_f32_rocm(*[some] * 11, s, d, B, C, 1)
backward = lambda B, s, C, d=64: lib.selfref_chunkwise_backward_f32_rocm(*[some] * 12, s, d, B, C, 1)
ONE, OTHER = 0x1000, 0x2000
on = lambda stream: lib.nlh_set_stream(ctypes.c_void_p(stream))
switch_behind = lambda call, stream: fake.behind_next(call, ctypes.cast(lib.nlh_set_stream, ctypes.c_void_p), stream)
def said():
    fake.join_other()
    out = [tuple(line.split(" ")) for line in fake.what_was_said().decode().splitlines()]
    fake.say_nothing()
    return [(what, which, int(stream)) for what, which, stream in out]
def launches():
    return [(which, stream) for what, which, stream in said() if what == "launch"]
"""


@pytest.fixture(scope="module")
def on_host(tmp_path_factory):
    at = tmp_path_factory.mktemp("runtime")
    (at / "runtime.cpp").write_text(RUNTIME)
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-pthread", "-o", str(at / "runtime.so"), str(at / "runtime.cpp")])
    root = os.path.dirname(os.path.dirname(os.path.abspath(ffi.__file__)))

    def run(body):
        r = subprocess.run([sys.executable, "-c", DRIVER + body, str(at / "runtime.so")], cwd=root, capture_output=True, text=True,
                           timeout=100)
        assert r.returncode == 0, r.stdout + r.stderr

    return run


CALLS = [("forward", "2, 640, 64", "selfref_forward_kernel"), ("backward", "64, 1024, 64", "selfref_backward_kernel")]


@pytest.mark.parametrize("moment", ["hipStreamIsCapturing", "hipFuncSetAttribute"])
@pytest.mark.parametrize("call,sizes,kernel", CALLS)
def test_counters_and_their_kernel_on_one_stream(on_host, call, sizes, kernel, moment):
    """Another thread sets another stream while a call is under way."""
    on_host(f"""
on(ONE)
{call}({sizes})       # what is allocated once
said()
switch_behind(b"{moment}", OTHER)
{call}({sizes})
ran = launches()
clear = [s for name, s in ran if "clear_counters_kernel" in name]
kernel = [s for name, s in ran if "{kernel}" in name]
assert clear == kernel == [ONE], ran
""")


@pytest.mark.parametrize("call,sizes,kernel", CALLS)
def test_one_handle_for_a_stream_in_every_thread(on_host, call, sizes, kernel):
    """hipStreamPerThread: two threads' launches are not ordered, so they share no counters."""
    on_host(f"""
PER_THREAD = 2
on(PER_THREAD)
{call}({sizes})
ran = launches()
assert ran and not any("clear_counters_kernel" in name or "{kernel}" in name for name, _ in ran), ran
assert {{stream for _, stream in ran}} == {{PER_THREAD}}
on(ONE)      # which did not make it the owner
{call}({sizes})
assert any("{kernel}" in name for name, _ in launches())
""")


@pytest.mark.parametrize("call,sizes,kernel", CALLS)
def test_a_handle_that_comes_again(on_host, call, sizes, kernel):
    """A stream destroyed with work on it, its handle given to another one: the counters are cleared behind the work."""
    on_host(f"""
on(ONE)
{call}({sizes})
for _ in range(3):
    said()
    {call}({sizes})
    order = [(what, which) for what, which, stream in said() if stream == ONE and what != "query"]
    what = [w for w, _ in order]
    assert what == ["wait", "launch", "launch", "record"], order
    assert order[0][1] == order[3][1] and "clear_counters_kernel" in order[1][1] and "{kernel}" in order[2][1], order
lib.nlh_release_workspace()
on(None)     # which cannot be destroyed
{call}({sizes})
said()
{call}({sizes})
assert [what for what, _, stream in said() if what in ("wait", "launch", "record")] == ["launch", "launch"]
""")


def test_counters_that_grow_wait_for_their_last_user(on_host):
    on_host("""
on(ONE)
forward(2, 640, 64)
said()
forward(8, 640, 64)
order = [(what, which) for what, which, _ in said() if what in ("synchronize", "free", "alloc")]
assert order == [("synchronize", "event"), ("free", ""), ("alloc", "")], order
""")


def test_optional_scratch_is_allocated_beside_captures(on_host):
    """A capture of another stream ends with an allocation, a free or a wait in the mode that it has by default."""
    on_host("""
on(ONE)
inside = False
for size in ((2, 640, 64), (8, 640, 64)):
    forward(*size)
    for what, which, _ in said():
        inside = which == "relaxed" if what == "mode" else inside
        assert inside or what not in ("alloc", "free", "synchronize"), what
assert not inside
""")


@pytest.mark.parametrize("call,sizes,kernel", CALLS)
def test_a_release_waits_for_the_launch(on_host, call, sizes, kernel):
    """nlh_release_workspace from another thread while a call has its counters and has not launched their kernel."""
    on_host(f"""
on(ONE)
{call}({sizes})
said()
fake.behind_next(b"hipFuncSetAttribute", ctypes.cast(lib.nlh_release_workspace, ctypes.c_void_p), None)
{call}({sizes})
order = [which if what == "launch" else what for what, which, _ in said() if what in ("launch", "free")]
assert "free" in order and [o for o in order if "{kernel}" in o], order
assert max(i for i, o in enumerate(order) if "{kernel}" in o) < order.index("free"), order
""")


@pytest.mark.parametrize("step", ["hipStreamWaitEvent", "hipGetLastError"])   # behind the launch that clears them
@pytest.mark.parametrize("call,sizes,kernel", CALLS)
def test_no_kernel_on_counters_that_were_not_cleared(on_host, call, sizes, kernel, step):
    on_host(f"""
lib.nlh_set_error_mode(1)
on(ONE)
{call}({sizes})
said()
fake.fail_next(b"{step}")
{call}({sizes})
assert b"failed on purpose" in ctypes.string_at(lib.nlh_last_error())
assert not any("{kernel}" in name for name, _ in launches())
lib.nlh_clear_error()
{call}({sizes})
assert any("{kernel}" in name for name, _ in launches()) and ctypes.string_at(lib.nlh_last_error()) == b""
""")

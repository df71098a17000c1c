"""Which kernels a call of the C ABI launches, without a GPU: the library between a stand-in for the HIP runtime that writes down
every launch and a process of its own.  The stand-in's device has 256 CUs; the pointers that a call passes are never followed."""
import json
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "ditango_amd", "lib", "libditango_hip.so")

_RUNTIME = r"""
#include <cstddef>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <sys/syscall.h>
#include <unistd.h>
#include <vector>
struct Dim3 { unsigned x, y, z; };
static std::map<const void*, std::string>& names() { static std::map<const void*, std::string> m; return m; }
static std::mutex mu;
static std::string text;
static int wait_us = 0;
static thread_local Dim3 grid, block;
static thread_local size_t lds;
static thread_local void* queue;
extern "C" {
void** __hipRegisterFatBinary(const void*) { static void* handle; return &handle; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* device, unsigned, void*, void*, void*, void*, int*) { names()[host] = device; }
void __hipRegisterVar(void**, void*, char*, const char*, int, size_t, int, int) {}
int __hipPushCallConfiguration(Dim3 g, Dim3 b, size_t l, void* q) { grid = g; block = b; lds = l; queue = q; return 0; }
int __hipPopCallConfiguration(Dim3* g, Dim3* b, size_t* l, void** q) { *g = grid; *b = block; *l = lds; *q = queue; return 0; }
int hipDeviceGetAttribute(int* value, int, int) { *value = 256; return 0; }
int hipFuncSetAttribute(const void*, int, int) { return 0; }
int hipGetDevice(int* device) { *device = 0; return 0; }
const char* hipGetErrorString(int) { return "stand-in"; }
int hipGetLastError(void) { return 0; }
int hipGetSymbolAddress(void** p, const void*) { *p = reinterpret_cast<void*>(4096); return 0; }
int hipPointerGetAttributes(void*, const void*) { return 1; }
int hipLaunchKernel(const void* f, Dim3, Dim3, void**, size_t, void*) {
  {
    std::lock_guard<std::mutex> lock(mu);
    text += std::to_string(syscall(SYS_gettid)) + " " + names()[f] + "\n";
  }
  if (wait_us) usleep(wait_us);
  return 0;
}
const char* log_text(void) { return text.c_str(); }
void log_clear(void) { text.clear(); }
void log_wait(int us) { wait_us = us; }
}
"""

_PROCESS = r"""
import ctypes, json, sys, threading
runtime = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
runtime.log_text.restype = ctypes.c_char_p
lib = ctypes.CDLL(sys.argv[2])
i32, i64, vp, f32 = ctypes.c_int32, ctypes.c_int64, ctypes.c_void_p, ctypes.c_float
lib.dt_attn_merge_counters.restype = lib.dt_attn_workspace_bytes.restype = i64
lib.dt_last_error.restype = ctypes.c_char_p
AT = 1 << 20   # any aligned address

class Into(ctypes.Structure):
    _fields_ = [("out", vp), ("lse", vp), ("dtype", i32), ("n_states", i32), ("outs", vp), ("lses", vp), ("counters", vp), ("n_counters", i64)]

def call(B, Sq, H, D, lens, jobs, merged, fp16=False, max_jobs=0, workspace=True):
    # jobs: lists of chunks (host-listed), or None: max_jobs jobs listed on the device.  merged: the number of states, 0: no merge.
    n = len(lens)
    at = lambda k: (vp * max(k, 1))(*[AT] * max(k, 1))
    head = [vp(AT), i32(B), i32(Sq), i32(H), i32(D), i64(Sq * H * D), i64(H * D), i64(D), i32(n), at(n), at(n), (i32 * n)(*lens),
            (i64 * n)(*[x * H * D for x in lens]), i64(H * D), i64(D)]
    ws = [vp(AT if workspace else 0), i64(lib.dt_attn_workspace_bytes() if workspace else 0)]
    flags = i32(2 if fp16 else 0)
    counters = lib.dt_attn_merge_counters(B, Sq, H)
    into = Into(AT, AT, 2 if fp16 else 0, merged, ctypes.cast(at(merged), vp), ctypes.cast(at(merged), vp), AT, counters)
    if jobs is None:
        sched = [vp(AT), vp(AT), i32(max_jobs), vp(AT), i64(B * Sq * H * D), vp(AT), i64(B * H * Sq), i32(-1), vp(AT), vp(AT)]
        if merged: rc = lib.dt_attn_sched_merge_fwd(*head, *sched, ctypes.byref(into), f32(0), flags, *ws, vp(0))
        else: rc = lib.dt_attn_sched_seg_ws_fwd(*head, *sched, i32(0), vp(0), vp(0), vp(0), vp(0), f32(0), flags, *ws, vp(0))
    else:
        begin, chunks = [0], []
        for job in jobs:
            chunks += job
            begin.append(len(chunks))
        listed = [i32(len(jobs)), (i32 * len(begin))(*begin), (i32 * max(1, len(chunks)))(*chunks)]
        dst = [at(len(jobs)), at(len(jobs))]
        if merged: rc = lib.dt_attn_jobs_merge_fwd(*head, *listed, *dst, ctypes.byref(into), f32(0), flags, *ws, vp(0))
        else: rc = lib.dt_attn_seg_jobs_ws_fwd(*head, *listed, vp(0), vp(0), vp(0), vp(0), *dst, f32(0), flags, *ws, vp(0))
    assert rc == 0, lib.dt_last_error()

asked = json.loads(sys.stdin.read())
answer = []
for calls in asked["in turn"]:
    runtime.log_clear()
    call(**calls)
    answer.append([line.split(" ", 1) for line in runtime.log_text().decode().splitlines()])
    if calls["merged"]:   # what the library says of such a call beforehand
        B, Sq, H, D, jobs = (calls[k] for k in ("B", "Sq", "H", "D", "jobs"))
        tiles = lambda c: (calls["lens"][c] + 63) // 64
        longest = max(map(tiles, range(len(calls["lens"])))) if jobs is None else max(sum(map(tiles, job)) for job in jobs)
        need = lib.dt_attn_merges_in_launch(B, Sq, H, D, calls["max_jobs"] if jobs is None else len(jobs), int(jobs is not None), longest, calls["merged"])
        assert need == lib.dt_attn_merge_counters(B, Sq, H) if len(answer[-1]) == 1 else need in (0, lib.dt_attn_merge_counters(B, Sq, H)), calls
if asked["together"]:
    runtime.log_clear()
    runtime.log_wait(2000)
    start = threading.Barrier(len(asked["together"]))
    def work(c):
        start.wait()
        for _ in range(asked["times"]): call(**c)
    threads = [threading.Thread(target=work, args=(c,)) for c in asked["together"]]
    for t in threads: t.start()
    for t in threads: t.join()
    answer.append([line.split(" ", 1) for line in runtime.log_text().decode().splitlines()])
print(json.dumps(answer))
"""


def record(tmp_path, in_turn=(), together=(), times=0):
    """The launches, (thread, kernel) in the order in which they enter the queue, of every call of ``in_turn`` and then of the calls
    of ``together``, each made ``times`` times by a thread of its own while a launch takes 2 ms.  A call is the arguments of
    ``call`` above; one of ``in_turn`` that merges in its launch has to be one of which ``dt_attn_merges_in_launch`` says so."""
    source, runtime = tmp_path / "runtime.cpp", tmp_path / "runtime.so"
    source.write_text(_RUNTIME)
    subprocess.run(["g++", "-shared", "-fPIC", "-O1", "-o", str(runtime), str(source)], check=True)
    script = tmp_path / "process.py"
    script.write_text(_PROCESS)
    asked = json.dumps({"in turn": list(in_turn), "together": list(together), "times": times})
    run = subprocess.run([sys.executable, str(script), str(runtime), LIB], input=asked, capture_output=True, text=True, timeout=100)
    assert run.returncode == 0, run.stderr[-2000:]
    return json.loads(run.stdout)

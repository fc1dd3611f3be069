"""The bookkeeping of the library workspace (csrc/hip/workspace.hpp) on the host, over a
recorded stand-in for the device: calls of several streams and threads follow each
other, and a buffer that cannot grow leaves an empty one."""
import shutil
import subprocess
from pathlib import Path

import pytest

HIP = Path(__file__).resolve().parents[1] / "spsim_amd" / "csrc" / "hip"

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not installed")

PRELUDE = r"""
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <string>
#include <thread>
#include <vector>
#include "workspace.hpp"
using namespace spsim;
// Streams and events are small numbers; what is asked of the device is written down.
std::string logged;
bool memory = true, events = true, capture[8];
void put(const std::string &what) { logged += what + " "; }
struct Api {
  using Stream = int;
  using Event = int;
  static bool alloc(void **p, size_t n) {
    put((memory ? "alloc" : "none") + std::to_string(n));
    if (memory) *p = malloc(n);
    return memory;
  }
  static void free(void *p) { put("free"); ::free(p); }
  static bool synchronize() { put("sync"); return true; }
  static bool capturing(int s) { return capture[s]; }
  static bool lasting(int s) { return s == 0; }  // the default stream
  static bool record(int *e, int s) {
    if (events) *e = s;
    put(events ? "record" + std::to_string(s) : "norecord");
    return events;
  }
  static bool wait(int s, int e) { put("wait" + std::to_string(s) + "for" + std::to_string(e)); return true; }
};
using Shared = SharedWorkspace<Api>;
void *use(Shared &ws, int stream, size_t bytes) {
  Shared::Use u(stream);
  void *p = nullptr;
  if (!u.acquire(&ws) || u.get(bytes, &p) != WorkspaceResult::kOk) return nullptr;
  put("work");
  return p;
}
"""


def _run(tmp_path, body):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(PRELUDE + "int main() {\n  Shared ws;\n" + body + '\n  puts(logged.c_str());\n}\n')
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-pthread", f"-I{HIP}", str(src), "-o", str(exe)],
                   check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stderr
    return r.stdout.split()


def test_streams_follow_each_other(tmp_path):
    """Every call waits for the last one's event; a call that never looks at the
    buffer does nothing."""
    assert _run(tmp_path, """
  use(ws, 1, 100);
  { Shared::Use unused(5); }
  use(ws, 2, 100);
  use(ws, 1, 50);
  ws.release();""") == ["alloc125", "work", "record1", "wait2for1", "work", "record2", "wait1for2", "work", "record1",
                        "sync", "free"]


def test_the_default_stream_is_recorded_when_another_one_comes(tmp_path):
    """Calls on it alone record nothing and wait for nothing."""
    assert _run(tmp_path, """
  use(ws, 0, 100);
  use(ws, 0, 100);
  use(ws, 1, 100);
  use(ws, 0, 100);
  events = false;
  use(ws, 2, 100);""") == ["alloc125", "work", "work", "record0", "wait1for0", "work", "record1", "wait0for1", "work",
                           "norecord", "sync", "work", "norecord", "sync"]


def test_a_capture_neither_waits_nor_records(tmp_path):
    assert _run(tmp_path, """
  use(ws, 1, 100);
  capture[2] = true;
  use(ws, 2, 100);
  use(ws, 3, 100);
  ws.release();""") == ["alloc125", "work", "record1", "work", "wait3for1", "work", "record3", "sync", "free"]


def test_a_captured_buffer_outlives_growth(tmp_path):
    """It is kept through larger ones, eager or captured, until the release; a
    buffer that no capture was given is freed at once."""
    assert _run(tmp_path, """
  use(ws, 1, 100);
  use(ws, 1, 200);
  capture[2] = true;
  use(ws, 2, 200);
  use(ws, 1, 400);
  use(ws, 2, 400);
  use(ws, 1, 800);
  use(ws, 1, 2000);
  ws.release();
  use(ws, 1, 100);
  ws.release();""") == ["alloc125", "work", "record1", "wait1for1", "sync", "free", "alloc250", "work", "record1",
                        "work", "wait1for1", "sync", "alloc500", "work", "record1", "work", "wait1for1", "sync",
                        "alloc1000", "work", "record1", "wait1for1", "sync", "free", "alloc2500", "work", "record1",
                        "sync", "free", "free", "free", "wait1for1", "alloc125", "work", "record1", "sync", "free"]


def test_growth_and_no_memory(tmp_path):
    """Growth frees the old buffer after the device is idle. Without memory for
    the larger one there is none, and the same call goes on with a smaller one."""
    assert _run(tmp_path, """
  use(ws, 1, 100);
  {
    Shared::Use u(1);
    void *p = nullptr;
    if (!u.acquire(&ws)) return 1;
    if (!u.holds(125) || u.holds(126)) return 2;
    memory = false;
    if (u.get(1000, &p) != WorkspaceResult::kNoMemory || p || u.holds(1)) return 3;
    memory = true;
    if (u.get(40, &p) != WorkspaceResult::kOk || !p) return 4;
    put("work");
  }
  ws.release();
  ws.release();""") == ["alloc125", "work", "record1", "wait1for1", "sync", "free", "none1250", "alloc50", "work",
                        "record1", "sync", "free"]


def test_without_events_the_call_waits_itself(tmp_path):
    assert _run(tmp_path, """
  events = false;
  use(ws, 1, 4);
  use(ws, 2, 4);
  ws.release();""") == ["alloc5", "work", "norecord", "sync", "work", "norecord", "sync", "sync", "free"]


def test_threads_take_turns(tmp_path):
    """From its first look at the buffer to its end a call has it alone."""
    assert _run(tmp_path, """
  std::atomic<int> inside{0}, clashes{0};
  std::vector<std::thread> threads;
  for (int t = 0; t < 4; ++t)
    threads.emplace_back([&, t] {
      for (int i = 0; i < 200; ++i) {
        Shared::Use u(t);
        void *p = nullptr;
        if (!u.acquire(&ws)) abort();
        if (inside.fetch_add(1) != 0) ++clashes;
        if (u.get(16 + i * 4 + t, &p) != WorkspaceResult::kOk) abort();
        ((char *)p)[15] = 1;
        std::this_thread::yield();
        inside.fetch_sub(1);
      }
    });
  for (auto &t : threads) t.join();
  logged.clear();
  put(std::to_string(clashes.load()));
  ws.release();""") == ["0", "sync", "free"]

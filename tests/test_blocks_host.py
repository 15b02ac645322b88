"""Block cache (csrc/sq_blocks.h) on the host, over a memory of its own that
refuses requests beyond its size and remembers the error of a refused one,
like the HIP runtime.  Each case is a few lines of C++; a failed CHECK prints
its line."""
import glob
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "siam-quantum_amd", "csrc")
HEAD = r"""
#include "sq_blocks.h"
#include <cstdio>
#include <cstdlib>
#include <map>
#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)
constexpr size_t G = size_t(1) << 30;
struct State {
  size_t size[2] = {288 * G, 288 * G}, used[2] = {0, 0}, pinned = 0, pinned_size = 64 * G;
  int dev = 0, error = 0, mallocs = 0;
  char* next = (char*)4096;
  std::map<void*, std::pair<size_t, int>> what;  // bytes, device (-1: host)
};
struct Mem {
  State* s;
  int malloc(void** p, size_t bytes, bool host) {
    size_t &u = host ? s->pinned : s->used[s->dev], m = host ? s->pinned_size : s->size[s->dev];
    if (u + bytes > m) return s->error = 2;
    u += bytes;
    ++s->mallocs;
    *p = s->next;
    s->next += 4096;
    s->what[*p] = {bytes, host ? -1 : s->dev};
    return 0;
  }
  int free(void* p, bool host) {
    const auto w = s->what.at(p);
    if (host != (w.second < 0)) std::abort();
    (host ? s->pinned : s->used[w.second]) -= w.first;
    s->what.erase(p);
    return 0;
  }
  void clear_error() { s->error = 0; }
  int device() { return s->dev; }
  size_t total() { return s->size[s->dev]; }
  size_t available() { return s->size[s->dev] - s->used[s->dev]; }
};
int main() {
  State st;
  BlockCache<Mem> c(Mem{&st});
"""


def _run(tmp_path, body):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(HEAD + body + "  return 0;\n}\n")
    subprocess.run(["g++", "-std=c++17", "-Wall", "-I", CSRC, str(src), "-o", str(exe), "-lpthread"], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout


@pytest.mark.parametrize("host", ["false", "true"])
def test_refused_request_leaves_no_error(tmp_path, host):
    """A request that succeeds once the cache is given back, and one that
    fails for good: the runtime's last error is clear after both."""
    _run(tmp_path, f"""
  st.size[0] = st.pinned_size = 4 * G;
  void* a = c.get(3 * G, {host});
  CHECK(a);
  c.put(a);
  void* b = c.get(1536 * (size_t(1) << 20) + 1, {host});  // the cached block holds it
  CHECK(b == a);
  c.put(b);
  b = c.get(G, {host});  // it is too large for this one
  CHECK(b && st.mallocs == 2);
  c.put(b);
  b = c.get(4 * G, {host});  // fits when both have gone
  CHECK(b);
  CHECK(st.error == 0);
  CHECK(!c.get(G, {host}));
  CHECK(st.error == 0);
  c.put(b);
""")


def test_smallest_fitting_block(tmp_path):
    """The smallest block of the same kind and device, at most twice the
    request; a released block is handed out again."""
    _run(tmp_path, """
  void* a = c.get(300, false); void* b = c.get(200, false); void* h = c.get(150, true);
  c.put(a); c.put(b); c.put(h);
  CHECK(c.get(150, false) == b);
  CHECK(c.get(150, true) == h);
  CHECK(c.get(149, false) != a);  // 300 > 2 * 149
  st.dev = 1;
  CHECK(c.get(200, false) != a);
  st.dev = 0;
  CHECK(c.get(200, false) == a);
  c.put(nullptr);
""")


def test_large_blocks_follow_their_user(tmp_path):
    """Device blocks above 256 MiB: 4 GiB without a large user, an eighth of
    the device beside that with one, nothing of it after it."""
    _run(tmp_path, """
  auto pass = [&](size_t big) {
    void* a = c.get(big, false); void* b = c.get(5 * G, false); void* s = c.get(100, false);
    c.put(a); c.put(b); c.put(s);
  };
  pass(17 * G);
  CHECK(c.cached(0) == 100);
  c.large_user(1);
  pass(17 * G);
  CHECK(c.cached(0) == 22 * G + 100);
  const int n = st.mallocs;
  pass(17 * G);
  CHECK(st.mallocs == n);  // all of them were there
  c.put(c.get(15 * G, false));  // takes the 17 GiB block and gives it back
  CHECK(c.cached(0) == 22 * G + 100);
  void* x = c.get(30 * G, false);
  c.put(x);  // 52 GiB would pass the eighth
  CHECK(c.cached(0) == 22 * G + 100);
  c.large_user(1); c.large_user(-1);
  CHECK(c.cached(0) == 22 * G + 100);
  c.large_user(-1);
  CHECK(c.cached(0) == 100);
  CHECK(c.trim() == 100 && c.cached(0) == 0 && st.used[0] == 0);
""")


def test_large_blocks_leave_half_the_device(tmp_path):
    """With less than half of the device free, by whomever, only the 4 GiB."""
    _run(tmp_path, """
  c.large_user(1);
  st.used[0] = 130 * G;  // another process, or another allocator of this one
  void* a = c.get(10 * G, false); void* b = c.get(10 * G, false);
  c.put(a);  // 138 GiB free
  CHECK(c.cached(0) == 0);
  c.put(b);  // 148 GiB free with a gone
  CHECK(c.cached(0) == 10 * G);
  a = c.get(10 * G, false);
  CHECK(a == b);
  st.used[0] += 10 * G;
  c.put(a);
  CHECK(c.cached(0) == 0);
""")


def test_pinned_and_devices_apart(tmp_path):
    """Pinned memory never passes 4 GiB, and each device has its own eighth."""
    _run(tmp_path, """
  c.large_user(1);
  void* h = c.get(5 * G, true); void* g = c.get(3 * G, true);
  c.put(h); c.put(g);
  CHECK(st.pinned == 3 * G);
  void* a = c.get(30 * G, false);
  c.put(a);
  st.dev = 1;
  void* b = c.get(30 * G, false);
  c.put(b);
  CHECK(c.cached(0) == 30 * G && c.cached(1) == 30 * G);
  CHECK(c.get(20 * G, false) == b);
  st.dev = 0;
  c.put(b);  // of the other device: not beyond the 4 GiB
  CHECK(c.cached(1) == 0 && st.used[1] == 0);
""")


def test_device_memory_in_one_place():
    """Every allocation of the library goes through the cache, which gives up
    its blocks when the device is full: no other source calls the runtime's."""
    calls = [(os.path.basename(f), line.strip()) for f in sorted(glob.glob(os.path.join(CSRC, "*")))
             for line in open(f) if re.search(r"\bhip(Host)?Malloc(Async)?\(", line.split("//")[0])]
    assert len(calls) == 1 and calls[0][0] == "sq_jk_engine.hip", calls

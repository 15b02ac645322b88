"""Block cache (csrc/sq_blocks.h) on the host, over a memory of its own that
refuses requests beyond its size and remembers the error of a refused one,
like the HIP runtime.  Each case is a few lines of C++; a failed CHECK prints
its line."""
import os
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

"""The block cache behind rfx_malloc / rfx_free (csrc/block_cache.h), built
with the host compiler over a runtime that hands out numbered addresses."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

RUNTIME = r"""
#include <cassert>
#include <cstdio>
#include <set>
#include "block_cache.h"
using rfx::BlockCache;

struct Device {  // shared by the copies of the runtime below
  std::map<void*, uint64_t> live;
  std::set<void*> ever_released;
  uint64_t limit = ~0ull, used = 0, next = 1 << 20;
  int dev = 0, bad_releases = 0, waits = 0;
  bool can_wait = true, capturing = false;
};
struct Fake {
  Device* d;
  bool alloc(void** p, uint64_t bytes) {
    if (d->used + bytes > d->limit) return false;
    *p = reinterpret_cast<void*>(d->next);
    d->next += (bytes + 4095) / 4096 * 4096;
    d->live[*p] = bytes;
    d->used += bytes;
    return true;
  }
  void release(void* p) {
    auto it = d->live.find(p);
    if (it == d->live.end()) { ++d->bad_releases; return; }
    d->used -= it->second;
    d->live.erase(it);
  }
  int device() { return d->dev; }
  bool idle() { ++d->waits; return d->can_wait; }
  uint64_t extent(void* p) { auto it = d->live.find(p); return it == d->live.end() ? 0 : it->second; }
  bool capturing() { return d->capturing; }
};
using Cache = BlockCache<Fake>;
void* get(Cache& c, uint64_t bytes) { void* p = nullptr; return c.take(&p, bytes) ? p : nullptr; }
// rfx_free: true where it reports success.
bool put(Cache& c, Device& d, void* p) {
  switch (c.give(p)) {
    case Cache::kKept: return true;
    case Cache::kFreedBefore: return false;
    case Cache::kCallerFrees: break;
  }
  if (!d.live.count(p)) return false;  // what the runtime refuses
  Fake{&d}.release(p);
  return true;
}
"""

CASES = {
    "a kept block is handed out again, to one owner": r"""
  void* a = get(c, 1000);
  assert(put(c, d, a));
  assert(get(c, 1000) == a);
  void* b = get(c, 1000);
  assert(b && b != a && d.live.count(a) && d.live.count(b));
""",
    "a second free is refused and changes nothing": r"""
  void* a = get(c, 1000);
  assert(put(c, d, a));
  assert(!put(c, d, a) && !put(c, d, a));
  assert(d.live.count(a));           // not given to the runtime behind the cache's back
  void* b = get(c, 1000);
  void* e = get(c, 1000);
  assert(b == a && e != a);          // and listed once
  assert(put(c, d, b) && put(c, d, e));
  void* big = get(c, 65ull << 20);   // not kept: the runtime refuses the second free
  assert(put(c, d, big) && !put(c, d, big));
""",
    "a block freed past the cache and its address reused": r"""
  void* a = get(c, 1 << 20);
  Fake{&d}.release(a);               // by the runtime, not by rfx_free
  d.live[a] = 4096, d.used += 4096;  // a smaller allocation at the same address
  assert(put(c, d, a) && !d.live.count(a));
  assert(get(c, 1 << 20) != a);
""",
    "frees that cannot wait go to the runtime": r"""
  void* a = get(c, 1000); void* b = get(c, 1000); void* e = get(c, 1000);
  d.can_wait = false;
  assert(put(c, d, a) && !d.live.count(a));
  d.can_wait = true, d.capturing = true;
  assert(put(c, d, b) && !d.live.count(b));
  d.capturing = false, d.dev = 1;
  assert(put(c, d, e) && !d.live.count(e));
""",
    "no more than 512 MiB is kept": r"""
  std::vector<void*> all;
  for (int i = 0; i < 12; ++i) all.push_back(get(c, 64ull << 20));
  for (int i = 0; i < 8; ++i) assert(put(c, d, all[i]));
  d.can_wait = false;  // nor is the device waited for once there is no room
  d.waits = 0;
  for (int i = 8; i < 12; ++i) assert(put(c, d, all[i]));
  assert(d.used == 512ull << 20 && d.waits == 0);
""",
    "kept blocks make room for the library's own allocations": r"""
  d.limit = 100 << 20;
  void* a = get(c, 60 << 20);
  void* in_use = get(c, 20 << 20);
  assert(put(c, d, a) && d.live.count(a));
  void* ws = nullptr;
  assert(c.alloc(&ws, 70 << 20) && ws && !d.live.count(a) && d.live.count(in_use));
  assert(!put(c, d, a));              // given back: the runtime refuses it
  Fake{&d}.release(ws);
  void* b = nullptr;
  assert(!c.alloc(&b, 90 << 20));     // in use: no room, nothing kept to give back
  assert(put(c, d, in_use) && d.live.count(in_use));
  d.capturing = true;                 // no waiting for the device then
  assert(!c.alloc(&b, 90 << 20) && d.live.count(in_use));
  d.capturing = false;
  assert(c.alloc(&b, 90 << 20));
""",
    "and for rfx_malloc": r"""
  d.limit = 100 << 20;
  void* a = get(c, 60 << 20);
  assert(put(c, d, a));
  void* b = get(c, 63 << 20);
  assert(b && !d.live.count(a) && put(c, d, b));
  void* e = get(c, (64 << 20) - 5);   // its rounded size fits once the kept block is gone
  assert(e && d.live.at(e) >= (64 << 20) - 5);
""",
    "kept blocks outlive a context and go back with the last one": r"""
  c.context_made(); c.context_made();
  void* a = get(c, 1000);
  assert(put(c, d, a));
  c.context_gone();
  assert(d.live.count(a) && get(c, 1000) == a && put(c, d, a));
  c.context_gone();
  assert(!d.live.count(a) && d.used == 0);
""",
    "kept bytes are counted by device": r"""
  void* a = get(c, 1000); void* b = get(c, 3 << 20);
  assert(c.kept(0) == 0 && put(c, d, a) && put(c, d, b));
  d.dev = 1;
  void* e = get(c, 2000);
  assert(put(c, d, e));
  assert(c.kept(0) + c.kept(1) == d.used && c.kept(1) == d.live.at(e));
""",
}


def test_every_device_allocation_can_reclaim_kept_blocks():
    """hipMalloc has one caller: the runtime under the cache."""
    csrc = os.path.join(ROOT, "redfox_amd", "csrc")
    calls = [(f, line.strip()) for f in sorted(os.listdir(csrc)) if f.endswith((".hip", ".cpp", ".h"))
             for line in open(os.path.join(csrc, f)) if re.search(r"hipMalloc(Async|Managed)?\s*\((?!%)", line)]
    assert calls == [("context.hip", "if (hipMalloc(p, bytes) == hipSuccess) return true;")]


def run(tmp_path, body):
    src = tmp_path / "check.cpp"
    src.write_text(RUNTIME + "int main() {\n  Device d;\n  Cache c(Fake{&d});\n" + body +
                   "  assert(!d.bad_releases);\n  return 0;\n}\n")
    exe = tmp_path / "check"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Wno-unused-variable",
                    "-I" + os.path.join(ROOT, "redfox_amd", "csrc"), str(src), "-o", str(exe)],
                   check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stderr


@pytest.mark.parametrize("case", list(CASES))
def test_block_cache(tmp_path, case):
    run(tmp_path, CASES[case])

"""Idle workspaces are given back where an allocation finds no room (CPU only: the header that does it, over
a device of a few bytes)."""
import subprocess

from cpp_volume_rendering_amd import build as B

SOURCE = r"""
#include "cvr_memory.hpp"
#include <cstdio>
#include <cstdlib>
#include <map>
static std::map<void*, size_t> held;
static size_t used = 0;
static const size_t room = 100;
extern "C" {
hipError_t hipMalloc(void** p, size_t n) {
  if (used + n > room) return hipErrorOutOfMemory;
  used += n;
  *p = std::malloc(1);
  held[*p] = n;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  if (!held.count(p)) std::abort();
  used -= held[p];
  held.erase(p);
  return hipSuccess;
}
hipError_t hipGetDevice(int* d) { *d = 1; return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
static int pins = 0, frees = 0;
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  ++pins;
  if (n > 1000) return hipErrorOutOfMemory;
  *p = std::malloc(n);
  return hipSuccess;
}
hipError_t hipHostFree(void* p) { ++frees; std::free(p); return hipSuccess; }
}
using namespace cvr;
int main() {
  void *a = nullptr, *b = nullptr, *c = nullptr;
  size_t an = 40, bn = 30, cn = 20;
  auto ok = [](hipError_t e) { return e == hipSuccess; };
  if (!ok(device_alloc(&a, an)) || !ok(device_alloc(&b, bn)) || !ok(device_alloc(&c, cn))) return 1;
  park_work(&a, &an, 1);
  park_work(&b, &bn, 1);
  park_work(&c, &cn, 0);  // another device's
  claim_work(&b);         // in use again
  float* p = nullptr;
  if (!ok(device_alloc(&p, 10)) || !a || used != 100) return 2;  // there is room: nothing is given back
  float* q = nullptr;
  if (!ok(device_alloc(&q, 35)) || a || an || !b || !c || used != 95) return 3;
  float* r = q;
  if (ok(device_alloc(&r, 6)) || r || used != 95) return 4;  // nothing idle is left
  park_work(&b, &bn, 1);
  if (!ok(device_alloc(&r, 30)) || b || bn || !c || used != 95) return 5;
  claim_work(&a);  // it is gone: its owner finds none
  if (a) return 6;

  // a pinned buffer grows and is kept for less; where there is none to be had, the next call tries again
  float* h = nullptr;
  size_t hn = 0;
  float* first = pinned_buffer(&h, &hn, 400);
  if (!first || hn != 400 || pinned_buffer(&h, &hn, 100) != first || pinned_buffer(&h, &hn, 400) != first || pins != 1) return 7;
  if (!pinned_buffer(&h, &hn, 500) || hn != 500 || pins != 2 || frees != 1) return 8;
  if (pinned_buffer(&h, &hn, 2000) || h || hn || frees != 2) return 9;
  return pinned_buffer(&h, &hn, 100) && hn == 100 && frees == 2 ? 0 : 10;
}
"""


def test_idle_workspaces_are_given_back(tmp_path):
    (tmp_path / "m.hip").write_text(SOURCE)
    subprocess.run([B.HIPCC, "-O1", "-std=c++17", f"-I{B.CSRC}", "-x", "hip", "--offload-host-only",
                    f"--offload-arch={B.ARCH}", str(tmp_path / "m.hip"), "-o", str(tmp_path / "m")], check=True,
                   capture_output=True)
    assert subprocess.run([str(tmp_path / "m")]).returncode == 0


def test_every_device_buffer_comes_from_it():
    for f in sorted(B.CSRC.glob("*.h*")):
        if f.name != "cvr_memory.hpp":
            assert "hipMalloc(" not in f.read_text(), f.name

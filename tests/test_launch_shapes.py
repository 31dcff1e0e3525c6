"""How frames are dealt out to launches, computed on the host (CPU only: the host half of the kernels'
header in a small program of its own)."""
import subprocess

import pytest

from cpp_volume_rendering_amd import build as B

SOURCE = r"""
#include "cvr_queue.hpp"
#include <cstdio>
#include <cstdlib>
using namespace cvr;
int main(int n, char** v) {
  if (n == 7) {
    const BatchShape b = batch_shape(std::atoi(v[1]), std::atoi(v[2]), std::atoi(v[3]), std::atoi(v[4]), std::atoi(v[5]), 1,
                                     std::atoi(v[6]));
    std::printf("%d %d %d\n", b.tiles_x, b.tiles_y, b.nq);
    for (int q = 0; q < b.nq; ++q) std::printf("%d\n", queue_tiles(b, q));
    return 0;
  }
  const int w = std::atoi(v[1]), h = std::atoi(v[2]), rays = std::atoi(v[3]), parts = std::atoi(v[4]);
  const QueueShape q = queue_shape(w, h, rays, parts, 64);
  std::printf("%d %d\n", q.tile_log2, q.blocks);
  for_launches(q, q.blocks, 256, [&](const QueueShape& s, int blocks) { std::printf("%d %d\n", s.first, blocks); });
}
"""


@pytest.fixture(scope="module")
def shapes(tmp_path_factory):
    d = tmp_path_factory.mktemp("shapes")
    (d / "shapes.hip").write_text(SOURCE)
    subprocess.run([B.HIPCC, "-O1", "-std=c++17", f"-I{B.INCLUDE}", f"-I{B.CSRC}", "-x", "hip", "--offload-host-only",
                    f"--offload-arch={B.ARCH}", str(d / "shapes.hip"), "-o", str(d / "shapes")], check=True,
                   capture_output=True)

    def run(*args):
        out = subprocess.run([str(d / "shapes"), *map(str, args)], check=True, capture_output=True, text=True).stdout
        return [tuple(map(int, line.split())) for line in out.splitlines()]

    return run


# ground truth (4 rays, shared), cone tracer and DOS (4, own), EBS (16, own), marches (32, shared)
@pytest.mark.parametrize("rays,parts", [(4, 4), (4, 1), (16, 1), (32, 4)])
@pytest.mark.parametrize("w,h", [(1, 1), (333, 64), (1024, 1024), (8191, 8190), (8192, 8192), (16384, 16384), (1 << 28, 1),
                                 (1, 1 << 28), (65537, 4095)])
def test_launches_cover_a_frame_within_the_limit_of_lanes(shapes, w, h, rays, parts):
    (log2, blocks), *launches = shapes(w, h, rays, parts)
    m, per_wg = 1 << log2, rays * 4 // parts
    pixels = -(-w // m) * -(-h // m) * m * m
    assert blocks == -(-pixels // per_wg) and m * m >= rays
    at = 0
    for first, n in launches:
        assert first == at and 0 < n and n * 256 < 1 << 32
        at += n
    assert at == blocks


# images a call may have (2^26 pixels, 2^32 in all), flat ones above all: a tile is 4 x 16 span pixels
@pytest.mark.parametrize("queues", [1, 8])
@pytest.mark.parametrize("w,h,tw_log2,span,jobs", [(1, 1, 2, 1, 1), (333, 64, 3, 1, 5), (8192, 8192, 2, 1, 64),
                                                   (1 << 26, 1, 2, 8, 64), (1 << 26, 1, 2, 1, 64), (1, 1 << 26, 5, 1, 64),
                                                   (1 << 26, 1, 2, 1, 32), (1 << 22, 16, 2, 1, 64)])
def test_batch_items_are_counted_in_32_bits(shapes, w, h, tw_log2, span, queues, jobs):
    (tx, ty, nq), *tiles = shapes(w, h, tw_log2, span, queues, jobs)
    assert tx == -(-w // (1 << tw_log2))
    assert ty == -(-h // ((64 >> tw_log2) * span))
    assert sum(t for t, in tiles) == tx * ty and len(tiles) == nq
    items = [t * 4 * jobs for t, in tiles]
    assert max(items) < (1 << 31) - (1 << 20)
    assert nq == (queues if sum(items) < (1 << 31) - (1 << 20) else 8)


EXITS = r"""
#include "cvr_cone.hpp"
#include <cstdio>
using namespace cvr;
int main() {
  const float G = 32.f, inf = INFINITY;
  for (float zero : {0.f, -0.f})
    for (float q : {0.f, 5.f, 32.f})
      if (axis_exit(zero, q, G) != inf) return 1;
  if (axis_exit(0.5f, 30.f, G) != 4.f || axis_exit(-0.5f, 3.f, G) != 6.f || axis_exit(1.f, 32.f, G) != 0.f) return 2;
  const float box[3] = {32.f, 16.f, 8.f};
  for (float e : {0.f, 1e-4f, -1e-4f})
    if (!in_box(box, f3{e, 4.f, 8.f + e}) || !in_box(box, f3{32.f + e, e, 8.f})) return 3;
  for (float q : {-0.01f, -inf, inf, NAN})
    if (in_box(box, f3{q, 4.f, 4.f}) || in_box(box, f3{4.f, q, 4.f}) || in_box(box, f3{4.f, 4.f, q})) return 3;
  if (in_box(box, f3{32.01f, 4.f, 4.f}) || in_box(box, f3{4.f, 16.01f, 4.f}) || in_box(box, f3{4.f, 4.f, 8.01f})) return 3;
  ConeSched S{};
  S.n = 64;
  S.log2_t0 = 0.f;
  for (float r : {8.f, 0.25f, inf}) {
    S.inv_log2_q = r;
    for (float t : {-inf, inf, NAN, -1000.f, 1e30f, 0.f, 3.7f})
      if (steps_up_to(t, S) < 0 || steps_up_to(t, S) > 64) return 4;
    if (steps_up_to(inf, S) != 64 || steps_up_to(-inf, S) != 0 || steps_up_to(NAN, S) != 0) return 5;
  }
  S.inv_log2_q = 8.f;
  return steps_up_to(2.f, S) == 17 && steps_up_to(1.99f, S) == 16 ? 0 : 6;
}
"""


def test_cones_along_an_axis_leave_by_the_others(tmp_path):
    (tmp_path / "e.hip").write_text(EXITS)
    subprocess.run([B.HIPCC, "-O1", "-std=c++17", f"-I{B.INCLUDE}", f"-I{B.CSRC}", "-x", "hip", "--offload-host-only",
                    f"--offload-arch={B.ARCH}", str(tmp_path / "e.hip"), "-o", str(tmp_path / "e")], check=True,
                   capture_output=True)
    assert subprocess.run([str(tmp_path / "e")]).returncode == 0

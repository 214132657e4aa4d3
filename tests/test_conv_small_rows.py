"""Where the pointwise loads of the small-launch kernel go, for every short K.

The kernel reads through a buffer descriptor and is told an address in two parts.  Only the lane's part is
sure to be compared with the buffer's end, so a load whose lane offset is inside the buffer has to
be inside it with its scalar offset as well, padding rows of the last K tiles included.  Checked on
the host over the header that the kernel uses.
"""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
KERNELS = os.path.join(ROOT, "mini-caffe_amd", "csrc", "kernels")

PROGRAM = r"""
#include "small_rows.h"
#include <cstdio>
#include <initializer_list>
using namespace mchip;

// Loads of all rows of a K tile's two half-waves for the blob's first and last pixels; returns how many
// leave the blob although the lane's offset does not, and how many real rows are not where they belong.
template <bool TAIL>
int faults(int K, int planes_in_blob, int first_plane, unsigned plane) {
  const unsigned bytes = planes_in_blob * plane;
  int bad = 0;
  for (int kt = 0; kt < (K + 31) / 32 * 2; ++kt)   // (the packed filter's rows are a multiple of 32)
    for (int half = 0; half < 2; ++half)
      for (int e = 0; e < 8; ++e)
        for (unsigned pixel : {0u, plane - 4u, 0x80000000u}) {
          const bool none = pixel == 0x80000000u;  // a column past the last pixel
          const unsigned own = (none ? pixel : pixel + first_plane * plane) + 8 * half * plane;
          const unsigned lane = small_lane_offset<TAIL>(own, kt, e, plane);
          const unsigned scalar = small_scalar_offset<TAIL>(kt, e, plane);
          const int row = 16 * kt + 8 * half + e;
          if (lane < bytes && lane + scalar >= bytes) ++bad;
          if (none ? lane < bytes : row < K && lane + scalar != pixel + (first_plane + row) * plane) ++bad;
        }
  return bad;
}

int main() {
  for (int K = 9; K <= 300; ++K)
    for (unsigned plane : {4u, 196u, 40000u})
      for (int images = 1; images <= 3; ++images) {
        const int planes = K * images, last = K * (images - 1);   // (or groups)
        const bool tail = small_needs_tail(K, (K + 31) / 32 * 32);
        const int now = tail ? faults<true>(K, planes, last, plane) : faults<false>(K, planes, last, plane);
        if (now) return std::printf("K %d plane %u images %d: %d\n", K, plane, images, now), 1;
        // the scalar offset alone does leave the blob where there is padding
        if ((faults<false>(K, planes, last, plane) > 0) != tail) return std::printf("K %d: no padding?\n", K), 2;
      }
  return 0;
}
"""


def test_no_load_goes_past_the_blob(tmp_path):
    source, exe = tmp_path / "rows.cc", str(tmp_path / "rows")
    source.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I" + KERNELS, str(source), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout


def test_the_kernel_uses_these_offsets():
    text = open(os.path.join(KERNELS, "igemm_small.h")).read()
    assert "small_lane_offset<TAIL>(voff" in text and "small_scalar_offset<TAIL>(kt_, e, x_cbytes)" in text
    assert "small_needs_tail(s.K, s.Kpad)" in open(os.path.join(KERNELS, "conv_igemm.hip")).read()

// Host-only driver of gx_detector_work_size and gx_detector_accumulate_ws, built with host-side
// ASan and UBSan by tests/test_host_detector_work.py: both refuse what gx_detector_accumulate
// refuses, the size follows the size rule without overflow at the descriptor's limits, and a missing
// or misaligned work buffer is refused before any device work.  The device pointers below are never
// dereferenced.  Prints "checks passed: <n>" and exits 0, or names the check that failed and exits 1.

#include <stdint.h>
#include <stdio.h>
#include <string.h>

#include "giwaxsim_amd.h"

static int n_checks = 0;
#define CHECK(cond)                                                                       \
  do {                                                                                    \
    ++n_checks;                                                                           \
    if (!(cond)) {                                                                        \
      fprintf(stderr, "line %d: %s (message '%s')\n", __LINE__, #cond, gx_last_error());  \
      return 1;                                                                           \
    }                                                                                     \
  } while (0)

static gx_detector valid(int64_t n_pix, int64_t n_orient, int64_t side, int64_t f64) {
  gx_detector d;
  memset(&d, 0, sizeof d);
  d.n_pix = n_pix;
  d.n_init = 1;
  d.n_orient = n_orient;
  d.cy = d.cx = d.cz = side;
  d.iq_f64 = f64;
  d.dq = 0.01;
  double *p = reinterpret_cast<double *>(static_cast<uintptr_t>(4096));
  d.h_axis = d.v_axis = d.init_R = d.orient_R = d.orient_w = p;
  d.iq = p;
  d.det = p;
  return d;
}

static int64_t size_of(const gx_detector &d) {
  int64_t n = -1;
  return gx_detector_work_size(&d, &n) == GX_OK ? n : -1;
}
// the work buffer's documented bound in doubles
static bool maps(const gx_detector &d) {
  const int64_t n = size_of(d);
  return n > 0 && n * 8 <= 64 * (d.n_orient + 9);
}

int main() {
  int64_t n = 7;
  double *p = reinterpret_cast<double *>(static_cast<uintptr_t>(4096));
  CHECK(gx_detector_work_size(nullptr, &n) == GX_ERR_ARG && n == 7);
  CHECK(gx_detector_accumulate_ws(nullptr, p, nullptr) == GX_ERR_ARG);
  gx_detector d = valid(512, 361, 131, 1);
  CHECK(gx_detector_work_size(&d, nullptr) == GX_ERR_ARG);
  CHECK(maps(d));
  CHECK(gx_detector_accumulate_ws(&d, nullptr, nullptr) == GX_ERR_ARG);
  CHECK(strstr(gx_last_error(), "work buffer") != nullptr);
  CHECK(gx_detector_accumulate_ws(&d, reinterpret_cast<double *>(static_cast<uintptr_t>(4096 + 32)), nullptr) ==
        GX_ERR_ARG);
  // what gx_detector_accumulate refuses
  const gx_detector zero = {};
  CHECK(gx_detector_work_size(&zero, &n) == GX_ERR_ARG && gx_detector_accumulate_ws(&zero, p, nullptr) == GX_ERR_ARG);
  gx_detector bad = d;
  bad.n_pix = 65537;
  CHECK(size_of(bad) == -1 && gx_detector_accumulate_ws(&bad, p, nullptr) == GX_ERR_ARG);
  bad = d;
  bad.n_init = 4;
  CHECK(size_of(bad) == -1);
  bad = d;
  bad.orient_w = nullptr;
  CHECK(size_of(bad) == -1 && gx_detector_accumulate_ws(&bad, p, nullptr) == GX_ERR_ARG);
  // the size rule
  CHECK(size_of(valid(34, 39, 61, 1)) == 0 && maps(valid(34, 40, 61, 1)));
  CHECK(maps(valid(34, 63, 61, 1)) && size_of(valid(34, 64, 61, 1)) == 0);
  CHECK(size_of(valid(34, 159, 61, 1)) == 0 && maps(valid(34, 160, 61, 1)));
  CHECK(size_of(valid(362, 64, 61, 0)) == 0 && maps(valid(364, 64, 61, 0)));
  CHECK(maps(valid(1026, 33, 61, 1)) && size_of(valid(1024, 31, 61, 1)) == 0);
  CHECK(size_of(valid(289, 16000, 61, 1)) == 0 && maps(valid(291, 16000, 61, 1)));
  CHECK(size_of(valid(291, 396, 61, 1)) == 0 && maps(valid(291, 397, 61, 1)));
  CHECK(size_of(valid(512, 0, 61, 1)) == 0);
  // limits of the maps: grid edge, grid bytes, orientations, pixels
  gx_detector e = valid(512, 361, 16, 0);
  e.cx = 4095;
  CHECK(maps(e));
  e.cx = 4096;
  CHECK(size_of(e) == 0);
  CHECK(maps(valid(512, 361, 812, 1)) && size_of(valid(512, 361, 813, 1)) == 0);
  CHECK(maps(valid(512, 361, 1023, 0)) && size_of(valid(512, 361, 1625, 0)) == 0);
  CHECK(maps(valid(65536, 1 << 24, 61, 1)) && size_of(valid(65536, (1 << 24) + 1, 61, 1)) <= 0);
  printf("checks passed: %d\n", n_checks);
  return 0;
}

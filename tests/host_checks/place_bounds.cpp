// Host check of near_depth (csrc/vh_math.h): a block's corners bound its voxels' pixels. For random
// cameras, with one lattice point of the block at or near the camera centre, fields of view from a few
// degrees to nearly 180, images from 1 x 1 to 16384 x 16384 and the corners' reciprocals off by up to
// 1 ulp, the block's rectangle is formed as the kernel forms it (block_place); wherever that puts it inside
// the image, every voxel's z has to lie in the range of the kernel's reciprocal and its pixel in the rectangle.
// Prints "blocks inside, of them with a corner below a millimetre, voxels outside"; with the argument "without" the
// bound on the corners' depth is left out, with "columns" the corners are the ends of the voxels' columns, summed as voxels
// are, as for a single frame (block_place_one).
#include <cinttypes>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <random>

#include "vh_math.h"

using namespace vh;

static int32_t bits(float x) {
  int32_t b;
  std::memcpy(&b, &x, 4);
  return b;
}

int main(int argc, char** argv) {
  const bool without = argc > 1 && !std::strcmp(argv[1], "without"), columns = argc > 1 && !std::strcmp(argv[1], "columns");
  std::mt19937_64 rng(7);
  std::uniform_real_distribution<double> uni(0.0, 1.0);
  int64_t inside = 0, near = 0, out = 0;
  for (int it = 0; it < 2000000; ++it) {
    const int W = (int)std::exp2(14 * uni(rng)), H = (int)std::exp2(14 * uni(rng));
    const float f = (float)(W * std::exp2(6 * uni(rng) - 5));
    const Intr K{f, (float)(f * (0.7 + 0.6 * uni(rng))), (float)(W * uni(rng)), (float)(H * uni(rng))};
    const float vox = (float)std::exp2(-10 + 8 * uni(rng));
    const int span = 1 << (int)(12 * uni(rng));
    const int b[3] = {(int)(rng() % (2 * span)) - span, (int)(rng() % (2 * span)) - span, (int)(rng() % (2 * span)) - span};
    // the camera by a lattice point: half of the time one of the block's corners, looking into the block
    const bool corner = it & 1;
    int at[3];
    double R[3][3], fwd[3], right[3], down[3];
    for (int r = 0; r < 3; ++r) {
      at[r] = corner ? 7 * (int)(rng() % 2) : (int)(rng() % 8);
      fwd[r] = corner ? (at[r] ? -1.0 : 1.0) * (it % 8 == 1 ? 1.0 : 0.2 + uni(rng)) : uni(rng) - 0.5;
      right[r] = uni(rng) - 0.5;
    }
    if (it % 16 == 0) {  // exact axes
      fwd[0] = fwd[1] = right[1] = right[2] = 0.0;
      fwd[2] = right[0] = 1.0;
    }
    const auto unit = [](double* x) {
      const double n = std::sqrt(x[0] * x[0] + x[1] * x[1] + x[2] * x[2]);
      for (int r = 0; r < 3; ++r) x[r] /= n;
    };
    const auto cross = [](const double* x, const double* y, double* z) {
      for (int r = 0; r < 3; ++r) z[r] = x[(r + 1) % 3] * y[(r + 2) % 3] - x[(r + 2) % 3] * y[(r + 1) % 3];
    };
    unit(fwd);
    cross(fwd, right, down);
    unit(down);
    cross(down, fwd, right);
    float T[12];
    for (int r = 0; r < 3; ++r) {
      R[r][0] = right[r], R[r][1] = down[r], R[r][2] = fwd[r];
      const double away = (uni(rng) - (corner ? 0.6 : 0.5)) * fwd[r] * std::exp2(-30 * uni(rng));
      for (int c = 0; c < 3; ++c) T[4 * r + c] = (float)R[r][c];
      T[4 * r + 3] = (float)((double)(b[r] * kB + at[r]) * vox + away);
    }
    BlockFrame h;
    block_frame_h(T, vox, K, h);
    float cb[3], hb[3];
    block_origin_cam(T, vox, b[0], b[1], b[2], cb);
    to_pixel_h(K, cb, hb);
    const float need = without ? 0.0f : near_depth(near_steps(h, near_image(W, H)), hb, near_image(W, H));
    bool zin = true;
    int32_t lu = INT32_MAX, hu = INT32_MIN, lv = INT32_MAX, hv = INT32_MIN;
    float zmin = INFINITY;
    for (int c = 0; c < 8; ++c) {
      const float c0 = (c & 1) ? 7.0f : 0.0f, c1 = (c & 2) ? 7.0f : 0.0f, c2 = (c & 4) ? 7.0f : 0.0f;
      float off[3];
      for (int r = 0; r < 3; ++r) off[r] = std::fma(c0, h.ax[r], std::fma(c1, h.ay[r], c2 * h.az[r]));
      float P[3];
      for (int r = 0; r < 3; ++r) {
        const float col = hb[r] + std::fma(c1, h.ay[r], c2 * h.az[r]);
        P[r] = !columns ? hb[r] + off[r] : c0 > 0.0f ? std::fma(c0, h.ax[r], col) : col;
      }
      const float z = P[2];
      float iz = 1.0f / z;
      const int ulp = (int)(rng() % 3);
      if (ulp) iz = std::nextafter(iz, ulp == 1 ? INFINITY : -INFINITY);
      const float u = P[0] * iz, v = P[1] * iz;
      zin = zin && z >= need && z >= 0x1p-60f && z <= 0x1p60f;
      zmin = std::fmin(zmin, z);
      lu = std::min(lu, bits((u - 0.5f) + kPixMagic));
      hu = std::max(hu, bits((u + 0.5f) + kPixMagic));
      lv = std::min(lv, bits((v - 0.5f) + kPixMagic));
      hv = std::max(hv, bits((v + 0.5f) + kPixMagic));
    }
    const int32_t mb = (int32_t)kPixMagicBits;
    if (!(zin && lu >= mb && hu <= mb + W - 1 && lv >= mb && hv <= mb + H - 1)) continue;
    ++inside;
    near += zmin < 1e-3f;
    for (int v = 0; v < kB3; ++v) {
      const float k = (float)(v >> 6), j = (float)((v >> 3) & 7), i = (float)(v & 7);
      float P[3];
      for (int r = 0; r < 3; ++r) {
        const float col = hb[r] + std::fma(j, h.ay[r], i * h.az[r]);
        P[r] = v >> 6 ? std::fma(k, h.ax[r], col) : col;
      }
      const float iz = 1.0f / P[2];
      const int32_t ub = bits(std::fma(P[0], iz, kPixMagic)), vb = bits(std::fma(P[1], iz, kPixMagic));
      out += !(P[2] >= kMinZ && P[2] <= kMaxZ && ub >= lu && ub <= hu && vb >= lv && vb <= hv);
    }
  }
  std::printf("%" PRId64 " %" PRId64 " %" PRId64 "\n", inside, near, out);
  return 0;
}

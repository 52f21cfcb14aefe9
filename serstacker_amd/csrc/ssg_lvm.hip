// ssg_lvm.hip -- the local-variance sharpness map on gfx950
// (compute_local_variance_map, core/proc/sharpness_measure/
// c_local_variance_sharpness_measure.cc:193-249): morphological gradient of the
// (pyrDown'ed) gray frame, its L1 norm and fourth-power sum, the cubed map plus
// 0.05 Q, and cv::resize INTER_LINEAR back to the frame size.
#include <type_traits>

#include "ssg_engine.hpp"

namespace ssg {

namespace {

__device__ __forceinline__ size_t gid() { return (size_t)blockIdx.x * 256 + threadIdx.x; }

// cv::COLOR_BGR2GRAY on float: b*0.114 + g*0.587 + r*0.299
__global__ void __launch_bounds__(256) k_bgr2gray(const float* src, int pitch, int w, int h, float* g) {
  const size_t i = gid();
  if (i >= (size_t)w * h) return;
  const int y = (int)(i / w), x = (int)(i - (size_t)y * w);
  const float* p = src + (size_t)y * pitch + 3 * x;
  g[i] = (p[0] * 0.114f + p[1] * 0.587f) + p[2] * 0.299f;
}

// dilate - erode with a (2r+1)^2 square, BORDER_REPLICATE
__global__ void __launch_bounds__(256) k_morph_grad(const float* m, int w, int h, int r, float* g) {
  const size_t i = gid();
  if (i >= (size_t)w * h) return;
  const int y = (int)(i / w), x = (int)(i - (size_t)y * w);
  float mx = -3.4e38f, mn = 3.4e38f;
  for (int dy = -r; dy <= r; ++dy) {
    const float* row = m + (size_t)min(max(y + dy, 0), h - 1) * w;
    for (int dx = -r; dx <= r; ++dx) {
      const float v = row[min(max(x + dx, 0), w - 1)];
      mx = fmaxf(mx, v);
      mn = fminf(mn, v);
    }
  }
  g[i] = mx - mn;
}

// per-block partial sums of |G| and G^4 in double
__global__ void __launch_bounds__(256) k_lvm_sums(const float* g, size_t n, double* partial) {
  __shared__ double s1[256], s4[256];
  double a = 0, b = 0;
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) {
    const double v = g[i];
    a += fabs(v);
    const double v2 = v * v;
    b += v2 * v2;
  }
  s1[threadIdx.x] = a;
  s4[threadIdx.x] = b;
  __syncthreads();
  for (int k = 128; k > 0; k >>= 1) {
    if (threadIdx.x < k) {
      s1[threadIdx.x] += s1[threadIdx.x + k];
      s4[threadIdx.x] += s4[threadIdx.x + k];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    partial[2 * blockIdx.x] = s1[0];
    partial[2 * blockIdx.x + 1] = s4[0];
  }
}

// map = G^3 * mapScale + add
__global__ void __launch_bounds__(256) k_lvm_map(const float* g, size_t n, float map_scale, float add, float* m) {
  const size_t i = gid();
  if (i >= n) return;
  const float v = g[i];
  m[i] = ((v * v) * v) * map_scale + add;
}

__global__ void __launch_bounds__(256) k_resize_linear(const float* src, int sw, int sh, float* dst, int dst_pitch,
                                                       int dw, int dh, double scale_x, double scale_y) {
  const size_t i = gid();
  if (i >= (size_t)dw * dh) return;
  const int y = (int)(i / dw), x = (int)(i - (size_t)y * dw);
  int x0, x1, y0, y1;
  float a0, a1, b0, b1;
  lin_tap(x, scale_x, sw, x0, x1, a0, a1);
  lin_tap_v(y, scale_y, sh, y0, y1, b0, b1);
  const float* r0 = src + (size_t)y0 * sw;
  const float* r1 = src + (size_t)y1 * sw;
  const float h0 = r0[x0] * a0 + r0[x1] * a1, h1 = r1[x0] * a0 + r1[x1] * a1;
  dst[(size_t)y * dst_pitch + x] = h0 * b0 + h1 * b1;
}

}  // namespace

namespace {
// an 8/16-bit image as dense f32 (exact)
__global__ void __launch_bounds__(256) k_int_to_f32(const uint8_t* src, int pitch, int w, int h, int u16, float* d) {
  const size_t i = gid();
  if (i >= (size_t)w * h) return;
  const int x = (int)(i % w), y = (int)(i / w);
  const uint8_t* row = src + (size_t)y * pitch;
  d[i] = u16 ? (float)((const uint16_t*)row)[x] : (float)row[x];
}
// cv::pyrDown's integer rounding on 8/16-bit data, (sum + 128) >> 8, applied to the float
// pyramid level (whose values are exact multiples of 1/256 for integer inputs)
__global__ void __launch_bounds__(256) k_round_half_up(float* v, size_t n) {
  const size_t i = gid();
  if (i < n) v[i] = floorf(v[i] + 0.5f);
}
}  // namespace

hipError_t launch_int_to_f32(const void* src, int pitch, int w, int h, bool u16, float* dst, hipStream_t s) {
  hipLaunchKernelGGL(k_int_to_f32, dim3((unsigned)(((size_t)w * h + 255) / 256)), dim3(256), 0, s,
                     (const uint8_t*)src, pitch, w, h, u16 ? 1 : 0, dst);
  return hipGetLastError();
}
hipError_t launch_round_half_up(float* v, size_t n, hipStream_t s) {
  hipLaunchKernelGGL(k_round_half_up, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, v, n);
  return hipGetLastError();
}

hipError_t launch_bgr2gray(const float* src, int pitch, int w, int h, float* g, hipStream_t s) {
  hipLaunchKernelGGL(k_bgr2gray, dim3((unsigned)(((size_t)w * h + 255) / 256)), dim3(256), 0, s, src, pitch, w, h, g);
  return hipGetLastError();
}
hipError_t launch_morph_grad(const float* m, int w, int h, int r, float* g, hipStream_t s) {
  hipLaunchKernelGGL(k_morph_grad, dim3((unsigned)(((size_t)w * h + 255) / 256)), dim3(256), 0, s, m, w, h, r, g);
  return hipGetLastError();
}
int lvm_sum_blocks(size_t n) { return (int)std::min<size_t>(1024, (n + 255) / 256); }
hipError_t launch_lvm_sums(const float* g, size_t n, double* partial, hipStream_t s) {
  hipLaunchKernelGGL(k_lvm_sums, dim3(lvm_sum_blocks(n)), dim3(256), 0, s, g, n, partial);
  return hipGetLastError();
}
hipError_t launch_lvm_map(const float* g, size_t n, float map_scale, float add, float* m, hipStream_t s) {
  hipLaunchKernelGGL(k_lvm_map, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, g, n, map_scale, add, m);
  return hipGetLastError();
}
hipError_t launch_resize_linear(const float* src, int sw, int sh, float* dst, int dst_pitch, int dw, int dh,
                                hipStream_t s) {
  const double sx = 1.0 / ((double)dw / sw), sy = 1.0 / ((double)dh / sh);
  hipLaunchKernelGGL(k_resize_linear, dim3((unsigned)(((size_t)dw * dh + 255) / 256)), dim3(256), 0, s, src, sw, sh,
                     dst, dst_pitch, dw, dh, sx, sy);
  return hipGetLastError();
}

// ---- the quality of a batch of 8/16-bit frames ----------------------------------------------------
// One tile of a level per block, all of the chain in LDS: average_bayer_planes of the raw cells, cv::pyrDown
// in whole numbers ((sum + 128) >> 8, REFLECT_101), then either the level stored for a further pyrDown
// (R = 0) or its morphological gradient and the tile's sums of G and G^4 in double.  Every value is the whole
// number that the float kernels above hold.
// What bounds it: the raw frames' one read.  24 frames of 4096x3000: 0.14 ms (4.3 TB/s); 1.30 ms in six launches per
// frame, each through memory.
namespace {
// The tile of the level is a wave's width with the gradient's halo R on each side (R = 0: STORE), 16 rows high
// without it; rows of the level and of its source are then whole wave steps
constexpr int QT_NW = WAVE, QT_H = 16, QT_R = 3;  // QT_R: the largest gradient radius
constexpr int QT_AW = 2 * QT_NW + 4;              // source pixels of a row, an even number

template <bool U16, bool BAYER, int R>
__global__ void __launch_bounds__(256) k_quality(const void* const* frames, long long fstride, int pitch, int wide, int aw,
                                                 int ah, int dw, int dh, uint16_t* out, double* part) {
  constexpr int TW = QT_NW - 2 * R, NH = QT_H + 2 * R, AH = 2 * NH + 3;
  __shared__ __align__(8) uint16_t av[AH][QT_AW];
  __shared__ int hs[AH][QT_NW];
  __shared__ uint16_t dn[NH][QT_NW];
  __shared__ double red[4][2];
  const int tid = threadIdx.x, lane = tid & (WAVE - 1), wv = tid / WAVE, f = blockIdx.z;
  // the frames by their pointers, or planes of a stride from the first
  const uint8_t* src = fstride ? (const uint8_t*)frames + f * fstride : (const uint8_t*)frames[f];
  const int x0 = blockIdx.x * TW, y0 = blockIdx.y * QT_H;
  const int ax0 = 2 * (x0 - R) - 2, ay0 = 2 * (y0 - R) - 2;
  auto at = [&](const uint8_t* row, int x) { return U16 ? (int)((const uint16_t*)row)[x] : (int)row[x]; };
  auto pixel = [&](int x, int y) {  // the source pixel (x, y), both inside
    if constexpr (BAYER) {
      const uint8_t* row = src + (size_t)(2 * y) * pitch;
      return (at(row, 2 * x) + at(row, 2 * x + 1) + at(row + pitch, 2 * x) + at(row + pitch, 2 * x + 1) + 2) >> 2;
    } else {
      return at(src + (size_t)y * pitch, x);
    }
  };
  // ---- the tile's source pixels, two per step (ax0 is even)
  constexpr int uw = QT_AW / 2, steps = uw * AH;
  using Raw = std::conditional_t<BAYER && U16, uint2, std::conditional_t<BAYER || U16, uint32_t, uint16_t>>;
  auto unpack = [](Raw u, Raw v) -> uint32_t {  // the two pixels of a load (v: the cells' second row)
    uint32_t a, b;
    if constexpr (BAYER && U16) {
      a = ((u.x & 0xffffu) + (u.x >> 16) + (v.x & 0xffffu) + (v.x >> 16) + 2) >> 2;
      b = ((u.y & 0xffffu) + (u.y >> 16) + (v.y & 0xffffu) + (v.y >> 16) + 2) >> 2;
    } else if constexpr (BAYER) {
      a = ((u & 0xffu) + (u >> 8 & 0xffu) + (v & 0xffu) + (v >> 8 & 0xffu) + 2) >> 2;
      b = ((u >> 16 & 0xffu) + (u >> 24) + (v >> 16 & 0xffu) + (v >> 24) + 2) >> 2;
    } else if constexpr (U16) {
      a = u & 0xffffu;
      b = u >> 16;
    } else {
      a = u & 0xffu;
      b = u >> 8;
    }
    return a | b << 16;
  };
  auto row_of = [&](int x, int y) {
    return src + (size_t)(BAYER ? 2 * y : y) * pitch + (size_t)x * (U16 ? 2 : 1) * (BAYER ? 2 : 1);
  };
  if (wide && ax0 >= 0 && ay0 >= 0 && ax0 + QT_AW <= aw && ay0 + AH <= ah) {
    // all inside: the loads of four steps are in flight before the first is used
    for (int i0 = tid; i0 < steps; i0 += 4 * 256) {
      Raw u[4], v[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int i = min(i0 + q * 256, steps - 1), ly = i / uw;
        const uint8_t* row = row_of(ax0 + 2 * (i - ly * uw), ay0 + ly);
        u[q] = *(const Raw*)row;
        if (BAYER) v[q] = *(const Raw*)(row + pitch);
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int i = min(i0 + q * 256, steps - 1), ly = i / uw;
        *(uint32_t*)&av[ly][2 * (i - ly * uw)] = unpack(u[q], BAYER ? v[q] : u[q]);
      }
    }
  } else {
    for (int i = tid; i < steps; i += 256) {
      const int ly = i / uw, lx = 2 * (i - ly * uw);
      const int x = ax0 + lx, y = border_interp(ay0 + ly, ah, BORDER_REFLECT101);
      uint32_t ab;
      if (wide && x >= 0 && x + 1 < aw) {
        const uint8_t* row = row_of(x, y);
        const Raw u = *(const Raw*)row;
        ab = unpack(u, BAYER ? *(const Raw*)(row + pitch) : u);
      } else {
        ab = (uint32_t)pixel(border_interp(x, aw, BORDER_REFLECT101), y) |
             (uint32_t)pixel(border_interp(x + 1, aw, BORDER_REFLECT101), y) << 16;
      }
      *(uint32_t*)&av[ly][lx] = ab;
    }
  }
  __syncthreads();
  // ---- pyrDown: rows, then columns
  for (int ly = wv; ly < AH; ly += 4) {
    const uint32_t p = *(const uint32_t*)&av[ly][2 * lane], q = *(const uint32_t*)&av[ly][2 * lane + 2];
    hs[ly][lane] =
        (int)(p & 0xffffu) + (int)av[ly][2 * lane + 4] + 4 * ((int)(p >> 16) + (int)(q >> 16)) + 6 * (int)(q & 0xffffu);
  }
  __syncthreads();
  for (int ly = wv; ly < NH; ly += 4) {
    const int v = (hs[2 * ly][lane] + hs[2 * ly + 4][lane] + 4 * (hs[2 * ly + 1][lane] + hs[2 * ly + 3][lane]) +
                   6 * hs[2 * ly + 2][lane] + 128) >> 8;
    if constexpr (R == 0) {
      if (x0 + lane < dw && y0 + ly < dh) out[((size_t)f * dh + y0 + ly) * dw + x0 + lane] = (uint16_t)v;
    } else {
      dn[ly][lane] = (uint16_t)v;
    }
  }
  if constexpr (R > 0) {
    __syncthreads();
    // ---- dilate - erode (BORDER_REPLICATE), G and G^4: four rows per thread, each row's extremes formed once
    constexpr int RPT = QT_H / 4;
    double s1 = 0, s4 = 0;
    const int x = x0 + lane, yb = y0 + wv * RPT;
    if (lane < TW && x < dw) {
      int col[2 * R + 1], mx[RPT + 2 * R], mn[RPT + 2 * R];
#pragma unroll
      for (int i = 0; i <= 2 * R; ++i) col[i] = min(max(x + i - R, 0), dw - 1) - (x0 - R);
#pragma unroll
      for (int i = 0; i < RPT + 2 * R; ++i) {
        // rows past the level belong to no pixel's window that is used; they stay in the tile
        const uint16_t* row = dn[min(min(max(yb + i - R, 0), dh - 1) - (y0 - R), NH - 1)];
        mx[i] = mn[i] = row[col[0]];
#pragma unroll
        for (int j = 1; j <= 2 * R; ++j) {
          const int v = row[col[j]];
          mx[i] = max(mx[i], v);
          mn[i] = min(mn[i], v);
        }
      }
#pragma unroll
      for (int k = 0; k < RPT; ++k) {
        if (yb + k >= dh) continue;
        int a = mx[k], b = mn[k];
#pragma unroll
        for (int i = 1; i <= 2 * R; ++i) {
          a = max(a, mx[k + i]);
          b = min(b, mn[k + i]);
        }
        const double g = (double)(a - b), g2 = g * g;
        s1 += g;
        s4 += g2 * g2;
      }
    }
    s1 = wave_sum(s1);
    s4 = wave_sum(s4);
    if (lane == 0) {
      red[wv][0] = s1;
      red[wv][1] = s4;
    }
    __syncthreads();
    if (tid < 2)
      part[(((size_t)f * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x) * 2 + tid] =
          ((red[0][tid] + red[1][tid]) + red[2][tid]) + red[3][tid];
  }
}

// the tiles' sums of a frame, in a fixed order
__global__ void __launch_bounds__(256) k_quality_fold(const double* part, int tiles, double* out) {
  __shared__ double red[4][2];
  const double* p = part + (size_t)blockIdx.x * tiles * 2;
  double s1 = 0, s4 = 0;
  for (int i = threadIdx.x; i < tiles; i += 256) {
    s1 += p[2 * i];
    s4 += p[2 * i + 1];
  }
  s1 = wave_sum(s1);
  s4 = wave_sum(s4);
  if ((threadIdx.x & (WAVE - 1)) == 0) {
    red[threadIdx.x / WAVE][0] = s1;
    red[threadIdx.x / WAVE][1] = s4;
  }
  __syncthreads();
  if (threadIdx.x < 2)
    out[2 * blockIdx.x + threadIdx.x] =
        ((red[0][threadIdx.x] + red[1][threadIdx.x]) + red[2][threadIdx.x]) + red[3][threadIdx.x];
}
}  // namespace

int quality_max_radius() { return QT_R; }
int quality_tiles(int dw, int dh, int r) {
  const int tw = QT_NW - 2 * r;
  return ((dw + tw - 1) / tw) * ((dh + QT_H - 1) / QT_H);
}

hipError_t launch_quality(const void* const* frames, long long fstride, bool u16, bool bayer, int pitch, bool wide, int aw,
                          int ah, int r, int n, uint16_t* out, double* part, double* sums, hipStream_t s) {
  const int dw = (aw + 1) / 2, dh = (ah + 1) / 2, rr = out ? 0 : r, tw = QT_NW - 2 * rr;
  const dim3 grid((dw + tw - 1) / tw, (dh + QT_H - 1) / QT_H, n);
#define SSG_Q(U, B, RR)                                                                                                \
  hipLaunchKernelGGL((k_quality<U, B, RR>), grid, dim3(256), 0, s, frames, fstride, pitch, wide ? 1 : 0, aw, ah, dw, dh, \
                     out, part)
#define SSG_QR(RR)                        \
  do {                                    \
    if (u16 && bayer) SSG_Q(true, true, RR);   \
    else if (u16) SSG_Q(true, false, RR);      \
    else if (bayer) SSG_Q(false, true, RR);    \
    else SSG_Q(false, false, RR);              \
  } while (0)
  switch (rr) {
    case 0: SSG_QR(0); break;
    case 1: SSG_QR(1); break;
    case 2: SSG_QR(2); break;
    case 3: SSG_QR(3); break;
    default: return hipErrorInvalidValue;
  }
#undef SSG_QR
#undef SSG_Q
  if (!out) hipLaunchKernelGGL(k_quality_fold, dim3(n), dim3(256), 0, s, part, quality_tiles(dw, dh, r), sums);
  return hipGetLastError();
}

}  // namespace ssg

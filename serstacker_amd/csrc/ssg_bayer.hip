// ssg_bayer.hip -- c_bayer_average on gfx950 (core/average/c_frame_accumulation.cc:988-1334).
//
// The reference adds a raw Bayer frame into a 3-channel float accumulator and
// counter.  With a remap set, destination pixel (x, y) takes the source point
// p = rmap(x, y), truncates it (src = (int)p), and gives the four taps of the
// source cell the side weights (src+1-p) and (p-src) -- computed in float, as
// the reference's int/float expression is -- multiplied in double with the
// pixel weight; each tap goes to the channel of its own Bayer position and the
// float accumulator takes the double sum rounded back to float (:1044-1081).
// Without a remap, every pixel adds its own value to its own channel
// (:996-1039).  These kernels do exactly that per pixel, frames in order, so
// results match the reference arithmetic bit for bit; a per-tap count of
// non-zero weights gives the integer per-cell sample counts.
//
// Layout: planes [c][h*w] for c = B, G, R (BAYER_B = 0, BAYER_G = 1,
// BAYER_R = 2, c_frame_accumulation.h:230-234).
#include "ssg_engine.hpp"

namespace ssg {

namespace {

constexpr int BY_TW = 64, BY_RPT = 4, BY_TH = BY_RPT * 4;  // batched tile: 64 x 16, 4 rows per thread

__device__ __forceinline__ int bayer_ch(unsigned pattern, int x, int y) {
  return (int)((pattern >> (2 * (((y & 1) << 1) | (x & 1)))) & 3u);
}

template <bool U16>
__device__ __forceinline__ float raw_value(const void* src, size_t idx, float scale) {
  if constexpr (U16) return (float)((const uint16_t*)src)[idx] * scale;
  else return ((const float*)src)[idx];
}

// the four taps of one destination pixel (reference :1049-1081), accumulated in
// registers; acc = (float)((double)acc + v * s)
template <bool U16>
__device__ __forceinline__ void bayer_gather(const void* src, int pitch, int w, int h, float scale, unsigned pattern,
                                             float px, float py, double wt, float acc[3], float cntr[3],
                                             unsigned cnt[3]) {
  const int sx = (int)px, sy = (int)py;
  if (!(sx >= 0 && sx < w - 1 && sy >= 0 && sy < h - 1)) return;
  const double ax = (double)((float)(sx + 1) - px), ay = (double)((float)(sy + 1) - py);
  const double bx = (double)(px - (float)sx), by = (double)(py - (float)sy);
  const double s[4] = {ax * ay * wt, bx * ay * wt, ax * by * wt, bx * by * wt};
  const size_t o = (size_t)sy * pitch + sx;
  const float v[4] = {raw_value<U16>(src, o, scale), raw_value<U16>(src, o + 1, scale),
                      raw_value<U16>(src, o + pitch, scale), raw_value<U16>(src, o + pitch + 1, scale)};
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int c = bayer_ch(pattern, sx + (k & 1), sy + (k >> 1));
    // select the channel without a dynamic register index
#pragma unroll
    for (int cc = 0; cc < 3; ++cc) {
      if (cc == c) {
        acc[cc] = (float)((double)acc[cc] + (double)v[k] * s[k]);
        cntr[cc] = (float)((double)cntr[cc] + s[k]);
        cnt[cc] += s[k] != 0.0;
      }
    }
  }
}

// ---- one add(src, weights) ------------------------------------------------------------------------
template <bool U16, bool MAP, int WMODE>  // WMODE 0 none, 1 u8 mask, 2 f32 weights
__global__ void __launch_bounds__(256) k_bayer_add(BayerState st, const void* src, int pitch, float scale,
                                                   const float* rmap, int rmap_pitch, const uint8_t* mask,
                                                   int mask_pitch, const float* wts, int wts_pitch) {
  const int x = blockIdx.x * 64 + (threadIdx.x & 63), y = blockIdx.y * 4 + (threadIdx.x >> 6);
  if (x >= st.w || y >= st.h) return;
  if (WMODE == 1 && !mask[(size_t)y * mask_pitch + x]) return;
  const size_t o = (size_t)y * st.w + x;
  if constexpr (!MAP) {
    const int cc = bayer_ch(st.pattern, x, y);
    const float v = raw_value<U16>(src, (size_t)y * pitch + x, scale);
    const size_t q = (size_t)cc * st.plane + o;
    if (WMODE == 2) {
      const float wt = wts[(size_t)y * wts_pitch + x];
      st.acc[q] = st.acc[q] + v * wt;
      st.cntr[q] = st.cntr[q] + wt;
      st.cnt[q] += wt != 0.f;
    } else {
      st.acc[q] = st.acc[q] + v;
      st.cntr[q] = st.cntr[q] + 1.f;
      st.cnt[q] += 1u;
    }
  } else {
    float acc[3], cntr[3];
    unsigned cnt[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      acc[c] = st.acc[(size_t)c * st.plane + o];
      cntr[c] = st.cntr[(size_t)c * st.plane + o];
      cnt[c] = st.cnt[(size_t)c * st.plane + o];
    }
    const float* mp = rmap + (size_t)y * rmap_pitch + 2 * x;
    const double wt = WMODE == 2 ? (double)wts[(size_t)y * wts_pitch + x] : 1.0;
    bayer_gather<U16>(src, pitch, st.w, st.h, scale, st.pattern, mp[0], mp[1], wt, acc, cntr, cnt);
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      st.acc[(size_t)c * st.plane + o] = acc[c];
      st.cntr[(size_t)c * st.plane + o] = cntr[c];
      st.cnt[(size_t)c * st.plane + o] = cnt[c];
    }
  }
}

// ---- batched: registered frames, fused map + base_remap mask + gather ---------------------------
// The map of frame k is the create_remap field of its transform (warp_xy, the
// same arithmetic as ssg_registration_create_remap); its mask is base_remap's
// (c_frame_registration.cc:1319-1338): remap of an all-255 mask (LINEAR,
// CONSTANT 0) >= 255, eroded 5x5 with BORDER_CONSTANT 255.  Each thread holds
// its pixels' accumulators in registers over all frames, in frame order.
//
// k_bayer_staged takes the batches whose maps keep a tile's source box within BY_SH rows of SPR units (BayerBox)
// for every frame, k_bayer_batch the others (bayer_box_fits).
constexpr int BY_SH = 21;  // staged rows: 16, their lower taps, and what a rotation of about 3 degrees adds
template <bool U16, int UNIT>
struct BayerBox {
  static constexpr int ES = U16 ? 2 : 4;
  static constexpr int PER = UNIT / ES;                        // elements of a unit
  static constexpr int SPR = (BY_TW + 4 + PER - 1) / PER + 1;  // units of a staged row
  static constexpr int LOADS = (BY_SH * SPR + 255) / 256;      // units per thread
  // how far apart a tile's positions may lie: from floor(min - 1/4), put back to a unit boundary, to
  // floor(max + 1/4) and its lower tap is less than this and 1/2 + 1 + 1 + (PER - 1), each position being off by
  // less than 1/8 (bayer_box_fits)
  static constexpr double SPAN_X = SPR * PER - PER - 1.75, SPAN_Y = BY_SH - 1 - 1.75;
  static_assert(SPAN_X >= BY_TW - 1 && SPAN_Y >= BY_TH - 1, "a translated tile fits");
};

// the extremes of a map over a rectangle (the maps are affine: at its corners); NaN positions give a
// rectangle that is inside nothing
template <int MOTION>
__device__ __forceinline__ void map_extremes(const MapCoef& mc, int rx0, int ry0, int rx1, int ry1, float& mnx,
                                             float& mxx, float& mny, float& mxy) {
  mnx = 1e30f, mxx = -1e30f, mny = 1e30f, mxy = -1e30f;
  const int cx[4] = {rx0, rx1, rx0, rx1}, cy[4] = {ry0, ry0, ry1, ry1};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float sx, sy;
    warp_xy<MOTION>(mc, cx[i], cy[i], sx, sy);
    mnx = fminf(mnx, sx); mxx = fmaxf(mxx, sx); mny = fminf(mny, sy); mxy = fmaxf(mxy, sy);
    if (sx != sx || sy != sy) mnx = -1e30f;
  }
}

// the tile and its erosion halo map strictly inside the frame: no mask test
template <int MOTION>
__device__ __forceinline__ bool bayer_interior(const BayerState& st, const MapCoef& mc, int x0, int y0) {
  float mnx, mxx, mny, mxy;
  map_extremes<MOTION>(mc, max(x0 - 2, 0), max(y0 - 2, 0), min(x0 + BY_TW + 1, st.w - 1),
                       min(y0 + BY_TH + 1, st.h - 1), mnx, mxx, mny, mxy);
  return mnx >= 0.25f && mny >= 0.25f && mxx <= (float)st.w - 1.25f && mxy <= (float)st.h - 1.25f;
}

// What a frame is to a tile: outside (its positions all beyond the frame, or NaN: no pixel is added), inside,
// or with pixels the mask may drop.  The box starts at a unit boundary; the corners' positions may round apart
// from a pixel's by less than 1/4 px.
enum : int { BY_OUTSIDE = 0, BY_INSIDE = 1, BY_BORDER = 2 };
template <int MOTION, bool U16, int UNIT>
__device__ __forceinline__ int bayer_plan(const BayerState& st, const MapCoef& mc, int x0, int y0, int& bx, int& by) {
  using Box = BayerBox<U16, UNIT>;
  float mnx, mxx, mny, mxy;
  map_extremes<MOTION>(mc, x0, y0, min(x0 + BY_TW - 1, st.w - 1), min(y0 + BY_TH - 1, st.h - 1), mnx, mxx, mny, mxy);
  if (!(mnx > -1e29f) || !(mxx > -1.f) || !(mxy > -1.f) || !(mnx < (float)st.w) || !(mny < (float)st.h)) return BY_OUTSIDE;
  const int ix = (int)floorf(mnx - 0.25f);
  bx = ix - ((ix % Box::PER) + Box::PER) % Box::PER;
  by = (int)floorf(mny - 0.25f);
  return bayer_interior<MOTION>(st, mc, x0, y0) ? BY_INSIDE : BY_BORDER;
}

// the eroded mask of a tile that is not inside the frame, into rmk: bit columns combined over x, five rows
// of it to combine over y (barriers)
template <int MOTION>
__device__ __forceinline__ void bayer_mask(const BayerState& st, const MapCoef& mc, int x0, int y0,
                                           uint8_t (*mk)[BY_TW + 4], uint8_t (*rmk)[BY_TW]) {
  for (int i = threadIdx.x; i < (BY_TH + 4) * (BY_TW + 4); i += 256) {
    const int ly = i / (BY_TW + 4), lx = i - ly * (BY_TW + 4);
    const int px = x0 - 2 + lx, py = y0 - 2 + ly;
    uint8_t v = 1;  // outside the destination: the erosion border value 255
    if ((unsigned)px < (unsigned)st.w && (unsigned)py < (unsigned)st.h) {
      float sx, sy;
      warp_xy<MOTION>(mc, px, py, sx, sy);
      v = remap_mask_u8(nullptr, 0, st.w, st.h, quant32(sx), quant32(sy)) >= 255;
    }
    mk[ly][lx] = v;
  }
  __syncthreads();
  for (int i = threadIdx.x; i < (BY_TH + 4) * BY_TW; i += 256) {
    const int ly = i / BY_TW, lx = i - ly * BY_TW;
    rmk[ly][lx] = mk[ly][lx] & mk[ly][lx + 1] & mk[ly][lx + 2] & mk[ly][lx + 3] & mk[ly][lx + 4];
  }
  __syncthreads();
}

// The staged tiles: a frame's source box goes to LDS by direct-to-LDS loads of UNIT bytes, the next frame's
// landing while this one's taps are summed (two boxes; one barrier a frame).  The four taps of a pixel fall
// on the four positions of the Bayer cell -- one R, one B, two G -- so each tap is read by channel, at the
// column and row of its parity, and every update is made once, without a mask; (double)(raw * scale) * s is
// fma(raw * s, scale, acc), the scale being a power of two.  A wave finds the boxes of 64 frames at a time,
// a frame per lane.
// What bounds it: vector operations, most of them the double-precision updates and their conversions.
// 32 raw frames of 4096x3000: 1.14 ms; 2.16 ms with sixteen two-byte gathers in flight per thread and the
// channel as a lane mask over three updates per tap (k_bayer_batch).
// EDGE: frames whose mask may drop pixels of the tile are among them (a kernel of its own code: the
// branches around a row's update keep its loads apart)
template <int MOTION, bool U16, int UNIT, bool EDGE>
__device__ __forceinline__ void bayer_tile(const BayerBatchArgs& a, int x0, int y0, int lane, int wv,
                                           uint8_t (*box)[BayerBox<U16, UNIT>::LOADS * 256 * UNIT],
                                           uint8_t (*mk)[BY_TW + 4], uint8_t (*rmk)[BY_TW]) {
  using Box = BayerBox<U16, UNIT>;
  constexpr int BP = Box::SPR * Box::PER;  // elements of a box row
  const BayerState& st = a.st;
  // pixels past the frame's edge repeat its last column or row; they are not stored
  const int x = x0 + lane, xc = min(x, st.w - 1);
  float acc[BY_RPT][3], cntr[BY_RPT][3];
  unsigned full[BY_RPT];    // frames whose row has no zero weight: a count each for B and R, two for G
  unsigned part[BY_RPT][3]; // counts of the other frames
#pragma unroll
  for (int r = 0; r < BY_RPT; ++r) {
    const size_t o = (size_t)min(y0 + wv * BY_RPT + r, st.h - 1) * st.w + xc;
    full[r] = 0;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      acc[r][c] = st.acc[(size_t)c * st.plane + o];
      cntr[r][c] = st.cntr[(size_t)c * st.plane + o];
      part[r][c] = 0;
    }
  }
  const int posx = a.pos_r & 1, posy = a.pos_r >> 1;
  const double dscale = U16 ? (double)a.scale : 1.0;
  const uint32_t rowb = (uint32_t)a.src_pitch * Box::ES;
  for (int k0 = 0; k0 < a.nframes; k0 += WAVE) {
    int bx = 0, by = 0;
    const int kl = k0 + lane;
    int plan = BY_OUTSIDE;
    if (kl < a.nframes && a.valid[kl]) {
      MapCoef mc;
#pragma unroll
      for (int i = 0; i < 8; ++i) mc.c[i] = a.maps[kl].c[i];
      plan = bayer_plan<MOTION, U16, UNIT>(st, mc, x0, y0, bx, by);
    }
    unsigned long long left = __ballot(plan == BY_INSIDE || plan == BY_BORDER);
    const unsigned long long border = __ballot(plan == BY_BORDER);
    if (!left) continue;
    auto stage = [&](int j, int buf) {  // the box of frame k0 + j
      const int jx = __builtin_amdgcn_readlane(bx, j), jy = __builtin_amdgcn_readlane(by, j);
      const rsrc_t rs = make_rsrc(a.frames[k0 + j], (uint32_t)st.h * rowb);
#pragma unroll
      for (int n = 0; n < Box::LOADS; ++n) {
        const int i = n * 256 + wv * WAVE + lane, row = i / Box::SPR, col = i - row * Box::SPR;
        // a unit that holds a pixel of the row lies in the row's memory (its start is a multiple of UNIT)
        if (row < BY_SH && (unsigned)(jy + row) < (unsigned)st.h && (unsigned)(jx + col * Box::PER) < (unsigned)st.w) {
          const uint32_t o = (uint32_t)(jy + row) * rowb + (uint32_t)(jx + col * Box::PER) * Box::ES;
          uint8_t* d = &box[buf][(n * 256 + wv * WAVE) * UNIT];
          if constexpr (UNIT == 16) bload_lds16(rs, d, o);
          else bload_lds4(rs, d, o);
        }
      }
    };
    int cur = 0;
    __syncthreads();  // the previous group's last box has been read
    stage(__builtin_ctzll(left), 0);
    for (; left; left &= left - 1, cur ^= 1) {
      const int j = __builtin_ctzll(left);
      __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): this wave's part of the box has landed
      __syncthreads();                     // every wave's has, and the other box has been read
      if (left & (left - 1)) stage(__builtin_ctzll(left & (left - 1)), cur ^ 1);
      const int jx = __builtin_amdgcn_readlane(bx, j), jy = __builtin_amdgcn_readlane(by, j);
      MapCoef mc;
#pragma unroll
      for (int i = 0; i < 8; ++i) mc.c[i] = a.maps[k0 + j].c[i];
      const bool edge = EDGE && (border >> j & 1) != 0;
      if (edge) bayer_mask<MOTION>(st, mc, x0, y0, mk, rmk);  // its barriers keep the frames' masks apart
      auto raw = [&](int o) {
        if constexpr (U16) return (double)((const uint16_t*)box[cur])[o];
        else return (double)((const float*)box[cur])[o];
      };
      int sx = 0, cr = 0;
      double wxr = 0, wxb = 0;
      bool xnz = true;
      auto columns = [&](float px) {  // R's column is that of its parity, B's the other one
        sx = (int)px;
        const float ax = (float)(sx + 1) - px, bxf = px - (float)sx;
        cr = (sx ^ posx) & 1;
        wxr = (double)(cr ? bxf : ax);
        wxb = (double)(cr ? ax : bxf);
        xnz = bxf != 0.f;
      };
      if constexpr (MOTION == MOTION_TRANSLATION) columns((float)xc + mc.c[0]);
#pragma unroll
      for (int r = 0; r < BY_RPT; ++r) {
        float px, py;
        warp_xy<MOTION>(mc, xc, min(y0 + wv * BY_RPT + r, st.h - 1), px, py);
        if constexpr (MOTION != MOTION_TRANSLATION) columns(px);
        const int sy = (int)py;
        const float ay = (float)(sy + 1) - py, byf = py - (float)sy;
        const bool below = ((sy ^ posy) & 1) != 0;  // R lies in row sy + 1
        const double wyr = (double)(below ? byf : ay), wyb = (double)(below ? ay : byf);
        if (edge) {
          const int ly = wv * BY_RPT + r;
          if (!(rmk[ly][lane] & rmk[ly + 1][lane] & rmk[ly + 2][lane] & rmk[ly + 3][lane] & rmk[ly + 4][lane])) continue;
          if (!(sx >= 0 && sx < st.w - 1 && sy >= 0 && sy < st.h - 1)) continue;
        }
        const int o0 = (sy - jy) * BP + sx - jx, cb = 1 - cr;
        const double sr = wxr * wyr, sb = wxb * wyb, p = wxb * wyr, q = wxr * wyb;
        const double s1 = below ? q : p, s2 = below ? p : q;  // the G taps of rows sy and sy + 1, in that order
        const double vr = raw(o0 + cr + (below ? BP : 0)), vb = raw(o0 + cb + (below ? 0 : BP));
        const double v1 = raw(o0 + (below ? cr : cb)), v2 = raw(o0 + BP + (below ? cb : cr));
        acc[r][2] = (float)fma(vr * sr, dscale, (double)acc[r][2]);
        acc[r][0] = (float)fma(vb * sb, dscale, (double)acc[r][0]);
        acc[r][1] = (float)fma(v1 * s1, dscale, (double)acc[r][1]);
        acc[r][1] = (float)fma(v2 * s2, dscale, (double)acc[r][1]);
        cntr[r][2] = (float)((double)cntr[r][2] + sr);
        cntr[r][0] = (float)((double)cntr[r][0] + sb);
        cntr[r][1] = (float)((double)cntr[r][1] + s1);
        cntr[r][1] = (float)((double)cntr[r][1] + s2);
        // ax, ay > 0: a weight is zero only where a lower tap's factor is
        if (!edge && __all(xnz && byf != 0.f)) {
          full[r] += 1;
        } else {
          part[r][2] += sr != 0.0;
          part[r][0] += sb != 0.0;
          part[r][1] += (s1 != 0.0) + (s2 != 0.0);
        }
      }
    }
  }
#pragma unroll
  for (int r = 0; r < BY_RPT; ++r) {
    const int y = y0 + wv * BY_RPT + r;
    if (x >= st.w || y >= st.h) continue;
    const size_t o = (size_t)y * st.w + x;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      st.acc[(size_t)c * st.plane + o] = acc[r][c];
      st.cntr[(size_t)c * st.plane + o] = cntr[r][c];
      st.cnt[(size_t)c * st.plane + o] += part[r][c] + (c == 1 ? 2 * full[r] : full[r]);
    }
  }
}

template <int MOTION, bool U16, int UNIT>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) k_bayer_staged(BayerBatchArgs a) {
  // a wave's loads write WAVE consecutive units from a uniform base
  __shared__ __align__(16) uint8_t box[2][BayerBox<U16, UNIT>::LOADS * 256 * UNIT];
  __shared__ uint8_t mk[BY_TH + 4][BY_TW + 4];
  __shared__ uint8_t rmk[BY_TH + 4][BY_TW];
  const int lane = threadIdx.x & (WAVE - 1), wv = __builtin_amdgcn_readfirstlane((int)threadIdx.x / WAVE);
  // the outermost ring of tiles first: the masks make them three times as long as the others, and the last
  // ones would be the launch's tail; then the inner tiles row by row
  const int X = (a.st.w + BY_TW - 1) / BY_TW, Y = (a.st.h + BY_TH - 1) / BY_TH, id = blockIdx.x;
  int tx, ty;
  if (X < 3 || Y < 3) {
    tx = id % X, ty = id / X;
  } else if (id < 2 * X) {
    tx = id % X, ty = id < X ? 0 : Y - 1;
  } else if (id < 2 * X + 2 * (Y - 2)) {
    const int i = id - 2 * X;
    tx = i & 1 ? X - 1 : 0, ty = 1 + (i >> 1);
  } else {
    const int i = id - 2 * X - 2 * (Y - 2);
    tx = 1 + i % (X - 2), ty = 1 + i / (X - 2);
  }
  const int x0 = tx * BY_TW, y0 = ty * BY_TH;
  bool inside = true;
  for (int k0 = 0; k0 < a.nframes; k0 += WAVE) {
    const int k = k0 + lane;
    int plan = BY_INSIDE;
    if (k < a.nframes && a.valid[k]) {
      MapCoef mc;
#pragma unroll
      for (int i = 0; i < 8; ++i) mc.c[i] = a.maps[k].c[i];
      int bx, by;
      plan = bayer_plan<MOTION, U16, UNIT>(a.st, mc, x0, y0, bx, by);
    }
    inside = inside && __all(plan == BY_INSIDE || plan == BY_OUTSIDE);
  }
  if (inside) bayer_tile<MOTION, U16, UNIT, false>(a, x0, y0, lane, wv, box, mk, rmk);
  else bayer_tile<MOTION, U16, UNIT, true>(a, x0, y0, lane, wv, box, mk, rmk);
}

// The batches that k_bayer_staged does not take.
template <int MOTION, bool U16>
__global__ void __launch_bounds__(256) k_bayer_batch(BayerBatchArgs a) {
  __shared__ uint8_t mk[BY_TH + 4][BY_TW + 4];
  __shared__ uint8_t rmk[BY_TH + 4][BY_TW];
  const BayerState& st = a.st;
  const int tid = threadIdx.x, lane = tid & (WAVE - 1), wv = tid / WAVE;
  const int x0 = blockIdx.x * BY_TW, y0 = blockIdx.y * BY_TH;
  const int x = x0 + lane;
  float acc[BY_RPT][3], cntr[BY_RPT][3];
  unsigned cnt[BY_RPT][3];
#pragma unroll
  for (int r = 0; r < BY_RPT; ++r) {
    const int y = y0 + wv * BY_RPT + r;
    const bool in = x < st.w && y < st.h;
    const size_t o = (size_t)y * st.w + x;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      acc[r][c] = in ? st.acc[(size_t)c * st.plane + o] : 0.f;
      cntr[r][c] = in ? st.cntr[(size_t)c * st.plane + o] : 0.f;
      cnt[r][c] = in ? st.cnt[(size_t)c * st.plane + o] : 0u;
    }
  }
  for (int k = 0; k < a.nframes; ++k) {
    if (!a.valid[k]) continue;
    MapCoef mc;
#pragma unroll
    for (int i = 0; i < 8; ++i) mc.c[i] = a.maps[k].c[i];
    const void* src = a.frames[k];
    const bool interior = bayer_interior<MOTION>(st, mc, x0, y0);
    if (!interior) {
      bayer_mask<MOTION>(st, mc, x0, y0, mk, rmk);
    }
#pragma unroll
    for (int r = 0; r < BY_RPT; ++r) {
      const int ly = wv * BY_RPT + r, y = y0 + ly;
      if (x >= st.w || y >= st.h) continue;
      if (!interior && !(rmk[ly][lane] & rmk[ly + 1][lane] & rmk[ly + 2][lane] & rmk[ly + 3][lane] & rmk[ly + 4][lane]))
        continue;
      float sx, sy;
      warp_xy<MOTION>(mc, x, y, sx, sy);
      bayer_gather<U16>(src, a.src_pitch, st.w, st.h, a.scale, st.pattern, sx, sy, 1.0, acc[r], cntr[r], cnt[r]);
    }
    if (!interior) __syncthreads();
  }
#pragma unroll
  for (int r = 0; r < BY_RPT; ++r) {
    const int y = y0 + wv * BY_RPT + r;
    if (x >= st.w || y >= st.h) continue;
    const size_t o = (size_t)y * st.w + x;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      st.acc[(size_t)c * st.plane + o] = acc[r][c];
      st.cntr[(size_t)c * st.plane + o] = cntr[r][c];
      st.cnt[(size_t)c * st.plane + o] = cnt[r][c];
    }
  }
}

// compute() (:1205-1238): avg = acc / cntr per channel (float division, 0 where
// cntr <= 0), interleaved BGR; mask = any channel's cntr > 0
__global__ void __launch_bounds__(256) k_bayer_compute(BayerState st, float* avg, int avg_pitch, uint8_t* mask,
                                                       int mask_pitch) {
  const int x = blockIdx.x * 64 + (threadIdx.x & 63), y = blockIdx.y * 4 + (threadIdx.x >> 6);
  if (x >= st.w || y >= st.h) return;
  const size_t o = (size_t)y * st.w + x;
  bool any = false;
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const float n = st.cntr[(size_t)c * st.plane + o];
    if (avg) avg[(size_t)y * avg_pitch + 3 * x + c] = n > 0.f ? st.acc[(size_t)c * st.plane + o] / n : 0.f;
    any |= n > 0.f;
  }
  if (mask) mask[(size_t)y * mask_pitch + x] = any ? 255 : 0;
}

// get_acc_counters() (:1240-1250): the counter scaled by (1, 0.5, 1), interleaved
__global__ void __launch_bounds__(256) k_bayer_counters(BayerState st, float* out, int out_pitch) {
  const int x = blockIdx.x * 64 + (threadIdx.x & 63), y = blockIdx.y * 4 + (threadIdx.x >> 6);
  if (x >= st.w || y >= st.h) return;
  const size_t o = (size_t)y * st.w + x;
  out[(size_t)y * out_pitch + 3 * x + 0] = st.cntr[o];
  out[(size_t)y * out_pitch + 3 * x + 1] = st.cntr[(size_t)st.plane + o] * 0.5f;
  out[(size_t)y * out_pitch + 3 * x + 2] = st.cntr[(size_t)2 * st.plane + o];
}

}  // namespace

unsigned bayer_pattern_bits(int colorid) {
  // generate_bayer_pattern_mask (:1267-1334): cell positions (0,0) (0,1) (1,0) (1,1)
  static const int tab[4][4] = {{2, 1, 1, 0}, {1, 2, 0, 1}, {1, 0, 2, 1}, {0, 1, 1, 2}};
  if (colorid < 8 || colorid > 11) return 0;
  unsigned bits = 0;
  for (int i = 0; i < 4; ++i) bits |= (unsigned)tab[colorid - 8][i] << (2 * i);
  return bits;
}

hipError_t launch_bayer_add(const BayerState& st, const void* src, int src_pitch, bool u16, float scale,
                            const float* rmap, int rmap_pitch, const uint8_t* mask, int mask_pitch,
                            const float* wts, int wts_pitch, hipStream_t s) {
  dim3 grid((st.w + 63) / 64, (st.h + 3) / 4);
  const int wm = wts ? 2 : (mask ? 1 : 0);
#define SSG_BA(U, M, W) \
  hipLaunchKernelGGL((k_bayer_add<U, M, W>), grid, dim3(256), 0, s, st, src, src_pitch, scale, rmap, rmap_pitch, \
                     mask, mask_pitch, wts, wts_pitch)
#define SSG_BA_W(U, M)            \
  do {                            \
    if (wm == 2) SSG_BA(U, M, 2); \
    else if (wm == 1) SSG_BA(U, M, 1); \
    else SSG_BA(U, M, 0);         \
  } while (0)
  if (u16) {
    if (rmap) SSG_BA_W(true, true);
    else SSG_BA_W(true, false);
  } else {
    if (rmap) SSG_BA_W(false, true);
    else SSG_BA_W(false, false);
  }
#undef SSG_BA_W
#undef SSG_BA
  return hipGetLastError();
}

// Whether the source box of every tile of a w x h frame fits the staged one.  The maps are affine, so a tile's
// positions are as far apart everywhere; below 2^18 their three roundings are off by less than 1/8 px in all.  A map
// with NaN or infinite values does not fit.
// Why the whole batch: with the kernels sharing one by tiles, a rotation out of the box among smaller ones made both
// run, 132 us for 8 frames of 640x480 where k_bayer_batch alone takes 93.
bool bayer_box_fits(int motion, const MapCoef& m, int w, int h, bool u16, int unit) {
  double a = 1, b = 0, c = 0, d = 1, tx, ty;
  if (motion == MOTION_TRANSLATION) {
    tx = m.c[0], ty = m.c[1];
  } else if (motion == MOTION_AFFINE) {
    a = m.c[0], b = m.c[1], tx = m.c[2], c = m.c[3], d = m.c[4], ty = m.c[5];
  } else {
    const double s = m.c[2];
    if (m.c[5] != 0.f || m.c[6] != 0.f) return false;  // a batch's maps turn about (0, 0)
    a = s * m.c[1], b = s * m.c[0], c = s * m.c[0], d = s * m.c[1], tx = m.c[3], ty = m.c[4];
    if (!(fabs(m.c[0]) <= 1.f && fabs(m.c[1]) <= 1.f)) return false;
  }
  a = fabs(a), b = fabs(b), c = fabs(c), d = fabs(d);
  const double top = 262144;
  if (!(a * w + b * h + fabs(tx) < top && c * w + d * h + fabs(ty) < top)) return false;
  const double sx = a * (BY_TW - 1) + b * (BY_TH - 1), sy = c * (BY_TW - 1) + d * (BY_TH - 1);
  const auto within = [&](auto box) { return sx <= decltype(box)::SPAN_X && sy <= decltype(box)::SPAN_Y; };
  if (unit == 16) return u16 ? within(BayerBox<true, 16>{}) : within(BayerBox<false, 16>{});
  return u16 ? within(BayerBox<true, 4>{}) : within(BayerBox<false, 4>{});
}

hipError_t launch_bayer_batch(int motion, bool u16, const BayerBatchArgs& a, hipStream_t s) {
  dim3 grid((a.st.w + BY_TW - 1) / BY_TW, (a.st.h + BY_TH - 1) / BY_TH);
#define SSG_STAGED(M, U, UNIT) \
  hipLaunchKernelGGL((k_bayer_staged<M, U, UNIT>), dim3(grid.x * grid.y), dim3(256), 0, s, a)
#define SSG_BB(M)                                                                          \
  do {                                                                                     \
    if (a.unit == 16 && u16) SSG_STAGED(M, true, 16);                                      \
    else if (a.unit == 16) SSG_STAGED(M, false, 16);                                       \
    else if (a.unit == 4 && u16) SSG_STAGED(M, true, 4);                                   \
    else if (a.unit == 4) SSG_STAGED(M, false, 4);                                         \
    else if (u16) hipLaunchKernelGGL((k_bayer_batch<M, true>), grid, dim3(256), 0, s, a);  \
    else hipLaunchKernelGGL((k_bayer_batch<M, false>), grid, dim3(256), 0, s, a);          \
  } while (0)
  switch (motion) {
    case MOTION_TRANSLATION: SSG_BB(MOTION_TRANSLATION); break;
    case MOTION_EUCLIDEAN:
    case MOTION_SCALED_EUCLIDEAN: SSG_BB(MOTION_EUCLIDEAN); break;
    case MOTION_AFFINE: SSG_BB(MOTION_AFFINE); break;
    default: return hipErrorInvalidValue;
  }
#undef SSG_BB
#undef SSG_STAGED
  return hipGetLastError();
}

hipError_t launch_bayer_compute(const BayerState& st, float* avg, int avg_pitch, uint8_t* mask, int mask_pitch,
                                hipStream_t s) {
  dim3 grid((st.w + 63) / 64, (st.h + 3) / 4);
  hipLaunchKernelGGL(k_bayer_compute, grid, dim3(256), 0, s, st, avg, avg_pitch, mask, mask_pitch);
  return hipGetLastError();
}

hipError_t launch_bayer_counters(const BayerState& st, float* out, int out_pitch, hipStream_t s) {
  dim3 grid((st.w + 63) / 64, (st.h + 3) / 4);
  hipLaunchKernelGGL(k_bayer_counters, grid, dim3(256), 0, s, st, out, out_pitch);
  return hipGetLastError();
}

}  // namespace ssg

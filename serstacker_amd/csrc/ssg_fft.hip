// ssg_fft.hip -- FFT phase-correlation translation estimate on gfx950.
//
// SerStacker has no phase correlation on this path (nearest code:
// core/proc/fft.cc:17-160); this is the pre-alignment the build defines:
// optional 2x2 binning, mean removal and separable Hann apodisation, zero
// padding to powers of two, 2-D FFT, normalised cross-power F conj(G) / |F conj(G)|
// with a gaussian weight (correlation peak of sigma 1 px), inverse FFT, integer
// peak and a 3-point gaussian refinement per axis in FP64.
//
// The frames are real, so their spectra are Hermitian and only the columns kx = 0 .. M / 2 are
// transformed and crossed. A frame's plane in memory (float2 [N][M], strip by strip) is touched four
// times -- k_pc_rows writes half of it, k_pc_cols reads that half and writes all, k_pc_rows_peak reads it:
//   k_pc_rows       forward row FFTs; the rows are binned, centred and apodised while they are loaded
//   k_pc_cols       a strip of columns whole in LDS: forward FFT, cross power, inverse FFT; then the
//                   inverse FFT of the mirrored columns M - kx, whose cross power is the conjugate
//   k_pc_rows_peak  inverse row FFTs and their largest value; the correlation surface itself is never
//                   written
//   k_pc_peak       the frame's peak; the rows around it once more for the fit's five samples
// The FFTs are radix-2 Stockham stages with table twiddles, three (or two) of them in registers between
// two exchanges through LDS.  A forward transform takes conjugate operands through the same operations
// at k and -k, so leaving the second half out changes no result; the inverse does not, so the mirrored
// columns are transformed too.
// The plane is two halves of strips ([strip][row][column of the strip], then column M / 2; the mirrored
// columns at the same places of the second half), so a strip is one contiguous block and the row kernels
// write and read runs of (rows of the block) * 64 B.
//
// What bounds it: the sweeps over the plane and the frame (about 140 MB for a raw 4096 x 3000 frame,
// padded to 2048 x 2048) and the transforms' arithmetic, about equal.  16 such frames: 1.13 ms; 3.90 ms
// with full complex planes, one LDS exchange per radix-2 stage and transposes in memory (seventeen 8-byte
// sweeps of the padded plane).  Packing two real rows into one complex FFT and radix-8 butterflies gave
// 0.84 ms; its last digits differ, and the dense flow that starts from the shifts magnifies a last digit
// without bound where the frames have no texture, so the operations stay as they were.
#include "ssg_engine.hpp"

namespace ssg {

namespace {

// ---- FFT in LDS: three radix-2 Stockham stages per pass (two at the end), natural order in and out ----
__device__ __forceinline__ float2 cadd(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ float2 csub(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ float2 cmul(float2 a, float2 w) {
  return make_float2(fmaf(a.x, w.x, -(a.y * w.y)), fmaf(a.x, w.y, a.y * w.x));
}

// LOGR radix-2 Stockham stages on the R = 1 << LOGR points of a group: stage t joins the halves of what is
// left, out index bit t is its branch, and the branches so far select the twiddle: w(t, m) is the stage's
// twiddle of k + m ns
template <int LOGR, int T = 0, class W>
__device__ __forceinline__ void stages(float2* v, W w) {
  if constexpr (T < LOGR) {
    constexpr int half = 1 << (LOGR - 1 - T);  // points left per branch, halved
    // v[m + (r << T)]: branch m (T bits), point r of 2 * half
    float2 o[1 << LOGR];
#pragma unroll
    for (int m = 0; m < (1 << T); ++m) {
      const float2 wm = w(std::integral_constant<int, T>{}, m);
#pragma unroll
      for (int r = 0; r < half; ++r) {
        const float2 u = v[m + (r << T)], x = cmul(v[m + ((r + half) << T)], wm);
        o[m + (r << (T + 1))] = cadd(u, x);
        o[m + (1 << T) + (r << (T + 1))] = csub(u, x);
      }
    }
#pragma unroll
    for (int i = 0; i < (1 << LOGR); ++i) v[i] = o[i];
    stages<LOGR, T + 1>(v, w);
  }
}

constexpr int FFT_PPT = 16;  // points per thread, held in registers between a pass's reads and writes

// Where point i of sequence c lies, and how the groups are dealt to the threads.  The strips keep the
// sequences (columns) side by side, the rows one after the other.  The low index bits are mixed with
// higher ones so that a three-stage pass's stride-8 writes spread over the LDS banks: 64 lanes of 8 B then
// take the two cycles their bytes need.  The mix is linear over exclusive or, so the place of i | j with
// no common bits is at(i, c) ^ step(j): one operation per point, j being a constant of the pass.
struct StripLayout {
  int lc;  // log2 of the columns
  __device__ __forceinline__ int at(int i, int c) const { return ((i ^ ((i >> 3) & 7)) << lc) + c; }
  __device__ __forceinline__ int step(int i) const { return (i ^ ((i >> 3) & 7)) << lc; }
  template <int LOGB>
  __device__ __forceinline__ void deal(int b, int& j, int& c) const {
    c = b & ((1 << lc) - 1);
    j = b >> lc;
  }
};
template <int LOGN>
struct RowLayout {
  __device__ __forceinline__ int step(int i) const { return i ^ ((i >> 5) & 31) ^ (((i >> 6) & 3) << 3); }
  // bits 3 and 4 also by the row: the strips' runs of 8 columns in 4 rows then lie in different banks
  __device__ __forceinline__ int at(int i, int c) const {
    return (c << LOGN) + (step(i) ^ (LOGN >= 5 ? (c & 3) << 3 : 0));
  }
  template <int LOGB>
  __device__ __forceinline__ void deal(int b, int& j, int& c) const {
    j = b & ((1 << LOGB) - 1);
    c = b >> LOGB;
  }
};

// Twiddles in LDS: exp(-2 pi i k / n), k < n / 2, as the stages with the longest steps read it (every entry
// or every second one), then a table of its own for each stage below, whose steps through the first table
// would fall into one LDS bank (stage s: 1 << s entries at n / 2 + (1 << s)).
template <int LOGN>
constexpr int TW_SIZE = LOGN > 2 ? 3 << (LOGN - 2) : 1 << (LOGN - 1);
template <int LOGN>
__device__ __forceinline__ void tw_load(float2* tw, const float2* twg) {
  constexpr int H = 1 << (LOGN - 1);
  for (int i = threadIdx.x; i < TW_SIZE<LOGN>; i += blockDim.x) {
    const int e = i - H, s = e > 0 ? 31 - __clz(e) : 0;
    tw[i] = i < H ? twg[i] : (e > 0 ? twg[(e - (1 << s)) << (LOGN - 1 - s)] : make_float2(0.f, 0.f));
  }
}
// entry k of stage S
template <int LOGN, int S>
__device__ __forceinline__ float2 tw_at(const float2* tw, int k) {
  if constexpr (S + 2 >= LOGN) return tw[k << (LOGN - 1 - S)];
  else return tw[(1 << (LOGN - 1)) + (1 << S) + k];
}

// one pass of LOGR stages over nseq sequences of 1 << LOGN points
template <int LOGN, int LOGR, int LOGNS, bool INV, class Layout>
__device__ __forceinline__ void fft_pass(float2* buf, const float2* tw, int nseq, const Layout& L) {
  constexpr int R = 1 << LOGR, G = FFT_PPT / R, LOGB = LOGN - LOGR;
  const int total = nseq << LOGB;
  float2 v[G][R];
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const int b = (int)threadIdx.x + g * (int)blockDim.x;
    if (b < total) {
      int j, c;
      L.template deal<LOGB>(b, j, c);
      const int a = L.at(j, c);
#pragma unroll
      for (int r = 0; r < R; ++r) v[g][r] = buf[a ^ L.step(r << LOGB)];
      const int k = j & ((1 << LOGNS) - 1);
      stages<LOGR>(v[g], [&](auto t, int m) {
        float2 w = tw_at<LOGN, LOGNS + decltype(t)::value>(tw, k + (m << LOGNS));  // exp(-2 pi i (k + m ns) / (2 ns 2^t))
        if (INV) w.y = -w.y;
        return w;
      });
    }
  }
  __syncthreads();
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const int b = (int)threadIdx.x + g * (int)blockDim.x;
    if (b < total) {
      int j, c;
      L.template deal<LOGB>(b, j, c);
      const int k = j & ((1 << LOGNS) - 1), a = L.at(((j - k) << LOGR) + k, c);
#pragma unroll
      for (int r = 0; r < R; ++r) buf[a ^ L.step(r << LOGNS)] = v[g][r];
    }
  }
  __syncthreads();
}

// the passes from stage LOGNS on: three stages while what is left is not two or four
template <int LOGN, bool INV, class Layout, int LOGNS = 0>
__device__ __forceinline__ void fft_lds(float2* buf, const float2* tw, int nseq, const Layout& L) {
  if constexpr (LOGNS < LOGN) {
    constexpr int LEFT = LOGN - LOGNS, LOGR = (LEFT == 2 || LEFT == 4) ? 2 : 3;
    fft_pass<LOGN, LOGR, LOGNS, INV>(buf, tw, nseq, L);
    fft_lds<LOGN, INV, Layout, LOGNS + LOGR>(buf, tw, nseq, L);
  }
}

// ---- loading --------------------------------------------------------------------------------------
struct PcSource {
  const void* const* frames;
  int pitch;    // elements
  int u16, binning;
  int wide;     // every frame's rows hold two binned pixels' samples at aligned addresses
  int bw, bh;   // binned size
};

__device__ __forceinline__ float pc_at(const void* src, int u16, size_t o) {
  return u16 ? (float)((const uint16_t*)src)[o] : ((const float*)src)[o];
}

// the binned pixels x, x + 1 (x even) of row y; 0 where they are outside
__device__ __forceinline__ float2 pc_pair(const PcSource& s, const void* src, int x, int y) {
  if (y >= s.bh || x >= s.bw) return make_float2(0.f, 0.f);
  const bool two = x + 1 < s.bw;
  if (s.binning == 2) {
    const size_t o = (size_t)(2 * y) * s.pitch + 2 * x, p = o + s.pitch;
    float a[4], b[4];
    if (s.wide && two) {
      if (s.u16) {
        const uint2 u = *(const uint2*)((const uint16_t*)src + o), v = *(const uint2*)((const uint16_t*)src + p);
        a[0] = (float)(u.x & 0xffffu); a[1] = (float)(u.x >> 16); a[2] = (float)(u.y & 0xffffu); a[3] = (float)(u.y >> 16);
        b[0] = (float)(v.x & 0xffffu); b[1] = (float)(v.x >> 16); b[2] = (float)(v.y & 0xffffu); b[3] = (float)(v.y >> 16);
      } else {
        const float4 u = *(const float4*)((const float*)src + o), v = *(const float4*)((const float*)src + p);
        a[0] = u.x; a[1] = u.y; a[2] = u.z; a[3] = u.w;
        b[0] = v.x; b[1] = v.y; b[2] = v.z; b[3] = v.w;
      }
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const bool in = i < 2 || two;
        a[i] = in ? pc_at(src, s.u16, o + i) : 0.f;
        b[i] = in ? pc_at(src, s.u16, p + i) : 0.f;
      }
    }
    return make_float2(((a[0] + a[1]) + (b[0] + b[1])) * 0.25f, ((a[2] + a[3]) + (b[2] + b[3])) * 0.25f);
  }
  const size_t o = (size_t)y * s.pitch + x;
  if (s.wide && two) {
    if (s.u16) {
      const uint32_t u = *(const uint32_t*)((const uint16_t*)src + o);
      return make_float2((float)(u & 0xffffu), (float)(u >> 16));
    }
    return *(const float2*)((const float*)src + o);
  }
  return make_float2(pc_at(src, s.u16, o), two ? pc_at(src, s.u16, o + 1) : 0.f);
}

// mean of the binned image (double accumulation)
constexpr int PC_PARTS = PC_PARTS_MAX;  // blocks per frame of the mean

// stage 1: double sums of the binned frame over row bands, one partial per block (PC_PARTS per frame);
// four rows' pairs in flight per thread
__global__ void __launch_bounds__(256) k_pc_mean_part(PcSource s, double* part) {
  __shared__ double red[256];
  const void* src = s.frames[blockIdx.y];
  const int y0 = (int)((long long)s.bh * blockIdx.x / PC_PARTS), y1 = (int)((long long)s.bh * (blockIdx.x + 1) / PC_PARTS);
  double sum = 0;
  for (int y = y0 + (threadIdx.x >> 6); y < y1; y += 4)
    for (int x = 2 * (threadIdx.x & 63); x < s.bw; x += 512) {
      float2 v[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = pc_pair(s, src, x + 128 * i, y);
#pragma unroll
      for (int i = 0; i < 4; ++i) sum += (double)v[i].x + (double)v[i].y;
    }
  red[threadIdx.x] = sum;
  __syncthreads();
  for (int k = 128; k > 0; k >>= 1) {
    if (threadIdx.x < k) red[threadIdx.x] += red[threadIdx.x + k];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[(size_t)blockIdx.y * PC_PARTS + blockIdx.x] = red[0];
}

// stage 2: the partials of a frame in order, then the mean
__global__ void k_pc_mean_fin(const double* part, int bw, int bh, float* mean) {
  if (threadIdx.x != 0) return;
  double s = 0;
  for (int i = 0; i < PC_PARTS; ++i) s += part[(size_t)blockIdx.x * PC_PARTS + i];
  mean[blockIdx.x] = (float)(s / ((double)bw * bh));
}

// ---- the plane ------------------------------------------------------------------------------------
// float2 offset of row y, column k <= M / 2 of a half: strips of C = 1 << lc columns, column M / 2 after them
__device__ __forceinline__ size_t plane_at(int y, int k, int N, int M, int lc) {
  return k == M / 2 ? (size_t)N * (M / 2) + y : ((size_t)(k >> lc) * N + y) * (1 << lc) + (k & ((1 << lc) - 1));
}
__device__ __forceinline__ size_t half_size(int N, int M) { return (size_t)N * (M / 2 + 1); }

// forward FFTs of 1 << lr rows per block, grid (row groups, frames); rows from the first row past the
// image up to N are zero and are not written (k_pc_cols takes them as zero)
template <int LOGM>
__global__ void __launch_bounds__(512) k_pc_rows(PcSource s, const float* mean, const float* wx, const float* wy,
                                                 const float2* twg, float2* plane, int N, int lc, int lr) {
  constexpr int M = 1 << LOGM;
  extern __shared__ float2 lds[];
  float2* tw = lds;
  float2* buf = lds + TW_SIZE<LOGM>;
  const void* src = s.frames[blockIdx.y];
  const float mu = mean[blockIdx.y];
  const int rows = 1 << lr, y0 = blockIdx.x << lr, T = blockDim.x;
  const RowLayout<LOGM> L;
  tw_load<LOGM>(tw, twg);
  for (int i = threadIdx.x; i < rows * (M / 2); i += T) {
    const int r = i >> (LOGM - 1), x = 2 * (i & (M / 2 - 1)), y = y0 + r;
    const float2 a = pc_pair(s, src, x, y);
    const bool in0 = y < s.bh && x < s.bw, in1 = y < s.bh && x + 1 < s.bw;
    const float v = y < s.bh ? wy[y] : 0.f;
    buf[L.at(x, r)] = make_float2(in0 ? (a.x - mu) * (wx[x] * v) : 0.f, 0.f);
    buf[L.at(x + 1, r)] = make_float2(in1 ? (a.y - mu) * (wx[x + 1] * v) : 0.f, 0.f);
  }
  __syncthreads();
  fft_lds<LOGM, false>(buf, tw, rows, L);
  float2* out = plane + (size_t)blockIdx.y * 2 * half_size(N, M);
  const int C = 1 << lc;
  for (int i = threadIdx.x; i < rows * (M / 2); i += T) {
    // in plane order: column of the strip, row of the group, strip
    const int c = i & (C - 1), r = (i >> lc) & (rows - 1), k = ((i >> (lc + lr)) << lc) + c;
    if (y0 + r < s.bh) out[plane_at(y0 + r, k, N, M, lc)] = buf[L.at(k, r)];
  }
  for (int r = threadIdx.x; r < rows; r += T)
    if (y0 + r < s.bh) out[plane_at(y0 + r, M / 2, N, M, lc)] = buf[L.at(M / 2, r)];
}

// R = F conj(G) / |F conj(G)| times the gaussian weight exp(-2 pi^2 s^2 (kx^2 + ky^2)) that makes the
// correlation peak a gaussian of sigma s = 1 px
__device__ __forceinline__ float2 pc_cross(float2 f, float2 g, int ix, int iy, int M, int N) {
  const float re = fmaf(f.x, g.x, f.y * g.y), im = fmaf(f.y, g.x, -(f.x * g.y));
  const float mag = sqrtf(fmaf(re, re, im * im));
  const float kx = (float)(ix < M / 2 ? ix : ix - M) / (float)M, ky = (float)(iy < N / 2 ? iy : iy - N) / (float)N;
  const float wgt = expf(-2.f * 9.8696044f * fmaf(kx, kx, ky * ky));  // 2 pi^2 s^2, s = 1
  return mag > 0.f ? make_float2(re / mag * wgt, im / mag * wgt) : make_float2(0.f, 0.f);
}

// A strip of columns of a frame (the last block of a frame: column M / 2 alone): forward FFT, then either
// stored (the reference spectrum) or crossed with the reference's strip, inverse FFT and stored.  A strip
// is 128 KB (a CU's LDS but the twiddles) for the 64-B runs its 8 columns of 2048 rows give the row
// kernels; strips of one index run together over the frames of a launch and share the reference's in L2.
template <int LOGN>
__global__ void __launch_bounds__(1024) k_pc_cols(float2* plane, float2* ref, const float2* twg, int M, int lc_strip,
                                                  int rows_in, int store_only) {
  constexpr int N = 1 << LOGN;
  extern __shared__ float2 lds[];
  float2* tw = lds;
  float2* buf = lds + TW_SIZE<LOGN>;
  const int strip = blockIdx.y, T = blockDim.x;
  const bool last = strip == (M / 2) >> lc_strip;
  const int lc = last ? 0 : lc_strip, C = 1 << lc, points = N << lc, k0 = strip << lc_strip;
  const size_t at = last ? (size_t)N * (M / 2) : (size_t)strip * points;
  const StripLayout L{lc};
  float2* P = plane + (size_t)blockIdx.x * 2 * half_size(N, M) + at;
  float2* Rf = ref + at;
  tw_load<LOGN>(tw, twg);
  const int have = rows_in << lc;
  for (int i = threadIdx.x; i < points; i += T)
    buf[L.at(i >> lc, i & (C - 1))] = i < have ? P[i] : make_float2(0.f, 0.f);
  __syncthreads();
  fft_lds<LOGN, false>(buf, tw, C, L);
  if (store_only) {
    for (int i = threadIdx.x; i < points; i += T) Rf[i] = buf[L.at(i >> lc, i & (C - 1))];
    return;
  }
  for (int i = threadIdx.x; i < points; i += T) {
    const int y = i >> lc, c = i & (C - 1), a = L.at(y, c);
    buf[a] = pc_cross(buf[a], Rf[i], k0 + c, y, M, N);
  }
  __syncthreads();
  // the mirrored columns' cross power, R(M - kx, ky) = conj R(kx, -ky), waits in registers
  float2 mir[FFT_PPT];
#pragma unroll
  for (int q = 0; q < FFT_PPT; ++q) {
    const int i = (int)threadIdx.x + q * T;
    if (i < points) {
      const float2 u = buf[L.at((N - (i >> lc)) & (N - 1), i & (C - 1))];
      mir[q] = make_float2(u.x, -u.y);
    }
  }
  __syncthreads();
  constexpr float sc = 1.f / (float)N;
  auto store = [&](float2* D) {
    for (int i = threadIdx.x; i < points; i += T) {
      const float2 u = buf[L.at(i >> lc, i & (C - 1))];
      D[i] = make_float2(u.x * sc, u.y * sc);
    }
  };
  fft_lds<LOGN, true>(buf, tw, C, L);
  store(P);
  if (last) return;  // column M / 2 is its own mirror
  __syncthreads();
#pragma unroll
  for (int q = 0; q < FFT_PPT; ++q) {
    const int i = (int)threadIdx.x + q * T;
    if (i < points) buf[L.at(i >> lc, i & (C - 1))] = mir[q];
  }
  __syncthreads();
  fft_lds<LOGN, true>(buf, tw, C, L);
  store(P + half_size(N, M));
}

// the columns k and M - k of row y (strip order of the first half) into row r of buf
template <int LOGM>
__device__ __forceinline__ void get_row(float2* buf, const RowLayout<LOGM>& L, int r, const float2* in, int y, int k,
                                        int N, int lc) {
  constexpr int M = 1 << LOGM;
  const size_t o = plane_at(y, k, N, M, lc);
  buf[L.at(k, r)] = in[o];
  if (k != 0 && k != M / 2) buf[L.at(M - k, r)] = in[o + half_size(N, M)];
}

// inverse FFTs of 1 << lr rows per block and their largest value with its index (first on ties) as the
// group's partial; grid (N >> lr groups, frames)
template <int LOGM>
__global__ void __launch_bounds__(512) k_pc_rows_peak(const float2* plane, const float2* twg, int N, int lc, int lr,
                                                      float* pv, int* pi) {
  constexpr int M = 1 << LOGM;
  extern __shared__ float2 lds[];
  float2* tw = lds;
  float2* buf = lds + TW_SIZE<LOGM>;
  __shared__ float sv[512 / WAVE];
  __shared__ int si[512 / WAVE];
  const int rows = 1 << lr, y0 = blockIdx.x << lr, T = blockDim.x, C = 1 << lc;
  const RowLayout<LOGM> L;
  const float2* in = plane + (size_t)blockIdx.y * 2 * half_size(N, M);
  tw_load<LOGM>(tw, twg);
  for (int i = threadIdx.x; i < rows * (M / 2); i += T) {
    const int c = i & (C - 1), r = (i >> lc) & (rows - 1), k = ((i >> (lc + lr)) << lc) + c;
    get_row<LOGM>(buf, L, r, in, y0 + r, k, N, lc);
  }
  for (int r = threadIdx.x; r < rows; r += T) get_row<LOGM>(buf, L, r, in, y0 + r, M / 2, N, lc);
  __syncthreads();
  fft_lds<LOGM, true>(buf, tw, rows, L);
  float best = -3.4e38f;
  int bi = y0 * M;
  for (int i = threadIdx.x; i < rows * M; i += T) {
    const float v = buf[L.at(i & (M - 1), i >> LOGM)].x * (1.f / (float)M);
    if (v > best) {  // the index rises along the loop: the first of equal values stays
      best = v;
      bi = y0 * M + i;
    }
  }
  auto take = [&](float v, int j) {
    if (v > best || (v == best && j < bi)) {
      best = v;
      bi = j;
    }
  };
#pragma unroll
  for (int k = WAVE / 2; k > 0; k >>= 1) take(__shfl_xor(best, k), __shfl_xor(bi, k));
  if ((threadIdx.x & (WAVE - 1)) == 0) {
    sv[threadIdx.x / WAVE] = best;
    si[threadIdx.x / WAVE] = bi;
  }
  __syncthreads();
  if (threadIdx.x == 0)
    for (int q = 1; q < T / WAVE; ++q) take(sv[q], si[q]);
  if (threadIdx.x == 0) {
    pv[(size_t)blockIdx.y * gridDim.x + blockIdx.x] = best;
    pi[(size_t)blockIdx.y * gridDim.x + blockIdx.x] = bi;
  }
}

// per frame: the largest of the groups' partials (first index on ties), the peak's row and its neighbours
// once more through the inverse FFT, then the 3-point fits in FP64
template <int LOGM>
__global__ void __launch_bounds__(768) k_pc_peak(const float2* plane, const float2* twg, int N, int lc, int groups,
                                                 int binning, const float* pv, const int* pi, double* out) {
  constexpr int M = 1 << LOGM;
  extern __shared__ float2 lds[];
  float2* tw = lds;
  float2* buf = lds + TW_SIZE<LOGM>;
  __shared__ float sv[64];
  __shared__ int si[64];
  const int t = threadIdx.x, T = blockDim.x;
  if (t < 64) {
    float best = -INFINITY;
    int bi = 0x7fffffff;
    for (int g = t; g < groups; g += 64) {
      const float v = pv[(size_t)blockIdx.x * groups + g];
      const int j = pi[(size_t)blockIdx.x * groups + g];
      if (v > best || (v == best && j < bi)) {
        best = v;
        bi = j;
      }
    }
    sv[t] = best;
    si[t] = bi;
  }
  tw_load<LOGM>(tw, twg);
  __syncthreads();
  for (int k = 32; k > 0; k >>= 1) {
    if (t < k) {
      const float v = sv[t + k];
      const int j = si[t + k];
      if (v > sv[t] || (v == sv[t] && j < si[t])) {
        sv[t] = v;
        si[t] = j;
      }
    }
    __syncthreads();
  }
  const int py = si[0] / M, px = si[0] - py * M;
  const float2* in = plane + (size_t)blockIdx.x * 2 * half_size(N, M);
  const RowLayout<LOGM> L;
  const int ys[3] = {py, (py + N - 1) % N, (py + 1) % N};
  for (int k = t; k <= M / 2; k += T)
#pragma unroll
    for (int r = 0; r < 3; ++r) get_row<LOGM>(buf, L, r, in, ys[r], k, N, lc);
  __syncthreads();
  fft_lds<LOGM, true>(buf, tw, 3, L);
  if (t == 0) {
    auto at = [&](int r, int x) { return (double)(buf[L.at(x, r)].x * (1.f / (float)M)); };
    const double r0 = at(0, px);
    // gaussian fit: a parabola through the logarithms (a plain parabola if a value is not positive)
    auto fit = [](double a, double b, double c) {
      if (a > 0 && b > 0 && c > 0) {
        a = log(a);
        b = log(b);
        c = log(c);
      }
      const double d = a - 2.0 * b + c;
      return d == 0.0 ? 0.0 : 0.5 * (a - c) / d;
    };
    const double cx = fit(at(0, (px + M - 1) % M), r0, at(0, (px + 1) % M)), cy = fit(at(1, px), r0, at(2, px));
    const int sx = px > M / 2 ? px - M : px, sy = py > N / 2 ? py - N : py;
    out[3 * blockIdx.x + 0] = ((double)sx + cx) * binning;
    out[3 * blockIdx.x + 1] = ((double)sy + cy) * binning;
    out[3 * blockIdx.x + 2] = r0;
  }
}

int ilog2(int n) {
  int l = 0;
  while ((1 << l) < n) ++l;
  return l;
}

// log2 of the columns of a strip: 8 (64-B runs), but at most 16384 points (128 KB of LDS).  A frame's blocks are its
// strips, so short ones are what fills the chip where the planes are small: strips of 16384 points at every size
// (64 columns of 256 rows) were two blocks of a 256 x 256 plane, 39 us for two frames of 451 x 344 binned by 2, a call
// of 131 us; now 89 us (95 with one row per block in memory, as before the strips).  1024 x 1024: 16 frames 319 -> 292 us.
int strip_log2(int M, int N) { return std::min({3, ilog2(M) - 1, std::max(1, 14 - ilog2(N))}); }

size_t tw_size(int n) { return n > 4 ? (size_t)n / 4 * 3 : (size_t)n / 2; }  // TW_SIZE

// a radix-8 group per thread where the block is small (fewer rounds between two barriers), else two
int threads_for(int points, int most) {
  const int per = points < 8192 && points / 8 <= most ? 8 : FFT_PPT;
  return std::max(64, (points / per + 63) / 64 * 64);
}

template <class F>
hipError_t allow_lds(F f, size_t bytes) {
  return bytes > 65536 ? hipFuncSetAttribute((const void*)f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes)
                       : hipSuccess;
}

// calls f(integral_constant<log2 n>) for n = 4 .. 4096
template <class F>
hipError_t by_log2(int l, F f) {
  switch (l) {
#define SSG_CASE(K) case K: return f(std::integral_constant<int, K>{});
    SSG_CASE(2) SSG_CASE(3) SSG_CASE(4) SSG_CASE(5) SSG_CASE(6) SSG_CASE(7) SSG_CASE(8) SSG_CASE(9) SSG_CASE(10)
    SSG_CASE(11) SSG_CASE(12)
#undef SSG_CASE
  }
  return hipErrorInvalidValue;
}

}  // namespace

// 8192 complex points at the most (64 KB of LDS, two blocks per CU), at most 32 rows, and no more than the plane
// has; down to 4 rows while the launch is below two blocks per CU
int pc_rows_log2(int M, int N, int nframes) {
  int lr = std::min({5, 13 - ilog2(M), ilog2(N)});
  while (lr > 2 && (long long)nframes * (N >> lr) < 512) --lr;
  return lr;
}
size_t pc_plane(int M, int N) { return 2 * (size_t)N * (M / 2 + 1); }

hipError_t launch_pc_mean(const void* const* frames, bool u16, int pitch, bool wide, int bw, int bh, int binning,
                          float* mean, double* part, int nframes, hipStream_t s) {
  constexpr int MOST = 32768;  // frames per launch: a grid's second dimension ends at 65535
  for (int f0 = 0; f0 < nframes; f0 += MOST) {
    const int n = std::min(MOST, nframes - f0);
    const PcSource src{frames + f0, pitch, u16 ? 1 : 0, binning, wide ? 1 : 0, bw, bh};
    double* p = part + (size_t)PC_PARTS * f0;
    hipLaunchKernelGGL(k_pc_mean_part, dim3(PC_PARTS, n), dim3(256), 0, s, src, p);
    hipLaunchKernelGGL(k_pc_mean_fin, dim3(n), dim3(64), 0, s, p, bw, bh, mean + f0);
  }
  return hipGetLastError();
}

hipError_t launch_pc_rows(const void* const* frames, bool u16, int pitch, bool wide, int bw, int bh, int binning,
                          const float* mean, const float* wx, const float* wy, const float2* tw_m, float2* plane, int M,
                          int N, int nframes, hipStream_t s) {
  const PcSource src{frames, pitch, u16 ? 1 : 0, binning, wide ? 1 : 0, bw, bh};
  const int lr = pc_rows_log2(M, N, nframes), lc = strip_log2(M, N);
  const dim3 grid((bh + (1 << lr) - 1) >> lr, nframes);
  const size_t lds = sizeof(float2) * (tw_size(M) + ((size_t)M << lr));
  return by_log2(ilog2(M), [&](auto l) {
    const hipError_t e = allow_lds(k_pc_rows<decltype(l)::value>, lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_pc_rows<decltype(l)::value>, grid, dim3(threads_for(M << lr, 512)), lds, s, src, mean, wx, wy, tw_m,
                       plane, N, lc, lr);
    return hipGetLastError();
  });
}

hipError_t launch_pc_cols(float2* plane, float2* ref, const float2* tw_n, int M, int N, int bh, bool store_only,
                          int nframes, hipStream_t s) {
  const int lc = strip_log2(M, N);
  const size_t lds = sizeof(float2) * (tw_size(N) + ((size_t)N << lc));
  return by_log2(ilog2(N), [&](auto l) {
    const hipError_t e = allow_lds(k_pc_cols<decltype(l)::value>, lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_pc_cols<decltype(l)::value>, dim3(nframes, ((M / 2) >> lc) + 1), dim3(threads_for(N << lc, 1024)), lds,
                       s, plane, ref, tw_n, M, lc, bh, store_only ? 1 : 0);
    return hipGetLastError();
  });
}

hipError_t launch_pc_peak(const float2* plane, const float2* tw_m, int M, int N, int lr, int binning, int nframes,
                          float* pv, int* pi, double* out, hipStream_t s) {
  const int lc = strip_log2(M, N), groups = N >> lr;
  const size_t lds = sizeof(float2) * (tw_size(M) + ((size_t)M << lr));
  const size_t lds3 = sizeof(float2) * (tw_size(M) + 3 * (size_t)M);
  return by_log2(ilog2(M), [&](auto l) {
    hipError_t e = allow_lds(k_pc_rows_peak<decltype(l)::value>, lds);
    if (e == hipSuccess) e = allow_lds(k_pc_peak<decltype(l)::value>, lds3);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_pc_rows_peak<decltype(l)::value>, dim3(groups, nframes), dim3(threads_for(M << lr, 512)), lds, s,
                       plane, tw_m, N, lc, lr, pv, pi);
    hipLaunchKernelGGL(k_pc_peak<decltype(l)::value>, dim3(nframes), dim3(threads_for(3 * M, 768)), lds3, s, plane, tw_m, N, lc,
                       groups, binning, pv, pi, out);
    return hipGetLastError();
  });
}

}  // namespace ssg

// RMSNorm and fused residual-add + RMSNorm for gfx950.
//
// Semantics (reference src/fused_decode/reference.py:14-30):
//   rms:     y = round(x * rsqrt(mean(x^2) + eps) * w)
//   add_rms: s = x + r (float32); ro = round(s); y = round(s * rsqrt(mean(s^2) + eps) * w)
// The norm always sees the float32 sum, never the rounded residual.
//
// Four kernels:
//   rms_rows_kernel - unit column stride, rows of any alignment and n >= 8: n <= 256
//                     (several rows per wave) and what the next two don't take up
//                     to n = 8192.
//   rms_wave_kernel - unit column stride, n % 8 == 0, 16-byte aligned rows,
//                     n <= 8192: one wave per row, the row in registers.
//   rms_vec_kernel  - the same layouts for 8192 < n <= 16384: one 256-thread
//                     workgroup per row. Both make one HBM pass: every byte is read
//                     once and written once.
//   rms_gen_kernel  - any strides and any n: two passes over the row (the second
//                     pass re-reads through L2).
// Reduction: wave64 shuffles, then one LDS exchange across the workgroup's waves.
#include "fd_device.h"
#include "fd_gemv.h"
#include "fd_host.h"
#include "fd_internal.h"

namespace fd {

template <int NT>
__device__ __forceinline__ float block_sum(float v, float* red) {
  v = wave_sum(v);
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = threadIdx.x / kWave;
  constexpr int NWAVE = NT / kWave;
  if (NWAVE == 1) return v;
  __syncthreads();  // `red` may still be read from a previous call
  if (lane == 0) red[wave] = v;
  __syncthreads();
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < NWAVE; ++i) s += red[i];
  return s;
}

// T: activation type; W: weight type; VPT: 8-element vectors per thread.
template <typename T, typename W, int NT, int VPT, bool ADD>
__global__ __launch_bounds__(NT) void rms_vec_kernel(T* y, T* ro, const T* x, const T* r,
                                                     const W* __restrict__ w, RowGrid grid,
                                                     RowStrides lx, RowStrides lr,
                                                     RowStrides ly, RowStrides lro, int n,
                                                     float eps) {
  __shared__ float red[NT / kWave];
  const RowPos p = row_pos(grid, blockIdx.x);
  const T* xr = x + row_off(lx, p);
  const T* rr = ADD ? r + row_off(lr, p) : nullptr;
  float v[VPT][8];
  float ss = 0.f;
#pragma unroll
  for (int j = 0; j < VPT; ++j) {
    const int k = (j * NT + threadIdx.x) * 8;
    if (k < n) {
      typename Vec8<T>::type a = load8<T>(xr + k);
      if (ADD) {
        typename Vec8<T>::type b = load8<T>(rr + k);
#pragma unroll
        for (int i = 0; i < 8; ++i) v[j][i] = to_f32(a[i]) + to_f32(b[i]);
      } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) v[j][i] = to_f32(a[i]);
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) ss += v[j][i] * v[j][i];
    }
  }
  ss = block_sum<NT>(ss, red);
  const float inv = rsqrtf(ss / (float)n + eps);
  T* yr = y + row_off(ly, p);
  T* ror = ADD ? ro + row_off(lro, p) : nullptr;
#pragma unroll
  for (int j = 0; j < VPT; ++j) {
    const int k = (j * NT + threadIdx.x) * 8;
    if (k < n) {
      float wf[8];
      load8_f32<W>(w + k, wf);
      typename Vec8<T>::type o;
      if (ADD) {
        typename Vec8<T>::type s;
#pragma unroll
        for (int i = 0; i < 8; ++i) s[i] = from_f32<T>(v[j][i]);
        store8<T>(ror + k, s);
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) o[i] = from_f32<T>(v[j][i] * inv * wf[i]);
      store8<T>(yr + k, o);
    }
  }
}

// One wave per row, four rows per workgroup: the reduction is wave shuffles
// only, and each lane keeps VPL vectors of its row in registers. Activations
// stream through nontemporal loads and stores (read and written exactly once).
// The norm weight (n * sizeof(W) bytes, L2-resident, shared by every row) is
// staged once per workgroup in LDS: its loads go out before the row's, and the
// output pass reads it from LDS, so it holds no registers while the row loads
// are in flight. Without the residual the kernel is held to 64 VGPRs up to n =
// 4096 (the row packed, widened again in the output pass), so eight waves per
// SIMD keep every row of an 8192 x 4096 norm resident at once.
template <typename W>
__host__ __device__ constexpr int norm_w_chunks_per_thread(int vpl) {
  return vpl * (int)sizeof(W) / 8 > 0 ? vpl * (int)sizeof(W) / 8 : 1;  // n <= vpl * 512
}

template <typename T, typename W, int VPL, bool ADD>
__global__ __launch_bounds__(256, !ADD && VPL <= 8 ? 8 : 1) void rms_wave_kernel(T* y, T* ro, const T* x, const T* r,
                                                      const W* __restrict__ w, RowGrid grid,
                                                      RowStrides lx, RowStrides lr,
                                                      RowStrides ly, RowStrides lro, int n,
                                                      uint32_t rows, float eps) {
  typedef typename Vec8<T>::type V8;
  constexpr int WPT = norm_w_chunks_per_thread<W>(VPL);
  extern __shared__ __align__(16) u32x4 wsm[];  // the norm weight, n * sizeof(W) bytes
  const int wchunks = n * (int)sizeof(W) / 16;
  const u32x4* wsrc = reinterpret_cast<const u32x4*>(w);
  u32x4 wr[WPT];
#pragma unroll
  for (int i = 0; i < WPT; ++i) {
    const int c = threadIdx.x + i * 256;
    wr[i] = wsrc[c < wchunks ? c : 0];
  }
  const uint32_t row = blockIdx.x * 4 + threadIdx.x / kWave;
  const bool live = row < rows;  // the last workgroup's waves past the rows only stage the weight
  const int lane = threadIdx.x & (kWave - 1);
  const RowPos p = row_pos(grid, live ? row : 0);
  const T* xr = x + row_off(lx, p);
  const T* rr = ADD ? r + row_off(lr, p) : nullptr;
  V8 a[VPL], b[VPL];
#pragma unroll
  for (int j = 0; j < VPL; ++j) {
    const int k = (j * kWave + lane) * 8;
    if (live && k < n) {
      a[j] = load8_nt<T>(xr + k);
      if (ADD) b[j] = load8_nt<T>(rr + k);
    }
  }
#pragma unroll
  for (int i = 0; i < WPT; ++i) {
    const int c = threadIdx.x + i * 256;
    if (c < wchunks) wsm[c] = wr[i];
  }
  __syncthreads();
  if (!live) return;
  // rms: the row stays packed in registers and its packed pairs are squared
  // with v_dot2, so nothing is widened before the output pass; add_rms keeps
  // the float32 sums x + r and writes residual_out = round(sum) in the first
  // pass (it does not depend on the norm), so those stores overlap the reduction.
  float v[ADD ? VPL : 1][8];
  float ss = 0.f;
  T* ror = ADD ? ro + row_off(lro, p) : nullptr;
#pragma unroll
  for (int j = 0; j < VPL; ++j) {
    const int k = (j * kWave + lane) * 8;
    if (k >= n) continue;
    if constexpr (ADD) {
      V8 s;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        v[j][i] = to_f32(a[j][i]) + to_f32(b[j][i]);
        ss += v[j][i] * v[j][i];
        s[i] = from_f32<T>(v[j][i]);
      }
      __builtin_nontemporal_store(__builtin_bit_cast(u32x4, s), reinterpret_cast<u32x4*>(ror + k));
    } else {
      const u32x4 pk = __builtin_bit_cast(u32x4, a[j]);
#pragma unroll
      for (int i = 0; i < 4; ++i) ss = sq_dot2<T>(pk[i], ss);
    }
  }
  ss = wave_sum(ss);
  const float inv = rsqrtf(ss / (float)n + eps);
  T* yr = y + row_off(ly, p);
  const W* wl = reinterpret_cast<const W*>(wsm);
#pragma unroll
  for (int j = 0; j < VPL; ++j) {
    const int k = (j * kWave + lane) * 8;
    if (k < n) {
      Raw8<W> wv;
      wv.load(wl + k);
      V8 o;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float x = ADD ? v[ADD ? j : 0][i] : to_f32(a[j][i]);
        o[i] = from_f32<T>(x * inv * wv[i]);
      }
      __builtin_nontemporal_store(__builtin_bit_cast(u32x4, o), reinterpret_cast<u32x4*>(yr + k));
    }
  }
}

// LPR lanes per row (a power of two; 64 / LPR rows per wave), VPL vectors of 8 per
// lane, RPT rows per lane group, every row's loads issued before the first
// reduction. Vectors are loaded and stored as 2-byte aligned 16-byte words, which
// gfx950 does in one instruction at any address, so rows may start anywhere. Where
// n % 8 != 0 the last vector lies at n - 8: its first elements, which the vector
// before it holds too, are left out of the sum and written twice with one value
// (every load of a row comes before its first store, so in place as well).
//
// Short rows are why LPR varies: with a wave per row an attention head's norm (n =
// 128) uses 16 of 64 lanes and moves 512 bytes per wave before it ends. Of the 32
// query heads of 2048 tokens (float16, views of a QKV buffer, float32 weight): n =
// 64 / 80 / 128 / 256 13.8 / 14.5 / 15.1 / 17.2 us with a wave per row, 4.3 / 6.0 /
// 7.0 / 12.5 here (n = 128: 4.8 TB/s), and one token's in 2.0 either way. Rows that are not
// 16-byte aligned, which a workgroup per row reads twice in 2-byte loads: 2048 x 4097
// 15.9 -> 8.8 us, 8192 x 1025 18.5 -> 9.7, 4096 x 8191 68.8 -> 27.0, 65536 x 100 42.0
// -> 6.9, one row of 4097 6.1 -> 4.3. Aligned rows past 256 stay with the wave kernel,
// whose weights sit in LDS (4096 x 8192 23.0 us).
template <typename T, typename W, int LPR, int VPL, int RPT, bool ADD>
__global__ __launch_bounds__(256) void rms_rows_kernel(T* y, T* ro, const T* x, const T* r, const W* __restrict__ w,
                                                       RowGrid grid, RowStrides lx, RowStrides lr, RowStrides ly,
                                                       RowStrides lro, int n, uint32_t rows, float eps) {
  typedef typename Vec8<T>::type V8;
  constexpr int RPP = 256 / LPR;  // rows of a pass of the workgroup
  const int l = threadIdx.x % LPR;
  const int nv = (n + 7) / 8;
  int k[VPL], skip[VPL];  // first element; elements the vector before it has
  bool in[VPL];
#pragma unroll
  for (int j = 0; j < VPL; ++j) {
    const int v = j * LPR + l;
    in[j] = v < nv;
    k[j] = v * 8 + 8 <= n ? v * 8 : n - 8;
    skip[j] = v * 8 - k[j];
  }
  uint32_t row[RPT];
  V8 a[RPT][VPL], b[RPT][ADD ? VPL : 1];
#pragma unroll
  for (int t = 0; t < RPT; ++t) {
    row[t] = (blockIdx.x * RPT + t) * RPP + threadIdx.x / LPR;
    const RowPos p = row_pos(grid, row[t] < rows ? row[t] : 0);
    const T* xr = x + row_off(lx, p);
    const T* rr = ADD ? r + row_off(lr, p) : nullptr;
#pragma unroll
    for (int j = 0; j < VPL; ++j) {
      a[t][j] = load8_any<T>(xr + k[j]);
      if constexpr (ADD) b[t][j] = load8_any<T>(rr + k[j]);
    }
  }
  RawAny<W> wv[VPL];  // the lane's weights, the same for each of its rows
#pragma unroll
  for (int j = 0; j < VPL; ++j) wv[j].load(w + k[j]);
#pragma unroll
  for (int t = 0; t < RPT; ++t) {
    auto value = [&](int j, int i) {
      const float f = to_f32(a[t][j][i]);
      return ADD ? f + to_f32(b[t][ADD ? j : 0][i]) : f;
    };
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < VPL; ++j)
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float f = value(j, i), q = in[j] && i >= skip[j] ? f : 0.f;
        ss += q * q;
      }
    if constexpr (LPR >= 64) ss = xlane_sum<32>(ss);
    if constexpr (LPR >= 32) ss = xlane_sum<16>(ss);
    if constexpr (LPR >= 16) ss = xlane_sum<8>(ss);
    if constexpr (LPR >= 8) ss = xlane_sum<4>(ss);
    if constexpr (LPR >= 4) ss = xlane_sum<2>(ss);
    if constexpr (LPR >= 2) ss = xlane_sum<1>(ss);
    const float inv = rsqrtf(ss / (float)n + eps);
    const RowPos p = row_pos(grid, row[t]);
    T* yr = y + row_off(ly, p);
    T* ror = ADD ? ro + row_off(lro, p) : nullptr;
#pragma unroll
    for (int j = 0; j < VPL; ++j) {
      V8 o, s;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float f = value(j, i);
        o[i] = from_f32<T>(f * inv * wv[j][i]);
        if constexpr (ADD) s[i] = from_f32<T>(f);
      }
      if (in[j] && row[t] < rows) {
        if constexpr (ADD) store8_any<T>(ror + k[j], s);
        store8_any<T>(yr + k[j], o);
      }
    }
  }
}

template <typename T, bool ADD>
__global__ __launch_bounds__(256) void rms_gen_kernel(T* y, T* ro, const T* x, const T* r,
                                                      const void* __restrict__ w, int w_dtype,
                                                      int64_t w_stride, RowGrid grid,
                                                      RowStrides lx, RowStrides lr,
                                                      RowStrides ly, RowStrides lro, int64_t n,
                                                      float eps) {
  __shared__ float red[4];
  const RowPos p = row_pos(grid, blockIdx.x);
  const T* xr = x + row_off(lx, p);
  const T* rr = ADD ? r + row_off(lr, p) : nullptr;
  float ss = 0.f;
  for (int64_t k = threadIdx.x; k < n; k += 256) {
    float s = to_f32(xr[k * lx.col]);
    if (ADD) s += to_f32(rr[k * lr.col]);
    ss += s * s;
  }
  ss = block_sum<256>(ss, red);
  const float inv = rsqrtf(ss / (float)n + eps);
  T* yr = y + row_off(ly, p);
  T* ror = ADD ? ro + row_off(lro, p) : nullptr;
  for (int64_t k = threadIdx.x; k < n; k += 256) {
    float s = to_f32(xr[k * lx.col]);
    if (ADD) {
      s += to_f32(rr[k * lr.col]);
      ror[k * lro.col] = from_f32<T>(s);
    }
    yr[k * ly.col] = from_f32<T>(s * inv * load_any(w, w_dtype, k * w_stride));
  }
}

namespace {

template <typename T, typename W, int VPT, bool ADD>
void launch_vec(void* y, void* ro, const void* x, const void* r, const void* w,
                const fd_rows& lx, const fd_rows& lr, const fd_rows& ly, const fd_rows& lro,
                int64_t rows, float eps, hipStream_t st) {
  constexpr int NT = 256;
  hipLaunchKernelGGL((rms_vec_kernel<T, W, NT, VPT, ADD>), dim3((unsigned)rows), dim3(NT), 0,
                     st, static_cast<T*>(y), static_cast<T*>(ro), static_cast<const T*>(x),
                     static_cast<const T*>(r), static_cast<const W*>(w), row_grid(lx),
                     row_strides(lx), row_strides(lr), row_strides(ly), row_strides(lro),
                     (int)lx.n, eps);
}

template <typename T, typename W, int VPL, bool ADD>
void launch_wave(void* y, void* ro, const void* x, const void* r, const void* w,
                 const fd_rows& lx, const fd_rows& lr, const fd_rows& ly, const fd_rows& lro,
                 int64_t rows, float eps, hipStream_t st) {
  const size_t lds = (size_t)(lx.n * (int64_t)sizeof(W) + 15) / 16 * 16;  // the staged norm weight
  hipLaunchKernelGGL((rms_wave_kernel<T, W, VPL, ADD>), dim3((unsigned)((rows + 3) / 4)),
                     dim3(256), lds, st, static_cast<T*>(y), static_cast<T*>(ro),
                     static_cast<const T*>(x), static_cast<const T*>(r),
                     static_cast<const W*>(w), row_grid(lx), row_strides(lx), row_strides(lr),
                     row_strides(ly), row_strides(lro), (int)lx.n, (uint32_t)rows, eps);
}

template <typename T, typename W, int LPR, int VPL, int RPT, bool ADD>
void launch_rows_r(void* y, void* ro, const void* x, const void* r, const void* w, const fd_rows& lx,
                   const fd_rows& lr, const fd_rows& ly, const fd_rows& lro, int64_t rows, float eps,
                   hipStream_t st) {
  constexpr int per = 256 / LPR * RPT;
  hipLaunchKernelGGL((rms_rows_kernel<T, W, LPR, VPL, RPT, ADD>), dim3((unsigned)((rows + per - 1) / per)),
                     dim3(256), 0, st, static_cast<T*>(y), static_cast<T*>(ro), static_cast<const T*>(x),
                     static_cast<const T*>(r), static_cast<const W*>(w), row_grid(lx), row_strides(lx),
                     row_strides(lr), row_strides(ly), row_strides(lro), (int)lx.n, (uint32_t)rows, eps);
}

template <typename T, typename W, bool ADD>
void launch_rows(void* y, void* ro, const void* x, const void* r, const void* w, const fd_rows& lx,
                 const fd_rows& lr, const fd_rows& ly, const fd_rows& lro, int64_t rows, float eps, hipStream_t st) {
  const int64_t nv = (lx.n + 7) / 8;
#define FD_ROWS(LPR, VPL, RPT) launch_rows_r<T, W, LPR, VPL, RPT, ADD>(y, ro, x, r, w, lx, lr, ly, lro, rows, eps, st)
  // several rows per lane group once one each would already fill the GPU
#define FD_ROWS_SHORT(LPR)                                            \
  do {                                                                \
    if (rows >= (int64_t)device_cus() * 8 * (256 / LPR)) FD_ROWS(LPR, 1, 4); else FD_ROWS(LPR, 1, 1); \
  } while (0)
  if (nv <= 8) FD_ROWS_SHORT(8);
  else if (nv <= 16) FD_ROWS_SHORT(16);
  else if (nv <= 32) FD_ROWS_SHORT(32);
  else if (nv <= 64) FD_ROWS(64, 1, 1);
  else if (nv <= 128) FD_ROWS(64, 2, 1);
  else if (nv <= 192) FD_ROWS(64, 3, 1);
  else if (nv <= 256) FD_ROWS(64, 4, 1);
  else if (nv <= 384) FD_ROWS(64, 6, 1);
  else if (nv <= 512) FD_ROWS(64, 8, 1);
  else if (nv <= 768) FD_ROWS(64, 12, 1);
  else FD_ROWS(64, 16, 1);
#undef FD_ROWS_SHORT
#undef FD_ROWS
}

template <typename T, typename W, bool ADD>
void pick_vpt(void* y, void* ro, const void* x, const void* r, const void* w,
              const fd_rows& lx, const fd_rows& lr, const fd_rows& ly, const fd_rows& lro,
              int64_t rows, float eps, hipStream_t st) {
  // Rows up to 8192 elements: one wave per row (VPL vectors per lane).
  const int64_t lanes_vecs = (lx.n + 8 * kWave - 1) / (8 * kWave);
  if (lanes_vecs <= 2) {
    launch_wave<T, W, 2, ADD>(y, ro, x, r, w, lx, lr, ly, lro, rows, eps, st);
    return;
  }
  if (lanes_vecs <= 4) {
    launch_wave<T, W, 4, ADD>(y, ro, x, r, w, lx, lr, ly, lro, rows, eps, st);
    return;
  }
  if (lanes_vecs <= 8) {
    launch_wave<T, W, 8, ADD>(y, ro, x, r, w, lx, lr, ly, lro, rows, eps, st);
    return;
  }
  if (lanes_vecs <= 16) {
    launch_wave<T, W, 16, ADD>(y, ro, x, r, w, lx, lr, ly, lro, rows, eps, st);
    return;
  }
  const int64_t vecs = (lx.n + 8 * 256 - 1) / (8 * 256);
  if (vecs <= 1)
    launch_vec<T, W, 1, ADD>(y, ro, x, r, w, lx, lr, ly, lro, rows, eps, st);
  else if (vecs <= 2)
    launch_vec<T, W, 2, ADD>(y, ro, x, r, w, lx, lr, ly, lro, rows, eps, st);
  else if (vecs <= 4)
    launch_vec<T, W, 4, ADD>(y, ro, x, r, w, lx, lr, ly, lro, rows, eps, st);
  else
    launch_vec<T, W, 8, ADD>(y, ro, x, r, w, lx, lr, ly, lro, rows, eps, st);
}

template <typename T, bool ADD>
void dispatch_rows_w(int w_dtype, void* y, void* ro, const void* x, const void* r, const void* w, const fd_rows& lx,
                     const fd_rows& lr, const fd_rows& ly, const fd_rows& lro, int64_t rows, float eps,
                     hipStream_t st) {
  if (w_dtype == FD_F32)
    launch_rows<T, float, ADD>(y, ro, x, r, w, lx, lr, ly, lro, rows, eps, st);
  else if (w_dtype == FD_BF16)
    launch_rows<T, bf16, ADD>(y, ro, x, r, w, lx, lr, ly, lro, rows, eps, st);
  else
    launch_rows<T, f16, ADD>(y, ro, x, r, w, lx, lr, ly, lro, rows, eps, st);
}

template <typename T, bool ADD>
void dispatch_w(int w_dtype, void* y, void* ro, const void* x, const void* r, const void* w,
                const fd_rows& lx, const fd_rows& lr, const fd_rows& ly, const fd_rows& lro,
                int64_t rows, float eps, hipStream_t st) {
  if (w_dtype == FD_F32)
    pick_vpt<T, float, ADD>(y, ro, x, r, w, lx, lr, ly, lro, rows, eps, st);
  else if (w_dtype == FD_BF16)
    pick_vpt<T, bf16, ADD>(y, ro, x, r, w, lx, lr, ly, lro, rows, eps, st);
  else
    pick_vpt<T, f16, ADD>(y, ro, x, r, w, lx, lr, ly, lro, rows, eps, st);
}

constexpr int64_t kVecMaxN = 256 * 8 * 8;
constexpr int64_t kShortN = 256;    // rows of at most half a wave's vectors
constexpr int64_t kRowsMaxN = 8192;  // 16 vectors of 8 per lane

bool vec_ok(const void* p, const fd_rows& l, int elem) {
  return rows_vectorizable(p, l, elem) && l.n <= kVecMaxN;
}

int rms_common(bool add, void* y, void* ro, const void* x, const void* r, const void* w,
               int w_dtype, int64_t w_stride, const fd_rows* lx, const fd_rows* lr,
               const fd_rows* ly, const fd_rows* lro, float eps, int act_dtype, void* stream) {
  if (!check_act_dtype(act_dtype) || !check_any_dtype(w_dtype, "w_dtype")) return FD_EINVAL;
  if (!y || !x || !w || !lx || !ly) return set_error(FD_EINVAL, "null pointer argument");
  if (add && (!ro || !r || !lr || !lro)) return set_error(FD_EINVAL, "null residual argument");
  if (!check_rows(*lx, "x") || !check_rows(*ly, "out") || !same_grid(*lx, *ly, "out"))
    return FD_EINVAL;
  if (add && (!check_rows(*lr, "residual") || !check_rows(*lro, "residual_out") ||
              !same_grid(*lx, *lr, "residual") || !same_grid(*lx, *lro, "residual_out")))
    return FD_EINVAL;
  if (!(eps >= 0.f) || eps == INFINITY) return set_error(FD_EINVAL, "eps must be a finite value >= 0");
  const int64_t rows = lx->a * lx->b * lx->c;
  if (rows == 0 || lx->n == 0) return FD_OK;
  if (rows > 0x7fffffffLL) return set_error(FD_EUNSUPPORTED, "too many rows (>= 2^31)");
  hipStream_t st = static_cast<hipStream_t>(stream);
  const fd_rows& LR = add ? *lr : *lx;
  const fd_rows& LRO = add ? *lro : *ly;
  bool vec = vec_ok(x, *lx, 2) && vec_ok(y, *ly, 2) && w_stride == 1 &&
             (reinterpret_cast<uintptr_t>(w) % 16) == 0;
  if (add) vec = vec && vec_ok(r, *lr, 2) && vec_ok(ro, *lro, 2);
  // Rows of unit column stride that the wave kernels don't take, and the short
  // rows that they take with most lanes idle.
  const bool unit = lx->col == 1 && ly->col == 1 && (!add || (lr->col == 1 && lro->col == 1)) && w_stride == 1;
  const bool by_rows = unit && lx->n >= 8 && lx->n <= (vec ? kShortN : kRowsMaxN);
  if (by_rows) {
#define FD_RMS_ROWS(T, A) \
  dispatch_rows_w<T, A>(w_dtype, y, ro, x, r, w, *lx, LR, *ly, LRO, rows, eps, st)
    if (act_dtype == FD_F16) {
      if (add) FD_RMS_ROWS(f16, true); else FD_RMS_ROWS(f16, false);
    } else {
      if (add) FD_RMS_ROWS(bf16, true); else FD_RMS_ROWS(bf16, false);
    }
#undef FD_RMS_ROWS
  } else if (vec) {
    if (act_dtype == FD_F16) {
      if (add)
        dispatch_w<f16, true>(w_dtype, y, ro, x, r, w, *lx, LR, *ly, LRO, rows, eps, st);
      else
        dispatch_w<f16, false>(w_dtype, y, ro, x, r, w, *lx, LR, *ly, LRO, rows, eps, st);
    } else {
      if (add)
        dispatch_w<bf16, true>(w_dtype, y, ro, x, r, w, *lx, LR, *ly, LRO, rows, eps, st);
      else
        dispatch_w<bf16, false>(w_dtype, y, ro, x, r, w, *lx, LR, *ly, LRO, rows, eps, st);
    }
  } else {
#define FD_RMS_GEN(T, A)                                                                     \
  hipLaunchKernelGGL((rms_gen_kernel<T, A>), dim3((unsigned)rows), dim3(256), 0, st,         \
                     static_cast<T*>(y), static_cast<T*>(ro), static_cast<const T*>(x),      \
                     static_cast<const T*>(r), w, w_dtype, w_stride, row_grid(*lx),          \
                     row_strides(*lx), row_strides(LR), row_strides(*ly), row_strides(LRO),   \
                     lx->n, eps)
    if (act_dtype == FD_F16) {
      if (add) FD_RMS_GEN(f16, true); else FD_RMS_GEN(f16, false);
    } else {
      if (add) FD_RMS_GEN(bf16, true); else FD_RMS_GEN(bf16, false);
    }
#undef FD_RMS_GEN
  }
  return check_launch();
}

}  // namespace

int rms_rows(void* y, const void* x, const void* w, int w_dtype, int64_t rows, int64_t n,
             float eps, int act_dtype, hipStream_t st) {
  fd_rows l;
  l.a = 1;
  l.b = 1;
  l.c = rows;
  l.sa = 0;
  l.sb = 0;
  l.sc = n;
  l.col = 1;
  l.n = n;
  return rms_common(false, y, nullptr, x, nullptr, w, w_dtype, 1, &l, nullptr, &l, nullptr, eps,
                    act_dtype, st);
}

}  // namespace fd

extern "C" int fd_rms_norm(void* y, const void* x, const void* w, int w_dtype, int64_t w_stride,
                           const fd_rows* lx, const fd_rows* ly, float eps, int act_dtype,
                           void* stream) {
  return fd::rms_common(false, y, nullptr, x, nullptr, w, w_dtype, w_stride, lx, nullptr, ly,
                        nullptr, eps, act_dtype, stream);
}

extern "C" int fd_add_rms_norm(void* y, void* residual_out, const void* x, const void* residual,
                               const void* w, int w_dtype, int64_t w_stride, const fd_rows* lx,
                               const fd_rows* lr, const fd_rows* ly, const fd_rows* lro,
                               float eps, int act_dtype, void* stream) {
  return fd::rms_common(true, y, residual_out, x, residual, w, w_dtype, w_stride, lx, lr, ly,
                        lro, eps, act_dtype, stream);
}

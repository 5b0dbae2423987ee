// Streaming elementwise kernels for gfx950: SwiGLU and rotate-half RoPE.
//
// Both run on the row grid of fd_rows (up to three leading dims with arbitrary
// strides, including 0 for broadcast operands). The vector kernels move one
// 16-byte vector per operand per thread, with nontemporal loads and stores for
// the activations (each byte is touched once); the generic kernels take any
// column stride and any row length.
#include "fd_device.h"
#include "fd_gemv.h"
#include "fd_host.h"

namespace fd {

constexpr int kPwThreads = 256;

// Elements `skip` to 7 of a vector (skip 0: one store).
template <typename T>
__device__ __forceinline__ void store8_from(T* p, const typename Vec8<T>::type& v, uint32_t skip) {
  if (skip == 0) {
    store8_any<T>(p, v);
    return;
  }
#pragma unroll
  for (uint32_t i = 1; i < 8; ++i)
    if (i >= skip) p[i] = v[i];
}

// ---------------------------------------------------------------------------
// SwiGLU: y = round(silu(g) * u), float32 math (reference.py:33-35, stable sigmoid
// as kernels.py:448-451).

//
// Rows of unit column stride at any element address (one 16-byte word per operand
// and thread, aligned or not). Where n % 8 != 0 a row's last thread loads the 8
// elements up to its end and stores only those past the thread before it, so that
// no element one thread writes matters to another (the operation may be in place).
// Rows of 14335 by this kernel and element by element: 2048 of them 35.9 and 79.3
// us (14336: 29.6), 64 3.4 and 3.8, one 2.2 and 1.9; 2048 x 1025 4.6 and 7.0.
// ALIGNED (rows of whole, 16-byte aligned vectors) leaves the last thread's case
// out, which costs 1.2% at 2048 x 14336.
template <typename T, bool ALIGNED>
__global__ __launch_bounds__(kPwThreads) void swiglu_vec_kernel(T* y, const T* g, const T* u,
                                                                RowGrid grid, FastDiv vpr,
                                                                RowStrides sg, RowStrides su,
                                                                RowStrides sy, uint32_t total, uint32_t n) {
  const uint32_t v = blockIdx.x * kPwThreads + threadIdx.x;
  if (v >= total) return;
  uint32_t cv;
  const uint32_t row = vpr.divmod(v, cv);
  const uint32_t k = ALIGNED || cv * 8 + 8 <= n ? cv * 8 : n - 8;
  const RowPos p = row_pos(grid, row);
  typename Vec8<T>::type a, b, o;
  if constexpr (ALIGNED) {
    a = load8_nt<T>(g + row_off(sg, p) + k);
    b = load8_nt<T>(u + row_off(su, p) + k);
  } else {
    a = load8_any<T>(g + row_off(sg, p) + k);
    b = load8_any<T>(u + row_off(su, p) + k);
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) o[i] = from_f32<T>(silu_stable(to_f32(a[i])) * to_f32(b[i]));
  if constexpr (ALIGNED)
    store8_nt<T>(y + row_off(sy, p) + k, o);
  else
    store8_from<T>(y + row_off(sy, p) + k, o, cv * 8 - k);
}

template <typename T>
__global__ __launch_bounds__(kPwThreads) void swiglu_gen_kernel(T* y, const T* g, const T* u,
                                                                RowGrid grid, FastDiv n,
                                                                RowStrides sg, RowStrides su,
                                                                RowStrides sy, uint32_t total) {
  const uint32_t e = blockIdx.x * kPwThreads + threadIdx.x;
  if (e >= total) return;
  uint32_t k;
  const uint32_t row = n.divmod(e, k);
  const RowPos p = row_pos(grid, row);
  const float a = to_f32(g[row_off(sg, p) + (int64_t)k * sg.col]);
  const float b = to_f32(u[row_off(su, p) + (int64_t)k * su.col]);
  y[row_off(sy, p) + (int64_t)k * sy.col] = from_f32<T>(silu_stable(a) * b);
}

// ---------------------------------------------------------------------------
// y = round(a + r) in float32: the residual of a product that another library
// wrote (row_add above the GEMV's rows, kernels.py:657-672 order), in one pass
// where float32 copies of both operands, their sum and its rounding take four
// (777 x 4096 float16: 27 -> 5.7 us). Rows as swiglu_vec_kernel's; r may
// have any strides (0 = broadcast) and dtype.
template <typename T, typename R>
__global__ __launch_bounds__(kPwThreads) void add_rows_kernel(T* y, const T* a, const R* r, RowGrid grid,
                                                              FastDiv vpr, RowStrides sa, RowStrides sr,
                                                              RowStrides sy, uint32_t n, uint32_t total) {
  const uint32_t v = blockIdx.x * kPwThreads + threadIdx.x;
  if (v >= total) return;
  uint32_t cv;
  const uint32_t row = vpr.divmod(v, cv);
  const uint32_t k = cv * 8;
  const RowPos p = row_pos(grid, row);
  const T* ar = a + row_off(sa, p);
  const R* rr = r + row_off(sr, p);
  T* yr = y + row_off(sy, p);
  if (n < 8 || sr.col != 1) {
    const uint32_t end = n < k + 8 ? n : k + 8;
    for (uint32_t i = k; i < end; ++i) yr[i] = from_f32<T>(to_f32(ar[i]) + to_f32(rr[i * sr.col]));
    return;
  }
  const uint32_t kc = k + 8 <= n ? k : n - 8;
  const typename Vec8<T>::type x = load8_any<T>(ar + kc);
  RawAny<R> q;
  q.load(rr + kc);
  typename Vec8<T>::type o;
#pragma unroll
  for (int i = 0; i < 8; ++i) o[i] = from_f32<T>(to_f32(x[i]) + q[i]);
  store8_from<T>(yr + kc, o, k - kc);
}

// ---------------------------------------------------------------------------
// RoPE, rotate-half pairing (reference.py:38-47):
//   y[j]     = x[j] * c[j]     - x[j+h] * s[j]
//   y[j + h] = x[j+h] * c[j+h] + x[j] * s[j+h]

// HPT rows per thread: when cos/sin do not vary along the innermost row dim
// (stride 0 there, e.g. one table row shared by all heads of a token), a thread
// handles HPT consecutive rows of that dim and loads its cos/sin vectors once.
template <typename T, typename C, int HPT>
__global__ __launch_bounds__(kPwThreads) void rope_vec_kernel(T* y, const T* x, const C* cs,
                                                              const C* sn, RowGrid grid,
                                                              FastDiv vpr, RowStrides sx,
                                                              RowStrides sc, RowStrides ss,
                                                              RowStrides sy, uint32_t h,
                                                              uint32_t total) {
  const uint32_t v = blockIdx.x * kPwThreads + threadIdx.x;
  if (v >= total) return;
  uint32_t jv;
  const uint32_t grp = vpr.divmod(v, jv);
  const uint32_t j = jv * 8;
  const RowPos p = row_pos(grid, grp * HPT);
  const C* cr = cs + row_off(sc, p);
  const C* sr = sn + row_off(ss, p);
  float c1[8], c2[8], s1[8], s2[8];
  load8_f32<C>(cr + j, c1);
  load8_f32<C>(cr + j + h, c2);
  load8_f32<C>(sr + j, s1);
  load8_f32<C>(sr + j + h, s2);
  const T* xr = x + row_off(sx, p);
  T* yr = y + row_off(sy, p);
  typename Vec8<T>::type x1[HPT], x2[HPT];
#pragma unroll
  for (int t = 0; t < HPT; ++t) {
    x1[t] = load8_nt<T>(xr + t * sx.sc + j);
    x2[t] = load8_nt<T>(xr + t * sx.sc + j + h);
  }
#pragma unroll
  for (int t = 0; t < HPT; ++t) {
    typename Vec8<T>::type o1, o2;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float a = to_f32(x1[t][i]), b = to_f32(x2[t][i]);
      o1[i] = from_f32<T>(a * c1[i] - b * s1[i]);
      o2[i] = from_f32<T>(b * c2[i] + a * s2[i]);
    }
    store8_nt<T>(yr + t * sy.sc + j, o1);
    store8_nt<T>(yr + t * sy.sc + j + h, o2);
  }
}

template <typename T>
__global__ __launch_bounds__(kPwThreads) void rope_gen_kernel(T* y, const T* x, const void* cs,
                                                              const void* sn, int cs_dtype,
                                                              RowGrid grid, FastDiv hd,
                                                              RowStrides sx, RowStrides sc,
                                                              RowStrides ss, RowStrides sy,
                                                              uint32_t total) {
  const uint32_t e = blockIdx.x * kPwThreads + threadIdx.x;
  if (e >= total) return;
  uint32_t j;
  const uint32_t row = hd.divmod(e, j);
  const int64_t h = hd.d;
  const RowPos p = row_pos(grid, row);
  const T* xr = x + row_off(sx, p);
  const int64_t cb = row_off(sc, p), sb = row_off(ss, p);
  const float a = to_f32(xr[j * sx.col]);
  const float b = to_f32(xr[(j + h) * sx.col]);
  const float c1 = load_any(cs, cs_dtype, cb + j * sc.col);
  const float c2 = load_any(cs, cs_dtype, cb + (j + h) * sc.col);
  const float s1 = load_any(sn, cs_dtype, sb + j * ss.col);
  const float s2 = load_any(sn, cs_dtype, sb + (j + h) * ss.col);
  T* yr = y + row_off(sy, p);
  yr[j * sy.col] = from_f32<T>(a * c1 - b * s1);
  yr[(j + h) * sy.col] = from_f32<T>(b * c2 + a * s2);
}

namespace {

// Work items (vectors, elements or pairs) of one launch are counted in 32 bits.
constexpr int64_t kMaxPwWork = 0xffffffffLL - kPwThreads;

inline unsigned blocks_for(int64_t work) {
  return (unsigned)((work + kPwThreads - 1) / kPwThreads);
}

// Row layout with the last dim halved: the vector rope kernel addresses pairs
// (j, j+h), so alignment is needed at both j and h.
inline bool rope_rows_vec(const void* p, const fd_rows& l, int elem) {
  fd_rows half = l;
  half.n = l.n / 2;
  return rows_vectorizable(p, half, elem);
}

}  // namespace
}  // namespace fd

using namespace fd;

extern "C" int fd_swiglu(void* y, const void* gate, const void* up, const fd_rows* lg,
                         const fd_rows* lu, const fd_rows* ly, int act_dtype, void* stream) {
  if (!check_act_dtype(act_dtype)) return FD_EINVAL;
  if (!y || !gate || !up || !lg || !lu || !ly) return set_error(FD_EINVAL, "null pointer argument");
  if (!check_rows(*lg, "gate") || !check_rows(*lu, "up") || !check_rows(*ly, "out") ||
      !same_grid(*lg, *lu, "up") || !same_grid(*lg, *ly, "out"))
    return FD_EINVAL;
  const int64_t rows = lg->a * lg->b * lg->c;
  const int64_t total = rows * lg->n;
  if (total == 0) return FD_OK;
  if (total > kMaxPwWork) return set_error(FD_EUNSUPPORTED, "swiglu tensor too large (>= 2^32 elements)");
  hipStream_t st = static_cast<hipStream_t>(stream);
  const RowGrid grid = row_grid(*lg);
  const bool aligned = rows_vectorizable(gate, *lg, 2) && rows_vectorizable(up, *lu, 2) &&
                       rows_vectorizable(y, *ly, 2);
  // other rows in vectors too once these make a workgroup for every CU; below,
  // the per-element kernel's eight times as many threads finish sooner
  const bool vec = aligned || (lg->col == 1 && lu->col == 1 && ly->col == 1 && lg->n >= 8 &&
                               total >= (int64_t)8 * kPwThreads * device_cus());
  if (vec) {
    const uint32_t vectors = (uint32_t)((lg->n + 7) / 8), tv = (uint32_t)rows * vectors;
    const FastDiv vpr(vectors);
#define FD_SWIGLU_VEC(T, A)                                                                    \
  hipLaunchKernelGGL((swiglu_vec_kernel<T, A>), dim3(blocks_for(tv)), dim3(kPwThreads), 0, st, \
                     (T*)y, (const T*)gate, (const T*)up, grid, vpr, row_strides(*lg),         \
                     row_strides(*lu), row_strides(*ly), tv, (uint32_t)lg->n)
    if (act_dtype == FD_F16) {
      if (aligned) FD_SWIGLU_VEC(f16, true); else FD_SWIGLU_VEC(f16, false);
    } else {
      if (aligned) FD_SWIGLU_VEC(bf16, true); else FD_SWIGLU_VEC(bf16, false);
    }
#undef FD_SWIGLU_VEC
  } else {
    const FastDiv nd((uint32_t)lg->n);
#define FD_SWIGLU_GEN(T)                                                                       \
  hipLaunchKernelGGL(swiglu_gen_kernel<T>, dim3(blocks_for(total)), dim3(kPwThreads), 0, st,   \
                     (T*)y, (const T*)gate, (const T*)up, grid, nd, row_strides(*lg),          \
                     row_strides(*lu), row_strides(*ly), (uint32_t)total)
    if (act_dtype == FD_F16) FD_SWIGLU_GEN(f16); else FD_SWIGLU_GEN(bf16);
#undef FD_SWIGLU_GEN
  }
  return check_launch();
}

extern "C" int fd_add_rows(void* y, const void* a, const void* r, int r_dtype, const fd_rows* la,
                           const fd_rows* lr, const fd_rows* ly, int act_dtype, void* stream) {
  if (!check_act_dtype(act_dtype) || !check_any_dtype(r_dtype, "r_dtype")) return FD_EINVAL;
  if (!y || !a || !r || !la || !lr || !ly) return set_error(FD_EINVAL, "null pointer argument");
  if (!check_rows(*la, "a") || !check_rows(*lr, "r") || !check_rows(*ly, "out") || !same_grid(*la, *lr, "r") ||
      !same_grid(*la, *ly, "out"))
    return FD_EINVAL;
  const int64_t rows = la->a * la->b * la->c, vectors = (la->n + 7) / 8;
  if (rows == 0 || la->n == 0) return FD_OK;
  if (la->n > 1 && (la->col != 1 || ly->col != 1))
    return set_error(FD_EUNSUPPORTED, "a and out need unit column stride");
  if (rows > kMaxPwWork || vectors > kMaxPwWork / rows || la->n > kMaxPwWork)
    return set_error(FD_EUNSUPPORTED, "tensor too large");
  auto span = [](const fd_rows& l, int dt) {
    return ((l.a - 1) * l.sa + (l.b - 1) * l.sb + (l.c - 1) * l.sc + (l.n - 1) * l.col + 1) * dtype_bytes(dt);
  };
  // r may be y element for element (a dim of one has no stride); any other overlap is read after it is written
  auto same = [](int64_t dim, int64_t s, int64_t t) { return dim == 1 || s == t; };
  if (overlaps(y, span(*ly, act_dtype), r, span(*lr, r_dtype)) &&
      !(y == r && act_dtype == r_dtype && same(ly->a, ly->sa, lr->sa) && same(ly->b, ly->sb, lr->sb) &&
        same(ly->c, ly->sc, lr->sc) && same(ly->n, ly->col, lr->col)))
    return set_error(FD_EUNSUPPORTED, "y must not overlap r, other than as r itself");
  hipStream_t st = static_cast<hipStream_t>(stream);
  const uint32_t tv = (uint32_t)(rows * vectors);
#define FD_ADD_ROWS(T, R)                                                                                    \
  hipLaunchKernelGGL((add_rows_kernel<T, R>), dim3(blocks_for(tv)), dim3(kPwThreads), 0, st, (T*)y,          \
                     (const T*)a, (const R*)r, row_grid(*la), FastDiv((uint32_t)vectors), row_strides(*la), \
                     row_strides(*lr), row_strides(*ly), (uint32_t)la->n, tv)
#define FD_ADD_ROWS_R(T)                                 \
  do {                                                   \
    if (r_dtype == FD_F32) FD_ADD_ROWS(T, float);        \
    else if (r_dtype == FD_BF16) FD_ADD_ROWS(T, bf16);   \
    else FD_ADD_ROWS(T, f16);                            \
  } while (0)
  if (act_dtype == FD_F16) FD_ADD_ROWS_R(f16); else FD_ADD_ROWS_R(bf16);
#undef FD_ADD_ROWS_R
#undef FD_ADD_ROWS
  return check_launch();
}

extern "C" int fd_rope(void* y, const void* x, const void* cos, const void* sin, int cs_dtype,
                       const fd_rows* lx, const fd_rows* lc, const fd_rows* ls,
                       const fd_rows* ly, int act_dtype, void* stream) {
  if (!check_act_dtype(act_dtype) || !check_any_dtype(cs_dtype, "cs_dtype")) return FD_EINVAL;
  if (!y || !x || !cos || !sin || !lx || !lc || !ls || !ly)
    return set_error(FD_EINVAL, "null pointer argument");
  if (!check_rows(*lx, "x") || !check_rows(*lc, "cos") || !check_rows(*ls, "sin") ||
      !check_rows(*ly, "out") || !same_grid(*lx, *lc, "cos") || !same_grid(*lx, *ls, "sin") ||
      !same_grid(*lx, *ly, "out"))
    return FD_EINVAL;
  if (lx->n % 2 != 0) return set_error(FD_EINVAL, "rope last dimension must be even");
  const int64_t rows = lx->a * lx->b * lx->c;
  const int64_t h = lx->n / 2;
  const int64_t total = rows * h;
  if (total == 0) return FD_OK;
  if (total > kMaxPwWork) return set_error(FD_EUNSUPPORTED, "rope tensor too large (>= 2^32 pairs)");
  hipStream_t st = static_cast<hipStream_t>(stream);
  const RowGrid grid = row_grid(*lx);
  const int cse = cs_dtype == FD_F32 ? 4 : 2;
  const bool vec = rope_rows_vec(x, *lx, 2) && rope_rows_vec(y, *ly, 2) &&
                   rope_rows_vec(cos, *lc, cse) && rope_rows_vec(sin, *ls, cse);
  if (vec) {
    // rows sharing cos/sin along the innermost row dim are handled 4 per thread
    const int hpt = (lc->sc == 0 && ls->sc == 0 && lx->c % 4 == 0) ? 4 : 1;
    const uint32_t tv = (uint32_t)(total / 8 / hpt);
    const FastDiv vpr((uint32_t)(h / 8));
#define FD_ROPE_VEC(T, C)                                                                       \
  do {                                                                                          \
  if (hpt == 4)                                                                                 \
    hipLaunchKernelGGL((rope_vec_kernel<T, C, 4>), dim3(blocks_for(tv)), dim3(kPwThreads), 0,   \
                       st, (T*)y, (const T*)x, (const C*)cos, (const C*)sin, grid, vpr,         \
                       row_strides(*lx), row_strides(*lc), row_strides(*ls), row_strides(*ly),  \
                       (uint32_t)h, tv);                                                        \
  else                                                                                          \
    hipLaunchKernelGGL((rope_vec_kernel<T, C, 1>), dim3(blocks_for(tv)), dim3(kPwThreads), 0,   \
                       st, (T*)y, (const T*)x, (const C*)cos, (const C*)sin, grid, vpr,         \
                       row_strides(*lx), row_strides(*lc), row_strides(*ls), row_strides(*ly),  \
                       (uint32_t)h, tv);                                                        \
  } while (0)
    if (act_dtype == FD_F16) {
      if (cs_dtype == FD_F32) FD_ROPE_VEC(f16, float);
      else if (cs_dtype == FD_BF16) FD_ROPE_VEC(f16, bf16);
      else FD_ROPE_VEC(f16, f16);
    } else {
      if (cs_dtype == FD_F32) FD_ROPE_VEC(bf16, float);
      else if (cs_dtype == FD_BF16) FD_ROPE_VEC(bf16, bf16);
      else FD_ROPE_VEC(bf16, f16);
    }
#undef FD_ROPE_VEC
  } else {
    const FastDiv hd((uint32_t)h);
#define FD_ROPE_GEN(T)                                                                         \
  hipLaunchKernelGGL(rope_gen_kernel<T>, dim3(blocks_for(total)), dim3(kPwThreads), 0, st,     \
                     (T*)y, (const T*)x, cos, sin, cs_dtype, grid, hd, row_strides(*lx),       \
                     row_strides(*lc), row_strides(*ls), row_strides(*ly), (uint32_t)total)
    if (act_dtype == FD_F16) FD_ROPE_GEN(f16); else FD_ROPE_GEN(bf16);
#undef FD_ROPE_GEN
  }
  return check_launch();
}

// GEMV (M <= 16) with the weight stored [K, N]: linear_decode on a transposed view,
// e.g. a checkpoint that keeps its projections as [in, out].
//
//   y[m,n] = round(sum_k x[m,k] * w[k,n] + bias[n] + row_add[m,n])
//
// Streaming again: every weight byte once from HBM. A lane loads 16 bytes, 8
// columns of one k; 32 lanes cover the workgroup's 256 columns (512 bytes of a
// weight row) and the wave's two lane groups two k pairs. The two rows of a pair
// are interleaved into (k, k+1) halves (v_perm) and folded against x[m, k..k+1]
// with v_dot2, the exact products and float32 sums of the [N, K] kernels. x sits
// in LDS as [k pair][row], so a lane reads its pair's rows as 16-byte vectors.
// N / 256 workgroups are too few for the GPU at the decode widths, so K is split
// over workgroups too, whose float32 sums go through caller scratch and a second
// launch, added in order.
//
// What bounds it, with cold weights in a graph: the weight stream up to 4 rows, the
// perms and v_dot2s beside it from 8. bfloat16, 1 / 4 / 8 / 16 rows: N = K = 4096
// 11.0 / 11.8 / 13.3 / 15.3 us, of which the sum 2.9; N = 4096, K = 14336 22.9 /
// 23.7 / 25.4 / 32.1; N = 28672, K = 4096 40.0 / 41.1 / 42.6 / 59.2. The kernel for
// any strides, which reads 2 bytes of every 128-byte line per workgroup, takes
// 118 at N = K = 4096. Narrower tiles are slower (4 rows, K = 14336: 128 columns
// 24.9, 64 columns 25.8; N = 28672: 44.7, 48.5): shorter runs of each weight row.
#include "fd_gemv.h"

namespace fd {


constexpr int kKnCols = 256;              // columns of a tile
constexpr int kKnLanes = kKnCols / 8;     // lanes of a weight row
constexpr int kKnGroups = kWave / kKnLanes;  // k pairs of a wave's load
static_assert(kKnGroups == 2, "the final exchange is one step");

// k pairs a lane holds of one x stage, and that stage's k (8 waves of two lane
// groups): two buffers of 8 * pairs registers beside the 8 * MB sums.
constexpr int kn_pairs(int mb) { return mb <= 8 ? 4 : 2; }
constexpr int kn_chunk(int mb) { return 2 * kn_pairs(mb) * kMaxWaves * kKnGroups; }

__device__ __forceinline__ float kn_dot2(uint32_t a, uint32_t b, float acc, f16) {
  return __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2, a), __builtin_bit_cast(f16x2, b), acc, false);
}
__device__ __forceinline__ float kn_dot2(uint32_t a, uint32_t b, float acc, bf16) {
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, a), __builtin_bit_cast(bf16x2, b), acc, false);
}

// MB: activation rows held (M rounded up; the others are zero and never stored).
// PART: float32 sums of this K split to `partial` [split][M][N], else the output.
template <typename T, int MB, bool PART>
__global__ __launch_bounds__(kMaxWaves * kWave) void gemv_kn_kernel(T* y, float* partial, const T* x, const T* w,
                                                                    int M, int N, int K, int64_t sxm, int64_t sxk,
                                                                    int64_t swk, int64_t sym, int64_t syn, Epi e,
                                                                    int tiles, int splits, bool xvec) {
  constexpr int XV = MB < 4 ? MB : 4;  // rows of one LDS read
  constexpr int NP = kn_pairs(MB), CHUNK = kn_chunk(MB);
  typedef uint32_t xvec_t __attribute__((ext_vector_type(XV)));
  __shared__ __align__(16) uint32_t xs[2][CHUNK / 2 * MB];
  __shared__ __align__(16) float part[kMaxWaves * MB * kKnCols];
  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int grp = lane / kKnLanes, chunk = lane % kKnLanes;
  const int tile = (int)blockIdx.x % tiles, split = (int)blockIdx.x / tiles;
  const int chunks = (K + CHUNK - 1) / CHUNK;
  const int c0 = (int)((int64_t)chunks * split / splits), c1 = (int)((int64_t)chunks * (split + 1) / splits);
  const int col = tile * kKnCols + chunk * 8;
  const T* wc = w + (col < N ? col : 0);  // columns past N (a multiple of 8): never stored

  // pair i of this lane in a chunk: k = 2 * ((i * kMaxWaves + wave) * kKnGroups + grp)
  struct Rows {
    u32x4 a[NP], b[NP];
  };
  auto issue = [&](Rows& q, int c) {
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int k = c * CHUNK + 2 * ((i * kMaxWaves + wave) * kKnGroups + grp);
      q.a[i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(wc + (int64_t)(k < K ? k : 0) * swk));
      q.b[i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(wc + (int64_t)(k + 1 < K ? k + 1 : 0) * swk));
    }
  };
  // stage chunk c of x: thread -> row m = t % MB, 8 k from 8 * (t / MB); zeros past M and K
  constexpr int OCT = CHUNK / 8;                                     // 8-k groups of a chunk
  constexpr int PER = (OCT * MB + kMaxWaves * kWave - 1) / (kMaxWaves * kWave);  // per thread
  auto load_x = [&](u32x4 (&v)[PER], int c) {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int t = tid + i * kMaxWaves * kWave;
      const int m = t % MB, k = c * CHUNK + 8 * (t / MB);
      const bool in = t < OCT * MB && m < M;
      v[i] = u32x4{0u, 0u, 0u, 0u};
      if (in && xvec && k + 8 <= K) {
        v[i] = *reinterpret_cast<const u32x4*>(x + m * sxm + k);
      } else if (in) {
        typename Vec8<T>::type o = __builtin_bit_cast(typename Vec8<T>::type, v[i]);
#pragma unroll
        for (int j = 0; j < 8; ++j)
          if (k + j < K) o[j] = x[m * sxm + (k + j) * sxk];
        v[i] = __builtin_bit_cast(u32x4, o);
      }
    }
  };
  auto store_x = [&](const u32x4 (&v)[PER], int buf) {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int t = tid + i * kMaxWaves * kWave;
      const int m = t % MB, p = 4 * (t / MB);
      if (t < OCT * MB) {
#pragma unroll
        for (int j = 0; j < 4; ++j) xs[buf][(p + j) * MB + m] = v[i][j];
      }
    }
  };

  float acc[8][MB];
#pragma unroll
  for (int j = 0; j < 8; ++j)
#pragma unroll
    for (int m = 0; m < MB; ++m) acc[j][m] = 0.f;
  auto consume = [&](const Rows& q, int c, int buf) {
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int p = (i * kMaxWaves + wave) * kKnGroups + grp, k = c * CHUNK + 2 * p;
      u32x4 a = q.a[i], b = q.b[i];
      if (c * CHUNK + CHUNK > K) {  // the last chunk: rows past K are zero
        if (k >= K) a = u32x4{0u, 0u, 0u, 0u};
        if (k + 1 >= K) b = u32x4{0u, 0u, 0u, 0u};
      }
      uint32_t pr[8];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        pr[2 * j] = __builtin_amdgcn_perm(b[j], a[j], 0x05040100u);
        pr[2 * j + 1] = __builtin_amdgcn_perm(b[j], a[j], 0x07060302u);
      }
#pragma unroll
      for (int m = 0; m < MB; m += XV) {
        const xvec_t xv = *reinterpret_cast<const xvec_t*>(&xs[buf][p * MB + m]);
#pragma unroll
        for (int h = 0; h < XV; ++h)
#pragma unroll
          for (int j = 0; j < 8; ++j) acc[j][m + h] = kn_dot2(pr[j], xv[h], acc[j][m + h], T{});
      }
    }
  };

  Rows qa, qb;
  u32x4 xr[PER];
  if (c0 < c1) {
    load_x(xr, c0);
    issue(qa, c0);
    store_x(xr, 0);
  }
  auto step = [&](Rows& cur, Rows& nxt, int c) {
    const int buf = (c - c0) & 1;
    const bool more = c + 1 < c1;
    if (more) {
      load_x(xr, c + 1);
      issue(nxt, c + 1);
    }
    __syncthreads();  // chunk c's x is in xs[buf]; every wave is done with chunk c - 1's
    consume(cur, c, buf);
    if (more) store_x(xr, buf ^ 1);
  };
  for (int c = c0; c < c1; c += 2) {
    step(qa, qb, c);
    if (c + 1 < c1) step(qb, qa, c + 1);
  }

  // the two lane groups: each keeps half of its lanes' 8 columns
#pragma unroll
  for (int m = 0; m < MB; ++m) {
    f32x4 v;
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = xlane_keep_sum<32>(acc[j][m], acc[j + 4][m], lane);
    *reinterpret_cast<f32x4*>(&part[(wave * MB + m) * kKnCols + chunk * 8 + grp * 4]) = v;
  }
  __syncthreads();
  for (int t = tid; t < M * kKnCols; t += kMaxWaves * kWave) {
    const int m = t / kKnCols, n = tile * kKnCols + t % kKnCols;
    if (n >= N) continue;
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < kMaxWaves; ++i) sum += part[(i * MB + m) * kKnCols + t % kKnCols];
    if constexpr (PART)
      partial[((int64_t)split * M + m) * N + n] = sum;
    else
      y[m * sym + n * syn] = from_f32<T>(epilogue(e, sum, m, n));
  }
}

// The K splits' sums, added in split order, then the epilogue.
template <typename T>
__global__ __launch_bounds__(256) void gemv_kn_sum_kernel(T* y, const float* partial, int M, int N, int splits,
                                                          int64_t sym, int64_t syn, Epi e) {
  const int n = (int)(blockIdx.x * 256 + threadIdx.x), m = (int)blockIdx.y;
  if (n >= N) return;
  const float* p = partial + (int64_t)m * N + n;
  const int64_t step = (int64_t)M * N;
  float sum = 0.f;
  for (int i = 0; i < splits; ++i) sum += p[i * step];
  y[m * sym + n * syn] = from_f32<T>(epilogue(e, sum, m, n));
}

namespace {

// K splits: about one workgroup on every CU, each with at least one chunk of x.
int kn_mb(int64_t M) { return M <= 2 ? 2 : M <= 4 ? 4 : M <= 8 ? 8 : 16; }
int kn_splits(int64_t M, int64_t N, int64_t K) {
  const int64_t chunk = kn_chunk(kn_mb(M));
  const int64_t tiles = (N + kKnCols - 1) / kKnCols, chunks = (K + chunk - 1) / chunk;
  int64_t s = device_cus() / tiles;
  if (s > chunks) s = chunks;
  return s < 1 ? 1 : (int)s;
}

template <typename T, int MB>
void kn_launch(void* y, float* scratch, const void* x, const void* w, int M, int N, int K, int64_t sxm, int64_t sxk,
               int64_t swk, int64_t sym, int64_t syn, const Epi& e, int splits, bool xvec, hipStream_t st) {
  const int tiles = (N + kKnCols - 1) / kKnCols;
  const dim3 grid((unsigned)(tiles * splits)), block(kMaxWaves * kWave);
  if (splits == 1) {
    hipLaunchKernelGGL((gemv_kn_kernel<T, MB, false>), grid, block, 0, st, (T*)y, scratch, (const T*)x, (const T*)w, M,
                       N, K, sxm, sxk, swk, sym, syn, e, tiles, splits, xvec);
    return;
  }
  hipLaunchKernelGGL((gemv_kn_kernel<T, MB, true>), grid, block, 0, st, (T*)y, scratch, (const T*)x, (const T*)w, M, N,
                     K, sxm, sxk, swk, sym, syn, e, tiles, splits, xvec);
  hipLaunchKernelGGL(gemv_kn_sum_kernel<T>, dim3((unsigned)((N + 255) / 256), (unsigned)M), dim3(256), 0, st, (T*)y,
                     scratch, M, N, splits, sym, syn, e);
}

}  // namespace
}  // namespace fd

using namespace fd;

extern "C" int fd_linear_kn_scratch(int64_t M, int64_t N, int64_t K, int64_t* bytes) {
  if (M < 0 || N < 0 || K < 0) return set_error(FD_EINVAL, "negative size");
  if (!bytes) return set_error(FD_EINVAL, "null pointer argument");
  *bytes = 0;
  if (M == 0 || N == 0 || K == 0) return FD_OK;
  const int s = kn_splits(M, N, K);
  if (s > 1) *bytes = (int64_t)s * M * N * 4;
  return FD_OK;
}

extern "C" int fd_linear_kn(void* y, const void* x, const void* w, const void* bias, int bias_dtype,
                            const void* row_add, int row_dtype, int64_t M, int64_t N, int64_t K, int64_t sxm,
                            int64_t sxk, int64_t swk, int64_t sb, int64_t srm, int64_t srn, int64_t sym, int64_t syn,
                            float* scratch, int64_t scratch_bytes, int act_dtype, void* stream) {
  if (!check_act_dtype(act_dtype)) return FD_EINVAL;
  if (M < 0 || M > 16 || N < 0 || K <= 0) return set_error(FD_EINVAL, "M must be in [0, 16], N >= 0 and K positive");
  if (sxm < 0 || sxk < 0 || swk < 0 || sb < 0 || srm < 0 || srn < 0 || sym < 0 || syn < 0)
    return set_error(FD_EINVAL, "negative stride");
  if (bias && bias_dtype != act_dtype && bias_dtype != FD_F32)
    return set_error(FD_EINVAL, "bias must match x or be float32");
  if (row_add && !check_any_dtype(row_dtype, "row_dtype")) return FD_EINVAL;
  if (M == 0 || N == 0) return FD_OK;
  if (!y || !x || !w) return set_error(FD_EINVAL, "null pointer argument");
  if (N % 8 != 0 || !aligned16(w) || (K > 1 && swk % 8 != 0))
    return set_error(FD_EUNSUPPORTED, "the [K, N] GEMV needs N %% 8 == 0 and 16-byte aligned weight rows");
  if (N > 0x7fffffffLL - kKnCols || K > 0x7fffffffLL - 512) return set_error(FD_EUNSUPPORTED, "too large");
  // one row of a column is written while the others' bias or broadcast row_add is still to be read
  const int64_t ny = span_bytes(M, N, sym, syn, 2);
  if ((bias && overlaps(y, ny, bias, span_bytes(1, N, 0, sb, dtype_bytes(bias_dtype)))) ||
      row_add_meets(row_add, row_dtype, srm, srn, y, act_dtype, sym, syn, M, N))
    return set_error(FD_EUNSUPPORTED, "y must not overlap bias, or row_add other than as row_add itself");
  int splits = kn_splits(M, N, K);
  if (!scratch) scratch_bytes = 0;
  while (splits > 1 && scratch_bytes < (int64_t)splits * M * N * 4) --splits;
  Epi e{};
  e.bias = bias;
  e.bias_dtype = bias_dtype;
  e.sb = sb;
  e.row = row_add;
  e.row_dtype = row_dtype;
  e.srm = srm;
  e.srn = srn;
  const bool xvec = sxk == 1 && aligned16(x) && (M == 1 || sxm % 8 == 0);
  hipStream_t st = static_cast<hipStream_t>(stream);
#define FD_KN(T, MB)                                                                                                \
  kn_launch<T, MB>(y, scratch, x, w, (int)M, (int)N, (int)K, sxm, sxk, swk, sym, syn, e, splits, xvec, st)
#define FD_KN_M(T)                                                                             \
  do {                                                                                         \
    switch (kn_mb(M)) {                                                                        \
      case 2: FD_KN(T, 2); break;                                                              \
      case 4: FD_KN(T, 4); break;                                                              \
      case 8: FD_KN(T, 8); break;                                                              \
      default: FD_KN(T, 16);                                                                   \
    }                                                                                          \
  } while (0)
  if (act_dtype == FD_F16) FD_KN_M(f16); else FD_KN_M(bf16);
#undef FD_KN_M
#undef FD_KN
  return check_launch();
}

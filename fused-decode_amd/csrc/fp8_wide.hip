// E4M3-weight products for more rows than the decode kernels take (M > 16): the
// tiled MFMA GEMM behind linear_decode_fp8 and the gate/up half of the fp8 MLP.
//
//   y[m,n] = round(scale[n] * sum_k e4m3(w[n,k]) * x[m,k] + bias[n] + row_add[m,n])
//
// The activations stay fp16/bf16: codes are decoded exactly to the activation
// type after their LDS read (as in the decode kernels) and
// v_mfma_f32_16x16x32 adds exact products in float32.
//
// A workgroup owns BN weight rows x BM activation rows and walks K in stages of
// 128. Both tiles of a stage go to LDS by DMA (global_load_lds_dwordx4: BN * 128
// code bytes, nontemporal where one row block reads them, and BM * 256
// activation bytes), D - 1 stages ahead of the one being multiplied, with one
// barrier a stage. The DMAs are inline assembly, so the compiler sees plain LDS
// reads and schedules and waits for those itself; the vmcnt waits are explicit.
// Waves split the tile WN x WM, and each stage's K in two halves (KG = 2): two
// waves per SIMD, each with the whole wave tile, so one's LDS reads hide
// under the other's MFMAs without a third wave tile's worth of operand reads.
// The halves' sums meet in LDS at the end.
//
// LDS layout: a tile row is 8 (codes) or 16 (activations) chunks of 16 bytes,
// chunk c at slot c ^ (row mod chunks), so the 8 lanes of a read (8 rows, one
// chunk) hit distinct bank groups and a DMA instruction still fills 1 KiB in
// lane order. A workgroup starts its K sweep at its own stage, so that they do
// not all read one line of every weight row at once. k order: MFMA step s of K half h takes k = 64 h + 16 g + 8 s + j
// for lane group g, so a lane's 16 codes of one read feed both steps.
//
// What bounds it, at 120 bfloat16 rows and the widths of Llama-3-8B (H = 4096, I =
// 14336): gate/up 39 us (44 on another card, where the times below are longer alike),
// of which its loads alone take 24 (117 MB of codes from HBM and twice that in
// activations from L2, which a tile of all rows reads once per 128 weight rows),
// its LDS reads, decodes and MFMAs alone 19, launch and output 9; down 23 us and 6
// for the sum over K splits. No unit is full: matrix cores busy 29% of the cycles
// (20% in down), LDS 13%, and the waves issue, wait to issue and wait for loads or
// the barrier for a third of theirs each. A layer's MLP 834 -> 74 us against the
// float32 product of the decoded weights that these rows took before (the weights
// written out in float32 and read again). The output first left the kernel as 2-byte
// stores with the scales loaded per tile: 62 us for gate/up.
#include <type_traits>

#include "fd_dma.h"
#include "fd_gemv.h"

namespace fd {

constexpr int kWideK = 128;  // K elements of a stage

enum WideEpi { WIDE_OUT = 0, WIDE_PART = 1, WIDE_SWIGLU = 2 };

// One 16-byte-per-lane DMA into LDS at byte address `lds` (wave-uniform; lane L
// lands at 16 L). The s_nop is the wait state a load that reads m0 needs after
// the write of m0. (m0 is a reserved register, which the compiler warns of; the clobber
// still keeps it from reusing a value of its own across the asm.)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
template <bool NT>
__device__ __forceinline__ void wide_dma(const void* src, unsigned lds) {
  if constexpr (NT)
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off nt" ::"s"(lds), "v"(src)
                 : "memory", "m0");
  else
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds), "v"(src)
                 : "memory", "m0");
}
#pragma clang diagnostic pop

// This wave's LDS reads have returned and its LDS writes are done, then the
// workgroup's barrier; nothing moves across.
__device__ __forceinline__ void wide_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// Row pitch (floats) of the sums in LDS: 16 bytes past the tile, so that a
// wave's 16 rows of one column fall into different banks.
template <int BN> constexpr int kWidePitch = BN + 4;

constexpr size_t wide_stage_bytes(int bn, int bm) { return (size_t)bn * kWideK + (size_t)bm * kWideK * 2; }
// Dynamic LDS of a launch: D stages, or what the halves' sums take at the end.
constexpr size_t wide_lds(int bn, int bm, int d) {
  const size_t ring = wide_stage_bytes(bn, bm) * d, sums = (size_t)2 * bm * (bn + 4) * 4;
  return ring > sums ? ring : sums;
}

template <typename T, int WN, int WM, int NT, int MT, int D, int EPI>
__global__ __launch_bounds__(2 * WN * WM * kWave) void fp8_wide_kernel(
    T* y, float* partial, const T* x, const uint8_t* w, const float* wscale, int M, int N, int K, int64_t sxm,
    int64_t swn, int64_t sym, int64_t syn, Epi e, int mtiles, int splits) {
  typedef typename Vec8<T>::type V8;
  constexpr int BN = WN * NT * 16, BM = WM * MT * 16, NW = 2 * WN * WM;
  constexpr int AOPS = BN / 8 / NW, BOPS = BM / 4 / NW;  // DMA instructions per stage and wave
  constexpr int OPS = AOPS + BOPS;
  static_assert(AOPS >= 1 && BOPS >= 1 && AOPS * 8 * NW == BN && BOPS * 4 * NW == BM, "the waves share a stage evenly");
  extern __shared__ __align__(16) u32x4 wide_smem[];
  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int kg = wave & 1, wm = (wave >> 1) % WM, wn = (wave >> 1) / WM;
  const int r = lane & 15, g = lane >> 4;

  // Block -> (tile, K split). Consecutive blocks go to the eight XCDs in turn:
  // with K splits the split is the fastest index, so that an XCD's L2 holds few
  // K ranges of x; without, each XCD takes a contiguous run of tiles, the row
  // blocks of one weight tile next to each other.
  int tile, split = 0;
  {
    const int b = (int)blockIdx.x, total = (int)gridDim.x;
    if (splits > 1) {
      split = b % splits;
      tile = b / splits;
    } else {
      const int xcd = b & 7, q = total >> 3, rem = total & 7;
      tile = xcd * q + (xcd < rem ? xcd : rem) + (b >> 3);
    }
  }
  const int ntile = tile / mtiles, m0 = (tile - ntile * mtiles) * BM;
  const int half_n = N / 2;  // SWIGLU: gate rows; up row j is row half_n + j
  const int stages_all = (K + kWideK - 1) / kWideK;
  const int s0 = (int)((int64_t)stages_all * split / splits);
  const int ns = (int)((int64_t)stages_all * (split + 1) / splits) - s0;
  const int off = ns > 0 ? tile % ns : 0;
  auto stage_k = [&](int s) {  // first k of this block's s-th stage
    const int u = s + off;
    return (s0 + (u >= ns ? u - ns : u)) * kWideK;
  };

  // weight row of tile row t (past N: a row that exists, never stored)
  auto wrow = [&](int t) -> int64_t {
    if constexpr (EPI == WIDE_SWIGLU) {
      // per wave: NT/2 gate tiles, then the matching up tiles
      const int wv = t / (NT * 16), q = t % (NT * 16);
      const int j = ntile * (BN / 2) + wv * (NT * 8) + q % (NT * 8);
      const int jc = j < half_n ? j : half_n - 1;
      return q < NT * 8 ? jc : half_n + jc;
    } else {
      const int n = ntile * BN + t;
      return n < N ? n : N - 1;
    }
  };

  const unsigned lds0 = lds_addr(wide_smem);
  constexpr unsigned kStage = (unsigned)wide_stage_bytes(BN, BM);
  const uint8_t* ap[AOPS];
  int ak[AOPS];
#pragma unroll
  for (int i = 0; i < AOPS; ++i) {
    const int t = (wave * AOPS + i) * 8 + lane / 8;
    ap[i] = w + wrow(t) * swn;
    ak[i] = ((lane & 7) ^ (t & 7)) * 16;
  }
  const T* bp[BOPS];
  int bk[BOPS];
#pragma unroll
  for (int i = 0; i < BOPS; ++i) {
    const int t = (wave * BOPS + i) * 4 + lane / 16;
    const int m = m0 + t;
    bp[i] = x + (int64_t)(m < M ? m : M - 1) * sxm;
    bk[i] = ((lane & 15) ^ (t & 15)) * 8;
  }
  const bool once = mtiles == 1;  // this block alone reads its codes
  auto issue = [&](int s) {
    const int k0 = stage_k(s);
    const unsigned base = lds0 + (unsigned)(s % D) * kStage;
#pragma unroll
    for (int i = 0; i < AOPS; ++i) {
      const int k = k0 + ak[i];
      const uint8_t* p = ap[i] + (k < K ? k : 0);
      const unsigned to = base + (unsigned)(wave * AOPS + i) * 1024u;
      if (once)
        wide_dma<true>(p, to);
      else
        wide_dma<false>(p, to);
    }
#pragma unroll
    for (int i = 0; i < BOPS; ++i) {
      const int k = k0 + bk[i];
      wide_dma<false>(bp[i] + (k < K ? k : 0), base + (unsigned)(BN * 128) + (unsigned)(wave * BOPS + i) * 1024u);
    }
  };

  f32x4 acc[NT][MT];
#pragma unroll
  for (int n = 0; n < NT; ++n)
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[n][m] = f32x4{0.f, 0.f, 0.f, 0.f};

  // this lane's chunks in a stage (u32x4 entries): codes of k 64 kg + 16 g, and
  // the activations of its two steps
  int fa[NT], fb[MT][2];
#pragma unroll
  for (int n = 0; n < NT; ++n) {
    const int t = (wn * NT + n) * 16 + r;
    fa[n] = t * 8 + ((kg * 4 + g) ^ (t & 7));
  }
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int t = (wm * MT + m) * 16 + r;
      fb[m][s] = BN * 8 + t * 16 + ((kg * 8 + 2 * g + s) ^ (t & 15));
    }

  const int pre = ns < D - 1 ? ns : D - 1;
  for (int s = 0; s < pre; ++s) issue(s);
  for (int s = 0; s < ns; ++s) {
    // stages issued so far end at s + D - 2: D - 2 of them may stay in flight
    if (s + D - 2 < ns)
      wait_vm<OPS*(D - 2)>();
    else
      wait_vm<0>();
    const int k0 = stage_k(s);
    if (k0 + kWideK > K) {  // K tail: activations past K are zero
      const unsigned base = lds0 + (unsigned)(s % D) * kStage + (unsigned)(BN * 128);
#pragma unroll
      for (int i = 0; i < BOPS; ++i)
        if (k0 + bk[i] >= K) ds_zero16(base + (unsigned)(wave * BOPS + i) * 1024u + (unsigned)lane * 16u);
    }
    wide_barrier();  // stage s has landed everywhere; every wave is done with stage s - 1
    if (s + D - 1 < ns) issue(s + D - 1);
    const u32x4* st = wide_smem + (size_t)(s % D) * (kStage / 16);
    u32x4 bf[2][MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      bf[0][m] = st[fb[m][0]];
      bf[1][m] = st[fb[m][1]];
    }
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      u32x4 a0, a1;
      fp8x16_decode<T>(st[fa[n]], a0, a1);
#pragma unroll
      for (int m = 0; m < MT; ++m)
        acc[n][m] = mfma16(__builtin_bit_cast(V8, a0), __builtin_bit_cast(V8, bf[0][m]), acc[n][m]);
#pragma unroll
      for (int m = 0; m < MT; ++m)
        acc[n][m] = mfma16(__builtin_bit_cast(V8, a1), __builtin_bit_cast(V8, bf[1][m]), acc[n][m]);
    }
  }

  // The K halves meet in LDS, each wave tile row-major [activation row][weight
  // row] so that the output leaves in 16-byte pieces along a row: thread t takes
  // the same OC output columns of every row it writes, and loads their scales
  // and bias once.
  wide_barrier();
  float* sums = reinterpret_cast<float*>(wide_smem);
#pragma unroll
  for (int n = 0; n < NT; ++n)
#pragma unroll
    for (int m = 0; m < MT; ++m)
      *reinterpret_cast<f32x4*>(sums + (size_t)(kg * BM + (wm * MT + m) * 16 + r) * kWidePitch<BN> +
                                (wn * NT + n) * 16 + 4 * g) = acc[n][m];
  constexpr int OUT = EPI == WIDE_SWIGLU ? BN / 2 : BN;  // output columns of a tile row
  constexpr int OC = EPI == WIDE_PART ? 4 : 8;           // output columns a thread takes
  constexpr int TPR = OUT / OC;                          // threads per row
  static_assert((NW * kWave) % TPR == 0, "a thread keeps its columns");
  const int oc = tid % TPR * OC;
  // column of the sums: SWIGLU per wave NT * 8 gate then NT * 8 up columns
  const int sc = EPI == WIDE_SWIGLU ? oc / (NT * 8) * (NT * 16) + oc % (NT * 8) : oc;
  const int c0 = ntile * OUT + oc, cols = EPI == WIDE_SWIGLU ? half_n : N;
  float s1[OC], s2[OC];  // scales; SWIGLU: of the gate and the up rows; OUT: s2 the bias
#pragma unroll
  for (int i = 0; i < OC; ++i) {
    const int c = c0 + i < cols ? c0 + i : cols - 1;
    s1[i] = EPI == WIDE_PART ? 1.f : wscale[c];
    s2[i] = EPI == WIDE_SWIGLU          ? wscale[half_n + c]
            : EPI == WIDE_OUT && e.bias ? load_any(e.bias, e.bias_dtype, c * e.sb)
                                        : 0.f;
  }
  const bool whole = c0 + OC <= cols;
  const bool wide_store =
      EPI != WIDE_PART && whole && syn == 1 && sym % 8 == 0 && (reinterpret_cast<uintptr_t>(y) & 15) == 0;
  wide_barrier();
  for (int t = tid / TPR; t < BM; t += NW * kWave / TPR) {
    const int row = m0 + t;
    if (row >= M || c0 >= cols) break;
    const float* p0 = sums + (size_t)t * kWidePitch<BN> + sc;
    const float* p1 = p0 + (size_t)BM * kWidePitch<BN>;
    float v[OC];
#pragma unroll
    for (int i = 0; i < OC; i += 4) {
      const f32x4 q = *reinterpret_cast<const f32x4*>(p0 + i) + *reinterpret_cast<const f32x4*>(p1 + i);
#pragma unroll
      for (int j = 0; j < 4; ++j) v[i + j] = q[j];
    }
    if constexpr (EPI == WIDE_PART) {
      float* to = partial + ((int64_t)split * M + row) * N + c0;
      if (N % 4 == 0) {
        *reinterpret_cast<f32x4*>(to) = f32x4{v[0], v[1], v[2], v[3]};
      } else {
#pragma unroll
        for (int i = 0; i < OC; ++i)
          if (c0 + i < N) to[i] = v[i];
      }
    } else {
      V8 o;
      if constexpr (EPI == WIDE_SWIGLU) {
#pragma unroll
        for (int i = 0; i < OC; i += 4) {
          const f32x4 q = *reinterpret_cast<const f32x4*>(p0 + NT * 8 + i) +
                          *reinterpret_cast<const f32x4*>(p1 + NT * 8 + i);
#pragma unroll
          for (int j = 0; j < 4; ++j) o[i + j] = swiglu_out<T>(v[i + j] * s1[i + j], q[j] * s2[i + j]);
        }
      } else {
#pragma unroll
        for (int i = 0; i < OC; ++i) {
          float f = v[i] * s1[i] + s2[i];
          if (e.row && c0 + i < N) f += load_any(e.row, e.row_dtype, row * e.srm + (c0 + i) * e.srn);
          o[i] = from_f32<T>(f);
        }
      }
      T* to = y + (int64_t)row * sym + c0 * syn;
      if (wide_store) {
        store8<T>(to, o);
      } else {
#pragma unroll
        for (int i = 0; i < OC; ++i)
          if (c0 + i < cols) to[i * syn] = o[i];
      }
    }
  }
}

// The K splits' sums, added in split order, then the channel scale and the
// epilogue: one thread per four columns of a row (ceil(N / 4) per row).
template <typename T>
__global__ __launch_bounds__(256) void fp8_wide_sum_kernel(T* y, const float* partial, const float* wscale, int M,
                                                           int N, int splits, int64_t sym, int64_t syn, Epi e,
                                                           FastDiv quads, uint32_t total) {
  const uint32_t v = blockIdx.x * 256 + threadIdx.x;
  if (v >= total) return;
  uint32_t q;
  const uint32_t m = quads.divmod(v, q);
  const int c = (int)q * 4;
  const float* p = partial + (int64_t)m * N + c;
  const int64_t step = (int64_t)M * N;
  float s[4] = {0.f, 0.f, 0.f, 0.f};
  if (N % 4 == 0) {
    f32x4 a = *reinterpret_cast<const f32x4*>(p);
    for (int i = 1; i < splits; ++i) a += *reinterpret_cast<const f32x4*>(p + i * step);
#pragma unroll
    for (int i = 0; i < 4; ++i) s[i] = a[i];
  } else {
    for (int i = 0; i < splits; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (c + j < N) s[j] += p[i * step + j];
  }
#pragma unroll
  for (int j = 0; j < 4; ++j)
    if (c + j < N) y[(int64_t)m * sym + (c + j) * syn] = from_f32<T>(epilogue(e, s[j] * wscale[c + j], m, c + j));
}

namespace {

struct WideArgs {
  void* y;
  float* partial;
  const void* x;
  const uint8_t* w;
  const float* scale;
  int M, N, K;
  int64_t sxm, swn, sym, syn;
  Epi e;
  hipStream_t st;
};

template <typename T, int WN, int WM, int NT, int MT, int D, int EPI>
int wide_launch(const WideArgs& a, int splits) {
  constexpr int BN = WN * NT * 16, BM = WM * MT * 16;
  constexpr size_t lds = wide_lds(BN, BM, D);
  static_assert(lds <= kMaxLds, "a launch fits the LDS of a CU");
  const int64_t nt = (a.N + BN - 1) / BN, mt = (a.M + BM - 1) / BM;
  if (nt * mt * splits > 0x7fffffffLL) return set_error(FD_EUNSUPPORTED, "too many tiles");
  auto kernel = fp8_wide_kernel<T, WN, WM, NT, MT, D, EPI>;
  if (!allow_lds(kernel, lds)) return set_error(FD_ELAUNCH, "cannot raise the LDS limit to %zu bytes", lds);
  hipLaunchKernelGGL(kernel, dim3((unsigned)(nt * mt * splits)), dim3(2 * WN * WM * kWave), lds, a.st,
                     static_cast<T*>(a.y), a.partial, static_cast<const T*>(a.x), a.w, a.scale, a.M, a.N, a.K, a.sxm,
                     a.swn, a.sym, a.syn, a.e, (int)mt, splits);
  return FD_OK;
}

// Activation rows of a tile: 32, 64, 96 or 128, whichever takes the least time for
// all M rows. A tile's time is about that of its rows and 74 more (gate/up at the
// widths of Llama-3-8B: 25.0, 28.0, 33.4 and 39.2 us with one tile of 32, 64, 96 and 128
// a weight tile). Gate/up of 32 rows 25.0 us (31.1 in the tile of 64, 40.6 in that of
// 128), 64 rows 28.0 (39.6, 38.6), 96 rows 33.4 (40.9 in that of 128), 120 rows 39.2
// (73.5 in four tiles of 32, 48.1 in two of 64), 192 rows 60.8 in two of 96 (71.7 in
// two of 128), 288 rows 90.5 in three (105.8).
inline int wide_bm(int64_t M) {
  auto cost = [&](int64_t bm) { return (M + bm - 1) / bm * (bm + 74); };
  int best = 32;
  for (int bm : {64, 96, 128})
    if (cost(bm) < cost(best)) best = bm;
  return best;
}

// Tiles of 128 weight rows, with as many stages as the LDS holds. Tiles of 64
// weight rows read the activations twice as often (gate/up of 32, 64 and 120 rows
// 26.4, 33.6, 50.5 us) and two waves a SIMD beat one with twice the tile (120 rows:
// 39.2 against 41.4 and 47.4).
template <typename T, int EPI>
int wide_rows(const WideArgs& a, int splits) {
  switch (wide_bm(a.M)) {
    case 32: return wide_launch<T, 4, 1, 2, 2, 6, EPI>(a, splits);
    case 64: return wide_launch<T, 2, 2, 4, 2, 4, EPI>(a, splits);
    case 96: return wide_launch<T, 2, 2, 4, 3, 4, EPI>(a, splits);
    default: return wide_launch<T, 2, 2, 4, 4, 3, EPI>(a, splits);
  }
}

// K splits of a product: enough for one workgroup on every CU, each with at
// least four stages, which is where the next split's sums cost what its share
// of the stages saves (N = 4096, K = 14336, 64 rows without the sum kernel: 2 / 4 /
// 8 splits 38.2 / 22.7 / 15.7 us; 120 rows 60.4 / 34.5 / 23.1).
int wide_splits(int64_t M, int64_t N, int64_t K) {
  const int64_t tiles = ((N + 127) / 128) * ((M + wide_bm(M) - 1) / wide_bm(M));
  const int64_t stages = (K + kWideK - 1) / kWideK;
  int64_t s = device_cus() / tiles;
  if (s > stages / 4) s = stages / 4;
  return s < 1 ? 1 : (int)s;
}

int wide_check(const void* x, const void* w8, int64_t M, int64_t N, int64_t K, int64_t sxm, int64_t swn) {
  if (K % 16 != 0 || !aligned16(x) || !aligned16(w8) || (M > 1 && sxm % 8 != 0) || (N > 1 && swn % 16 != 0))
    return set_error(FD_EUNSUPPORTED, "the fp8 kernels need K %% 16 == 0 and 16-byte aligned rows");
  // the kernel's int indexes run to the end of the last tile of 128 rows and stage of 128 k
  if (M > 0x7fffffffLL - 128 || N > 0x7fffffffLL - 128 || K > 0x7fffff00LL)
    return set_error(FD_EUNSUPPORTED, "too large");
  return FD_OK;
}

}  // namespace
}  // namespace fd

using namespace fd;

extern "C" int fd_linear_fp8_wide_scratch(int64_t M, int64_t N, int64_t K, int64_t* bytes) {
  if (M < 0 || N < 0 || K < 0) return set_error(FD_EINVAL, "negative size");
  if (!bytes) return set_error(FD_EINVAL, "null pointer argument");
  *bytes = 0;
  if (M == 0 || N == 0 || K == 0) return FD_OK;
  const int s = wide_splits(M, N, K);
  if (s > 1) *bytes = (int64_t)s * M * N * 4;
  return FD_OK;
}

extern "C" int fd_linear_fp8_wide(void* y, const void* x, const void* w8, const float* w_scale, const void* bias,
                                  int bias_dtype, const void* row_add, int row_dtype, int64_t M, int64_t N,
                                  int64_t K, int64_t sxm, int64_t swn, int64_t sb, int64_t srm, int64_t srn,
                                  int64_t sym, int64_t syn, float* scratch, int64_t scratch_bytes, int act_dtype,
                                  void* stream) {
  if (!check_act_dtype(act_dtype)) return FD_EINVAL;
  if (M < 0 || N < 0 || K <= 0) return set_error(FD_EINVAL, "M and N must be >= 0 and K positive");
  if (sxm < 0 || swn < 0 || sb < 0 || srm < 0 || srn < 0 || sym < 0 || syn < 0)
    return set_error(FD_EINVAL, "negative stride");
  if (bias && bias_dtype != act_dtype && bias_dtype != FD_F32)
    return set_error(FD_EINVAL, "bias must match x or be float32");
  if (row_add && !check_any_dtype(row_dtype, "row_dtype")) return FD_EINVAL;
  if (M == 0 || N == 0) return FD_OK;
  if (!y || !x || !w8 || !w_scale) return set_error(FD_EINVAL, "null pointer argument");
  int rc = wide_check(x, w8, M, N, K, sxm, swn);
  if (rc != FD_OK) return rc;
  // tiles are stored while other workgroups still read their operands
  const int64_t ny = span_bytes(M, N, sym, syn, 2);
  if (overlaps(y, ny, x, span_bytes(M, K, sxm, 1, 2)) || overlaps(y, ny, w8, span_bytes(N, K, swn, 1, 1)) ||
      overlaps(y, ny, w_scale, N * 4) ||
      (bias && overlaps(y, ny, bias, span_bytes(1, N, 0, sb, dtype_bytes(bias_dtype)))) ||
      row_add_meets(row_add, row_dtype, srm, srn, y, act_dtype, sym, syn, M, N))
    return set_error(FD_EUNSUPPORTED, "y must not overlap an operand, other than as row_add itself");
  const int64_t quads = (N + 3) / 4;
  int splits = wide_splits(M, N, K);
  if (!scratch) scratch_bytes = 0;
  if (scratch && !aligned16(scratch)) return set_error(FD_EUNSUPPORTED, "scratch must be 16-byte aligned");
  while (splits > 1 && scratch_bytes < (int64_t)splits * M * N * 4) --splits;
  WideArgs a{y,        scratch, x,   static_cast<const uint8_t*>(w8), w_scale, (int)M, (int)N, (int)K, sxm, swn, sym,
             syn,      Epi{},   static_cast<hipStream_t>(stream)};
  a.e.bias = bias;
  a.e.bias_dtype = bias_dtype;
  a.e.sb = sb;
  a.e.row = row_add;
  a.e.row_dtype = row_dtype;
  a.e.srm = srm;
  a.e.srn = srn;
  if (splits == 1) {
    rc = act_dtype == FD_F16 ? wide_rows<f16, WIDE_OUT>(a, 1) : wide_rows<bf16, WIDE_OUT>(a, 1);
  } else {
    rc = act_dtype == FD_F16 ? wide_rows<f16, WIDE_PART>(a, splits) : wide_rows<bf16, WIDE_PART>(a, splits);
    if (rc == FD_OK) {
      const uint32_t total = (uint32_t)(M * quads);  // splits > 1: few tiles, so M * N is small
      const unsigned blocks = (unsigned)((total + 255) / 256);
      if (act_dtype == FD_F16)
        hipLaunchKernelGGL(fp8_wide_sum_kernel<f16>, dim3(blocks), dim3(256), 0, a.st, static_cast<f16*>(y), scratch,
                           w_scale, a.M, a.N, splits, sym, syn, a.e, FastDiv((uint32_t)quads), total);
      else
        hipLaunchKernelGGL(fp8_wide_sum_kernel<bf16>, dim3(blocks), dim3(256), 0, a.st, static_cast<bf16*>(y),
                           scratch, w_scale, a.M, a.N, splits, sym, syn, a.e, FastDiv((uint32_t)quads), total);
    }
  }
  if (rc != FD_OK) return rc;
  return check_launch();
}

extern "C" int fd_gate_up_fp8_wide(void* mid, const void* x, const void* w_gate_up8, const float* gate_up_scale,
                                   int64_t M, int64_t H, int64_t I, int64_t sxm, int act_dtype, void* stream) {
  if (!check_act_dtype(act_dtype)) return FD_EINVAL;
  if (M < 0 || H <= 0 || I <= 0) return set_error(FD_EINVAL, "M must be >= 0, H and I positive");
  if (sxm < 0) return set_error(FD_EINVAL, "negative stride");
  if (M == 0) return FD_OK;
  if (!mid || !x || !w_gate_up8 || !gate_up_scale) return set_error(FD_EINVAL, "null pointer argument");
  int rc = wide_check(x, w_gate_up8, M, 2 * I, H, sxm, H);
  if (rc != FD_OK) return rc;
  const int64_t nm = M * I * 2;  // stored while other workgroups still read
  if (overlaps(mid, nm, x, span_bytes(M, H, sxm, 1, 2)) || overlaps(mid, nm, w_gate_up8, 2 * I * H) ||
      overlaps(mid, nm, gate_up_scale, 2 * I * 4))
    return set_error(FD_EINVAL, "mid must not overlap x or the weights");
  WideArgs a{mid, nullptr, x,     static_cast<const uint8_t*>(w_gate_up8), gate_up_scale, (int)M, (int)(2 * I), (int)H, sxm,
             H,   I,       1,     Epi{}, static_cast<hipStream_t>(stream)};
  rc = act_dtype == FD_F16 ? wide_rows<f16, WIDE_SWIGLU>(a, 1) : wide_rows<bf16, WIDE_SWIGLU>(a, 1);
  if (rc != FD_OK) return rc;
  return check_launch();
}

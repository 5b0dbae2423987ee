// MFMA GEMV in workgroups of one, three or four octets of weight rows (8, 24 or
// 32), for outputs that 16-row tiles divide unevenly over the CUs or that leave
// many of them idle (oct_rows).
//
// The stream, the ring and the unit's k order are those of gemv_mfma_dma_kernel
// (fd_dma.h); a unit's activations are read once for all its weight rows: one MFMA
// tile of 8 rows (rows 8-15 repeat them and are never stored), or rows 0-15 and
// rows 16-23 (the second tile's rows 8-15 repeated) or 16-31. Wave n writes tile n.
//
// What bounds it: the bytes that the busiest CU takes in, weights and activations
// alike. A workgroup of 16 rows by itself on a CU takes about 16 bytes a clock
// however many units it keeps in flight (1024 x 4096 to 4096 x 11032, four or eight
// waves, one to three units each: within 3% of each other), so its time falls only
// with its rows or with the activations read per row.
#include "fd_dma.h"

namespace fd {

template <typename T, typename W, int OCT, int NW, int D, int BR>
__global__ __launch_bounds__(NW * kWave) void gemv_mfma_oct_kernel(T* y, const T* x, const W* w, const float* wscale,
                                                                   int M, int N, int K, int64_t sxm, int64_t swn,
                                                                   int64_t sym, int64_t syn, Epi e) {
  typedef typename Vec8<T>::type V8;
  constexpr bool F8 = sizeof(W) == 1;
  constexpr int CPR = F8 ? 8 : 16, EPC = F8 ? 16 : 8;  // 16-byte chunks of a weight row's unit, elements of one
  constexpr int ROWS = 8 * OCT, TILES = (OCT + 1) / 2, LAST = OCT % 2 ? 8 : 16;  // LAST: rows of the last tile
  constexpr int AE = ROWS * CPR, AOPS = AE / kWave, RPI = kWave / CPR;
  constexpr int NT = F8 ? 2 : 4, NA = TILES * NT, NR = NA + 4;  // LDS reads per unit: A of a tile, of all, all
  constexpr int SLOT = AE + BR * 16, OPS = AOPS + BR / 4;
  static_assert(NW >= TILES && TILES <= 2, "a wave for each tile");
  extern __shared__ __align__(16) u32x4 oct_lds[];  // ring [NW][D][SLOT]
  __shared__ f32x4 part[TILES][NW * kWave];
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int r = lane & 15, g = lane >> 4;
  const int64_t n0 = (int64_t)blockIdx.x * ROWS;
  const W* wrow[AOPS];
  int wch[AOPS];
#pragma unroll
  for (int i = 0; i < AOPS; ++i) {
    const int row = RPI * i + lane / CPR;
    const int64_t n = n0 + row;
    wrow[i] = w + (n < N ? n : 0) * swn;
    wch[i] = ((lane % CPR) ^ (row % CPR)) * EPC;
  }
  const T* xrow[BR / 4];
  int xch[BR / 4];
#pragma unroll
  for (int i = 0; i < BR / 4; ++i) {
    const int row = 4 * i + (lane >> 4);
    xrow[i] = x + (row < M ? row : 0) * sxm;
    xch[i] = ((lane & 15) ^ row) * 8;
  }
  const int units = (K + kUnit - 1) / kUnit;
  const int mine = wave < units ? (units - wave + NW - 1) / NW : 0;
  const int off = sweep_offset(units);
  u32x4* const ring = oct_lds + wave * (D * SLOT);
  auto issue = [&](int j) {  // the same instruction count in every unit; chunks past K read the row's first
    const int k0 = sweep_unit(wave, j, NW, off, units) * kUnit;
    u32x4* slot = ring + (j % D) * SLOT;
    const bool whole = k0 + kUnit <= K;
#pragma unroll
    for (int i = 0; i < AOPS; ++i) {
      const int k = k0 + wch[i];
      dma16_nt(wrow[i] + (whole || k < K ? k : 0), slot + i * kWave);
    }
#pragma unroll
    for (int i = 0; i < BR / 4; ++i) {
      const int k = k0 + xch[i];
      dma16(xrow[i] + (whole || k < K ? k : 0), slot + AE + i * kWave);
    }
  };
  const unsigned ring0 = lds_addr(ring);
  const int rb = r % BR;
  unsigned fa[NA], fb[4];  // this lane's fragment entries within a slot (bytes)
#pragma unroll
  for (int t = 0; t < NA; ++t) {
    const int c = F8 ? 2 * g + t % NT : t % NT * 4 + g;
    const int row = t / NT * 16 + (t / NT == TILES - 1 ? r % LAST : r);
    fa[t] = ring0 + (unsigned)(row * CPR + (c ^ (row % CPR))) * 16u;
  }
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    const int c = F8 ? g * 4 + s : s * 4 + g;
    fb[s] = ring0 + (unsigned)(AE + rb * 16 + (c ^ rb)) * 16u;
  }
  f32x4 acc[TILES];
#pragma unroll
  for (int n = 0; n < TILES; ++n) acc[n] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto consume = [&](int j) {
    const unsigned so = (unsigned)(j % D) * (SLOT * 16u);
    const int k0 = sweep_unit(wave, j, NW, off, units) * kUnit;
    if (k0 + kUnit > K) {  // K tail: zero the entries fetched past K
#pragma unroll
      for (int i = 0; i < AOPS; ++i)
        if (k0 + wch[i] >= K) ds_zero16(ring0 + so + (unsigned)(i * kWave + lane) * 16u);
#pragma unroll
      for (int i = 0; i < BR / 4; ++i)
        if (k0 + xch[i] >= K) ds_zero16(ring0 + so + (unsigned)(AE + i * kWave + lane) * 16u);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
    u32x4 v[NR];
#pragma unroll
    for (int t = 0; t < NA; ++t) v[t] = ds_read16(fa[t] + so);
#pragma unroll
    for (int s = 0; s < 4; ++s) v[NA + s] = ds_read16(fb[s] + so);
    wait_lds_all(v);
    u32x4 af[TILES][4];
#pragma unroll
    for (int n = 0; n < TILES; ++n) {
      if constexpr (F8) {
        fp8x16_decode<T>(v[n * NT], af[n][0], af[n][1]);
        fp8x16_decode<T>(v[n * NT + 1], af[n][2], af[n][3]);
      } else {
#pragma unroll
        for (int s = 0; s < 4; ++s) af[n][s] = v[n * NT + (s & (NT - 1))];
      }
    }
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int n = 0; n < TILES; ++n)
        acc[n] = mfma16(__builtin_bit_cast(V8, af[n][s]), __builtin_bit_cast(V8, v[NA + s]), acc[n]);
  };

  // bias, row_add and channel scale, loaded before the stream by every wave for the
  // tile of its parity (wave n writes tile n)
  const int tile = wave % TILES;
  const int64_t nt0 = n0 + 16 * tile, nend = n0 + ROWS < N ? n0 + ROWS : N;
  const TileEpi tep = tile_epi_loads<F8>(e, wscale, wrow[0], lane, nt0, M, (int)nend);
  const int pre = mine < D ? mine : D;
  for (int j = 0; j < pre; ++j) issue(j);
  int j = 0;
  for (; j + D <= mine; ++j) {  // D units in flight: the D-1 after unit j may stay outstanding
    wait_vm<OPS*(D - 1)>();
    consume(j);
    if (j + D < mine) issue(j + D);
  }
  wait_vm<0>();
  for (; j < mine; ++j) consume(j);
#pragma unroll
  for (int n = 0; n < TILES; ++n) part[n][wave * kWave + lane] = acc[n];
  __syncthreads();
  // the last workgroup's second tile may start past N: it has no output rows, and no
  // row of sums either (Epi::ss holds ceil(N / 16) of them)
  if (wave >= TILES || nt0 >= N) return;
  f32x4 s = part[tile][lane];
  for (int i = 1; i < NW; ++i) s += part[tile][i * kWave + lane];
  mfma_tile_out_plain<T, F8>(y, s, lane, nt0, e, tep, M, (int)nend, sym, syn);
}

namespace {

template <typename T, typename W, int OCT, int NW, int D, int BR>
int oct_run(void* y, const void* x, const void* w, const float* ws, int M, int N, int K, int64_t sxm, int64_t swn,
            int64_t sym, int64_t syn, const Epi& e, hipStream_t st) {
  constexpr int ROWS = 8 * OCT;
  constexpr size_t ring = (size_t)NW * D * (ROWS * (sizeof(W) == 1 ? 8 : 16) + BR * 16) * 16;
  static_assert(ring + (size_t)(OCT + 1) / 2 * NW * kWave * 16 <= kMaxLds, "a launch fits the LDS of a CU");
  auto kernel = gemv_mfma_oct_kernel<T, W, OCT, NW, D, BR>;
  if (!allow_lds(kernel, ring)) return set_error(FD_ELAUNCH, "cannot raise the LDS limit to %zu bytes", ring);
  hipLaunchKernelGGL(kernel, dim3((unsigned)(((int64_t)N + ROWS - 1) / ROWS)), dim3(NW * kWave), ring, st,
                     static_cast<T*>(y), static_cast<const T*>(x), static_cast<const W*>(w), ws, M, N, K, sxm, swn,
                     sym, syn, e);
  return FD_OK;
}

}  // namespace

// The rows whose busiest CU takes in the fewest bytes for each k: its rounds of
// workgroups times their weights and staged activations. Measured against 16 rows,
// 8 / 16 activation rows (us):
//   fp16  1501 x 11032  8 rows   16.0 / 19.6 -> 12.3 / 15.7
//         5000 x 4096   24 rows  11.5 / 12.9 ->  9.7 / 10.3
//         6144 x 14336  24 rows  38.0 / 40.1 -> 29.8 / 31.2
//   E4M3  1911 x 6432   8 rows    8.6 / 10.2 ->  6.9 /  8.4
//         5000 x 4096   24 rows   8.4 / 10.3 ->  6.8 /  7.9
//         9016 x 2560   24 rows   8.9 / 10.8 ->  8.0 /  9.5  (32 rows: 9.0 / 10.3)
//         16384 x 2048  32 rows   9.2 / 12.4 ->  8.5 /  9.5  (24 rows: 9.3 / 11.5)
//         28672 x 4096  32 rows  24.7 / 30.4 -> 22.5 / 25.3
// With fp16 weights only while one round is enough: past it these workgroups, alone
// on their CU, leave HBM idle while they start and end (8192 x 4096 in 32 rows: 12.9 /
// 14.4 -> 14.8 / 15.3; 21536 x 3536 in 24: 39.0 -> 40.0 at 16). Row sums come in
// 16-row tiles, which 32 rows keep. Fewer than eight units leave waves idle.
int oct_rows(int M, int N, int K, int wbytes, bool sums) {
  if (M < 5 || (K + kUnit - 1) / kUnit < 8) return 0;
  const int64_t cus = device_cus();
  auto rounds = [&](int rows) { return (((int64_t)N + rows - 1) / rows + cus - 1) / cus; };
  auto bytes = [&](int rows) { return rounds(rows) * (rows * wbytes + dma_rows(M) * 2); };
  int best = 16;
  if (!sums)
    for (int rows : {8, 24})
      if (bytes(rows) < bytes(best) && (wbytes == 1 || rounds(rows) == 1)) best = rows;
  if (wbytes == 1 && bytes(32) < bytes(best)) best = 32;
  return best == 16 ? 0 : best;
}

// Waves and units in flight, by measurement: eight waves where one workgroup has a
// CU to itself and its units are small (E4M3 5000 x 4096 at 8 rows: 6.8 us against 7.4
// for four; fp16 1024 x 4096: 5.4 against 6.1), else four, of which several
// workgroups share a CU (E4M3 28672 x 4096: 22.5 against 27.5).
template <typename T, typename W>
int launch_oct(int rows, int M, void* y, const void* x, const void* w, const float* ws, int N, int K, int64_t sxm,
               int64_t swn, int64_t sym, int64_t syn, const Epi& e, hipStream_t st) {
#define FD_RUN(OCT, NW, BR) return oct_run<T, W, OCT, NW, 2, BR>(y, x, w, ws, M, N, K, sxm, swn, sym, syn, e, st)
  const bool few = M <= 8;
  if (rows == 8) {
    if (few) FD_RUN(1, 8, 8); else FD_RUN(1, 8, 16);
  }
  if (rows == 24) {
    if constexpr (sizeof(W) == 1)
      if (few && ((int64_t)N + 23) / 24 <= device_cus()) FD_RUN(3, 8, 8);
    if (few) FD_RUN(3, 4, 8); else FD_RUN(3, 4, 16);
  }
  if constexpr (sizeof(W) == 1)
    if (rows == 32) {
      if (few) FD_RUN(4, 4, 8); else FD_RUN(4, 4, 16);
    }
#undef FD_RUN
  return set_error(FD_EINVAL, "no launch of %d weight rows", rows);
}

#define FD_OCT(T, W)                                                                                            \
  template int launch_oct<T, W>(int, int, void*, const void*, const void*, const float*, int, int, int64_t, int64_t, \
                                int64_t, int64_t, const Epi&, hipStream_t)
FD_OCT(f16, f16);
FD_OCT(bf16, bf16);
FD_OCT(f16, uint8_t);
FD_OCT(bf16, uint8_t);
#undef FD_OCT

}  // namespace fd

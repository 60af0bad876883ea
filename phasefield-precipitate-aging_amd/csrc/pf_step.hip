// pf_step.hip -- fused KKS phase-field step for gfx950 (MI355X).
//
// One launch replaces the reference's per-step sequence (src/main.cpp:289-305):
//   boundaries -> fictitious compositions -> boundaries -> 4 Laplacians ->
//   boundaries -> Cahn-Hilliard || Allen-Cahn   (29 launches, 24 host syncs)
// and, on nucleation steps, the nucleation pass (src/discretization.cu:1079-1177).
// The per-strip arithmetic is pf::march (pf_march.h).  This kernel maps one
// wave to one (strip, row chunk), four adjacent strips per block, with blocks
// renumbered so that each of the 8 XCDs (each with its own L2) works on a
// contiguous band of the domain and halo re-reads stay inside one L2.
#include <hip/hip_runtime.h>

#include "pf_march.h"

namespace pf {

template <typename T, int BC, Mask MASK, bool NUC, int DEPTH>
__global__ __launch_bounds__(WAVE * WPB) void step_kernel(
    const T* __restrict__ iCr, const T* __restrict__ iNb, const T* __restrict__ ipd,
    const T* __restrict__ ipl, T* __restrict__ oCr, T* __restrict__ oNb, T* __restrict__ opd,
    T* __restrict__ opl, int Nx, int Ny, int pitch, int strips, int chunks, int rows, int remap,
    StepParams P, NucParams N, Scratch S) {
  const int nwaves = strips * chunks;
  const int nblocks = (nwaves + WPB - 1) / WPB;
  const int b = (remap ? xcd_remap(blockIdx.x, nblocks) : (int)blockIdx.x) * WPB +
                __builtin_amdgcn_readfirstlane((int)(threadIdx.x / WAVE));  // wave-uniform
  if (b >= nwaves) return;  // whole wave exits; no barriers in this kernel
  march<T, BC, MASK, NUC, DEPTH>(iCr, iNb, ipd, ipl, oCr, oNb, opd, opl, Nx, Ny, pitch,
                                 b % strips, b / strips, rows, P, N, S);
}

int default_rows(int nx, int ny) {
  // enough blocks to fill 256 CUs several times over, long enough chunks to
  // amortise the two halo rows
  const int Nx = nx - 2, Ny = ny - 2;
  const int strips = (Nx + STRIP - 1) / STRIP;
  int rows = 16;
  while (rows > 4 && (long)strips * ((Ny + rows - 1) / rows) < 16384) rows >>= 1;
  return rows;
}

template <typename T, int BC, Mask MASK, bool NUC, int DEPTH>
static hipError_t launch_step_t(int nx, int ny, const StepParams& P, const T* iCr, const T* iNb,
                                const T* ipd, const T* ipl, T* oCr, T* oNb, T* opd, T* opl,
                                const NucParams& N, const Scratch& S, const TileConfig& tc,
                                hipStream_t st) {
  const int Nx = nx - 2, Ny = ny - 2;
  const int rows = tc.rows > 0 ? tc.rows : default_rows(nx, ny);
  const int strips = (Nx + STRIP - 1) / STRIP;
  const int chunks = (Ny + rows - 1) / rows;
  const int blocks = (strips * chunks + WPB - 1) / WPB;
  hipLaunchKernelGGL((step_kernel<T, BC, MASK, NUC, DEPTH>), dim3(blocks), dim3(WAVE * WPB),
                     0, st, iCr, iNb, ipd, ipl, oCr, oNb, opd, opl, Nx, Ny, nx, strips, chunks,
                     rows, tc.remap, P, N, S);
  return hipGetLastError();
}

// The plain five-point step without nucleation (every step but one in ~900)
// is instantiated for prefetch depths 2, 3 and 6; the rarer variants use 3.
template <typename T, int BC>
static hipError_t launch_plain(int nx, int ny, const StepParams& P, const T* iCr, const T* iNb,
                               const T* ipd, const T* ipl, T* oCr, T* oNb, T* opd, T* opl,
                               const NucParams& N, const Scratch& S, const TileConfig& tc,
                               hipStream_t st) {
  if (tc.depth == 2)
    return launch_step_t<T, BC, FIVE, false, 2>(nx, ny, P, iCr, iNb, ipd, ipl, oCr, oNb, opd,
                                                 opl, N, S, tc, st);
  if (tc.depth == 6)
    return launch_step_t<T, BC, FIVE, false, 6>(nx, ny, P, iCr, iNb, ipd, ipl, oCr, oNb, opd,
                                                 opl, N, S, tc, st);
  return launch_step_t<T, BC, FIVE, false, 3>(nx, ny, P, iCr, iNb, ipd, ipl, oCr, oNb, opd, opl,
                                               N, S, tc, st);
}

template <typename T>
hipError_t launch_step(int nx, int ny, int bc, const StepParams& P, const T* iCr, const T* iNb,
                       const T* ipd, const T* ipl, T* oCr, T* oNb, T* opd, T* opl,
                       const NucParams* nuc, const Scratch& S, const TileConfig& tc,
                       hipStream_t st) {
  NucParams N{};
  if (nuc) N = *nuc;
#define PF_LAUNCH(BCV, MASK)                                                                    \
  do {                                                                                          \
    if (nuc)                                                                                    \
      return launch_step_t<T, BCV, MASK, true, 3>(nx, ny, P, iCr, iNb, ipd, ipl, oCr, oNb, opd, \
                                                  opl, N, S, tc, st);                           \
    if (MASK != FIVE)                                                                           \
      return launch_step_t<T, BCV, MASK, false, 3>(nx, ny, P, iCr, iNb, ipd, ipl, oCr, oNb,     \
                                                   opd, opl, N, S, tc, st);                     \
    return launch_plain<T, BCV>(nx, ny, P, iCr, iNb, ipd, ipl, oCr, oNb, opd, opl, N, S, tc,    \
                                st);                                                            \
  } while (0)
  const bool five = folded_five_point(P.m), nine = symmetric_nine_point(P.m);
  if (bc == 0) {
    if (five) PF_LAUNCH(0, FIVE);
    if (nine) PF_LAUNCH(0, NINE);
    PF_LAUNCH(0, ANY);
  }
  if (five) PF_LAUNCH(1, FIVE);
  if (nine) PF_LAUNCH(1, NINE);
  PF_LAUNCH(1, ANY);
#undef PF_LAUNCH
}

// ---- K steps per launch (marchk, K = 2, 3 or 4) ----

template <typename T, int BC, int K, int DEPTH, bool MODES, Mask MASK = FIVE>
__global__ __launch_bounds__(WAVE * WPB) void stepk_kernel(
    const T* __restrict__ iCr, const T* __restrict__ iNb, const T* __restrict__ ipd,
    const T* __restrict__ ipl, T* __restrict__ oCr, T* __restrict__ oNb, T* __restrict__ opd,
    T* __restrict__ opl, int Nx, int Ny, int pitch, int strips, int chunks, int rows, int remap,
    StepParams P) {
  const int nwaves = strips * chunks;
  const int nblocks = (nwaves + WPB - 1) / WPB;
  const int b = (remap ? xcd_remap(blockIdx.x, nblocks) : (int)blockIdx.x) * WPB +
                __builtin_amdgcn_readfirstlane((int)(threadIdx.x / WAVE));  // wave-uniform
  if (b >= nwaves) return;
  marchk<T, BC, K, DEPTH, WAVE - 2 * K, false, MODES, MASK>(
      iCr, iNb, ipd, ipl, oCr, oNb, opd, opl, Nx, Ny, pitch, b % strips, b / strips, rows, P);
}

// Four steps: the rows behind of the four levels' windows live in LDS (8 KiB
// per wave, 32 KiB per block of WPB = 4 waves); 231-247 VGPRs allow two waves
// per SIMD and the register budget is set to match.  At three waves per SIMD
// (168 VGPRs) it spills and takes twice as long.  FP64 4096^2, us per launch: on
// a domain full of particles 324-334, bound by FP64 issue (380 before the sums
// of update_cell were nested and its constant addends kept in vector registers);
// without precipitates 269 at 4.3 TB/s, bound by its 1.17 GB of traffic (331
// before the modes, MODE_ROWS).
template <typename T, int BC, int DEPTH, bool MODES, Mask MASK = FIVE, bool FAIR = false>
__global__ __launch_bounds__(WAVE * WPB) __attribute__((amdgpu_waves_per_eu(2, 2)))
void step4_kernel(const T* __restrict__ iCr, const T* __restrict__ iNb,
                  const T* __restrict__ ipd, const T* __restrict__ ipl, T* __restrict__ oCr,
                  T* __restrict__ oNb, T* __restrict__ opd, T* __restrict__ opl, int Nx, int Ny,
                  int pitch, int strips, int chunks, int rows, int remap, StepParams P) {
  constexpr int K = 4;
  constexpr int PER_WAVE = K * 4 * WAVE;  // levels x values x lanes
  __shared__ double win_lds[WPB * PER_WAVE];
  const int nwaves = strips * chunks;
  const int nblocks = (nwaves + WPB - 1) / WPB;
  const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / WAVE));  // wave-uniform
  const int b = (remap ? xcd_remap(blockIdx.x, nblocks) : (int)blockIdx.x) * WPB + w;
  if (b >= nwaves) return;
  marchk<T, BC, K, DEPTH, WAVE - 2 * K, true, MODES, MASK, FAIR>(
      iCr, iNb, ipd, ipl, oCr, oNb, opd, opl, Nx, Ny, pitch, b % strips, b / strips, rows, P,
      (LdsPtr)win_lds + w * PER_WAVE);
}

// Four steps on a small grid.  A march takes some ten iterations of four
// dependent levels however short its chunks are, and a small grid has too few
// waves to hide them: 7 us of latency.  Here a block takes a tile of TX x TY
// output cells with a halo of four, one cell per thread, and all threads go
// through the four levels together, exchanging a level's values through LDS
// (two buffers, so one barrier per level).  The cells of the halo are computed
// by every block that needs them, (TX + 8)(TY + 8) / (TX TY) times the work,
// which is why larger grids march.
template <typename T, int BC, int TX, int TY>
__global__ __launch_bounds__((TX + 8) * (TY + 8)) void tile4_kernel(
    const T* __restrict__ iCr, const T* __restrict__ iNb, const T* __restrict__ ipd,
    const T* __restrict__ ipl, T* __restrict__ oCr, T* __restrict__ oNb, T* __restrict__ opd,
    T* __restrict__ opl, int Nx, int Ny, int pitch, int tiles_x, StepParams P) {
  constexpr int K = 4, W = TX + 2 * K, H = TY + 2 * K, CELLS = W * H;
  __shared__ double buf[2][4][CELLS];
  const int b = xcd_remap(blockIdx.x, gridDim.x);
  const int tid = threadIdx.x;
  const int tx = tid % W, ty = tid / W;
  const int gx = (b % tiles_x) * TX + tx - K, gy = (b / tiles_x) * TY + ty - K;
  Raw<T> r;
  load_row(r, iCr, iNb, ipd, ipl, (size_t)(1 + bc_map<BC>(gy, Ny)) * pitch * sizeof(T),
           (uint32_t)(1 + bc_map<BC>(gx, Nx)) * (uint32_t)sizeof(T));
  // neighbours; on the tile's rim, whose values no output needs, the cell itself
  const int w = tx > 0 ? tid - 1 : tid, e = tx < W - 1 ? tid + 1 : tid;
  const int s = ty > 0 ? tid - W : tid, n = ty < H - 1 ? tid + W : tid;
  const Addends ad = addends(P);
  Point v;
  Centre c;
  derive<T>(ad, r, v, c);
#pragma unroll
  for (int l = 0; l < K; l++) {
    double(*f)[CELLS] = buf[l & 1];
    f[0][tid] = v.pd;
    f[1][tid] = v.pl;
    f[2][tid] = v.mu0;
    f[3][tid] = v.mu1;
    __syncthreads();
    const double own[4] = {v.pd, v.pl, v.mu0, v.mu1};
    double lap[4], o[4];
#pragma unroll
    for (int q = 0; q < 4; q++) lap[q] = five_point(P.m, f[q][s], f[q][w], own[q], f[q][e], f[q][n]);
    update_cell(P, ad, lap, v, c, o[0], o[1], o[2], o[3]);
    if (l < K - 1) {
      derive<T>(ad, Raw<T>{(T)o[0], (T)o[1], (T)o[2], (T)o[3]}, v, c);
    } else if (tx >= K && tx < K + TX && ty >= K && ty < K + TY && gx < Nx && gy < Ny) {
      store4(oCr, oNb, opd, opl, (size_t)(1 + gy) * pitch + 1 + gx, o[0], o[1], o[2], o[3]);
      store_ghost_images<T, BC>(oCr, oNb, opd, opl, gx, gy, Nx, Ny, pitch, o[0], o[1], o[2],
                                o[3]);
    }
  }
}

// Side of the tiles of a small grid, 0 where it marches.  A tile of 8, 12 or 16
// is 4, 7 or 9 waves; with one tile per CU (256) the smallest that covers the
// grid is the fastest, then two of 12 per CU, then two of 16.  us per launch
// (FP64, back to back), march / tiles of 8 / 12 / 16: 128^2 7.6 / 4.3 / 4.9 /
// 5.5, 192^2 7.7 / 5.6 / 4.9 / 5.6, 256^2 8.8 / 6.5 / 6.2 / 5.7, 131 x 515
// 8.8 / 7.0 / 6.2 / 7.3, 340^2 10.1 / 9.3 / 9.1 / 7.5, 384^2 10.2 / 10.4 / 9.4
// / 10.1, 512^2 (14 / - / - / 14.3) and up the march.
static int tile_side(int Nx, int Ny) {
  auto tiles = [&](int side) {
    return (long)((Nx + side - 1) / side) * ((Ny + side - 1) / side);
  };
  for (int side : {8, 12, 16})
    if (tiles(side) <= 256) return side;
  for (int side : {12, 16})
    if (tiles(side) <= 512) return side;
  return 0;
}

// Chunk height of the four-step kernel from a model of its launch on
// MI355X: 256 CUs x 4 SIMDs hold 2048 waves at two waves per SIMD.  A wave's
// time is proportional to its rows plus the 3 rows (K - 1) its levels
// recompute per chunk; a SIMD running two waves delivers 1.3x one wave's
// throughput, so a full round of resident waves costs 2/1.3 wave-times and a
// last partial round of at most one wave per SIMD costs one.  The height
// that minimises (rows + 3) x (rounds) is the measured best, or within 0.7%
// of it, from 1024^2 to 8192^2 (e.g. 10 rows at 1024^2, 38 at 2048^2, 75 at
// 4096^2, 119 at 8192^2).
static int rows4_model(int strips, int Ny) {
  constexpr long RESIDENT = 2048;
  constexpr double PAIR = 2.0 / 1.3, HALO = 3.0;
  int best = 1;
  double best_cost = 1e300;
  for (int rows = 1; rows <= min(Ny, 128); rows++) {
    const long waves = (long)strips * ((Ny + rows - 1) / rows);
    const long full = waves / RESIDENT, rem = waves % RESIDENT;
    const double tail = rem == 0 ? 0.0 : (rem <= RESIDENT / 2 ? 1.0 : PAIR);
    const double cost = (rows + HALO) * (PAIR * (double)full + tail);
    if (cost < best_cost) {
      best_cost = cost;
      best = rows;
    }
  }
  return best;
}

// Chunks of this height and more run the march with modes (matrix and quiet
// rows apart, pf_march.h).  The 2K rows of a chunk's prologue, which are dense or
// matrix but never quiet, and three times the code do not pay on short chunks
// (2 rows, 256^2: 10.5 against 8.8 us per launch) unless the waves share their
// SIMDs fairly (fair_shares).  From here on, us per launch without / with modes:
//   FP64 4096^2, 75 rows, four steps: no precipitate 300 / 265, one particle's
//   tail over the domain 314 / 282, particles everywhere 324 / 328;
//   FP64 2048^2, 38 rows: 80.0 / 65.6, 86.5 / 88.3 with particles everywhere;
//   FP32 8192^2, 48 rows, three steps: 790 / 567, 802 / 818.
constexpr int MODE_ROWS = 32;
// The same for nine-point masks, whose rows cost more.  us per four-step launch
// with four particles in the domain / particles everywhere, without, then with
// modes: FP64 1021 x 1543, 15 rows: 42.3 / 45.0, 40.6 / 46.5; 2048 x 1536, 28
// rows: 67.1 / 73.9, 53.8 / 76.8; 2000^2, 37 rows: 82.0 / 89.7, 65.6 / 92.9.
// FP32 shares its SIMDs fairly besides, where fair_shares says so (2000^2: 82.8
// / 83.1, 64.0 / 88.7, 62.0 / 84.8); in FP64 that spills (2000^2: 89.5 / 102.5).
constexpr int NINE_MODE_ROWS = 20;

// Whether the four-step launch shares its SIMDs fairly (FAIR, pf_march.h): where
// all of it is resident at once, two waves on most SIMDs, and the chunks are
// long enough to be cut in quarters.  The launch then ends with its slowest
// wave, and where a domain has both matrix and precipitates the modes make
// waves differ more, so the two go together.  us per launch with four
// particles in the domain / particles everywhere, FAIR without modes, modes
// without FAIR, both:
//   FP64 2048 x 1536, 28 rows: 59.3 / 65.4, 49.7 / 70.2, 49.0 / 66.1;
//   FP64 1700 x 1500, 23 rows: 51.2 / 56.5, 45.5 / 58.8, 44.3 / 57.6;
//   FP64 1021 x 1543, 15 rows: 38.2 / 39.3, 35.5 / 42.7, 35.5 / 41.1;
//   FP32 1800 x 1450, 24 rows: 52.9 / 53.5, 43.7 / 59.4, 41.1 / 57.6;
//   FP32 1400 x 1100, 14 rows: 35.9 / 36.8, 33.1 / 39.8, 31.5 / 38.1.
// FP32 takes it on long chunks too (2048^2, 38 rows: 67.5 / 86.5 with modes
// alone, 65.8 / 81.2; 2400 x 2300, 49 rows: 79.2 / 108.4, 76.2 / 101.6); FP64,
// nearer its traffic there and with some registers spilled, does not (2048^2:
// 71.5 / 88.7, 79.5 / 86.6).  With later rounds the waves are staggered anyway
// and the rule holds the old ones back (4096^2, 60 rows: 329 / 357), and on
// chunks of one trip it holds back the prologues (700^2, 6 rows: 17.9 / 18.9).
static bool fair_shares(long waves, int rows, int storage_bytes) {
  return waves > 1024 && waves <= 2048 && rows >= 12 &&
         (storage_bytes == 4 || rows < MODE_ROWS);
}

int default_rows_k(int k, int nx, int ny, int storage_bytes) {
  // The intermediate levels recompute (K-1)K rows per chunk in all, so chunks
  // are longer than the one-step kernel's while the grid still fills the chip.
  // Two steps: FP64 storage is near the HBM bound and prefers more waves in
  // flight (16 rows at 4096^2); FP32 storage is bound by arithmetic and
  // prefers less recomputation (32).  Three steps are bound by arithmetic in
  // both and take 48 rows at 4096^2.  Four steps: rows4_model.
  const int Nx = nx - 2, Ny = ny - 2;
  const int sw = WAVE - 2 * k;
  const int strips = (Nx + sw - 1) / sw;
  if (k == 4) return rows4_model(strips, Ny);
  int rows = k == 3 ? 48 : (storage_bytes == 8 ? 16 : 32);
  const long min_waves = k == 3 ? 4096 : 8192;
  while (rows > 6 && (long)strips * ((Ny + rows - 1) / rows) < min_waves) rows >>= 1;
  return rows;
}

template <typename T, int BC, int K, int DEPTH>
static hipError_t launch_stepk_t(int nx, int ny, const StepParams& P, const T* iCr,
                                 const T* iNb, const T* ipd, const T* ipl, T* oCr, T* oNb,
                                 T* opd, T* opl, int rows_cfg, int remap, hipStream_t st) {
  const int Nx = nx - 2, Ny = ny - 2;
  const int rows = rows_cfg > 0 ? rows_cfg : default_rows_k(K, nx, ny, (int)sizeof(T));
  const int sw = WAVE - 2 * K;
  const int strips = (Nx + sw - 1) / sw;
  const int chunks = (Ny + rows - 1) / rows;
  const int blocks = (strips * chunks + WPB - 1) / WPB;
#define PF_LAUNCH_MARCH(KERNEL)                                                                 \
  hipLaunchKernelGGL(KERNEL, dim3(blocks), dim3(WAVE * WPB), 0, st, iCr, iNb, ipd, ipl, oCr,    \
                     oNb, opd, opl, Nx, Ny, nx, strips, chunks, rows, remap, P)
  if constexpr (K != 3) {
    if (!folded_five_point(P.m)) {
      if constexpr (K == 4) {
        constexpr bool F32 = sizeof(T) == sizeof(float);
        if (rows < NINE_MODE_ROWS)
          PF_LAUNCH_MARCH((step4_kernel<T, BC, 3, false, NINE>));
        else if (F32 && fair_shares((long)strips * chunks, rows, (int)sizeof(T)))
          PF_LAUNCH_MARCH((step4_kernel<T, BC, F32 ? 3 : 4, true, NINE, F32>));
        else
          PF_LAUNCH_MARCH((step4_kernel<T, BC, 4, true, NINE>));
      } else {
        PF_LAUNCH_MARCH((stepk_kernel<T, BC, K, 3, false, NINE>));
      }
      return hipGetLastError();
    }
  }
  if constexpr (K == 4) {
    const int tile = rows_cfg == 0 ? tile_side(Nx, Ny) : 0;
    if (tile) {
      const int tiles_x = (Nx + tile - 1) / tile, tiles = tiles_x * ((Ny + tile - 1) / tile);
      const dim3 threads((tile + 8) * (tile + 8));
#define PF_LAUNCH_TILE(S)                                                                       \
  hipLaunchKernelGGL((tile4_kernel<T, BC, S, S>), dim3(tiles), threads, 0, st, iCr, iNb, ipd,   \
                     ipl, oCr, oNb, opd, opl, Nx, Ny, nx, tiles_x, P)
      if (tile == 8)
        PF_LAUNCH_TILE(8);
      else if (tile == 12)
        PF_LAUNCH_TILE(12);
      else
        PF_LAUNCH_TILE(16);
#undef PF_LAUNCH_TILE
      return hipGetLastError();
    }
    if (fair_shares((long)strips * chunks, rows, (int)sizeof(T)))
      PF_LAUNCH_MARCH((step4_kernel<T, BC, 3, true, FIVE, true>));
    else if (rows >= MODE_ROWS)
      PF_LAUNCH_MARCH((step4_kernel<T, BC, 4, true>));
    else
      PF_LAUNCH_MARCH((step4_kernel<T, BC, DEPTH, false>));
  } else if constexpr (K == 3 && sizeof(T) == sizeof(float)) {
    if (rows >= MODE_ROWS)
      PF_LAUNCH_MARCH((stepk_kernel<T, BC, K, 3, true>));
    else
      PF_LAUNCH_MARCH((stepk_kernel<T, BC, K, DEPTH, false>));
  } else {
    PF_LAUNCH_MARCH((stepk_kernel<T, BC, K, DEPTH, false>));
  }
#undef PF_LAUNCH_MARCH
  return hipGetLastError();
}

template <typename T>
hipError_t launch_stepk(int k, int nx, int ny, int bc, const StepParams& P, const T* iCr,
                        const T* iNb, const T* ipd, const T* ipl, T* oCr, T* oNb, T* opd,
                        T* opl, const TileConfig& tc, hipStream_t st) {
  const int rows = k == 4 ? tc.rows4 : k == 3 ? tc.rows3 : tc.rows2;
  const int depth = k == 4 ? tc.depth4 : k == 3 ? tc.depth3 : tc.depth2;
#define PF_LAUNCHK(BCV, KV, D)                                                             \
  return launch_stepk_t<T, BCV, KV, D>(nx, ny, P, iCr, iNb, ipd, ipl, oCr, oNb, opd, opl, \
                                       rows, tc.remap, st)
#define PF_LAUNCHK_D(BCV, KV)          \
  do {                                 \
    if (depth == 2) PF_LAUNCHK(BCV, KV, 2); \
    if (depth == 6) PF_LAUNCHK(BCV, KV, 6); \
    PF_LAUNCHK(BCV, KV, 3);            \
  } while (0)
  if (k == 4) {
    if (bc == 0) PF_LAUNCHK_D(0, 4);
    PF_LAUNCHK_D(1, 4);
  }
  if (k == 3) {
    if (bc == 0) PF_LAUNCHK_D(0, 3);
    PF_LAUNCHK_D(1, 3);
  }
  if (bc == 0) PF_LAUNCHK_D(0, 2);
  PF_LAUNCHK_D(1, 2);
#undef PF_LAUNCHK_D
#undef PF_LAUNCHK
}

template hipError_t launch_stepk<double>(int, int, int, int, const StepParams&, const double*,
                                         const double*, const double*, const double*, double*,
                                         double*, double*, double*, const TileConfig&,
                                         hipStream_t);
template hipError_t launch_stepk<float>(int, int, int, int, const StepParams&, const float*,
                                        const float*, const float*, const float*, float*, float*,
                                        float*, float*, const TileConfig&, hipStream_t);

template hipError_t launch_step<double>(int, int, int, const StepParams&, const double*,
                                        const double*, const double*, const double*, double*,
                                        double*, double*, double*, const NucParams*,
                                        const Scratch&, const TileConfig&, hipStream_t);
template hipError_t launch_step<float>(int, int, int, const StepParams&, const float*,
                                       const float*, const float*, const float*, float*, float*,
                                       float*, float*, const NucParams*, const Scratch&,
                                       const TileConfig&, hipStream_t);

}  // namespace pf

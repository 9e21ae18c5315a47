// Wide-workgroup fused shrink + expand of batch rows: one workgroup of 16 waves per
// (16-token tile, range of output columns), for launches too small to fill
// the GPU with 4-wave workgroups, where the time is one workgroup's chain of
// memory round trips.
//
// The 16 waves split K, so that for K up to 1024 a wave's whole K range (and
// for K = 4096 half of it) is one round trip; their partials meet in LDS, summed
// pairwise and rounded once to the model dtype; then every wave expands
// 128 bytes of each of the tile's y rows per step.  The first step's B and y
// loads need nothing from the shrink and issue right behind its first loads, so
// the expand waits on LDS only.  Products are MFMA with fp32 sums and the
// epilogue is the expand's, as in the other fused kernel.  In fp32 the sums over K
// are kept in short chains, so that they are no less exact than a lane's share
// of K and a tree over 64 lanes (delta against 64 bits, K = 2048, rank 16: 1.2e-7, a
// wave per row 1.4e-7, one running sum per wave 2.3e-7; 64 x 60 rows, 2048 ->
// 1024, rank 16: 24 us, a wave per row 155 us).
//
// Tiles are 16 consecutive positions of one batch row, straight from the
// row -> slot map and the row lengths, with no plan and no scratch, at any K,
// N, row stride and element alignment: 16-byte accesses at element alignment
// (global memory allows them), and the elements past the last whole chunk of K
// or N one by one.  Ranks go in passes of 16 * JT, up to kWideRankMax.  Many
// rows of few positions at low ranks stay with the plain kernels
// (plain_rows_faster).
#include <algorithm>
#include <cmath>

#include "pl_common.h"

namespace {

constexpr int kWWaves = 16;
constexpr int kWThreads = 64 * kWWaves;
constexpr int kWRankBlock = 32;    // ranks of B held per expand block
constexpr int kWYBytes = 128;      // bytes of each y row a wave covers per expand step

struct pl_wide_args {
  const void* x;
  int64_t ldx;
  int32_t K;
  int32_t kw;  // K per wave, a multiple of one wave load
  void* y;
  int64_t ldy;
  int32_t N;
  int32_t cols;    // output columns per workgroup, a multiple of a 16-wave step
  int32_t slices;  // workgroups per tile
  const char* arena;
  const pl_slot_entry* table;
  int32_t num_slots;
  int32_t num_modules;
  int32_t module;
  const int32_t* row_slot;
  const int32_t* seq_lens;
  int32_t row_len;
  int32_t row_tiles;  // 16-position tiles per row
  int32_t tiles;      // rows * row_tiles
  int32_t epilogue;
};

// 16 bytes at element alignment.
typedef uint32_t pl_u32x4_el __attribute__((ext_vector_type(4), aligned(2)));
__device__ __forceinline__ pl_u32x4 pl_ld16_el_or0(const void* p, bool ok) {
  return *reinterpret_cast<const pl_u32x4_el*>(ok ? p : static_cast<const void*>(pl_zero16));
}

template <int DT>
struct pl_wide_shape {
  typedef typename pl_traits<DT>::T T;
  enum { kCols = kWYBytes / (int)sizeof(T) };  // columns per wave per step
  enum { kStepCols = kWWaves * kCols };        // columns per workgroup step
  enum { kPad = 16 / (int)sizeof(T) };
  enum { kTRow = kWideRankMax + kPad };  // staged intermediate [token][rank]
  enum { kDRow = kCols + kPad };         // per-wave delta tile [token][column]
};

template <int DT, int JT>
__global__ __launch_bounds__(kWThreads) void pl_lora_wide_rows(pl_wide_args a) {
  typedef typename pl_traits<DT>::T T;
  typedef typename pl_traits<DT>::T4 T4;
  typedef typename pl_traits<DT>::T8 T8;
  typedef pl_wide_shape<DT> S;
  constexpr int E = pl_traits<DT>::E;
  constexpr int kInstr = 4 * E;         // K (or ranks) covered by one wave load
  constexpr int kWCC = JT == 1 ? 4 : 2; // 16-byte chunks per lane per shrink step
  constexpr int kStep = kWCC * kInstr;  // K per shrink step
  constexpr int kPass = 16 * JT;        // ranks per shrink pass
  constexpr int kRSteps = kWRankBlock / kInstr;
  constexpr int kCT = S::kCols / 16;
  constexpr int kYLanes = S::kCols * (int)sizeof(T) / 16;
  constexpr int kYRows = 64 / kYLanes;
  constexpr int kYLoads = 16 / kYRows;
  union lds_t {
    pl_f32x4 red[kWWaves][JT][64];
    T delta[kWWaves][16 * S::kDRow];
  };
  __shared__ lds_t lds;
  __shared__ __attribute__((aligned(16))) T tt[16 * S::kTRow];

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int li = lane & 15;
  const int lg = lane >> 4;

  // a tile's column ranges run on one XCD: they reread its x rows and A
  const pl_xcd_slot ws = pl_xcd_map(a.slices);
  if (ws.g >= a.tiles) return;
  const int b = ws.g / a.row_tiles;
  const int m0 = (ws.g - b * a.row_tiles) * 16;
  const int len = min(min(a.seq_lens[b], a.row_len) - m0, 16);
  const int s = a.row_slot[b];
  if (len <= 0 || s <= 0 || s >= a.num_slots) return;
  const pl_slot_entry e = a.table[(int64_t)s * a.num_modules + a.module];
  const int rank = min(e.rank, kWideRankMax);  // the host guarantees rank <= kWideRankMax
  if (rank <= 0) return;
  const int r8 = e.rank8;
  const int K = a.K;
  const int N = a.N;
  const int64_t tok0 = (int64_t)b * a.row_len + m0;
  const T* __restrict__ x = reinterpret_cast<const T*>(a.x) + (tok0 + min(li, len - 1)) * a.ldx;
  const bool xok = li < len;
  const T* __restrict__ A = reinterpret_cast<const T*>(a.arena + e.a_off);
  const T* __restrict__ Bc = reinterpret_cast<const T*>(a.arena + e.b_off);

  // ---- expand set-up
  const int c1 = min(N, (ws.j + 1) * a.cols);
  const int c0 = ws.j * a.cols + wave * S::kCols;
  const int yq = lane % kYLanes;
  const int yr0 = lane / kYLanes;
  T* yrow[kYLoads];
  bool yok[kYLoads];
#pragma unroll
  for (int i = 0; i < kYLoads; ++i) {
    const int r = yr0 + kYRows * i;
    yok[i] = r < len;
    yrow[i] = reinterpret_cast<T*>(a.y) + (tok0 + min(r, len - 1)) * a.ldy + yq * E;
  }
  auto load_b = [&](pl_u32x4 (&bf)[kRSteps][kCT], int cb, int rb) {
#pragma unroll
    for (int q = 0; q < kRSteps; ++q) {
      // B's MFMA blocks: the 16-column tile at nb (nt columns), rank block
      // j0 (wb wide) starts at nb*r8 + j0*nt
      const int j0 = rb + q * kInstr;
      const int wb = min(kInstr, r8 - j0);
#pragma unroll
      for (int ct = 0; ct < kCT; ++ct) {
        const int nb = cb + ct * 16;
        const int nt = min(16, N - nb);
        bf[q][ct] = pl_ld16_or0(Bc + (int64_t)nb * r8 + (int64_t)j0 * nt + li * wb + lg * E,
                                nb + li < c1 && j0 + lg * E < r8);
      }
    }
  };
  auto load_y = [&](pl_u32x4 (&yv)[kYLoads], int cb) {
#pragma unroll
    for (int i = 0; i < kYLoads; ++i)
      yv[i] = pl_ld16_el_or0(yrow[i] + cb, yok[i] && cb + yq * E + E <= c1);
  };
  pl_u32x4 bf[kRSteps][kCT], yv[kYLoads];

  // ---- shrink: t[token][j] = T(sum_k x[token][k] * A[j][k]), every rank pass
  const int k0 = wave * a.kw;
  const int k1 = min(K, k0 + a.kw);
  for (int rb = 0; rb < rank; rb += kPass) {
    pl_f32x4 acc[JT];
#pragma unroll
    for (int jt = 0; jt < JT; ++jt) acc[jt] = pl_f32x4{0.f, 0.f, 0.f, 0.f};
    auto load_k = [&](pl_u32x4 (&xf)[kWCC], pl_u32x4 (&af)[JT][kWCC], int kb) {
#pragma unroll
      for (int cc = 0; cc < kWCC; ++cc) {
        const int k = kb + cc * kInstr;
        xf[cc] = pl_ld16_el_or0(x + k + lg * E, xok && k + lg * E + E <= k1);
      }
#pragma unroll
      for (int jt = 0; jt < JT; ++jt) {
        // rank tile of A's MFMA blocks (rt rows): the block of columns k
        // starts at t0*K + k*rt and is wb wide
        const int t0 = rb + jt * 16;
        const int rt = min(16, rank - t0);
#pragma unroll
        for (int cc = 0; cc < kWCC; ++cc) {
          const int k = kb + cc * kInstr;
          const int wb = min(kInstr, K - k);
          af[jt][cc] = pl_ld16_el_or0(A + (int64_t)t0 * K + (int64_t)k * rt + li * wb + lg * E,
                                      li < rt && k + lg * E + E <= k1);
        }
      }
    };
    auto mfma_k = [&](const pl_u32x4 (&xf)[kWCC], const pl_u32x4 (&af)[JT][kWCC]) {
#pragma unroll
      for (int jt = 0; jt < JT; ++jt)
#pragma unroll
        for (int cc = 0; cc < kWCC; ++cc) acc[jt] = pl_mfma_chunk_short<DT>(xf[cc], af[jt][cc], acc[jt]);
    };
    pl_u32x4 xf[kWCC], af[JT][kWCC];
    load_k(xf, af, k0);
    if (rb == 0) {
      load_b(bf, c0, 0);
      load_y(yv, c0);
    }
    __builtin_amdgcn_sched_barrier(0);
    mfma_k(xf, af);
    for (int kb = k0 + kStep; kb < k1; kb += kStep) {
      load_k(xf, af, kb);
      __builtin_amdgcn_sched_barrier(0);
      mfma_k(xf, af);
    }
    const int kt = K - K % E;  // the elements past the last whole chunk of K
    if (kt < k1 && kt >= k0) {
      const int n = lg == 0 ? K - kt : 0;
      T xe[E], ae[E];
#pragma unroll
      for (int q = 0; q < E; ++q) xe[q] = (xok && q < n) ? x[kt + q] : (T)0.f;
#pragma unroll
      for (int jt = 0; jt < JT; ++jt) {
        const int j = rb + jt * 16 + li;
        const T* __restrict__ Aj = A + (j < rank ? pl_tile_off<DT>(j, kt, rank, K) : 0);
#pragma unroll
        for (int q = 0; q < E; ++q) ae[q] = (j < rank && q < n) ? Aj[q] : (T)0.f;
        acc[jt] = pl_mfma_chunk_short<DT>(__builtin_bit_cast(pl_u32x4, xe), __builtin_bit_cast(pl_u32x4, ae), acc[jt]);
      }
    }

    // the 16 wave partials summed pairwise, rounded once to T;
    // acc[jt][v] holds (token 4*lg+v, rank rb + jt*16 + li)
    if (rb > 0) __syncthreads();  // the previous pass's sums are read
#pragma unroll
    for (int jt = 0; jt < JT; ++jt) lds.red[wave][jt][lane] = acc[jt];
    __syncthreads();
    if (tid < JT * 256) {
      const int jt = tid >> 8;
      const int l = (tid >> 2) & 63;
      const int v = tid & 3;
      float p[kWWaves];
#pragma unroll
      for (int w = 0; w < kWWaves; ++w) p[w] = lds.red[w][jt][l][v];
#pragma unroll
      for (int h = kWWaves / 2; h > 0; h /= 2)
#pragma unroll
        for (int w = 0; w < h; ++w) p[w] += p[w + h];
      const int j = rb + jt * 16 + (l & 15);
      tt[((l >> 4) * 4 + v) * S::kTRow + j] = (T)(j < rank ? p[0] : 0.f);
    } else if (kPass < kInstr && tid < JT * 256 + 16 * (kInstr - kPass)) {
      // the ranks past the pass that an expand block reads: zeros, until a later pass writes them
      const int i = tid - JT * 256;
      tt[(i / (kInstr - kPass)) * S::kTRow + rb + kPass + i % (kInstr - kPass)] = (T)0.f;
    }
  }
  __syncthreads();

  // ---- expand over this wave's columns
  const float scale = e.scale;
  const float scale_t = pl_round<DT>(scale);
  T* __restrict__ dw = lds.delta[wave];
  for (int cb = c0; cb < c1; cb += S::kStepCols) {
    pl_f32x4 d[kCT];
#pragma unroll
    for (int ct = 0; ct < kCT; ++ct) d[ct] = pl_f32x4{0.f, 0.f, 0.f, 0.f};
    for (int rb = 0; rb < r8; rb += kWRankBlock) {
      if (rb > 0 || cb > c0) load_b(bf, cb, rb);
      if (rb == 0 && cb > c0) load_y(yv, cb);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int q = 0; q < kRSteps; ++q) {
        if (rb + q * kInstr < r8) {
          const pl_u32x4 tf =
              *reinterpret_cast<const pl_u32x4*>(tt + li * S::kTRow + rb + q * kInstr + lg * E);
#pragma unroll
          for (int ct = 0; ct < kCT; ++ct) d[ct] = pl_mfma_chunk<DT>(bf[q][ct], tf, d[ct]);
        }
      }
    }
    // d[ct][v] = delta(column cb + ct*16 + 4*lg + v, token li): scale and round,
    // then through this wave's LDS tile to the row-major layout of y
#pragma unroll
    for (int ct = 0; ct < kCT; ++ct) {
      T4 dd;
#pragma unroll
      for (int v = 0; v < 4; ++v) dd[v] = (T)pl_delta<DT>(d[ct][v], scale, scale_t, a.epilogue);
      *reinterpret_cast<T4*>(dw + li * S::kDRow + ct * 16 + lg * 4) = dd;
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
#pragma unroll
    for (int i = 0; i < kYLoads; ++i) {
      const int r = yr0 + kYRows * i;
      const pl_u32x4 dv = *reinterpret_cast<const pl_u32x4*>(dw + r * S::kDRow + yq * E);
      const int n = c1 - (cb + yq * E);
      T* yp = yrow[i] + cb;
      if (yok[i] && n >= E) {
        pl_u32x4 out;
        if constexpr (E == 8) {
          T8 yy = __builtin_bit_cast(T8, yv[i]);
          const T8 dd = __builtin_bit_cast(T8, dv);
#pragma unroll
          for (int q = 0; q < 8; ++q) yy[q] = (T)((float)yy[q] + (float)dd[q]);
          out = __builtin_bit_cast(pl_u32x4, yy);
        } else {
          out = __builtin_bit_cast(pl_u32x4, __builtin_bit_cast(pl_f32x4, yv[i]) + __builtin_bit_cast(pl_f32x4, dv));
        }
        *reinterpret_cast<pl_u32x4_el*>(yp) = out;
      } else if (yok[i] && n > 0) {
        const T* dd = dw + r * S::kDRow + yq * E;
        for (int q = 0; q < n; ++q) yp[q] = (T)((float)yp[q] + (float)dd[q]);
      }
    }
    // the next step rewrites the tile only after these reads (in-order LDS)
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  }
}

// Whether the plain row kernels (a wave per row, a thread per output) are
// the faster ones: with few positions per tile and low ranks the matrix cores
// multiply padding, and a round of 16-wave workgroups costs 7 us whatever its
// tiles hold.  Estimates of both in us, fitted to 2,370 sizes (1 to 16384
// positions in rows of 1 to 1024, ranks 1 to 256, K and N 1 to 16384), where
// the pick takes 1% more than the faster path on average and this kernel
// alone took 16% more.  Plain / this kernel, bf16: 4096 rows of 1, 768 -> 768,
// rank 1 17 / 66 us, rank 16 70 / 67; 4096 -> 4096, rank 1 76 / 154, rank 16 350 /
// 154; fp32: 64 rows of 1, 4096 -> 4096, rank 1 13 / 24, rank 16 130 / 24.
bool plain_rows_faster(int es, double T, double tiles, double per, double slices, double K, double N, double rank) {
  const double k64 = std::ceil(K / 64) * 64, n256 = std::ceil(N / 256) * 256;
  const double plain = 3 + 0.2 * rank + 1.2e-3 * rank * K +
                       1e-6 * T * (rank * (0.14 * k64 + 0.39 * n256) + es * (0.05 * K + 1.36 * N));
  const double r16 = std::max(rank, 16.0), f = es == 4 ? 1 : 0;
  const double round = 1.2 + 5.4 * per + (1 + 2 * f) * 2.8e-5 * r16 * K + (1 + f) * 0.044 * per * r16;
  const double wide = std::max(1.0, tiles * slices / 650) * round + 0.18e-6 * T * N * es;
  return 1.1 * std::max(plain, 10.0) < wide;  // two launches: never under 10
}

template <int DT>
void launch_wide_rows(const pl_wide_args& a, int32_t rank_cap, dim3 grid, hipStream_t s) {
  if (rank_cap <= 16)
    hipLaunchKernelGGL((pl_lora_wide_rows<DT, 1>), grid, dim3(kWThreads), 0, s, a);
  else
    hipLaunchKernelGGL((pl_lora_wide_rows<DT, 2>), grid, dim3(kWThreads), 0, s, a);
}

}  // namespace

int pl_wide_rows_launch(int32_t dtype, const void* x, int64_t ldx, int32_t K, void* y, int64_t ldy,
                        int32_t N, const void* arena, const pl_slot_entry* table, int32_t num_slots,
                        int32_t num_modules, int32_t module, const int32_t* row_slot,
                        const int32_t* seq_lens, int32_t rows, int32_t row_len, int32_t rank_cap,
                        int32_t epilogue, void* stream) {
  const int64_t row_tiles = ((int64_t)row_len + 15) / 16;
  const int64_t tiles = rows * row_tiles;
  if (rank_cap < 1 || rank_cap > kWideRankMax || tiles > (int64_t)1 << 24) return PL_WIDE_DECLINED;
  // y may lie over x: the workgroup of a tile reads all of its x rows before it
  // writes y, but several column ranges, or several tiles, run side by side
  const pl_overlap overlap = pl_row_overlap(x, ldx, K, y, ldy, N, (int64_t)rows * row_len, pl_elem_size(dtype));
  if (overlap == pl_overlap::across) return PL_WIDE_DECLINED;
  const int step_cols = dtype == PL_F32 ? (int)pl_wide_shape<PL_F32>::kStepCols
                                        : (int)pl_wide_shape<PL_BF16>::kStepCols;
  // column ranges until the launch has about two workgroups per CU: each
  // range repeats the tile's shrink
  const int64_t steps = (N + step_cols - 1) / step_cols;
  const int64_t want = overlap == pl_overlap::own_row ? 1 : std::max<int64_t>(1, 512 / std::max<int64_t>(1, tiles));
  const int64_t per = (steps + std::min(want, steps) - 1) / std::min(want, steps);
  pl_wide_args a;
  a.cols = (int32_t)(per * step_cols);
  a.slices = (int32_t)((steps + per - 1) / per);
  if (!pl_grid_fits(pl_xcd_grid(tiles, a.slices), kWThreads)) return PL_WIDE_DECLINED;
  if (pl_grid_fits((int64_t)rows * row_len * (((int64_t)N + 255) / 256), 256) &&  // the plain kernels' grid
      plain_rows_faster(pl_elem_size(dtype), (double)rows * row_len, (double)tiles, (double)per, a.slices, K,
                        N, rank_cap))
    return PL_WIDE_DECLINED;
  a.x = x;
  a.ldx = ldx;
  a.K = K;
  const int instr = 4 * pl_chunk_elems(dtype);
  const int64_t per_wave = ((int64_t)K + kWWaves - 1) / kWWaves;
  a.kw = (int32_t)((per_wave + instr - 1) / instr * instr);
  a.y = y;
  a.ldy = ldy;
  a.N = N;
  a.arena = reinterpret_cast<const char*>(arena);
  a.table = table;
  a.num_slots = num_slots;
  a.num_modules = num_modules;
  a.module = module;
  a.row_slot = row_slot;
  a.seq_lens = seq_lens;
  a.row_len = row_len;
  a.row_tiles = (int32_t)row_tiles;
  a.tiles = (int32_t)tiles;
  a.epilogue = epilogue;
  const dim3 grid((unsigned)pl_xcd_grid(tiles, a.slices));
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  switch (dtype) {
    case PL_BF16: launch_wide_rows<PL_BF16>(a, rank_cap, grid, s); break;
    case PL_F16: launch_wide_rows<PL_F16>(a, rank_cap, grid, s); break;
    default: launch_wide_rows<PL_F32>(a, rank_cap, grid, s); break;
  }
  return pl_launch_status("pl_lora_apply_rows");
}

// Shrink and expand of long adapter segments as two streaming launches
// (prefill and large batches), gfx950.
//
// The shrink reads x once and leaves the intermediate t = T(x·Aᵀ), rounded
// once to the model dtype, in a workspace row per plan position; the expand
// streams y.  Each launch has one access pattern and a grid of its own: the
// expand's workgroups are short and sweep y's rows in order, which a
// read-modify-write wants (a probe over 705 MB of 28 KB rows: 5.7 TB/s with
// 2 KB of each row per workgroup, 5.0 TB/s when a workgroup walks whole
// rows).  Against one fused launch, whose workgroups run both phases, the
// second launch costs about 5 us, and that is paid back by large and wide
// outputs and by ranks above 32 (sgmv.long_ok).  bf16, before -> after:
//   4096 -> 2 x 14336, rank 32, 24740 tokens  642 -> 564 us (5.4 TB/s in the expand)
//   2048 -> 8192, rank 64, 4593 tokens         78 -> 46 us
//   14336 -> 4096, rank 32, 24740 tokens      268 -> 230 us
// and against the split shrink and expand above rank 64:
//   4096 -> 4096, rank 128, 4138 tokens        68 -> 43 us
//   14336 -> 4096, rank 128, 11557 tokens     338 -> 182 us
//
// Both kernels work on units of consecutive 16-token tiles of one XCD's plan
// positions.  The weights of a unit's slot are loaded once for all of its
// tiles: an A chunk feeds every tile's MFMAs, and an expand wave holds its
// columns' B in registers while the tiles' y rows stream past.  A unit whose
// tiles belong to several slots runs once per slot.
//
// What bounds them: a large expand the read-modify-write of y; the shrink at
// one or two workgroups per CU the latency of its K turns and the LDS traffic
// of its operands.  Splitting K over workgroups (fp32 planes, summed by the
// last to arrive) was slower at every size; 8 waves per workgroup left fewer,
// larger workgroups to balance over the CUs (rank 32 prefill 578 against 564 us).
//
// In fp32 the sums over K are kept in short chains (K = 4096, error of the delta
// against 64 bits: rank 64 2.1e-7, the fused launch 5.9e-7; rank 128 2.5e-7,
// the split pair 3.5e-7; 6.0e-7 with one running sum per wave).
#include <algorithm>

#include "pl_common.h"

namespace {

constexpr int kLJobs = PL_MAX_STACKED_MODULES;
constexpr int kLWaves = 4;        // waves per workgroup of both kernels
constexpr int kLUnitMax = 4;      // tiles per expand unit
constexpr int kLRowBytes = 256;   // bytes of each y row an expand wave owns

struct pl_long_args {
  const void* x;
  int64_t ldx;
  int32_t K;
  int32_t kw;        // shrink: K per wave, whole pairs of steps; 0: steps in turn (ranks above 64, fp32)
  const char* arena;
  const pl_slot_entry* table;
  int32_t num_modules;
  const int32_t* tok;
  const pl_group* groups;
  const int32_t* meta;
  int32_t group_cap;
  int32_t sub;       // 16-token tiles per plan group (1 or 4)
  int32_t epilogue;
  int32_t n_jobs;    // modules served, all fed the same x
  int32_t n_chunks;  // column chunks of all jobs together
  int32_t chunk0[kLJobs];
  int32_t module[kLJobs];
  void* t[kLJobs];   // intermediate [plan position][ldt], model dtype
  int32_t ldt;
  int32_t passes;    // rank passes of the shrink
  void* y[kLJobs];
  int64_t ldy[kLJobs];
  int32_t N[kLJobs];
};

struct pl_long_tile {
  int slot;   // 0: no tile
  int start;  // first plan position
  int len;    // tokens, 0..16
};

// The tiles of unit u on XCD x: tile L = u*NT + i is sub-tile L % sub of the
// group at plan position x + 8 * (L / sub).  Every record loads at once, with
// the count of positions in use, before any is looked at.
template <int NT>
__device__ __forceinline__ void pl_long_unit(const pl_long_args& a, int x, int u,
                                             pl_long_tile (&tl)[NT]) {
  pl_group grp[NT];
#pragma unroll
  for (int i = 0; i < NT; ++i) {
    const int L = u * NT + i;
    grp[i] = a.groups[min(x + kXcds * (a.sub == 1 ? L : L >> 2), a.group_cap - 1)];
  }
  const int n_groups = min(a.meta[3], a.group_cap);  // positions in use
#pragma unroll
  for (int i = 0; i < NT; ++i) {
    const int L = u * NT + i;
    const int off = a.sub == 1 ? 0 : (L & 3) * 16;
    const int len = min(grp[i].len - off, 16);
    const bool on = x + kXcds * (a.sub == 1 ? L : L >> 2) < n_groups && len > 0 && grp[i].slot > 0;
    tl[i].slot = on ? grp[i].slot : 0;
    tl[i].start = on ? grp[i].start + off : 0;
    tl[i].len = on ? len : 0;
  }
}

// ------------------------------------------------------------------ shrink

// A wave's x loads take whole 128-byte lines, 8 rows per load, and reach the
// MFMA layout through the wave's own LDS tile: reading x straight in MFMA
// layout, lanes 64 bytes apart, streams at 4.0-5.3 TB/s, in lines at 6.1-6.7.
template <int DT, int RT>
struct pl_long_xtile {
  typedef typename pl_traits<DT>::T T;
  enum { kPad = 16 / (int)sizeof(T) };
  enum { kRow = 128 / (int)sizeof(T) + kPad };  // elements per staged row
  enum { kBytes = 16 * RT * kRow * (int)sizeof(T) };
};

// A's blocks (16 rows x 64 bytes, contiguous) load in lane order, lane l
// taking piece l % 4 of row l / 4, and are staged piece-major: the 16-byte
// piece p of row r at p * 320 + r * 16, so that both the writes and the MFMA
// reads (lane (li, lg): piece lg of row li) are free of bank conflicts.
// Loaded in MFMA order, lanes 64 bytes apart, an L2-resident stream of such
// blocks runs at 17 TB/s, in lane order at 30 TB/s (256 CUs, 1 KB blocks).
constexpr int kLAPiece = 320;
constexpr int kLABlock = 4 * kLAPiece;

template <int DT, int JT, int RT>
constexpr int pl_long_stage_bytes() {
  return (int)pl_long_xtile<DT, RT>::kBytes + JT * 2 * kLABlock;
}

template <int DT, int JT, int RT>
constexpr int pl_long_shrink_lds() {
  return kLWaves * (pl_long_stage_bytes<DT, JT, RT>() > RT * JT * 1024 ? pl_long_stage_bytes<DT, JT, RT>()
                                                                             : RT * JT * 1024);
}

// SHARE: the waves take shares of K (a.kw), else K steps in turn.
template <int DT, int JT, int RT, int SB, bool XNT, bool SHARE>
__device__ __forceinline__ void pl_long_shrink_run(const pl_long_args& a, int job, int rb,
                                                   const pl_slot_entry& e,
                                                   const pl_long_tile (&tl)[RT],
                                                   const int (&xt)[2 * RT], char* smem) {
  typedef typename pl_traits<DT>::T T;
  typedef pl_long_xtile<DT, RT> X;
  constexpr int E = pl_traits<DT>::E;
  constexpr int kInstr = 4 * E;
  constexpr int kCC = 2;
  constexpr int kStep = kCC * kInstr;  // 128 bytes of each x row
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int li = lane & 15;
  const int lg = lane >> 4;
  const int xr = lane >> 3;
  const int xp = lane & 7;
  const int K = a.K;
  const int rank = e.rank;
  const T* __restrict__ A = reinterpret_cast<const T*>(a.arena + e.a_off);
  const T* __restrict__ x = reinterpret_cast<const T*>(a.x);
  const T* xrow[2 * RT];
#pragma unroll
  for (int i = 0; i < 2 * RT; ++i) xrow[i] = x + (int64_t)xt[i] * a.ldx + xp * E;
  char* stage = smem + wave * SB;
  T* __restrict__ xw = reinterpret_cast<T*>(stage);
  char* __restrict__ aw = stage + X::kBytes;
  T* __restrict__ t = reinterpret_cast<T*>(a.t[job]);

  pl_f32x4 acc[RT][JT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int jt = 0; jt < JT; ++jt) acc[rt][jt] = pl_f32x4{0.f, 0.f, 0.f, 0.f};
  auto load = [&](pl_u32x4 (&xf)[2 * RT], pl_u32x4 (&af)[JT][kCC], int kb) {
    // rows past a tile's tokens repeat its last one (their sums are not
    // stored); K past the range reads zeros
#pragma unroll
    for (int i = 0; i < 2 * RT; ++i) {
      if constexpr (XNT)
        xf[i] = pl_ld16_nt_or0(xrow[i] + kb, kb + xp * E < K);
      else
        xf[i] = pl_ld16_or0(xrow[i] + kb, kb + xp * E < K);
    }
#pragma unroll
    for (int jt = 0; jt < JT; ++jt) {
      // rank tile of A's MFMA blocks (rt rows): the block of columns k
      // starts at t0*K + k*rt and is wb wide
      const int t0 = rb + jt * 16;
      const int rt = min(16, rank - t0);
#pragma unroll
      for (int cc = 0; cc < kCC; ++cc) {
        const int k = kb + cc * kInstr;
        const int wb = min(kInstr, K - k);
        af[jt][cc] = pl_ld16_or0(A + (int64_t)t0 * K + (int64_t)k * rt + (lane >> 2) * wb + (lane & 3) * E,
                                 (lane >> 2) < rt && k + (lane & 3) * E < K);
      }
    }
  };
  auto mfma = [&](const pl_u32x4 (&xf)[2 * RT], const pl_u32x4 (&af)[JT][kCC]) {
#pragma unroll
    for (int i = 0; i < 2 * RT; ++i)
      *reinterpret_cast<pl_u32x4*>(xw + (xr + 8 * i) * X::kRow + xp * E) = xf[i];
#pragma unroll
    for (int jt = 0; jt < JT; ++jt)
#pragma unroll
      for (int cc = 0; cc < kCC; ++cc)
        *reinterpret_cast<pl_u32x4*>(aw + (jt * kCC + cc) * kLABlock + (lane & 3) * kLAPiece + (lane >> 2) * 16) = af[jt][cc];
    pl_u32x4 am[JT][kCC];
#pragma unroll
    for (int jt = 0; jt < JT; ++jt)
#pragma unroll
      for (int cc = 0; cc < kCC; ++cc)
        am[jt][cc] = *reinterpret_cast<const pl_u32x4*>(aw + (jt * kCC + cc) * kLABlock + lg * kLAPiece + li * 16);
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      pl_u32x4 xm[kCC];
#pragma unroll
      for (int cc = 0; cc < kCC; ++cc)
        xm[cc] = *reinterpret_cast<const pl_u32x4*>(xw + (rt * 16 + li) * X::kRow + cc * kInstr + lg * E);
#pragma unroll
      for (int jt = 0; jt < JT; ++jt)
#pragma unroll
        for (int cc = 0; cc < kCC; ++cc) acc[rt][jt] = pl_mfma_chunk_short<DT>(xm[cc], am[jt][cc], acc[rt][jt]);
    }
  };
  // a step past the range loads only zeros
  pl_u32x4 xa[2 * RT], aa[JT][kCC], xb[2 * RT], ab[JT][kCC];
  constexpr int next = SHARE ? kStep : kLWaves * kStep;
  const int k1 = SHARE ? min(K, (wave + 1) * a.kw) : K;
  int kb = wave * (SHARE ? a.kw : kStep);
  load(xa, aa, kb);
  for (; kb + 2 * next < k1; kb += 2 * next) {
    load(xb, ab, kb + next);
    __builtin_amdgcn_sched_barrier(0);
    mfma(xa, aa);
    load(xa, aa, kb + 2 * next);
    __builtin_amdgcn_sched_barrier(0);
    mfma(xb, ab);
  }
  if (kb < k1) {
    load(xb, ab, kb + next);
    __builtin_amdgcn_sched_barrier(0);
    mfma(xa, aa);
    __builtin_amdgcn_sched_barrier(0);
    mfma(xb, ab);
  }

  // the wave partials summed in wave order; acc[rt][jt][v] holds
  // (token 4*lg+v, rank rb + jt*16 + li)
  pl_f32x4(*red)[RT * JT][64] = reinterpret_cast<pl_f32x4(*)[RT * JT][64]>(smem);
  __syncthreads();  // every wave's x tile is read
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int jt = 0; jt < JT; ++jt) red[wave][rt * JT + jt][lane] = acc[rt][jt];
  __syncthreads();
#pragma unroll
  for (int q0 = 0; q0 < RT * JT; q0 += kLWaves) {
    const int q = q0 + wave;
    if (q < RT * JT) {
      pl_f32x4 s = red[0][q][lane];
#pragma unroll
      for (int w = 1; w < kLWaves; ++w) s += red[w][q][lane];
      const int rt = q / JT;
      const int j = rb + (q % JT) * 16 + li;
      int start = tl[0].start, len = tl[0].len;
#pragma unroll
      for (int i = 1; i < RT; ++i)
        if (rt == i) {
          start = tl[i].start;
          len = tl[i].len;
        }
      if (j < a.ldt) {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int row = lg * 4 + v;
          if (row < len) t[(int64_t)(start + row) * a.ldt + j] = (T)(j < rank ? s[v] : 0.f);
        }
      }
    }
  }
}

template <int DT, int JT, int RT, bool XNT, bool SHARE>
__global__ __launch_bounds__(64 * kLWaves, RT * JT <= 4 ? 3 : 2) void pl_long_shrink(pl_long_args a) {
  __shared__ __attribute__((aligned(16))) char smem[pl_long_shrink_lds<DT, JT, RT>()];
  const int xcd = (int)(blockIdx.x % kXcds);
  int rest = (int)(blockIdx.x / kXcds);
  // (job, rank pass) fastest: they read the same x
  const int job = rest % a.n_jobs;
  rest /= a.n_jobs;
  const int rb = rest % a.passes * (16 * JT);
  const int unit = rest / a.passes;
  pl_long_tile tl[RT];
  pl_long_unit<RT>(a, xcd, unit, tl);
  int any = 0;
#pragma unroll
  for (int i = 0; i < RT; ++i) any |= tl[i].slot;
  if (any == 0) return;
  const int xr = (threadIdx.x & 63) >> 3;
  int xt[2 * RT];
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int h = 0; h < 2; ++h)
      xt[2 * i + h] = tl[i].len > 0 ? a.tok[tl[i].start + min(xr + 8 * h, tl[i].len - 1)] : 0;
  // one run per slot among the unit's tiles (mostly one)
  int todo = 0;
#pragma unroll
  for (int i = 0; i < RT; ++i) todo |= tl[i].slot != 0 ? 1 << i : 0;
  bool wrote = false;
#pragma unroll 1
  while (todo != 0) {
    int slot = 0;
#pragma unroll
    for (int i = RT - 1; i >= 0; --i)
      if (todo >> i & 1) slot = tl[i].slot;
    pl_long_tile run[RT];
#pragma unroll
    for (int i = 0; i < RT; ++i) {
      run[i] = {slot, tl[i].start, tl[i].slot == slot ? tl[i].len : 0};
      if (tl[i].slot == slot) todo &= ~(1 << i);
    }
    const pl_slot_entry e = a.table[(int64_t)slot * a.num_modules + a.module[job]];
    if (rb >= e.rank) continue;
    if (wrote) __syncthreads();  // the previous run's sums are read
    wrote = true;
    if (JT > 1 && e.rank - rb <= 16)
      pl_long_shrink_run<DT, 1, RT, pl_long_stage_bytes<DT, JT, RT>(), XNT, SHARE>(a, job, rb, e, run, xt, smem);
    else if (JT > 2 && e.rank - rb <= 32)
      pl_long_shrink_run<DT, JT < 2 ? JT : 2, RT, pl_long_stage_bytes<DT, JT, RT>(), XNT, SHARE>(a, job, rb, e, run, xt, smem);
    else
      pl_long_shrink_run<DT, JT, RT, pl_long_stage_bytes<DT, JT, RT>(), XNT, SHARE>(a, job, rb, e, run, xt, smem);
  }
}

// ------------------------------------------------------------------ expand

// Above two rank steps a wave owns half the columns, so that its B fits the
// registers of three workgroups per CU (rank 256, 5915 tokens, 4096 columns:
// 51 -> 40 us; rank 128, 4138 tokens: 24.7 -> 23.1 us).
template <int DT, int RSMAX>
struct pl_long_shape {
  typedef typename pl_traits<DT>::T T;
  enum { kCols = (RSMAX > 2 ? kLRowBytes / 2 : kLRowBytes) / (int)sizeof(T) };  // columns per wave
  enum { kChunk = kLWaves * kCols };       // columns per workgroup
  enum { kPad = 16 / (int)sizeof(T) };
  enum { kDRow = kCols + kPad };
};

// One run of tiles of one slot; RS: rank steps of one MFMA wave load.
template <int DT, int RS, int RSMAX, int kTRow>
__device__ __forceinline__ void pl_long_expand_run(const pl_long_args& a, int job, int chunk,
                                                   const pl_slot_entry& e, int n_tiles,
                                                   const int (&tlen)[kLUnitMax],
                                                   const int* __restrict__ ltok,
                                                   const typename pl_traits<DT>::T* __restrict__ lt,
                                                   typename pl_traits<DT>::T* __restrict__ dw) {
  typedef typename pl_traits<DT>::T T;
  typedef typename pl_traits<DT>::T4 T4;
  typedef typename pl_traits<DT>::T8 T8;
  typedef pl_long_shape<DT, RSMAX> S;
  constexpr int E = pl_traits<DT>::E;
  constexpr int kRStep = 4 * E;
  constexpr int CT = S::kCols / 16;                          // 16-column MFMA tiles per wave
  constexpr int kYLanes = S::kCols * (int)sizeof(T) / 16;    // lanes per y row
  constexpr int kYRows = 64 / kYLanes;
  constexpr int kYLoads = 16 / kYRows;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int li = lane & 15;
  const int lg = lane >> 4;
  const int N = a.N[job];
  const int r8 = e.rank8;
  const T* __restrict__ Bc = reinterpret_cast<const T*>(a.arena + e.b_off);
  T* __restrict__ y = reinterpret_cast<T*>(a.y[job]);
  const int64_t ldy = a.ldy[job];
  const float scale = e.scale;
  const float scale_t = pl_round<DT>(scale);
  const int yq = lane % kYLanes;
  const int yr0 = lane / kYLanes;

  const int cb = chunk * S::kChunk + wave * S::kCols;
  if (cb >= N) return;
  const bool cok = cb + yq * E < N;
  auto load = [&](pl_u32x4 (&yv)[kYLoads], int i) {
    const bool on = i < n_tiles;
    const int len = on ? tlen[i] : 0;
#pragma unroll
    for (int q = 0; q < kYLoads; ++q) {
      const int r = yr0 + kYRows * q;
      yv[q] = pl_ld16_nt_or0(y + (int64_t)ltok[(on ? i : 0) * 16 + r] * ldy + cb + yq * E, r < len && cok);
    }
  };
  pl_u32x4 ya[kYLoads], yb[kYLoads];
  load(ya, 0);
  pl_u32x4 bf[RS][CT];
#pragma unroll
  for (int s = 0; s < RS; ++s) {
    // B's MFMA blocks: the 16-column tile at nb (nt columns), rank block
    // j0 (wb wide) starts at nb*r8 + j0*nt
    const int j0 = s * kRStep;
    const int wb = min(kRStep, r8 - j0);
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
      const int nb = cb + ct * 16;
      const int nt = min(16, N - nb);
      bf[s][ct] = pl_ld16_or0(Bc + (int64_t)nb * r8 + (int64_t)j0 * nt + li * wb + lg * E,
                              li < nt && j0 + lg * E < r8);
    }
  }
  auto apply = [&](const pl_u32x4 (&yv)[kYLoads], int i) {
    pl_u32x4 tf[RS];
#pragma unroll
    for (int s = 0; s < RS; ++s)
      tf[s] = *reinterpret_cast<const pl_u32x4*>(lt + (i * 16 + li) * kTRow + s * kRStep + lg * E);
    pl_f32x4 d[CT];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) d[ct] = pl_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < RS; ++s)
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) d[ct] = pl_mfma_chunk<DT>(bf[s][ct], tf[s], d[ct]);
    // d[ct][v] = delta(column cb + ct*16 + 4*lg + v, token li): scale and round,
    // then through this wave's LDS tile to the row-major layout of y
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
      T4 dd;
#pragma unroll
      for (int v = 0; v < 4; ++v) dd[v] = (T)pl_delta<DT>(d[ct][v], scale, scale_t, a.epilogue);
      *reinterpret_cast<T4*>(dw + li * S::kDRow + ct * 16 + lg * 4) = dd;
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    const int len = tlen[i];
#pragma unroll
    for (int q = 0; q < kYLoads; ++q) {
      const int r = yr0 + kYRows * q;
      const pl_u32x4 dv = *reinterpret_cast<const pl_u32x4*>(dw + r * S::kDRow + yq * E);
      if (r < len && cok) {
        pl_u32x4 out;
        if constexpr (E == 8) {
          T8 yy = __builtin_bit_cast(T8, yv[q]);
          const T8 dd = __builtin_bit_cast(T8, dv);
#pragma unroll
          for (int c = 0; c < 8; ++c) yy[c] = (T)((float)yy[c] + (float)dd[c]);
          out = __builtin_bit_cast(pl_u32x4, yy);
        } else {
          out = __builtin_bit_cast(pl_u32x4, __builtin_bit_cast(pl_f32x4, yv[q]) +
                                                 __builtin_bit_cast(pl_f32x4, dv));
        }
        pl_st16_nt(y + (int64_t)ltok[i * 16 + r] * ldy + cb + yq * E, out);
      }
    }
    // the next tile rewrites the LDS tile only after these reads (in-order LDS)
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  };
  for (int i = 0; i < n_tiles; i += 2) {
    load(yb, i + 1);
    __builtin_amdgcn_sched_barrier(0);
    apply(ya, i);
    if (i + 1 >= n_tiles) break;
    load(ya, i + 2);
    __builtin_amdgcn_sched_barrier(0);
    apply(yb, i + 1);
  }
}

template <int DT, int RSMAX, int NT>
__global__ __launch_bounds__(64 * kLWaves, RSMAX <= 4 ? 3 : 2) void pl_long_expand(pl_long_args a) {
  typedef typename pl_traits<DT>::T T;
  typedef pl_long_shape<DT, RSMAX> S;
  __shared__ __attribute__((aligned(16))) T delta[kLWaves][16 * S::kDRow];
  constexpr int kTRow = RSMAX * 4 * pl_traits<DT>::E + S::kPad;
  __shared__ __attribute__((aligned(16))) T lt[NT * 16 * kTRow];
  __shared__ int ltok[kLUnitMax * 16];
  const int xcd = (int)(blockIdx.x % kXcds);
  const int rest = (int)(blockIdx.x / kXcds);
  const int cg = rest % a.n_chunks;
  const int unit = rest / a.n_chunks;
  int job = 0;
#pragma unroll
  for (int j = 1; j < kLJobs; ++j)
    if (j < a.n_jobs && cg >= a.chunk0[j]) job = j;
  pl_long_tile tl[NT];
  pl_long_unit<NT>(a, xcd, unit, tl);
  int slot[kLUnitMax], ts[kLUnitMax], tlen[kLUnitMax];
#pragma unroll
  for (int i = 0; i < kLUnitMax; ++i) {
    slot[i] = i < NT ? tl[i < NT ? i : 0].slot : 0;
    ts[i] = i < NT ? tl[i < NT ? i : 0].start : 0;
    tlen[i] = i < NT ? tl[i < NT ? i : 0].len : 0;
  }
  if ((slot[0] | slot[1] | slot[2] | slot[3]) == 0) return;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tid = threadIdx.x;
  if (tid < kLUnitMax * 16) {
    int st = 0, ln = 0;
#pragma unroll
    for (int i = 0; i < kLUnitMax; ++i)
      if (tid >> 4 == i) {
        st = ts[i];
        ln = tlen[i];
      }
    ltok[tid] = ln > 0 ? a.tok[st + min(tid & 15, ln - 1)] : 0;
  }
  // the unit's intermediate, in lane order: zeros past a tile's tokens and
  // past the slot's padded rank
  {
    constexpr int E = pl_traits<DT>::E;
    constexpr int kPieces = RSMAX * 4;  // 16-byte pieces per row
    const T* t = reinterpret_cast<const T*>(a.t[job]);
    int r8s[NT];
#pragma unroll
    for (int i = 0; i < NT; ++i) r8s[i] = a.table[(int64_t)tl[i].slot * a.num_modules + a.module[job]].rank8;
#pragma unroll
    for (int i0 = 0; i0 < NT * 16 * kPieces; i0 += 64 * kLWaves) {
      const int idx = i0 + tid;
      const int row = idx / kPieces, p = idx % kPieces;
      int st = 0, ln = 0, r8 = 0;
#pragma unroll
      for (int i = 0; i < NT; ++i)
        if (row >> 4 == i) {
          st = ts[i];
          ln = tlen[i];
          r8 = r8s[i];
        }
      if (idx < NT * 16 * kPieces)
        *reinterpret_cast<pl_u32x4*>(lt + row * kTRow + p * E) =
            pl_ld16_or0(t + (int64_t)(st + min(row & 15, max(ln - 1, 0))) * a.ldt + p * E, (row & 15) < ln && p * E < r8);
    }
  }
  __syncthreads();
  T* dw = delta[wave];
  // runs of consecutive tiles of one slot
  for (int i0 = 0; i0 < NT;) {
    int s0 = 0;
    int rs[kLUnitMax], rl[kLUnitMax];
    int n = 0;
#pragma unroll
    for (int i = 0; i < kLUnitMax; ++i)
      if (i == i0) s0 = slot[i];
#pragma unroll
    for (int q = 0; q < kLUnitMax; ++q) {
      int st = 0, ln = 0, sl = -1;
#pragma unroll
      for (int i = 0; i < kLUnitMax; ++i)
        if (i == i0 + q && i < NT) {
          st = ts[i];
          ln = tlen[i];
          sl = slot[i];
        }
      rs[q] = st;
      rl[q] = ln;
      if (n == q && sl == s0) ++n;
    }
    if (s0 > 0) {
      const pl_slot_entry e = a.table[(int64_t)s0 * a.num_modules + a.module[job]];
      const int chunk = cg - a.chunk0[job];
      const int* lk = ltok + i0 * 16;
      const T* lti = lt + i0 * 16 * kTRow;
      if (e.rank > 0) {
        const int r = (e.rank8 + 4 * pl_traits<DT>::E - 1) / (4 * pl_traits<DT>::E);
        if (RSMAX == 1 || r == 1)
          pl_long_expand_run<DT, 1, RSMAX, kTRow>(a, job, chunk, e, n, rl, lk, lti, dw);
        else if (RSMAX == 2 || r == 2)
          pl_long_expand_run<DT, 2 < RSMAX ? 2 : RSMAX, RSMAX, kTRow>(a, job, chunk, e, n, rl, lk, lti, dw);
        else if (RSMAX == 4 || r <= 4)
          pl_long_expand_run<DT, 4 < RSMAX ? 4 : RSMAX, RSMAX, kTRow>(a, job, chunk, e, n, rl, lk, lti, dw);
        else
          pl_long_expand_run<DT, RSMAX, RSMAX, kTRow>(a, job, chunk, e, n, rl, lk, lti, dw);
      }
    }
    i0 += n;
  }
}

// ------------------------------------------------------------------ host

int64_t long_units(const pl_long_args& a, int nt) {
  const int64_t tiles = ((int64_t)a.group_cap + kXcds - 1) / kXcds * a.sub;
  return (tiles + nt - 1) / nt;
}

template <int DT, int JT, int RT, bool SHARE>
void launch_shrink_xnt(const pl_long_args& a, hipStream_t s) {
  const dim3 grid((unsigned)(long_units(a, RT) * kXcds * a.n_jobs * a.passes));
  // x is streamed only when one workgroup reads each of its rows
  if (a.n_jobs * a.passes == 1)
    hipLaunchKernelGGL((pl_long_shrink<DT, JT, RT, true, SHARE>), grid, dim3(64 * kLWaves), 0, s, a);
  else
    hipLaunchKernelGGL((pl_long_shrink<DT, JT, RT, false, SHARE>), grid, dim3(64 * kLWaves), 0, s, a);
}

template <int DT, int JT, int RT>
void launch_shrink_rt(const pl_long_args& a, hipStream_t s) {
  // shares in 16 bits up to rank 64 (one pass of 16 ranks at most: always)
  if constexpr (DT == PL_F32)
    launch_shrink_xnt<DT, JT, RT, false>(a, s);
  else if constexpr (JT == 1)
    launch_shrink_xnt<DT, JT, RT, true>(a, s);
  else
    a.kw > 0 ? launch_shrink_xnt<DT, JT, RT, true>(a, s) : launch_shrink_xnt<DT, JT, RT, false>(a, s);
}

template <int DT>
void launch_long_shrink(const pl_long_args& a, int jt, int rt, hipStream_t s) {
  if (jt == 1)
    rt == 2 ? launch_shrink_rt<DT, 1, 2>(a, s) : launch_shrink_rt<DT, 1, 1>(a, s);
  else if (jt == 2)
    rt == 2 ? launch_shrink_rt<DT, 2, 2>(a, s) : launch_shrink_rt<DT, 2, 1>(a, s);
  else
    rt == 2 ? launch_shrink_rt<DT, 4, 2>(a, s) : launch_shrink_rt<DT, 4, 1>(a, s);
}

template <int DT, int NT>
void launch_expand_nt(const pl_long_args& a, int ranks, hipStream_t s) {
  const dim3 grid((unsigned)(long_units(a, NT) * kXcds * a.n_chunks));
  const int rs = (ranks + 4 * pl_traits<DT>::E - 1) / (4 * pl_traits<DT>::E);
  const dim3 block(64 * kLWaves);
  if (rs <= 1) hipLaunchKernelGGL((pl_long_expand<DT, 1, NT>), grid, block, 0, s, a);
  else if (rs <= 2) hipLaunchKernelGGL((pl_long_expand<DT, 2, NT>), grid, block, 0, s, a);
  else if (rs <= 4) hipLaunchKernelGGL((pl_long_expand<DT, 4, NT>), grid, block, 0, s, a);
  else hipLaunchKernelGGL((pl_long_expand<DT, 8, NT>), grid, block, 0, s, a);
}

template <int DT>
void launch_long_expand(const pl_long_args& a, int ranks, int nt, hipStream_t s) {
  if (nt == 4) launch_expand_nt<DT, 4>(a, ranks, s);
  else if (nt == 2) launch_expand_nt<DT, 2>(a, ranks, s);
  else launch_expand_nt<DT, 1>(a, ranks, s);
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

int32_t long_ldt(int32_t ldt) { return (ldt + 31) / 32 * 32; }

}  // namespace

extern "C" int64_t pl_lora_long_workspace_bytes(int32_t dtype, int64_t tokens, int32_t ldt) {
  if ((dtype != PL_F32 && dtype != PL_BF16 && dtype != PL_F16) || tokens < 0 || ldt <= 0 ||
      ldt > (dtype == PL_F32 ? PL_LONG_MAX_RANK / 2 : PL_LONG_MAX_RANK))
    return 0;
  return std::max<int64_t>(1, tokens) * long_ldt(ldt) * pl_elem_size(dtype);
}

extern "C" int pl_lora_long_stacked(int32_t dtype, const void* x, int64_t ldx, int32_t K,
                                    int32_t n_modules, const int32_t* modules, void* const* y,
                                    const int64_t* ldy, const int32_t* N, const void* arena,
                                    const pl_slot_entry* table, int32_t num_modules, int32_t ldt,
                                    const int32_t* tok, const pl_group* groups,
                                    const int32_t* meta, int64_t group_cap, int32_t group_tokens,
                                    int64_t tokens, void* const* ws, int64_t ws_bytes,
                                    int32_t epilogue, void* stream) {
  if (dtype != PL_F32 && dtype != PL_BF16 && dtype != PL_F16) {
    pl_set_error("unsupported dtype code %d", dtype);
    return PL_ERR_ARG;
  }
  if (!x || !arena || !table || !tok || !groups || !meta || !modules || !y || !ldy || !N || !ws) {
    pl_set_error("pl_lora_long: null pointer");
    return PL_ERR_ARG;
  }
  if (n_modules < 1 || n_modules > kLJobs) {
    pl_set_error("pl_lora_long serves 1..%d modules (got %d)", kLJobs, n_modules);
    return PL_ERR_ARG;
  }
  if (group_tokens != PL_GROUP_TOKENS_SHORT && group_tokens != PL_GROUP_TOKENS_LONG) {
    pl_set_error("group_tokens must be 16 or 64 (got %d)", group_tokens);
    return PL_ERR_ARG;
  }
  const int64_t need = pl_lora_long_workspace_bytes(dtype, tokens, ldt);
  if (need == 0) {
    pl_set_error("pl_lora_long takes ranks up to %d (slot rank capacity %d) of >= 0 tokens (%lld)",
                 dtype == PL_F32 ? PL_LONG_MAX_RANK / 2 : PL_LONG_MAX_RANK, ldt, (long long)tokens);
    return PL_ERR_LIMIT;
  }
  if (epilogue != PL_EPI_FALLBACK && epilogue != PL_EPI_TRITON) {
    pl_set_error("bad epilogue mode %d", epilogue);
    return PL_ERR_ARG;
  }
  const int E = pl_chunk_elems(dtype);
  const int es = pl_elem_size(dtype);
  if (K <= 0 || ldx < K || K % E != 0 || (ldx * es) % 16 != 0 || !aligned16(x) ||
      !aligned16(arena)) {
    pl_set_error("pl_lora_long needs K > 0, a multiple of %d, and 16-byte aligned x rows "
                 "(K=%d ldx=%lld)", E, K, (long long)ldx);
    return PL_ERR_ALIGN;
  }
  if (group_cap < 0 || group_cap > (int64_t)1 << 24) {
    pl_set_error("group capacity %lld out of range", (long long)group_cap);
    return PL_ERR_LIMIT;
  }
  const int rs = (ldt + 4 * E - 1) / (4 * E);  // rank steps of the expand
  const int chunk = kLWaves * (rs > 2 ? kLRowBytes / 2 : kLRowBytes) / es;  // columns per expand workgroup
  pl_long_args a;
  int64_t n_chunks = 0;
  for (int j = 0; j < n_modules; ++j) {
    if (num_modules <= 0 || modules[j] < 0 || modules[j] >= num_modules) {
      pl_set_error("module index %d out of range [0, %d)", modules[j], num_modules);
      return PL_ERR_ARG;
    }
    if (!y[j] || N[j] <= 0 || ldy[j] < N[j]) {
      pl_set_error("bad output %d: N=%d ldy=%lld", j, N[j], (long long)ldy[j]);
      return PL_ERR_ARG;
    }
    if (N[j] % E != 0 || (ldy[j] * es) % 16 != 0 || !aligned16(y[j])) {
      pl_set_error("pl_lora_long needs N a multiple of %d and 16-byte aligned y rows", E);
      return PL_ERR_ALIGN;
    }
    if (!ws[j] || !aligned16(ws[j]) || ws_bytes < need) {
      pl_set_error("pl_lora_long workspace %d: %lld bytes at %p, this call needs %lld, 16-byte aligned", j,
                   (long long)ws_bytes, ws[j], (long long)need);
      return PL_ERR_ARG;
    }
    for (int i = 0; i < j; ++i)
      if (ws[i] == ws[j]) {
        pl_set_error("each module of a stacked launch needs its own workspace");
        return PL_ERR_ARG;
      }
    a.module[j] = modules[j];
    a.t[j] = ws[j];
    a.y[j] = y[j];
    a.ldy[j] = ldy[j];
    a.N[j] = N[j];
    a.chunk0[j] = (int32_t)n_chunks;
    n_chunks += (N[j] + chunk - 1) / chunk;
  }
  for (int j = n_modules; j < kLJobs; ++j) {
    a.module[j] = 0;
    a.t[j] = nullptr;
    a.y[j] = nullptr;
    a.ldy[j] = 0;
    a.N[j] = 0;
    a.chunk0[j] = (int32_t)n_chunks;
  }
  const int sub = group_tokens / 16;
  const int64_t tiles = (group_cap + kXcds - 1) / kXcds * kXcds * sub;
  // Shrink: two tiles per workgroup share each A load once the launch has
  // 512 tiles (8192 tokens), above rank 64 from 320 on; below, one tile, for
  // more workgroups (bf16, K = 4096: rank 32 with 260 tiles 12 against 17 us, 520
  // tiles 16 against 13; rank 64 with 354 tiles 17.4 against 17.0, fewer of them
  // in use 13 against 18; rank 128 with 260 tiles 21 against 23, 354 tiles 24
  // against 22; fp32 to rank 32 from 1024 on: 9152 -> 3072, rank 32, 512 tiles 128
  // against 112, 896 tiles 186 against 173, 1024 tiles 195 against 213).  Passes of 32 ranks balance better over the CUs than passes
  // of 64 (rank 64, 520 tiles 16 against 18 us; K = 14336 44 against 56) until
  // they make 1536 workgroups, when rereading x costs more (K = 14336, rank 128,
  // 1040 tiles: 195 against 130 us).
  const int rt = tiles >= (ldt > 64 ? 320 : dtype == PL_F32 && ldt <= 32 ? 1024 : 512) ? 2 : 1;
  const int64_t blocks = tiles / rt * n_modules * ((ldt + 31) / 32);
  const int jt = ldt <= 16 ? 1 : ldt <= 32 || blocks < 1536 ? 2 : 4;
  // Expand: tiles per workgroup, which share the workgroup's B: 4 above rank
  // 32 (2048 -> 8192, rank 64, 5773 tokens: 4 tiles 53, 2 tiles 60, 1 tile
  // 64 us), 2 below (4096 -> 2 x 14336, rank 32, 11557 tokens: 272, 270 and
  // 288 us), while that leaves at least 512 or 1024 workgroups.  Rows that are
  // not whole 128-byte lines take one tile, so that workgroups which share a
  // line run side by side (3080 -> 5000, 5900 tokens: 1 tile 29, 4 tiles 34 us).
  bool lines = true;
  for (int j = 0; j < n_modules; ++j) lines = lines && (ldy[j] * es) % 128 == 0;
  const int unit = !lines || tiles * n_chunks < 2048 ? 1 : ldt > 32 ? 4 : 2;
  a.passes = (ldt + 16 * jt - 1) / (16 * jt);
  a.sub = sub;
  a.group_cap = (int32_t)group_cap;
  a.n_jobs = n_modules;
  a.n_chunks = (int32_t)n_chunks;
  if (n_chunks > 1 << 24 || !pl_grid_fits(long_units(a, rt) * kXcds * n_modules * a.passes, 64 * kLWaves) ||
      !pl_grid_fits(long_units(a, unit) * kXcds * n_chunks, 64 * kLWaves)) {
    pl_set_error("pl_lora_long: grid of %lld groups too large", (long long)group_cap);
    return PL_ERR_LIMIT;
  }
  if (group_cap == 0) return PL_OK;
  a.x = x;
  a.ldx = ldx;
  a.K = K;
  // In 16 bits the ranks of the fused kernel get its shares of K per wave, so
  // that each sum is the same additions in the same order and either kernel
  // gives the same bits: a Linear alone and with its siblings may take
  // different ones.  (Steps in turn instead: 32768 tokens, 4096 -> 14336, rank 32
  // 280 us both; 4096 tokens, 14336 -> 4096, rank 64 52.1, shares 51.4; 16384
  // tokens, 2048 -> 8192, rank 40 87.4 and 88.4; above rank 64, where the rule
  // does not look at the outputs, turns: 8192 tokens, 8192 -> 2048, rank 256
  // 84.8, shares 87.3.)
  const int64_t pair = 16 * E;
  const int64_t share = ((int64_t)K + kLWaves - 1) / kLWaves;
  a.kw = dtype != PL_F32 && ldt <= 64 ? (int32_t)((share + pair - 1) / pair * pair) : 0;
  a.arena = reinterpret_cast<const char*>(arena);
  a.table = table;
  a.num_modules = num_modules;
  a.tok = tok;
  a.groups = groups;
  a.meta = meta;
  a.epilogue = epilogue;
  a.ldt = long_ldt(ldt);
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  switch (dtype) {
    case PL_BF16:
      launch_long_shrink<PL_BF16>(a, jt, rt, s);
      launch_long_expand<PL_BF16>(a, ldt, unit, s);
      break;
    case PL_F16:
      launch_long_shrink<PL_F16>(a, jt, rt, s);
      launch_long_expand<PL_F16>(a, ldt, unit, s);
      break;
    default:
      launch_long_shrink<PL_F32>(a, jt, rt, s);
      launch_long_expand<PL_F32>(a, ldt, unit, s);
      break;
  }
  return pl_launch_status("pl_lora_long");
}

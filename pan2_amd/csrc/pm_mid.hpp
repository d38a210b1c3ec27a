// Small-tile GEMM engine of libpanmuon (pm_tile_gemm_kernel), for stages whose
// 256 x 256 tiles would leave most of the chip idle: a lone or mid-size matrix
// is bound there by one tile's serial chain (K loop, then a 10 us epilogue) on
// a few CUs. Here a stage runs as 64 x 64 tiles (two blocks to a CU) or
// 128 x 128 tiles (one block of 8 waves, persistent when items are equally
// long), chosen per stage and group by the host (choose_engine).
//
// Every element is accumulated as in the 256-tile engine: the same
// v_mfma_f32_16x16x32_bf16 over the same k order and K-split chunks, rounded
// at the same points, so results do not depend on the tile. Tiles cover the
// matrix's own extents rounded up to the tile, and K stops at the last 64-deep
// unit that holds data (777 x 1900 runs 13 of the 16 units its 1024-padded
// side has); what lies beyond stays unwritten and is never multiplied in.
//
// Measured (per launch, GRAM / SYMM / UPDATE, us, 256-tile engine -> here):
// lone 1024 x 4096 29+9 / 30 / 36 -> 14+5 / 7.8 / 14 (K-split GRAM + reduce);
// 256 x 1000 23 / 15 / 17 -> 7.0 / 5.2 / 5.0; the 15 matrices of a width-1024
// block 142 / 52 / 100 -> 64 / 40 / 100 (UPDATE stays on 256). At 4 of 5120 x
// 5120 the 128 tile runs 558 / 573 / 1084 against 457 / 470 / 810: its
// operands cross the L2 twice as often, so large stages keep 256.
//
// A unit (64 k of both operands) is copied to LDS as there, four units deep:
// with cold L2s at each launch, a copy takes about 2 us, and one or two units
// in flight (tried) ran the K loop 1.3-1.7x longer. Fragments are read a unit
// ahead. T = 128 with 4 waves of 64 x 64 was 10-20% slower than 8 waves of
// 64 x 32 (nothing covers a lone wave's waits).
#pragma once

namespace pm {

constexpr int kMtRun = 16;  // consecutive items an XCD takes at once (xcd_runs)
constexpr int kMtRing = 4;  // LDS slots, each one unit of both operands
static_assert(kWsLayout == (kTiledX | kTiledS), "the copies and epilogues assume panel layouts of X and S");

// Blocks of NW waves in a 2 x NW/2 grid over the T x T tile.
template <int T, int NW>
struct MtTile {
  static_assert((T == 64 && NW == 4) || (T == 128 && NW == 8), "tile edge and waves");
  static constexpr int kOp = T * 128;          // one operand of one unit: T rows (or columns) x 64 k
  static constexpr int kRows = T / 2;          // a wave's rows and columns of the tile
  static constexpr int kCols = 2 * T / NW;
  static constexpr int kQi = kRows / 16;       // 16 x 16 MFMA tiles
  static constexpr int kQj = kCols / 16;
  static constexpr int kCopies = T / 8 / NW;   // 1 KiB copies per operand, unit and wave
  static constexpr int kThreads = 64 * NW;
};
// a wave's place in the grid
template <int NW> __device__ __forceinline__ int mt_wr(int wave) { return wave / (NW / 2); }
template <int NW> __device__ __forceinline__ int mt_wc(int wave) { return wave % (NW / 2); }

// Operands, tile and K range (in units of 64 k) of one work item.
struct MtJob {
  const uint16_t* L;
  const uint16_t* R;
  int ldl, ldr, ti, tj, u0, u1;
};

// Extents the stage's tiles cover: the matrix's own, or the padded ones when
// the 256-tile engine, which reads whole padded operands, runs another stage of
// the group.
template <class D> __device__ __forceinline__ int mt_rows(const D& d, const GemmArgs& a) { return a.pad ? d.Mp : d.M; }
template <class D> __device__ __forceinline__ int mt_cols(const D& d, const GemmArgs& a) { return a.pad ? d.Np : d.N; }
template <int STAGE, int T, class D>
__device__ __forceinline__ int mt_tiles(const D& d, const GemmArgs& a) {
  return (STAGE == ST_GRAM || STAGE == ST_SYMM) ? mt_sym_tiles(mt_rows(d, a), T)
                                                : mt_full_tiles(mt_rows(d, a), mt_cols(d, a), T);
}

template <int STAGE, int T, bool SPLIT, class D>
__device__ __forceinline__ MtJob mt_decode(const D& d, int lt, const GemmArgs& args) {
  MtJob j;
  const int np = mt_edge_tiles(mt_rows(d, args), T);
  constexpr bool sym = STAGE == ST_GRAM || STAGE == ST_SYMM;
  j.u0 = 0;
  j.u1 = ((STAGE == ST_GRAM ? d.N : d.M) + 63) >> 6;
  if constexpr (SPLIT) {
    int tile, chunk;
    split_item(lt, mt_tiles<STAGE, T>(d, args), tile, chunk);
    const int per = (STAGE == ST_GRAM ? d.Np : d.Mp) / 64 / stage_split<STAGE>(d);
    j.u0 = chunk * per;
    j.u1 = imin(j.u1, j.u0 + per);
    lt = tile;
  }
  if (STAGE == ST_GRAM) {
    j.L = j.R = d.X[args.cur];
    j.ldl = j.ldr = d.Np;
  } else if (STAGE == ST_SYMM) {
    j.L = d.S[args.sl];
    j.R = d.S[args.sr];
    j.ldl = j.ldr = d.Mp;
  } else {
    j.L = d.S[args.sl];
    j.ldl = d.Mp;
    j.R = d.X[args.cur];
    j.ldr = d.Np;
  }
  if (sym) sym_tile(lt, np, j.ti, j.tj, 512 / T);
  else full_tile_cols(lt, np, mt_edge_tiles(mt_cols(d, args), T), j.ti, j.tj, 512 / T);
  return j;
}

// Copies of one unit into a ring slot: each wave issues kCopies 1 KiB copies
// per operand. Layouts of the slot as in the 256-tile engine (make_engine):
// a row-read operand's chunk c of row r at chunk c ^ ((r >> 1) & 7), a
// transposed one as 64 x 64 column blocks with the 32-byte chunk swizzle tsw.
template <int T, int NW, bool TR>
struct MtCopy {
  __amdgpu_buffer_rsrc_t l, r;
  int row[2], tr[2];  // lane offsets of copies of even / odd index
  const uint16_t* tbase;
  int64_t tpanel;
  int wave;

  __device__ __forceinline__ MtCopy(const MtJob& j, int w, int lane) : wave(w) {
    const int pl = (j.ti * T) >> 8, sl = (j.ti * T) & 255;
    l = panel_rsrc(j.L + (int64_t)pl * kTile * j.ldl + sl * kBK, (uint32_t)kTile * j.ldl * 2 - sl * 128);
    tbase = nullptr;
    tpanel = 0;
    if (TR) {
      tpanel = (int64_t)j.ldr * kTile;
      tbase = j.R + (int64_t)j.tj * (T / 64) * (kOpBytes / 2);
    } else {
      const int pr = (j.tj * T) >> 8, sr = (j.tj * T) & 255;
      r = panel_rsrc(j.R + (int64_t)pr * kTile * j.ldr + sr * kBK, (uint32_t)kTile * j.ldr * 2 - sr * 128);
    }
#pragma unroll
    for (int par = 0; par < 2; ++par) {
      const int sw = (4 * par + (lane >> 4)) & 7;
      row[par] = (lane >> 3) * 128 + (((lane & 7) ^ sw) << 4);
      const int tsw_l = ((lane >> 4) & 1) | (par << 1);
      tr[par] = (lane >> 3) * 128 + ((((((lane & 7) >> 1) ^ tsw_l) << 1) | (lane & 1)) << 4);
    }
  }
  __device__ __forceinline__ void operator()(char* slot, char* b, int u) const {
    constexpr int n = MtTile<T, NW>::kCopies;
#pragma unroll
    for (int i = 0; i < n; ++i) {
      const int q = wave * n + i;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(l, to_lds(slot + q * 1024), 16, row[i & 1], u * kOpBytes + q * 1024, 0,
                                               0);
    }
    const __amdgpu_buffer_rsrc_t rs =
        TR ? panel_rsrc(tbase + (int64_t)(u >> 2) * tpanel, (T / 64) * kOpBytes) : r;
#pragma unroll
    for (int i = 0; i < n; ++i) {
      const int q = wave * n + i;
      const int off = TR ? (q >> 3) * kOpBytes + (u & 3) * 8192 + (q & 7) * 1024 : u * kOpBytes + q * 1024;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, to_lds(b + q * 1024), 16, TR ? tr[i & 1] : row[i & 1], off, 0, 0);
    }
  }
};

// The MFMA fragments of one unit (two k-steps of 32) of this wave.
template <int T, int NW>
struct MtFrags {
  bf16x8 a[2][MtTile<T, NW>::kQi], b[2][MtTile<T, NW>::kQj];
};

// Each read's address is one offset from its ring buffer: through a chain of
// pointer sums the compiler loses the buffer and drains every copy in flight
// before the read.
template <int T, int NW, bool TR>
__device__ __forceinline__ void mt_read(const char* a, const char* b, MtFrags<T, NW>& f, int wave, int lane) {
  typedef MtTile<T, NW> C;
  const int r16 = lane & 15, g = lane >> 4;
  const int ao = mt_wr<NW>(wave) * C::kRows * 128, bo = mt_wc<NW>(wave) * C::kCols * 128;
  const int tsw_f = ((r16 >> 3) & 1) | ((g & 1) << 1);
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const int fo = r16 * 128 + (((4 * s + g) ^ ((r16 >> 1) & 7)) << 4);
#pragma unroll
    for (int i = 0; i < C::kQi; ++i) f.a[s][i] = *(const bf16x8*)(a + (ao + i * 2048 + fo));
#pragma unroll
    for (int i = 0; i < C::kQj; ++i) {
      if (TR) {
        const int col = mt_wc<NW>(wave) * C::kCols + 16 * i;
        const int o = (col >> 6) * 8192 + s * 4096 + (8 * g + (r16 >> 2)) * 128 + ((((col & 63) >> 4) ^ tsw_f) << 5) +
                      8 * (r16 & 3);
        f.b[s][i] = tr_pair(tr_read(b + o), tr_read(b + (o + 512)));
      } else {
        f.b[s][i] = *(const bf16x8*)(b + (bo + i * 2048 + fo));
      }
    }
  }
}

// Waits until at most n units of this wave's copies are in flight.
template <int T, int NW>
__device__ __forceinline__ void mt_wait(int n) {
  constexpr int c = 2 * MtTile<T, NW>::kCopies;
  if (n >= 3) wait_vmcnt<3 * c>();
  else if (n == 2) wait_vmcnt<2 * c>();
  else if (n == 1) wait_vmcnt<c>();
  else wait_vmcnt<0>();
}

struct MtRing {
  char* a[kMtRing];
  char* b[kMtRing];
};

// Unit u, whose fragments are in f[S % 2], from the ring (unit u in slot
// S = (u - u0) % kMtRing): once every wave's copies of u + 1 have landed and
// every wave has read u, refill u's slot with unit u + kMtRing, read u + 1's
// fragments, and run u's MFMAs behind those reads.
// STEADY: units u + 1 .. u + kMtRing exist, so nothing is conditional (a
// conditional copy or wait would make the compiler, which tracks copies into
// LDS along every path, drain them all before a read).
template <int T, int NW, bool TR, int S, bool STEADY>
__device__ __forceinline__ void mt_step(const MtRing& ring, const MtCopy<T, NW, TR>& copy, int u, int u1,
                                        MtFrags<T, NW> (&f)[2],
                                        f32x4 (&acc)[MtTile<T, NW>::kQi][MtTile<T, NW>::kQj], int lane) {
  typedef MtTile<T, NW> C;
  if (STEADY || u + 1 < u1) {
    if (STEADY) wait_vmcnt<(kMtRing - 2) * 2 * C::kCopies>();
    else mt_wait<T, NW>(imin(kMtRing - 2, u1 - 2 - u));
    wait_lgkmcnt<0>();
    block_barrier();
    mt_read<T, NW, TR>(ring.a[(S + 1) % kMtRing], ring.b[(S + 1) % kMtRing], f[(S + 1) & 1], copy.wave, lane);
    __builtin_amdgcn_sched_barrier(0);
    if (STEADY || u + kMtRing < u1) copy(ring.a[S], ring.b[S], u + kMtRing);
    __builtin_amdgcn_sched_barrier(0);
  }
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int i = 0; i < C::kQi; ++i)
#pragma unroll
      for (int j = 0; j < C::kQj; ++j) acc[i][j] = mfma_bf16(f[S & 1].a[s][i], f[S & 1].b[s][j], acc[i][j]);
}

// The fp32 tile of an epilogue in LDS, 64 rows of T. Column c of row r is at
// c ^ v(r): the four 16-lane groups of an accumulator store (rows 4 apart) and
// the eight 8-row runs of a column read fall in distinct banks, and runs of 8
// columns stay whole.
template <int T>
__device__ __forceinline__ float* mt_el(char* tile, int r, int c) {
  const int v = (((r >> 3) & 1) << 5) | ((((r >> 2) ^ (r >> 4)) & 1) << 4) | (((r >> 5) & 1) << 3);
  return (float*)(tile + (r * T + (c ^ v)) * 4);
}

// Epilogue of one tile, 64 rows at a time (T = 128: the waves of the upper
// half of the grid, then those of the lower): the accumulators go through the
// fp32 tile in LDS, so that every global access is a 16-byte run of a row, T/8
// lanes to a row of the tile. Element for element the arithmetic of
// gemm_epilogue. On a diagonal tile an element below the diagonal takes its
// mirror's accumulator, so symmetric products come out exactly symmetric.
// Global reads are requested ahead of the stores, so no load waits behind one.
template <int STAGE, int T, int NW, class D>
__device__ __forceinline__ void mt_epilogue(const GemmArgs& args, const D& d, int ti, int tj,
                                            const f32x4 (&acc)[MtTile<T, NW>::kQi][MtTile<T, NW>::kQj], int wave,
                                            int lane, char* tile) {
#pragma clang fp contract(off)
  typedef MtTile<T, NW> Tl;
  constexpr int kHalves = T / 64, kRuns = T / 8, kPasses = 64 * kRuns / Tl::kThreads;
  static_assert(kHalves == 1 || Tl::kRows == 64, "a half is one row of waves");
  constexpr bool kSym = STAGE == ST_GRAM || STAGE == ST_SYMM;
  const int tid = wave * 64 + lane;
  const bool diag = kSym && ti == tj;
  // runs of a half: 64 rows x T columns (row run n of this thread: row rr,
  // columns rc .. rc+7), or T columns x 64 rows (column cr, rows cc .. cc+7)
  auto rr = [&](int n) { return (tid + n * Tl::kThreads) / kRuns; };
  auto rc = [&](int n) { return (tid + n * Tl::kThreads) % kRuns * 8; };
  auto cr = [&](int n) { return (tid + n * Tl::kThreads) / 8; };
  auto cc = [&](int n) { return (tid + n * Tl::kThreads) % 8 * 8; };

  // the addend: S[sd] (symmetric, read in both orientations) or X
  const float ca = kSym ? args.b : args.a;
  const bool addend = STAGE != ST_GRAM && ca != 0.0f;
  const uint16_t* A = kSym ? d.S[args.sd] : d.X[args.cur];
  const int lda = kSym ? d.Mp : d.Np;
  u32x4 an[kHalves][kPasses], at[kHalves][kPasses];
#pragma unroll
  for (int h = 0; h < kHalves; ++h)
#pragma unroll
    for (int n = 0; n < kPasses; ++n) {
      an[h][n] = at[h][n] = (u32x4){0, 0, 0, 0};
      if (addend) an[h][n] = glb_load16(A + ws_off(ti * T + 64 * h + rr(n), tj * T + rc(n), lda, true));
      if (STAGE == ST_SYMM && addend) at[h][n] = glb_load16(A + ws_off(tj * T + cr(n), ti * T + 64 * h + cc(n), lda, true));
    }

  auto row_run = [&](int r, int c, float (&x)[8]) {
    const f32x4 lo = *(const f32x4*)mt_el<T>(tile, r, c), hi = *(const f32x4*)mt_el<T>(tile, r, c + 4);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      x[e] = lo[e];
      x[4 + e] = hi[e];
    }
  };
  auto col_run = [&](int r, int c, float (&x)[8]) {
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = *mt_el<T>(tile, r + e, c);
  };
  auto at_el = [&](const u32x4& v, int e) { return bf2f((uint16_t)(v[e >> 1] >> (16 * (e & 1)))); };
  auto pack = [&](const uint16_t (&h)[8]) {
    return (u32x4){(uint32_t)h[0] | ((uint32_t)h[1] << 16), (uint32_t)h[2] | ((uint32_t)h[3] << 16),
                   (uint32_t)h[4] | ((uint32_t)h[5] << 16), (uint32_t)h[6] | ((uint32_t)h[7] << 16)};
  };
  const float s = STAGE == ST_SYMM || !args.first ? 1.0f : scale_of(d, STAGE == ST_GRAM ? 0 : 1);
  const bool step = STAGE == ST_FINAL && args.mode == MODE_STEP;
  float wdf = 0.0f, neg = 0.0f;
  if (step) {
    if (args.lr_dev) {
      const float lr = *args.lr_dev;
      wdf = 1.0f - lr * args.wd;
      neg = -(lr * d.adj_ratio);
    } else {
      wdf = args.wdf_host;
      neg = d.neg_lr_host;
    }
  }

#pragma unroll
  for (int h = 0; h < kHalves; ++h) {
    if (h > 0) {  // the previous half's reads of the tile are done
      wait_lgkmcnt<0>();
      block_barrier();
    }
    if (kHalves == 1 || mt_wr<NW>(wave) == h) {
      const int g = lane >> 4, r16 = lane & 15, r0 = kHalves == 1 ? mt_wr<NW>(wave) * Tl::kRows : 0;
#pragma unroll
      for (int i = 0; i < Tl::kQi; ++i)
#pragma unroll
        for (int j = 0; j < Tl::kQj; ++j)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            *mt_el<T>(tile, r0 + 16 * i + 4 * g + e, mt_wc<NW>(wave) * Tl::kCols + 16 * j + r16) = acc[i][j][e];
    }
    wait_lgkmcnt<0>();
    block_barrier();
    const int p0 = ti * T + 64 * h, q0 = tj * T;  // of the half

    if constexpr (kSym) {
      uint16_t* C = d.S[args.sc];
      const float alpha = args.c;
      const int ld = d.Mp;
      // the gram form's first Z of a segment also goes out as Q = Z + qa·I
      const int sq = STAGE == ST_SYMM ? args.sq : -1;
      uint16_t* Q = sq >= 0 ? d.S[sq] : nullptr;
      // element (p, q) .. (p, q + 7)
      auto out = [&](const float (&x)[8], const u32x4& a, int p, int q) {
        uint16_t o[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = f2bf(STAGE == ST_GRAM ? x[e] * s : alpha * x[e] + ca * at_el(a, e));
        const int64_t off = ws_off(p, q, ld, true);
        const u32x4 v = pack(o);
        glb_store16(C + off, v);
        if (sq >= 0) glb_store16(Q + off, diag && p < d.M && p >= q && p < q + 8 ? add_diag(v, p - q, args.qa) : v);
      };
#pragma unroll
      for (int n = 0; n < kPasses; ++n) {
        const int r = rr(n), c = rc(n);
        float x[8];
        row_run(r, c, x);
        if (diag) {
          // tile row 64h + r: columns of this half's square mirror inside the
          // half; those left of it were written by the upper half
          if (c < 64 * h) continue;
          if (c < 64 * h + 64) {
            float y[8];
            col_run(c - 64 * h, 64 * h + r, y);
#pragma unroll
            for (int e = 0; e < 8; ++e) x[e] = c + e < 64 * h + r ? y[e] : x[e];
          }
        }
        out(x, an[h][n], p0 + r, q0 + c);
      }
#pragma unroll
      for (int n = 0; n < kPasses; ++n) {
        const int q = cr(n), p = cc(n);
        if (diag && q < 64 * h + 64) continue;
        float x[8];
        col_run(p, q, x);
        out(x, at[h][n], q0 + q, p0 + p);
      }
    } else {
      // O of a row run: bf16((a·X + acc)·s)
      auto update = [&](int n, uint16_t (&o)[8]) {
        float x[8];
        row_run(rr(n), rc(n), x);
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = f2bf((ca * at_el(an[h][n], e) + x[e]) * s);
      };
      if constexpr (STAGE == ST_UPDATE) {
        uint16_t* Xn = d.X[args.cur ^ 1];
#pragma unroll
        for (int n = 0; n < kPasses; ++n) {
          uint16_t o[8];
          update(n, o);
          glb_store16(Xn + ws_off(p0 + rr(n), q0 + rc(n), d.Np, true), pack(o));
        }
      } else {
        // ST_FINAL: element (p, q) of O is the param's (p, q), or (q, p) for a
        // tall param, whose rows are O's columns. p <- p·(1 - lr·wd) - lr·adj·O
        // (MODE_NS: O stored) on whatever part of a run lies inside the param.
        const bool tall = d.trans;
        if (tall) {
#pragma unroll
          for (int n = 0; n < kPasses; ++n) {  // O back into the tile, each thread its own runs
            uint16_t o[8];
            update(n, o);
            *(f32x4*)mt_el<T>(tile, rr(n), rc(n)) = (f32x4){bf2f(o[0]), bf2f(o[1]), bf2f(o[2]), bf2f(o[3])};
            *(f32x4*)mt_el<T>(tile, rr(n), rc(n) + 4) = (f32x4){bf2f(o[4]), bf2f(o[5]), bf2f(o[6]), bf2f(o[7])};
          }
          wait_lgkmcnt<0>();
          block_barrier();
        }
        const int32_t dt = d.p_dt;
        float p[kPasses][8];
        int row[kPasses], valid[kPasses];
        int64_t off[kPasses];
#pragma unroll
        for (int n = 0; n < kPasses; ++n) {
          row[n] = tall ? q0 + cr(n) : p0 + rr(n);
          const int col = tall ? p0 + cc(n) : q0 + rc(n);
          valid[n] = row[n] < d.rows ? d.cols - col : 0;
          off[n] = (int64_t)row[n] * d.p_ld + col;
          if (step) load8(d.param, dt, off[n], valid[n], p[n]);
        }
#pragma unroll
        for (int n = 0; n < kPasses; ++n) {
          float f[8];
          if (tall) {
            col_run(cc(n), cr(n), f);
          } else {
            uint16_t o[8];
            update(n, o);
#pragma unroll
            for (int e = 0; e < 8; ++e) f[e] = bf2f(o[e]);
          }
#pragma unroll
          for (int e = 0; e < 8; ++e) f[e] = step ? p[n][e] * wdf + f[e] * neg : f[e];
          store8(d.param, dt, off[n], valid[n], f);
        }
      }
    }
  }
}

// fp32 partials of item (chunk c, tile t): [wave][quad][lane] float4s
template <int T, int NW>
__device__ __forceinline__ f32x4* mt_partial(float* kpart, int tiles, int tile, int chunk, int wave, int lane) {
  constexpr int quads = MtTile<T, NW>::kQi * MtTile<T, NW>::kQj;
  return (f32x4*)kpart + (((int64_t)chunk * tiles + tile) * NW + wave) * (quads * 64) + lane;
}

// One Newton–Schulz stage over every matrix of the group: an item is a T x T
// tile, or (SPLIT) a chunk of a tile's K range. Block b takes items b,
// b + gridDim, ...; with fewer blocks than items (persistent) an item's first
// units are requested before the previous item's epilogue.
template <int STAGE, int T, int NW, bool SPLIT>
__global__ __launch_bounds__(64 * NW, T == 64 ? 2 : 1) void pm_tile_gemm_kernel(GemmArgs args) {
  typedef MtTile<T, NW> C;
  constexpr int kOp = C::kOp;
  constexpr bool TR = STAGE == ST_UPDATE || STAGE == ST_FINAL;
  __shared__ __attribute__((aligned(1024))) char a0[kOp], b0[kOp], a1[kOp], b1[kOp], a2[kOp], b2[kOp], a3[kOp], b3[kOp];
  __shared__ __attribute__((aligned(1024))) char tile_lds[SPLIT ? 16 : 64 * T * 4];
  MtRing ring;  // (set member by member: an aggregate initialiser of LDS addresses does not compile)
  ring.a[0] = a0; ring.b[0] = b0; ring.a[1] = a1; ring.b[1] = b1;
  ring.a[2] = a2; ring.b[2] = b2; ring.a[3] = a3; ring.b[3] = b3;
  typedef const __attribute__((address_space(4))) MatDesc* DescPtr;
  typedef const __attribute__((address_space(4))) int32_t* PrefixPtr;
  const DescPtr descs = (DescPtr)args.descs;
  const PrefixPtr prefix = (PrefixPtr)args.prefix;
  const int wave = wave_id(), lane = threadIdx.x & 63;
  const int total = args.total, grid = gridDim.x;
  int b = blockIdx.x, m, lt;
  auto decode = [&](int item) {
    const int t = xcd_runs<kMtRun>(item, total);
    m = find_matrix(prefix, args.n, t);
    lt = t - prefix[m];
    return mt_decode<STAGE, T, SPLIT>(descs[m], lt, args);
  };
  // the first units of an item (past its end: the last unit again, never read)
  auto start = [&](const MtJob& j) {
    const MtCopy<T, NW, TR> copy(j, wave, lane);
#pragma unroll
    for (int i = 0; i < kMtRing; ++i) copy(ring.a[i], ring.b[i], imin(j.u0 + i, j.u1 - 1));
  };
  MtJob job = decode(b);
  start(job);
  for (;;) {
    const MtCopy<T, NW, TR> copy(job, wave, lane);
    f32x4 acc[C::kQi][C::kQj];
#pragma unroll
    for (int i = 0; i < C::kQi; ++i)
#pragma unroll
      for (int j = 0; j < C::kQj; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
    MtFrags<T, NW> f[2];
    int u = job.u0;
    const int u1 = job.u1;
    wait_vmcnt<0>();  // the first units, and the previous epilogue's stores
    wait_lgkmcnt<0>();
    block_barrier();
    mt_read<T, NW, TR>(ring.a[0], ring.b[0], f[0], wave, lane);
    for (; u + 2 * kMtRing <= u1; u += kMtRing) {
      mt_step<T, NW, TR, 0, true>(ring, copy, u, u1, f, acc, lane);
      mt_step<T, NW, TR, 1, true>(ring, copy, u + 1, u1, f, acc, lane);
      mt_step<T, NW, TR, 2, true>(ring, copy, u + 2, u1, f, acc, lane);
      mt_step<T, NW, TR, 3, true>(ring, copy, u + 3, u1, f, acc, lane);
    }
    // at most 2·kMtRing - 1 units are left
#pragma unroll 1
    for (; u < u1; u += kMtRing) {
      mt_step<T, NW, TR, 0, false>(ring, copy, u, u1, f, acc, lane);
      if (u + 1 < u1) mt_step<T, NW, TR, 1, false>(ring, copy, u + 1, u1, f, acc, lane);
      if (u + 2 < u1) mt_step<T, NW, TR, 2, false>(ring, copy, u + 2, u1, f, acc, lane);
      if (u + 3 < u1) mt_step<T, NW, TR, 3, false>(ring, copy, u + 3, u1, f, acc, lane);
    }
    wait_lgkmcnt<0>();
    block_barrier();  // every wave has read the last unit
    const int mc = m, ltc = lt, ti = job.ti, tj = job.tj;
    b += grid;
    if (b < total) {
      job = decode(b);
      start(job);
    }
    if constexpr (SPLIT) {
      int tile, chunk;
      const int tiles = mt_tiles<STAGE, T>(descs[mc], args);
      split_item(ltc, tiles, tile, chunk);
      typedef __attribute__((address_space(1))) f32x4 glb_f32x4;
      glb_f32x4* dst = (glb_f32x4*)mt_partial<T, NW>(descs[mc].kpart, tiles, tile, chunk, wave, lane);
#pragma unroll
      for (int i = 0; i < C::kQi; ++i)
#pragma unroll
        for (int j = 0; j < C::kQj; ++j) dst[(i * C::kQj + j) * 64] = acc[i][j];
    } else {
      mt_epilogue<STAGE, T, NW>(args, descs[mc], ti, tj, acc, wave, lane, tile_lds);
    }
    if (b >= total) break;
  }
}

// The second launch of a K-split stage: one block per split tile adds the
// chunks' partials in chunk order and runs the stage's epilogue.
template <int STAGE, int T, int NW>
__global__ __launch_bounds__(64 * NW) void pm_tile_reduce_kernel(GemmArgs args) {
  typedef MtTile<T, NW> C;
  __shared__ __attribute__((aligned(1024))) char tile_lds[64 * T * 4];
  typedef const __attribute__((address_space(4))) MatDesc* DescPtr;
  typedef const __attribute__((address_space(4))) int32_t* PrefixPtr;
  typedef const __attribute__((address_space(1))) f32x4 glb_f32x4;
  const DescPtr descs = (DescPtr)args.descs;
  const PrefixPtr prefix = (PrefixPtr)args.prefix;
  const int wave = wave_id(), lane = threadIdx.x & 63;
  const int m = find_matrix(prefix, args.n, blockIdx.x);
  const int tile = blockIdx.x - prefix[m];
  const MtJob job = mt_decode<STAGE, T, false>(descs[m], tile, args);
  const int tiles = mt_tiles<STAGE, T>(descs[m], args), split = stage_split<STAGE>(descs[m]);
  float* const kpart = descs[m].kpart;
  f32x4 acc[C::kQi][C::kQj];
#pragma unroll
  for (int c = 0; c < kMaxKSplit; ++c) {
    if (c >= split) break;
    const glb_f32x4* src = (const glb_f32x4*)mt_partial<T, NW>(kpart, tiles, tile, c, wave, lane);
    f32x4 v[C::kQi][C::kQj];
#pragma unroll
    for (int i = 0; i < C::kQi; ++i)
#pragma unroll
      for (int j = 0; j < C::kQj; ++j) v[i][j] = src[(i * C::kQj + j) * 64];
#pragma unroll
    for (int i = 0; i < C::kQi; ++i)
#pragma unroll
      for (int j = 0; j < C::kQj; ++j) acc[i][j] = c == 0 ? v[i][j] : acc[i][j] + v[i][j];
  }
  mt_epilogue<STAGE, T, NW>(args, descs[m], job.ti, job.tj, acc, wave, lane, tile_lds);
}

}  // namespace pm

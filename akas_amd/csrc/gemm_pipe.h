// Pipelined FP8 tile engine for the sizes between decode and prefill, shared
// by the dense and the grouped expert GEMMs.
//
// C[m, n] = sum_kb ( A_kb[m, :] . B_kb[n, :] ) * as[m, kb] * ws[n / 128, kb]
//
// What bounds these sizes: a few hundred rows give one tile or less per CU,
// so nothing but the workgroup's own loads in flight covers the memory
// latency, and every k-block costs a round of load, barrier, LDS read,
// multiply and fold.  A kernel that stages one k-block ahead through
// registers spends about 1,300 cycles per k-block whatever its tile
// (128x128 tiles at M=300, K=2048, N=6144: 20.5 us, of which the products
// are 2).  So here:
//   * operands go global->LDS by DMA (global_load_lds, no staging
//     registers) through ST stages, and the wait at a step leaves the ST - 2
//     younger stages in flight (a counted vmcnt, not a full drain);
//   * G groups of waves take G k-blocks of the same tile per step, so a step
//     moves G times the bytes per barrier and a tile's k-loop is G times
//     shorter; their partial tiles are summed in group order in the epilogue.
// Steady state is then the rate at which the copies land: 57-66 GB/s per CU
// in every configuration measured here, about half of what line-wide loads
// into registers reach in the split kernel (gemm.hip).  The L1s have misses
// pending for 14 to 17% of the cycles only, and four fifths of the requests
// hit in L2; what holds it has not been found.  What is left is choosing the tile that covers the CUs with the
// fewest bytes (dense_cost in gemm.hip).  The weight scales that the dense
// kernel holds in registers are first used in the k-loop, where the compiler
// waits for every load before it: the stages ahead of the first step land
// together.
//
// The same launch, 128x128 register-staged tiles -> this engine
// (GEMM alone, us): M=300 K=2048 N=6144 20.3 -> 10.9; M=512 K=2048 N=2048
// 19.7 -> 9.2; M=300 K=8192 N=2048 61.0 -> 20.8; M=1000 K=8192 N=2048
// 64.5 -> 29.1; M=1000 K=2048 N=6144 25.8 -> 20.9.
// Reading the next step's fragments into registers under this step's
// products (no LDS latency left in a step) measured the same: the loads
// are the bound, not the LDS reads.
//
// A workgroup is G groups of WM x WN waves; wave (wm, wn) of a group owns
// rows wm*TM.. and columns wn*TN.. of the tile.  LDS tiles are 128-byte rows
// of 16-byte chunks, chunk c of row r at slot c ^ swizzle(r) (gemm_core.h);
// one DMA instruction fills 8 rows.  Products are B x A^T, so a lane holds
// output row l % 16 and four adjacent columns: one activation scale per
// lane and row tile.
#pragma once

#include "gemm_core.h"

namespace akas {
namespace pipe {

// Waits until at most N of the wave's global loads and none of its LDS
// accesses are outstanding (s_waitcnt: vmcnt N, lgkmcnt 0).
template <int N>
AKAS_DEV void wait_loads() {
  static_assert(N >= 0 && N < 64, "vmcnt is six bits");
  __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | ((N >> 4) << 14));
}

// Workgroup barrier that memory accesses are not moved across.  Unlike
// __syncthreads it does not drain the DMA in flight.
AKAS_DEV void barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

template <int N>
struct Int {
  static constexpr int value = N;
};

template <int BM_, int BN_, int WM, int WN, int G_, int ST>
struct Engine {
  static constexpr int BM = BM_, BN = BN_, G = G_;
  static constexpr int W = WM * WN, THREADS = 64 * W * G;
  static constexpr int TM = BM / WM, TN = BN / WN, MT = TM / 16, NT = TN / 16;
  static constexpr int TILE = (BM + BN) * 128;  // bytes of one k-block
  static constexpr int STAGE = G * TILE;
  static constexpr int AHEAD = ST - 1;          // stages issued ahead of the one multiplied
  // DMA instructions per wave and stage: A pieces, B pieces (8 rows each), scales
  static constexpr int PA = BM / 8 / W, PB = BN / 8 / W, LOADS = PA + PB + 1;
  static constexpr int SR = BM / 64;            // 64-row scale copies per k-block
  static_assert(BM % (8 * W) == 0 && BN % (8 * W) == 0 && BM % 64 == 0 && W % SR == 0,
                "the waves of a group share its copies evenly");
  static_assert(ST >= 2 && ST <= 4 && TN >= 32 && 128 % TN == 0, "stages, wave columns");

  // Every stage is a variable of its own, selected at compile time: the
  // compiler then sees that a read of one stage does not alias the DMA into
  // another, and adds no wait of its own.
  template <int S>
  static AKAS_DEV uint8_t* stage() {
    static __shared__ __attribute__((aligned(1024))) uint8_t buffer[STAGE];
    return buffer;
  }
  template <int S>
  static AKAS_DEV float* stage_scales() {
    static __shared__ __attribute__((aligned(256))) float buffer[G * BM];
    return buffer;
  }

  struct Acc {
    v4f t[MT][NT];  // lane l: row l % 16, columns 4 * (l / 16) .. +3
    AKAS_DEV void clear() {
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) t[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
    }
  };

  // Where this wave is: its group, its place in it, its rows and columns.
  int lane, g, w, a_row0, b_row0;
  AKAS_DEV explicit Engine(int tid) {
    lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    g = wave / W;
    w = wave % W;
    a_row0 = (w % WM) * TM;
    b_row0 = (w / WM) * TN;
  }

  // Tile row of this lane in the wave's A (B) piece i, and the byte offset
  // in a source row of the chunk it fetches.
  AKAS_DEV int a_piece_row(int i) const { return (w * PA + i) * 8 + (lane >> 3); }
  AKAS_DEV int b_piece_row(int i) const { return (w * PB + i) * 8 + (lane >> 3); }
  AKAS_DEV int piece_chunk(int row) const { return ((lane & 7) ^ swizzle(row)) << 4; }
  // Tile row whose activation scale this lane copies.  (Groups with more
  // waves than 64-row copies write the same scales more than once, so that
  // every wave has the same number of loads in flight.)
  AKAS_DEV int scale_row() const { return (w % SR) * 64 + lane; }

  // The DMA of step t into stage S: the group's k-block, clamped to the last
  // (a clamped copy is never multiplied).  plan.a(i, kb) / plan.b(i, kb) are
  // the addresses of this lane's 16 bytes of piece i, plan.s(kb) that of its
  // scale.
  template <int S, class Plan>
  AKAS_DEV void issue_a(const Plan& plan, int t, int kb0, int nkb) const {
    const int kb = kb0 + min(t * G + g, nkb - 1);
    uint8_t* base = stage<S>() + g * TILE;
#pragma unroll
    for (int i = 0; i < PA; ++i)
      __builtin_amdgcn_global_load_lds((const void*)plan.a(i, kb),
                                       (lds_void*)(base + (w * PA + i) * 1024), 16, 0, 0);
    __builtin_amdgcn_global_load_lds((const void*)plan.s(kb),
                                     (lds_void*)(stage_scales<S>() + g * BM + (w % SR) * 64), 4, 0, 0);
  }
  template <int S, class Plan>
  AKAS_DEV void issue_b(const Plan& plan, int t, int kb0, int nkb) const {
    const int kb = kb0 + min(t * G + g, nkb - 1);
    uint8_t* base = stage<S>() + g * TILE + BM * 128;
#pragma unroll
    for (int i = 0; i < PB; ++i)
      __builtin_amdgcn_global_load_lds((const void*)plan.b(i, kb),
                                       (lds_void*)(base + (w * PB + i) * 1024), 16, 0, 0);
  }
  template <int S, class Plan>
  AKAS_DEV void issue(const Plan& plan, int t, int kb0, int nkb) const {
    issue_a<S>(plan, t, kb0, nkb);
    issue_b<S>(plan, t, kb0, nkb);
  }

  // The stages ahead of the first step, B (known first where A rows are
  // gathered through a table) and A; then wait until stage 0 has landed.
  template <class Plan>
  AKAS_DEV void start_b(const Plan& plan, int kb0, int nkb) const {
    issue_b<0>(plan, 0, kb0, nkb);
    if constexpr (AHEAD > 1) issue_b<1>(plan, 1, kb0, nkb);
    if constexpr (AHEAD > 2) issue_b<2>(plan, 2, kb0, nkb);
  }
  template <class Plan>
  AKAS_DEV void start_a(const Plan& plan, int kb0, int nkb) const {
    issue_a<0>(plan, 0, kb0, nkb);
    if constexpr (AHEAD > 1) issue_a<1>(plan, 1, kb0, nkb);
    if constexpr (AHEAD > 2) issue_a<2>(plan, 2, kb0, nkb);
    // (deeper, run's constant waits would count a younger stage's B as A)
    static_assert(AHEAD <= 2, "B ahead of A: two stages at most");
    wait_loads<(PA + 1) * (AHEAD - 1)>();
  }

  // One k-block of stage S into acc: acc = fma(P, as * ws, acc) per product.
  // PAIRED: odd 16-column tiles take ws1 (gate and up rows interleaved).
  template <int S, bool PAIRED>
  AKAS_DEV void multiply(Acc& acc, float ws0, float ws1) const {
    const uint8_t* at = stage<S>() + g * TILE;
    const uint8_t* bt = at + BM * 128;
    const float* sc = stage_scales<S>() + g * BM;
    v8i af[MT];
    float c0[MT], c1[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      af[i] = lds_fragment(at, a_row0 + 16 * i, lane);
      const float s = sc[a_row0 + 16 * i + (lane & 15)];
      c0[i] = s * ws0;
      c1[i] = PAIRED ? s * ws1 : c0[i];
    }
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const v8i bf = lds_fragment(bt, b_row0 + 16 * j, lane);
      v4f cur[MT];
#pragma unroll
      for (int i = 0; i < MT; ++i) cur[i] = mfma_e4m3(bf, af[i]);
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        const float c = (j & 1) ? c1[i] : c0[i];
#pragma unroll
        for (int e = 0; e < 4; ++e) acc.t[i][j][e] = __builtin_fmaf(cur[i][e], c, acc.t[i][j][e]);
      }
    }
  }

  // Step t: stage S is waited for, stage S + AHEAD refilled, stage S
  // multiplied.  The barrier says that every wave's copies of stage S have
  // landed and that every wave is done with the stage that is refilled.
  // FULL steps all issue a stage, so their wait is a constant.
  template <int S, bool FULL, bool PAIRED, class Plan, class WS>
  AKAS_DEV void step(const Plan& plan, Acc& acc, int t, int steps, int kb0, int nkb, WS ws,
                     bool live) const {
    wait_loads<FULL ? LOADS * (AHEAD - 1) : 0>();
    barrier();
    if (FULL || t + AHEAD < steps) issue<(S + AHEAD) % ST>(plan, t + AHEAD, kb0, nkb);
    const int kb = t * G + g;
    if (live && (G == 1 || kb < nkb)) {
      const float2 v = ws(kb);
      multiply<S, PAIRED>(acc, v.x, v.y);
    }
  }

  // k-blocks [kb0, kb0 + nkb) into acc, after start_b and start_a (or
  // start).  ws(i) is the (ws0, ws1) pair of k-block kb0 + i; it must come
  // from registers (a global or LDS load there would wait for the copies in
  // flight).  A wave that is not `live` only copies: no row or column of its
  // tile is stored.
  template <class Plan>
  AKAS_DEV void start(const Plan& plan, int kb0, int nkb) const {
    issue<0>(plan, 0, kb0, nkb);
    if constexpr (AHEAD > 1) issue<1>(plan, 1, kb0, nkb);
    if constexpr (AHEAD > 2) issue<2>(plan, 2, kb0, nkb);
  }
  template <bool PAIRED, class Plan, class WS>
  AKAS_DEV void run(const Plan& plan, Acc& acc, int kb0, int nkb, WS ws, bool live = true) const {
    const int steps = (nkb + G - 1) / G;
    int t = 0;
    for (; t + ST + AHEAD <= steps; t += ST) {
      step<0, true, PAIRED>(plan, acc, t, steps, kb0, nkb, ws, live);
      step<1, true, PAIRED>(plan, acc, t + 1, steps, kb0, nkb, ws, live);
      if constexpr (ST > 2) step<2, true, PAIRED>(plan, acc, t + 2, steps, kb0, nkb, ws, live);
      if constexpr (ST > 3) step<3, true, PAIRED>(plan, acc, t + 3, steps, kb0, nkb, ws, live);
    }
    for (; t < steps; t += ST) {
      step<0, false, PAIRED>(plan, acc, t, steps, kb0, nkb, ws, live);
      if (t + 1 < steps) step<1, false, PAIRED>(plan, acc, t + 1, steps, kb0, nkb, ws, live);
      if constexpr (ST > 2)
        if (t + 2 < steps) step<2, false, PAIRED>(plan, acc, t + 2, steps, kb0, nkb, ws, live);
      if constexpr (ST > 3)
        if (t + 3 < steps) step<3, false, PAIRED>(plan, acc, t + 3, steps, kb0, nkb, ws, live);
    }
  }

  // float32 tile of wave (group q, place w), TN columns per row, in the
  // stages' memory (free after the loop): 16-byte chunk c of row r at slot
  // c ^ (r & SWZ), conflict-free for the accumulators' writes and for row reads.
  static constexpr int TILE_F32 = TM * TN * 4, PER_STAGE = STAGE / TILE_F32;
  static constexpr int SWZ = TN / 4 >= 16 ? 15 : TN / 4 - 1;
  AKAS_DEV uint8_t* partial(int q) const {
    const int slot = q * W + w, s = slot / PER_STAGE;
    uint8_t* base = stage<0>();
    if (s == 1) base = stage<1>();
    if constexpr (ST > 2) if (s == 2) base = stage<2>();
    if constexpr (ST > 3) if (s == 3) base = stage<3>();
    return base + (slot % PER_STAGE) * TILE_F32;
  }

  // Sums the groups' partial tiles (in group order) and hands the wave tile
  // out in pieces of eight adjacent columns: put(row, col, lo, hi) with row
  // and col relative to the workgroup's tile.  The groups share the pieces.
  template <class Put>
  AKAS_DEV void reduce(const Acc& acc, Put put) const {
    static_assert(PER_STAGE * ST >= W * G, "the partial tiles fit in the stages");
    __syncthreads();  // the stages are read no more, and no copy is in flight
    uint8_t* own = partial(g);
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        const int r = 16 * i + (lane & 15), c = 4 * j + (lane >> 4);
        *reinterpret_cast<v4f*>(own + r * (TN * 4) + ((c ^ (r & SWZ)) << 4)) = acc.t[i][j];
      }
    if constexpr (G > 1)
      __syncthreads();
    else
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");  // the wave reads its own tile
    constexpr int PER_ROW = TN / 8, PIECES = TM * PER_ROW;
#pragma unroll
    for (int it = 0; it < (PIECES + 64 * G - 1) / (64 * G); ++it) {
      const int u = (it * G + g) * 64 + lane;
      if (PIECES % (64 * G) != 0 && u >= PIECES) break;
      const int r = u / PER_ROW, c = (u % PER_ROW) * 2;
      v4f lo, hi;
#pragma unroll
      for (int q = 0; q < G; ++q) {
        const uint8_t* row = partial(q) + r * (TN * 4);
        const v4f l = *reinterpret_cast<const v4f*>(row + ((c ^ (r & SWZ)) << 4));
        const v4f h = *reinterpret_cast<const v4f*>(row + (((c + 1) ^ (r & SWZ)) << 4));
        lo = q == 0 ? l : lo + l;
        hi = q == 0 ? h : hi + h;
      }
      put(a_row0 + r, b_row0 + 4 * c, lo, hi);
    }
  }
};

// Eight adjacent output elements from element i: one or two 16-byte stores
// when `wide` (i and the buffer 16-byte aligned), else one by one.
template <int OUT>
AKAS_DEV void store_out8(void* out, int64_t i, const v4f& lo, const v4f& hi, bool wide) {
  if (!wide) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      store_out<OUT>(out, i + e, lo[e]);
      store_out<OUT>(out, i + 4 + e, hi[e]);
    }
  } else if constexpr (OUT == AKAS_DTYPE_F32) {
    *reinterpret_cast<v4f*>(reinterpret_cast<float*>(out) + i) = lo;
    *reinterpret_cast<v4f*>(reinterpret_cast<float*>(out) + i + 4) = hi;
  } else {
    u32x4 v;
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      if constexpr (OUT == AKAS_DTYPE_BF16) {
        v[e] = f32x2_to_bf16x2(lo[2 * e], lo[2 * e + 1]);
        v[2 + e] = f32x2_to_bf16x2(hi[2 * e], hi[2 * e + 1]);
      } else {
        v[e] = f32x2_to_f16x2(lo[2 * e], lo[2 * e + 1]);
        v[2 + e] = f32x2_to_f16x2(hi[2 * e], hi[2 * e + 1]);
      }
    }
    *reinterpret_cast<u32x4*>(reinterpret_cast<uint16_t*>(out) + i) = v;
  }
}

}  // namespace pipe
}  // namespace akas

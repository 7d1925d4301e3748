// Main loop for products of 33 to a few hundred rows on gfx950, between the
// decode kernels (weights bound) and the 256-row prefill tiles (matrix cores
// bound).
//
// A block is WN x WK waves of 64 columns: every wave holds all 32*RB rows of
// the tile, so each weight is decoded once, and the WK waves of a column group
// split the 16-k steps of a chunk.  (Splitting the rows over waves, as the
// prefill kernel does, decodes every weight once per wave, and splitting the
// columns further needs more LDS reads of A per MFMA.)  Operands are fetched
// global -> LDS directly over a ring of NST chunks.
//
// The loop is pipelined across chunks: the wait for the next chunk's loads and
// the barrier sit before the last MFMAs of the current one, whose operands are
// in registers, so the next chunk's first LDS reads and decode run in their
// shadow.  A chunk start that waits, reads and decodes first costs about 700
// cycles, more than the MFMAs of a 64-row chunk.
//
// What bounds it (128-row tile, 4096 -> 2 x 14336 at M = 100, 36.5 us; parts
// taken out one at a time): no global -> LDS loads 27.5, no MFMAs 30.9, neither
// 19.2 -- LDS reads, decode and loads together cost as much as the matrix work.
// Counters of that launch: matrix cores busy 50% of the cycles, VALU 36%, LDS 22%
// without bank conflicts, waves waiting for data or a barrier 34% of their time.
// The 64-row tiles of the narrow products wait more (44-59%, matrix cores 16-33%):
// a split of K leaves each block few chunks between its first loads and its hand-off.
// Measured and not better: loads issued by dedicated waves with a deeper weight
// ring (41 us), two stages (70), 64-k chunks (47), four waves per block (44),
// rings of four stages (25 against 25.6 us at 64 rows, and one block per CU).
#pragma once
#include "mm_prefill.h"

namespace mmmid {
using namespace mmpf;

// s_waitcnt vmcnt(VM) lgkmcnt(0)
template <int VM>
MM_DEV void wait_vm_lgkm() {
  static_assert(VM >= 0 && VM < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((VM & 15) | (7 << 4) | ((VM >> 4) << 14));
}

constexpr int MID_BK = 128;      // k per chunk
constexpr int MID_WK = 4;        // waves that split a chunk's steps
constexpr int MID_NST = 3;       // ring depth

template <bool INT4, int RB, int WN>
struct MidShape {
  static constexpr int BK = MID_BK, WK = MID_WK, NST = MID_NST;
  static constexpr int NWAVE = WN * WK, NTHR = NWAVE * 64;
  static constexpr int BM = 32 * RB, BN = 64 * WN;
  static constexpr int STEPS = BK / 16 / WK;          // 16-k steps of a wave per chunk
  static constexpr int SROWS = BK / 32;               // scale rows of a chunk (g >= 32)
  static constexpr int A_PIECES = BM * (BK / 8), B_PIECES = (BK / 8) * (BN / 4);
  static constexpr int S_PIECES = SROWS * (BN / 8);
  static_assert(A_PIECES % 64 == 0 && B_PIECES % 64 == 0, "whole wave loads");
  static constexpr int A_IT = (A_PIECES + NTHR - 1) / NTHR;
  static constexpr int B_IT = (B_PIECES + NTHR - 1) / NTHR;
  static constexpr int S_IT = (S_PIECES + NTHR - 1) / NTHR;
  static constexpr int LOADS = A_IT + B_IT + S_IT * (INT4 ? 2 : 1);
  static constexpr int A_BYTES = A_PIECES * 16, B_BYTES = B_PIECES * 16;
  static constexpr int S_BYTES = ((S_PIECES + 63) / 64) * 1024;
  static constexpr int B_OFF = A_BYTES, S_OFF = B_OFF + B_BYTES, Z_OFF = S_OFF + S_BYTES;
  static constexpr int STAGE = Z_OFF + (INT4 ? S_BYTES : 0);
  static constexpr int D_OFF = NST * STAGE;            // dump area of waves past an operand
  static constexpr int RED = NWAVE * 2 * 16 * 64 * 4;   // one row block of mid_reduce
  static constexpr int LDS_BYTES = D_OFF + 1024 > RED ? D_OFF + 1024 : RED;
};

// Chunks [c_beg, c_end) of MID_BK k into acc[rb][j] (this wave's share of each
// chunk's steps): rows 32*rb + 8*(v>>2) + 4*h + (v&3) and, for lane l32 of
// column group wn, LDS column 64*wn + 2*l32 + j (TM: 64*wn + 32*j + l32), as
// pf2_mainloop; `src` as there.  G128: g % 128 == 0 (a chunk lies in one group);
// otherwise g % 32 == 0 (a wave's share of a chunk does).  Requires K % 128 == 0.
template <bool INT4, int RB, int WN, bool G128, bool TM, class Src>
MM_DEV void mid_mainloop(const Src& src, int K, int g, int c_beg, int c_end, char* smem,
                         f32x16 (&acc)[RB][2]) {
  using Sh = MidShape<INT4, RB, WN>;
  constexpr int BK = MID_BK, WK = MID_WK, NST = MID_NST;
  constexpr int NWAVE = Sh::NWAVE, BN = Sh::BN, STEPS = Sh::STEPS, CW = 2;
  constexpr int PPR = BK / 8;                       // 16-byte pieces per A row
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wn = wave % WN, wk = wave / WN;
  const int l32 = lane & 31, h = lane >> 5;
  const int ngroups = K / g, ld = src.ld;
  auto asw = [](int r) { return r & 15; };

  const f16* a_src[Sh::A_IT];
#pragma unroll
  for (int i = 0; i < Sh::A_IT; ++i) {
    const int p = min((i * NWAVE + wave) * 64 + lane, Sh::A_PIECES - 1);
    a_src[i] = src.arow(p / PPR) + 8 * ((p % PPR) ^ asw(p / PPR));
  }
  // Marlin words: piece p is 4 columns of one word row, [16 word rows][BN].
  // Row-packed words (ROWP): a column's 16 words of a chunk are 64 contiguous
  // bytes, four pieces; piece pc of the q-th column in lane order lies at slot
  // 4*q + (pc ^ ((q >> 2) & 3)), so a load instruction reads 64-byte runs and the
  // lanes' LDS reads hit distinct banks.  Wave wk's two steps need piece wk
  // only: lane half h takes its words 2h (step 0) and 2h + 1 (step 1), one 8-byte
  // read per column, and the A pieces in the same k order.  4096 -> 2 x 14336 at
  // M = 64 25.5 us, as the Marlin words (the prefill kernel took 35.2).
  constexpr bool ROWP = is_rowpacked<Src>::value;
  static_assert(!ROWP || (BK == 128 && WK == 4), "one piece of a column per wave");
  const uint32_t* b_src[Sh::B_IT];
#pragma unroll
  for (int i = 0; i < Sh::B_IT; ++i) {
    const int p = min((i * NWAVE + wave) * 64 + lane, Sh::B_PIECES - 1);
    if constexpr (ROWP) {
      const int q = p >> 2, pc = (p & 3) ^ ((q >> 2) & 3);
      const int P = TM ? q : (q & ~63) + 2 * (q & 31) + ((q >> 5) & 1);
      b_src[i] = src.brow(P) + 4 * pc;
    } else {
      b_src[i] = src.bcol(4 * (p % (BN / 4)), 4) + (size_t)(p / (BN / 4)) * ld;
    }
  }
  int s_row[Sh::S_IT];
  const f16* s_src[Sh::S_IT];
  const f16* z_src[Sh::S_IT];
#pragma unroll
  for (int i = 0; i < Sh::S_IT; ++i) {
    const int p = min((i * NWAVE + wave) * 64 + lane, Sh::S_PIECES - 1);
    s_row[i] = p / (BN / 8);
    s_src[i] = src.scol(8 * (p % (BN / 8)), 8);
    z_src[i] = INT4 ? src.zcol(8 * (p % (BN / 8)), 8) : nullptr;
  }
  auto issue = [&](int ch, int st) {
    const int k0 = ch * BK;
    char* const base = smem + st * Sh::STAGE;
#pragma unroll
    for (int i = 0; i < Sh::S_IT; ++i) {
      const int wp = i * NWAVE + wave;
      const size_t off = (size_t)min(k0 / g + s_row[i], ngroups - 1) * ld;
      const bool live = wp * 64 < Sh::S_PIECES;
      gl2lds16(s_src[i] + off, live ? base + Sh::S_OFF + wp * 1024 : smem + Sh::D_OFF);
      if constexpr (INT4)
        gl2lds16(z_src[i] + off, live ? base + Sh::Z_OFF + wp * 1024 : smem + Sh::D_OFF);
    }
#pragma unroll
    for (int i = 0; i < Sh::B_IT; ++i) {
      const int wp = i * NWAVE + wave;
      gl2lds16(b_src[i] + (ROWP ? (size_t)(k0 / 8) : (size_t)(k0 / 8) * ld),
               wp * 64 < Sh::B_PIECES ? base + Sh::B_OFF + wp * 1024 : smem + Sh::D_OFF);
    }
#pragma unroll
    for (int i = 0; i < Sh::A_IT; ++i) {
      const int wp = i * NWAVE + wave;
      gl2lds16(a_src[i] + k0, wp * 64 < Sh::A_PIECES ? base + wp * 1024 : smem + Sh::D_OFF);
    }
  };

#pragma unroll
  for (int rb = 0; rb < RB; ++rb)
#pragma unroll
    for (int j = 0; j < CW; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[rb][j][v] = 0.0f;

  const int last = c_end - 1;
#pragma unroll
  for (int c = 0; c < NST - 1; ++c) issue(min(c_beg + c, last), c);

  const int colw = wn * 64 + (TM ? l32 : 2 * l32);
  constexpr int CS = TM ? 32 : 1;
  const uint32_t a_base = l32 * (BK * 2), asx = asw(l32);   // row blocks share the swizzle
  const uint32_t b_base = Sh::B_OFF + (h * BN + colw) * 4;
  f16x8 af[2][RB];
  f16x8 bq[2][CW];
  uint32_t wv[CW];
  u32x2 wp[CW];              // ROWP: both steps' words
  f16 sc[CW] = {}, nz[CW] = {};
  const uint32_t p_base = Sh::B_OFF + 64 * (wn * 64 + l32) + 16 * (wk ^ ((l32 >> 2) & 3)) + 8 * h;
  // LDS reads of step s (of this wave) of the chunk at ring position st.
  auto read = [&](int st, int s, int slot) {
    const int t = wk * STEPS + s;
    const char* const base = smem + st * Sh::STAGE;
    const uint32_t bo = b_base + t * 2 * BN * 4;
    if constexpr (ROWP) {
#pragma unroll
      for (int j = 0; j < CW; ++j) {
        if (s == 0) wp[j] = *(const u32x2*)(base + p_base + j * 32 * 64);
        wv[j] = wp[j][s];
      }
    } else if constexpr (TM) {
#pragma unroll
      for (int j = 0; j < CW; ++j) wv[j] = *(const uint32_t*)(base + bo + j * CS * 4);
    } else {
      const u32x2 w = *(const u32x2*)(base + bo);
      wv[0] = w.x, wv[1] = w.y;
    }
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
      af[slot][rb] =
          *(const f16x8*)(base + a_base + rb * 32 * BK * 2 +
                          (((ROWP ? 4 * wk + 2 * h + s : 2 * t + h) ^ asx) * 16));
  };
  auto read_scale = [&](int st, int k0) {
    // row of this wave's group among the staged rows
    const int row = G128 ? 0 : (k0 + 16 * STEPS * wk) / g - k0 / g;
    const char* const base = smem + st * Sh::STAGE + (row * BN + colw) * 2;
    if constexpr (TM) {
#pragma unroll
      for (int j = 0; j < CW; ++j) {
        sc[j] = *(const f16*)(base + Sh::S_OFF + j * CS * 2);
        if constexpr (INT4) nz[j] = *(const f16*)(base + Sh::Z_OFF + j * CS * 2);
      }
    } else {
      const f16x2 s2 = *(const f16x2*)(base + Sh::S_OFF);
      sc[0] = s2.x, sc[1] = s2.y;
      if constexpr (INT4) {
        const f16x2 z2 = *(const f16x2*)(base + Sh::Z_OFF);
        nz[0] = z2.x, nz[1] = z2.y;
      }
    }
#pragma unroll
    for (int j = 0; j < CW; ++j) {
      sc[j] = sanitize_scale(sc[j]);
      if constexpr (INT4) nz[j] = -clamp_zero(nz[j]);
    }
  };
  auto decode = [&](int slot) {
#pragma unroll
    for (int j = 0; j < CW; ++j)
      bq[slot][j] = WordDq<INT4>::run(wv[j], sc[j], nz[j]);
  };
  auto mfma = [&](int slot) {
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int j = 0; j < CW; ++j)
        acc[rb][j] =
            __builtin_amdgcn_mfma_f32_32x32x16_f16(af[slot][rb], bq[slot][j], acc[rb][j], 0, 0, 0);
#pragma unroll
    for (int i = 0; i < RB * CW; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);   // MFMA
      __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);   // DS read
      __builtin_amdgcn_sched_group_barrier(0x002, 9, 0);   // VALU
    }
  };
  // Next chunk: its loads are complete once at most the NST-2 chunks issued
  // after it are in flight; this wave's LDS reads of the stage that is refilled
  // next have returned (lgkmcnt 0).
  auto next_chunk = [&]() {
    wait_vm_lgkm<(NST - 2) * Sh::LOADS>();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  next_chunk();
  read(0, 0, 0);
  read_scale(0, c_beg * BK);
  decode(0);
  auto chunk = [&](int ch, auto stc) {
    constexpr int st = decltype(stc)::value, sn = (st + 1) % NST;
    // The stage of chunk ch - 1 was read by every wave before the last barrier.
    issue(min(ch + NST - 1, last), (st + NST - 1) % NST);
    static_assert(STEPS == 2, "one operand slot per step");
    read(st, 1, 1);
    mfma(0);
    decode(1);
    next_chunk();
    read(sn, 0, 0);
    read_scale(sn, min(ch + 1, last) * BK);
    mfma(1);
    decode(0);
  };
  for (int ch = c_beg; ch < c_end; ch += NST) {
    static_for(
        [&](auto stc) {
          constexpr int st = decltype(stc)::value;
          if (st == 0 || ch + st < c_end) chunk(ch + st, stc);
        },
        std::make_integer_sequence<int, NST>{});
  }
  wait_vmcnt<0>();
}

// Sums acc over the four waves of a column group, in wave order, one row block
// at a time through LDS (the ring's memory).  own[rb][j][i]: entry v = 4*wk + i
// of acc[rb][j] summed.
template <int RB, int WN>
MM_DEV void mid_reduce(char* smem, const f32x16 (&acc)[RB][2], f32x4 (&own)[RB][2]) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wn = wave % WN, wk = wave / WN;
  f32x4* const slots = (f32x4*)smem;
  auto at = [&](int w, int j, int v4) { return ((((w * WN + wn) * 2 + j) * 4 + v4) * 64) + lane; };
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    __syncthreads();       // the ring, or the previous row block, has been read
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int v4 = 0; v4 < 4; ++v4)
        slots[at(wk, j, v4)] = f32x4{acc[rb][j][4 * v4], acc[rb][j][4 * v4 + 1],
                                     acc[rb][j][4 * v4 + 2], acc[rb][j][4 * v4 + 3]};
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      f32x4 x = slots[at(0, j, wk)];
#pragma unroll
      for (int w = 1; w < MID_WK; ++w) x += slots[at(w, j, wk)];
      own[rb][j] = x;
    }
  }
}
}  // namespace mmmid

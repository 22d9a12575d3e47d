// The fp8 block-scaled GEMM of gemm_fp8.hip for chunks too small to fill the
// chip with 256 x 256 tiles: the same MFMA per 128-deep K block, the same
// promotion order per output and the same epilogue arithmetic, so the same
// bits, on smaller tiles. Included by gemm_fp8.hip only.
#pragma once

namespace qh {
namespace gemm_small {

using gemm::BK;
using gemm::kQkvRope;
using gemm::kSiluQuant;
using gemm::kStoreBf16;

// One workgroup of NW = NR x WT waves computes BM = 16 TM WT tokens x
// BR = 16 NR RT weight rows; a wave holds RT n-tiles (16 weight rows each) of
// 16 TM tokens. K
// blocks of weights and activations, and the block's activation scales,
// reach an NS-stage LDS ring by DMA NS - 1 blocks ahead.
template <int EPI, int NR, int WT, int RT, int TM, int KU, int NS>
struct Shape {
  static constexpr int NW = NR * WT;
  static constexpr int BR = 16 * NR * RT;
  static constexpr int BM = 16 * TM * WT;
  static constexpr int WBYTES = BR * BK;
  static constexpr int ABYTES = BM * BK;
  static constexpr int SC = BM > 64 ? 512 : 256;     // activation scales: a dword DMA per 64 tokens
  static constexpr int BLOCK = WBYTES + ABYTES + SC;  // one K block
  static constexpr int STAGE = KU * BLOCK;
  static constexpr int WI = 2 * NR * RT / NW;        // 1 KiB weight pieces per wave
  static constexpr int AI = BM / 8;                  // 1 KiB activation pieces
  static constexpr int AL = (AI + NW - 1) / NW;      // issued per wave
  static constexpr int BLOADS = WI + AL + 1;         // DMA instructions per wave and block
  static constexpr int LOADS = KU * BLOADS;          // and per step
  // the epilogue stages the tile in LDS: token rows, padded by 16 bytes
  static constexpr int OUTB = EPI == kSiluQuant ? BR / 2 : BR * 2;
  static constexpr int OROW = OUTB + 16;
  // beside it: a head's squares (kQkvRope) or the waves' group maxima
  static constexpr int EXTRA = EPI == kQkvRope ? (BR / 128) * 8 * TM * WT * 256
                               : EPI == kSiluQuant ? NR * BM * 4 : 0;
  // weight-block scale rows of the tile, all K blocks
  static constexpr int NB = EPI == kSiluQuant || (EPI == kQkvRope && BR == 256) ? 2 : 1;
  static constexpr int SBROW = 4 * MAX_NK;
  static constexpr int SBROWS = BR == 256 ? 2 : 1;
  // The last step reads ahead like the others, into registers that nobody uses:
  // up to scale KU ceil(nk / KU) + KU - 1 of a row, which for nk = 253 .. 255 and
  // four blocks a step lies past the last row. The pad keeps it inside.
  static constexpr int SB_END = 4 * ((MAX_NK - 1 + KU - 1) / KU * KU + KU);
  static constexpr int SB_PAD = SB_END > SBROW ? SB_END - SBROW : 0;
  static constexpr int LDS_LOOP = NS * STAGE + SBROWS * SBROW + SB_PAD;
  static constexpr int LDS_EPI = BM * OROW + EXTRA;
  static constexpr int LDS = LDS_LOOP > LDS_EPI ? LDS_LOOP : LDS_EPI;
  static_assert(BM <= 64 || (BM <= 128 && NW % 2 == 0), "the scale DMA covers the tile's tokens");
  static_assert(2 * NR * RT % NW == 0 && (NS - 1) * LOADS < 64, "DMA pieces");
  static_assert(EPI == kStoreBf16 || BR == 256 || (EPI == kQkvRope && BR == 128),
                "a fused epilogue needs whole heads, or the gate and up rows of a group");
  static_assert(EPI != kQkvRope || NR == 4, "a head's n-tiles lie over four waves, two each");
  static_assert(LDS <= 160 * 1024, "LDS");
  static_assert(NS * STAGE + (SBROWS - 1) * SBROW + SB_END <= LDS, "the read ahead's last scale");
};

// f(0) .. f(N - 1) with compile-time arguments: fragment arrays indexed by an
// unrolled loop's counter went to scratch in the largest variant.
template <typename F, int... I>
__device__ __forceinline__ void static_each(F& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F f) {
  static_each(f, std::make_integer_sequence<int, N>{});
}

template <int N>
__device__ __forceinline__ void wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"i"(N) : "memory");
}

template <int EPI, bool HW, int NR, int WT, int RT, int TM, int KU, int NS, int OCC>
__global__ __launch_bounds__(64 * NR * WT, OCC) void fp8_gemm_small_kernel(GemmArgs p) {
  using S = Shape<EPI, NR, WT, RT, TM, KU, NS>;
  constexpr int NW = S::NW;
  __shared__ __attribute__((aligned(1024))) uint8_t lds[S::LDS];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wr = wave % NR;          // the wave's rows
  const int tok0 = 16 * TM * (wave / NR);  // and first token of the tile
  const int g = lane >> 4;
  const int M = p.M;
  const int nk = p.K / BK;

  // ---- tile: XCD-contiguous chunks, then group_m tile rows per column sweep;
  // or the pieces, neighbours in launch order, of 256 x 256 tiles tile0 and up ----
  int tm, tn;
  {
    const int n = (int)gridDim.x, per = n / gemm::XCDS;
    int t = (int)blockIdx.x;
    if (t < per * gemm::XCDS) t = (t % gemm::XCDS) * per + t / gemm::XCDS;
    if (p.tile0 == 0)
      tile_at(t, p.group_m, (M + S::BM - 1) / S::BM, p.N / S::BR, tm, tn);
    else
      Pieces(p.tile0, M, p.N, S::BM, S::BR).at(t, tm, tn);
  }
  const int m0 = tm * S::BM;

  // n-tile u of this wave, in the tile's row order. A fused epilogue wants a
  // column's partner in the same lane: gate n-tile i beside up n-tile i, a
  // head's n-tile ib beside ib + 4.
  auto ntile = [&](int u) __attribute__((always_inline)) {
    if constexpr (EPI == kSiluQuant)
      return u < RT / 2 ? wr * (RT / 2) + u : 8 + wr * (RT / 2) + (u - RT / 2);
    else if constexpr (EPI == kQkvRope)
      return 8 * (u >> 1) + wr + 4 * (u & 1);
    else
      return wr * RT + u;
  };
  // first weight row of the tile's 8-row piece b
  auto piece_row = [&](int b) __attribute__((always_inline)) {
    if constexpr (EPI == kSiluQuant)
      return b < 16 ? 128 * tn + 8 * b : p.N / 2 + 128 * tn + 8 * (b - 16);
    else
      return S::BR * tn + 8 * b;
  };

  // ---- loads ---------------------------------------------------------------
  // 8-row pieces of 128 bytes a row: lane l fetches physical chunk l % 8 of row
  // l / 8, which holds logical chunk (l % 8) ^ (row % 8). Tokens past M lie
  // outside the descriptor and read zero.
  const uint32_t swz = (uint32_t)((((lane & 7) ^ (lane >> 3)) & 7) * 16);
  const i32x4 rb = buffer_rsrc(p.B, (uint32_t)((long)p.N * p.ldb));
  const uint32_t offb = (uint32_t)(lane >> 3) * (uint32_t)p.ldb + swz;
  const i32x4 ra = buffer_rsrc(p.A + (long)m0 * p.lda,
                               (uint32_t)((long)min(M - m0, S::BM) * p.lda));
  const uint32_t offa = (uint32_t)(lane >> 3) * (uint32_t)p.lda + swz;
  const i32x4 rsa = buffer_rsrc(p.sa, (uint32_t)nk * (uint32_t)p.ld_sa * 4u);
  const uint32_t offs = (uint32_t)lane * 4u;
  // DMA instruction op (0 .. LOADS - 1) of block kb into `stage`: weight
  // pieces, then activation pieces (every wave issues AL of them, the same
  // count for every wave's waits; a piece issued twice writes the same bytes
  // twice), then the block's activation scales.
  // Blocks past the last are issued too, through empty descriptors: the
  // counts stay the same to the end and nothing is fetched.
  auto issue = [&](int step, int stage, int idx) __attribute__((always_inline)) {
    const int kb = KU * step + idx / S::BLOADS, op = idx % S::BLOADS;
    uint8_t* st = lds + stage * S::STAGE + (idx / S::BLOADS) * S::BLOCK;
    auto live = [&](i32x4 r) __attribute__((always_inline)) {
      r[2] = kb < nk ? r[2] : 0;
      return r;
    };
    if (op < S::WI) {
      const int b = op * NW + wave;
      const uint32_t dst = lds_addr(st + b * 1024);
      const uint32_t so = (uint32_t)piece_row(b) * (uint32_t)p.ldb + (uint32_t)kb * BK;
      asm volatile(
          "s_mov_b32 m0, %0\n\t"
          "buffer_load_dwordx4 %1, %2, %3 offen lds"
          :
          : "s"(dst), "v"(offb), "s"(live(rb)), "s"(so)
          : "memory", "m0");
    } else if (op < S::WI + S::AL) {
      const int b = ((op - S::WI) * NW + wave) % S::AI;
      const uint32_t dst = lds_addr(st + S::WBYTES + b * 1024);
      const uint32_t so = (uint32_t)(8 * b) * (uint32_t)p.lda + (uint32_t)kb * BK;
      asm volatile(
          "s_mov_b32 m0, %0\n\t"
          "buffer_load_dwordx4 %1, %2, %3 offen lds"
          :
          : "s"(dst), "v"(offa), "s"(live(ra)), "s"(so)
          : "memory", "m0");
    } else {
      const int h = S::BM > 64 ? wave & 1 : 0;  // which 64 tokens
      const uint32_t dst = lds_addr(st + S::WBYTES + S::ABYTES + 256 * h);
      const uint32_t so = ((uint32_t)kb * (uint32_t)p.ld_sa + (uint32_t)(m0 + 64 * h)) * 4u;
      asm volatile(
          "s_mov_b32 m0, %0\n\t"
          "buffer_load_dword %1, %2, %3 offen lds"
          :
          : "s"(dst), "v"(offs), "s"(live(rsa)), "s"(so)
          : "memory", "m0");
    }
  };

  // The scale rows of the tile's 128-row weight blocks (sb, all K blocks) by
  // DMA ahead of everything else: wave r < SBROWS moves row r.
  uint8_t* const sb_lds = lds + NS * S::STAGE;
  if (wave < S::SBROWS) {
    const i32x4 rsb = buffer_rsrc(p.sb, (uint32_t)(p.N / 128) * (uint32_t)nk * 4u);
    const uint32_t so = (uint32_t)(piece_row(16 * wave) / 128) * (uint32_t)nk * 4u;
    for (int k = 0; k < nk; k += 64)
      asm volatile(
          "s_mov_b32 m0, %0\n\t"
          "buffer_load_dword %1, %2, %3 offen lds"
          :
          : "s"(lds_addr(sb_lds + wave * S::SBROW + 4 * k)), "v"(offs), "s"(rsb),
            "s"(so + 4u * (uint32_t)k)
          : "memory", "m0");
  }
  // n-tile u's scale row: 0 for a tile of one 128-row block
  auto sb_row = [&](int u) __attribute__((always_inline)) {
    return S::SBROWS == 1 ? 0 : ntile(u) >> 3;
  };
  constexpr int NB = S::NB;  // distinct scale rows of one wave
  auto sb_of = [](int u) { return NB == 2 && u >= RT / 2 ? 1 : 0; };

  const int frow = (lane & 15) * BK;
  const int c_lo = ((g ^ (lane & 7)) & 7) * 16;
  const int c_hi = (((g + 4) ^ (lane & 7)) & 7) * 16;
  auto frag = [&](const uint8_t* st, int i) __attribute__((always_inline)) {
    const uint8_t* q = st + i * 16 * BK + frow;
    const i32x4 lo = *reinterpret_cast<const i32x4*>(q + c_lo);
    const i32x4 hi = *reinterpret_cast<const i32x4*>(q + c_hi);
    return (v8i){lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
  };

  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  f32x4 acc[RT][TM];
#pragma unroll
  for (int u = 0; u < RT; ++u)
#pragma unroll
    for (int j = 0; j < TM; ++j) acc[u][j] = zero;

  // kQkvRope: what the epilogue reads, loaded ahead of the K loop: the lane's
  // token positions, its norm weights, and the arena rows of what it stores
  // (an arena has far fewer than 2^31 rows: their low words). In the epilogue
  // each was a round trip to memory, one after the other: the qkv projection of
  // 80 tokens on cold weights 15.5 -> 13.5 us, Qwen3-32B's of 192 tokens 28.8 ->
  // 26.8.
  constexpr int CHUNKS = S::OUTB / 16;                  // 16-byte pieces of a staged row
  constexpr int ITERS = (S::BM * CHUNKS + 64 * NW - 1) / (64 * NW);  // of them per thread
  static_assert(EPI != kQkvRope || (S::BM * CHUNKS % (64 * NW) == 0 && 64 * NW % S::BM == 0),
                "the arena rows of a thread");
  int pos[TM], arow[ITERS];
  uint2 wl, wh;
  if constexpr (EPI == kQkvRope) {
#pragma unroll
    for (int j = 0; j < TM; ++j)
      pos[j] = (int)p.rope.positions[min(m0 + tok0 + 16 * j + (lane & 15), M - 1)];
    const int head0 = tn * (S::BR / 128);
    const bool is_q = head0 < p.rope.n_q, is_v = head0 >= p.rope.n_q + p.rope.n_kv;
    const uint16_t* wt = (is_q ? p.rope.q_w : p.rope.k_w) + 16 * wr + 4 * g;
    wl = *reinterpret_cast<const uint2*>(wt);
    wh = *reinterpret_cast<const uint2*>(wt + 64);
    if (!is_q && p.rope.row_dst != nullptr) {
#pragma unroll
      for (int i = 0; i < ITERS; ++i) {
        const int t = is_v ? tid % S::BM : (tid + 64 * NW * i) / CHUNKS;
        arow[i] = (int)p.rope.row_dst[min(m0 + t, M - 1)];
      }
    }
  }

  // ---- K loop ----------------------------------------------------------------
  // Fragments and scales of block s + 1 are read from LDS while block s is
  // multiplied from registers, so a wave's LDS latency hides behind its own
  // MFMAs. A stage is free as soon as its fragments are in registers: block
  // s + NS goes into block s's stage.
  v8i xa[2][KU][TM], wb[2][KU][RT];
  float sa[2][KU][TM], sb[2][KU][NB];
  // read i (0 .. TM + RT - 1) of block s: activation fragments with their
  // scales, then weight fragments
  auto read = [&](int step, int stage, auto slot_c, auto idx_c) __attribute__((always_inline)) {
    constexpr int slot = decltype(slot_c)::value;
    constexpr int kk = decltype(idx_c)::value / (TM + RT), i = decltype(idx_c)::value % (TM + RT);
    const uint8_t* st = lds + stage * S::STAGE + kk * S::BLOCK;
    if constexpr (i < TM) {
      sa[slot][kk][i] = *reinterpret_cast<const float*>(st + S::WBYTES + S::ABYTES +
                                                        4 * (tok0 + 16 * i + (lane & 15)));
      xa[slot][kk][i] = frag(st + S::WBYTES + tok0 * BK, i);
    } else {
      constexpr int u = i - TM;
      if constexpr (u < NB)
        sb[slot][kk][u] = *reinterpret_cast<const float*>(
            sb_lds + sb_row(u * (RT / NB)) * S::SBROW + 4 * (KU * step + kk));
      wb[slot][kk][u] = frag(st, ntile(u));
    }
  };
#pragma unroll
  for (int s = 0; s < NS; ++s)
#pragma unroll
    for (int op = 0; op < S::LOADS; ++op) issue(s, s, op);
  wait_vm<(NS - 1) * S::LOADS>();
  wg_barrier();
  static_for<KU*(TM + RT)>([&](auto i_c) __attribute__((always_inline)) {
    read(0, 0, std::integral_constant<int, 0>{}, i_c);
  });
  int stage = 0;  // of block s
  auto step = [&](int s, auto slot_c) __attribute__((always_inline)) {
    constexpr int slot = decltype(slot_c)::value;
    // this wave's fragments of block s are in registers
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    const int next = stage == NS - 1 ? 0 : stage + 1;
    const int freed = stage;
    wait_vm<(NS - 2) * S::LOADS>();
    wg_barrier();  // publishes block s + 1, frees block s's stage
    stage = next;
    float sc[KU][NB][TM];
    int ea[KU][TM], eb[KU][NB];
#pragma unroll
    for (int kk = 0; kk < KU; ++kk) {
      // a block past the last multiplies zeros; its scales are not data
      const bool live = KU == 1 || KU * s + kk < nk;
#pragma unroll
      for (int j = 0; j < TM; ++j) {
        ea[kk][j] = (int)((__builtin_bit_cast(uint32_t, sa[slot][kk][j]) >> 23) & 0xffu);
#pragma unroll
        for (int b = 0; b < NB; ++b)
          sc[kk][b][j] = live ? sa[slot][kk][j] * sb[slot][kk][b] : 0.f;
      }
#pragma unroll
      for (int b = 0; b < NB; ++b)
        eb[kk][b] = live ? (int)((__builtin_bit_cast(uint32_t, sb[slot][kk][b]) >> 23) & 0xffu) : 0;
    }
    f32x4 t0 = zero, t1 = zero;  // products two and one MFMAs back
    auto promote = [&](auto q_c, const f32x4& t) __attribute__((always_inline)) {
      constexpr int q = decltype(q_c)::value;
      constexpr int u = q % (RT * TM) / TM, j = q % TM;
      const float c = sc[q / (RT * TM)][sb_of(u)][j];
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[u][j][r] += t[r] * c;
    };
    // Between MFMAs: block s + NS's DMA instructions and block s + 1's fragment
    // reads, spread evenly. Issued together ahead of the MFMAs, the DMA's 64
    // bytes a clock and the MFMAs run one after the other.
    constexpr int Q = KU * RT * TM, R = KU * (TM + RT);
    static_for<Q>([&](auto q_c) __attribute__((always_inline)) {
      constexpr int q = decltype(q_c)::value;
      constexpr int kk = q / (RT * TM), u = q % (RT * TM) / TM, j = q % TM;
      if constexpr (HW) {
        acc[u][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(
            wb[slot][kk][u], xa[slot][kk][j], acc[u][j], 0, 0, 0, eb[kk][sb_of(u)], 0, ea[kk][j]);
      } else {
        const f32x4 t = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(
            wb[slot][kk][u], xa[slot][kk][j], zero, 0, 0, 0, 127, 0, 127);
        if constexpr (q >= 2) promote(std::integral_constant<int, q - 2>{}, t0);
        t0 = t1;
        t1 = t;
      }
      static_for<(q + 1) * R / Q - q * R / Q>([&](auto i_c) __attribute__((always_inline)) {
        read(s + 1, next, std::integral_constant<int, 1 - slot>{},
             std::integral_constant<int, q * R / Q + decltype(i_c)::value>{});
      });
      static_for<(q + 1) * S::LOADS / Q - q * S::LOADS / Q>([&](auto i_c)
          __attribute__((always_inline)) {
        issue(s + NS, freed, q * S::LOADS / Q + decltype(i_c)::value);
      });
      __builtin_amdgcn_sched_barrier(0);
    });
    if constexpr (!HW) {
      if constexpr (Q >= 2) promote(std::integral_constant<int, Q - 2>{}, t0);
      promote(std::integral_constant<int, Q - 1>{}, t1);
    }
  };
  const int steps = (nk + KU - 1) / KU;
  for (int s = 0; s < steps; s += 2) {
    step(s, std::integral_constant<int, 0>{});
    if (s + 1 < steps) step(s + 1, std::integral_constant<int, 1>{});
  }
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
  wg_barrier();  // every wave is past its last fragment: the ring is free

  // ---- epilogues -----------------------------------------------------------------
  // A lane holds columns 16 nt + 4 g + r of token 16 j + lane % 16.
  typedef float f32x2_t __attribute__((ext_vector_type(2)));
  auto stage_bf16 = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < RT; ++u)
#pragma unroll
      for (int j = 0; j < TM; ++j) {
        const f32x2_t x0 = {acc[u][j][0], acc[u][j][1]}, x1 = {acc[u][j][2], acc[u][j][3]};
        const bf16x2 p0 = __builtin_convertvector(x0, bf16x2);
        const bf16x2 p1 = __builtin_convertvector(x1, bf16x2);
        *reinterpret_cast<uint2*>(lds + (tok0 + 16 * j + (lane & 15)) * S::OROW + 32 * ntile(u) + 8 * g) =
            make_uint2(__builtin_bit_cast(uint32_t, p0), __builtin_bit_cast(uint32_t, p1));
      }
  };
  // the staged rows, 16 bytes per thread: dst(token of the tile, 16-byte chunk)
  auto store_rows = [&](auto dst) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < ITERS; ++i) {
      const int c = tid + 64 * NW * i, t = c / CHUNKS, ch = c % CHUNKS;
      if (t < S::BM && m0 + t < M)
        *reinterpret_cast<uint4*>(dst(t, ch, i)) =
            *reinterpret_cast<const uint4*>(lds + t * S::OROW + 16 * ch);
    }
  };

  if constexpr (EPI == kStoreBf16) {
    stage_bf16();
    __syncthreads();
    uint8_t* C = (uint8_t*)p.C + (long)m0 * p.ldc * 2 + (long)tn * S::BR * 2;
    store_rows([&](int t, int ch, int i) __attribute__((always_inline)) {
      return C + (long)t * p.ldc * 2 + 16 * ch;
    });
  } else if constexpr (EPI == kSiluQuant) {
    float* red = reinterpret_cast<float*>(lds + S::BM * S::OROW);
    float amax[TM];
#pragma unroll
    for (int j = 0; j < TM; ++j) {
      float a = 0.f;
#pragma unroll
      for (int u = 0; u < RT / 2; ++u)
#pragma unroll
        for (int r = 0; r < 4; r += 2) {
          float g0 = acc[u][j][r], g1 = acc[u][j][r + 1];
          float u0 = acc[u + RT / 2][j][r], u1 = acc[u + RT / 2][j][r + 1];
          round_bf16_pair(g0, g1);
          round_bf16_pair(u0, u1);
          const float y0 = silu_mul(g0, u0), y1 = silu_mul(g1, u1);
          acc[u][j][r] = y0;
          acc[u][j][r + 1] = y1;
          a = fmaxf(a, fabsf(y0));
          a = fmaxf(a, fabsf(y1));
        }
      a = fmaxf(a, __shfl_xor(a, 16, kWave));
      a = fmaxf(a, __shfl_xor(a, 32, kWave));
      if (g == 0) red[wr * S::BM + tok0 + 16 * j + lane] = a;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < TM; ++j) {
      float a = 0.f;
#pragma unroll
      for (int w = 0; w < NR; ++w) a = fmaxf(a, red[w * S::BM + tok0 + 16 * j + (lane & 15)]);
      const float scale = group_scale(a, p.ue8m0 != 0);
      const double rinv = recip_exact(scale);
#pragma unroll
      for (int u = 0; u < RT / 2; ++u)
        *reinterpret_cast<uint32_t*>(lds + (tok0 + 16 * j + (lane & 15)) * S::OROW + 16 * ntile(u) +
                                     4 * g) =
            quant_e4m3_x4(acc[u][j][0], acc[u][j][1], acc[u][j][2], acc[u][j][3], rinv);
      const int m = m0 + tok0 + 16 * j + lane;
      if (wr == 0 && g == 0 && m < M) p.scales[(long)tn * p.ld_sa + m] = scale;
    }
    __syncthreads();
    uint8_t* out = (uint8_t*)p.C + (long)m0 * p.ldc + 128 * tn;
    store_rows([&](int t, int ch, int i) __attribute__((always_inline)) {
      return out + (long)t * p.ldc + 16 * ch;
    });
  } else {
    constexpr int PT = 16;              // arena page tokens (checked at launch)
    // the arguments are read here, through a pointer the compiler cannot see
    // through, so they hold no scalar registers across the K loop
    typedef const __attribute__((address_space(4))) QkvRope ConstRope;
    const __attribute__((address_space(4))) uint8_t* ka =
        (const __attribute__((address_space(4))) uint8_t*)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(ka));
    ConstRope& R = *reinterpret_cast<ConstRope*>(ka + offsetof(GemmArgs, rope));
    const int head0 = tn * (S::BR / 128);  // q heads, then k heads, then v heads
    const bool is_q = head0 < R.n_q, is_v = head0 >= R.n_q + R.n_kv;
    if (!is_v) {
      // the lane's cos and sin, on their way while the squares are summed
      uint2 cr[TM], sr[TM];
#pragma unroll
      for (int j = 0; j < TM; ++j) {
        const int ps = pos[j] < 0 ? 0 : (pos[j] >= R.max_pos ? R.max_pos - 1 : pos[j]);
        const uint16_t* cs = R.cos_sin + (long)ps * 128 + 16 * wr + 4 * g;
        cr[j] = *reinterpret_cast<const uint2*>(cs);
        sr[j] = *reinterpret_cast<const uint2*>(cs + 64);
      }
      float* sq = reinterpret_cast<float*>(lds + S::BM * S::OROW);
      // u's n-tile as (head of the tile, ib), as ntile() lays them out
      auto head_of = [](int u) __attribute__((always_inline)) { return u >> 1; };
      // u even: n-tile wr of its head, u odd: wr + 4
#pragma unroll
      for (int u = 0; u < RT; ++u)
#pragma unroll
        for (int j = 0; j < TM; ++j) {
          f32x4& v = acc[u][j];
          float x0 = v[0], x1 = v[1], x2 = v[2], x3 = v[3];
          round_bf16_pair(x0, x1);
          round_bf16_pair(x2, x3);
          v = (f32x4){x0, x1, x2, x3};
          sq[((head_of(u) * 8 + wr + 4 * (u & 1)) * TM * WT + tok0 / 16 + j) * 64 + lane] = sumsq4(x0, x1, x2, x3);
        }
      __syncthreads();
#pragma unroll
      for (int u = 0; u < RT; u += 2) {
        const uint32_t wlo[2] = {wl.x, wl.y}, whi[2] = {wh.x, wh.y};
#pragma unroll
        for (int j = 0; j < TM; ++j) {
          const float* q = sq + (head_of(u) * 8 * TM * WT + tok0 / 16 + j) * 64 + lane;
          float qs[8];
#pragma unroll
          for (int ib = 0; ib < 8; ++ib) qs[ib] = q[ib * TM * WT * 64];
          const float sg = ((qs[0] + qs[1]) + (qs[2] + qs[3])) + ((qs[4] + qs[5]) + (qs[6] + qs[7]));
          const float rstd = head_rstd(xor32_sum(xor16_sum(sg)), R.eps);
          const uint32_t cw[2] = {cr[j].x, cr[j].y}, sw[2] = {sr[j].x, sr[j].y};
          f32x4& lo = acc[u][j];
          f32x4& hi = acc[u + 1][j];
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int sh = 16 * (r & 1);
            const float a0 = head_norm(lo[r], rstd, bf16_to_f32((wlo[r >> 1] >> sh) & 0xffffu));
            const float b0 = head_norm(hi[r], rstd, bf16_to_f32((whi[r >> 1] >> sh) & 0xffffu));
            const float c = bf16_to_f32((cw[r >> 1] >> sh) & 0xffffu);
            const float s = bf16_to_f32((sw[r >> 1] >> sh) & 0xffffu);
            lo[r] = rope_first(a0, b0, c, s);
            hi[r] = rope_second(b0, a0, c, s);
          }
        }
      }
    }
    stage_bf16();
    __syncthreads();
    if (is_q) {
      uint8_t* Q = (uint8_t*)R.q_out + (long)m0 * R.ld_q * 2 + (long)head0 * 256;
      store_rows([&](int t, int ch, int i) __attribute__((always_inline)) {
        return Q + (long)t * R.ld_q * 2 + 16 * ch;
      });
    } else if (R.row_dst == nullptr) {
      const int h = head0 - R.n_q - (is_v ? R.n_kv : 0);
      uint8_t* D = (uint8_t*)(is_v ? R.v_out : R.k_out) + (long)m0 * R.ld_kv * 2 + (long)h * 256;
      store_rows([&](int t, int ch, int i) __attribute__((always_inline)) {
        return D + (long)t * R.ld_kv * 2 + 16 * ch;
      });
    } else if (!is_v) {
      // K page rows: 256 bytes per token and head
      uint8_t* KP = (uint8_t*)R.k_pool;
      const int h0 = head0 - R.n_q;
      store_rows([&](int t, int ch, int i) __attribute__((always_inline)) {
        const long r = arow[i];
        return KP + (((r >> 4) * R.n_kv + h0 + (ch >> 4)) * PT + (r & (PT - 1))) * 256 +
               16 * (ch & 15);
      });
    } else {
      // V^T pages: tokens fastest over the lanes, so consecutive tokens land
      // in consecutive slots of one 32-byte page row
      const int h0 = head0 - R.n_q - R.n_kv;
      const int t = tid % S::BM;
      const long r = arow[0];
      if (m0 + t < M) {
        uint16_t* V = R.v_pool + ((r >> 4) * R.n_kv + h0) * 128 * PT + (r & (PT - 1));
#pragma unroll
        for (int i = 0; i < S::BM * S::BR / (64 * NW); ++i) {
          const int d = tid / S::BM + 64 * NW / S::BM * i;
          V[d * PT] = *reinterpret_cast<const uint16_t*>(lds + t * S::OROW + 2 * d);
        }
      }
    }
  }
}

template <int EPI, bool HW, int NR, int WT, int RT, int TM, int KU, int NS, int OCC>
static int launch(GemmArgs a, qh_stream_t stream, const char* what) {
  using S = Shape<EPI, NR, WT, RT, TM, KU, NS>;
  const int tiles = a.tile0 == 0 ? ((a.M + S::BM - 1) / S::BM) * (a.N / S::BR)
                                 : (int)Pieces(a.tile0, a.M, a.N, S::BM, S::BR).count();
  a.group_m = 8;
  hipLaunchKernelGGL((fp8_gemm_small_kernel<EPI, HW, NR, WT, RT, TM, KU, NS, OCC>), dim3(tiles),
                     dim3(64 * S::NW), 0, (hipStream_t)stream, a);
  return launch_status(what);
}

// Launches tiling v of choose().
template <int EPI, bool HW>
static int launch_tiling(int v, const GemmArgs& a, qh_stream_t st, const char* what) {
  if constexpr (EPI == kStoreBf16) {
    switch (v) {
      case 0: return launch<EPI, HW, 2, 1, 1, 1, 4, 4, 1>(a, st, what);
      case 1: return launch<EPI, HW, 4, 1, 1, 1, 4, 3, 1>(a, st, what);
      case 2: return launch<EPI, HW, 4, 1, 1, 2, 4, 3, 1>(a, st, what);
      case 3: return launch<EPI, HW, 4, 2, 1, 2, 2, 3, 2>(a, st, what);
      case 4: return launch<EPI, HW, 4, 1, 2, 4, 1, 3, 2>(a, st, what);
      case 5: return launch<EPI, HW, 4, 2, 2, 4, 1, 4, 2>(a, st, what);
      default: return launch<EPI, HW, 4, 2, 4, 4, 1, 3, 2>(a, st, what);
    }
  } else if constexpr (EPI == kSiluQuant) {
    switch (v) {
      case 0: return launch<EPI, HW, 4, 1, 4, 1, 1, 4, 1>(a, st, what);
      case 1: return launch<EPI, HW, 8, 1, 2, 2, 1, 4, 2>(a, st, what);
      case 2: return launch<EPI, HW, 8, 1, 2, 4, 1, 3, 2>(a, st, what);
      default: return launch<EPI, HW, 4, 2, 4, 4, 1, 3, 2>(a, st, what);
    }
  } else {
    switch (v) {
      case 0: return launch<EPI, HW, 4, 1, 2, 1, 1, 4, 1>(a, st, what);
      case 1: return launch<EPI, HW, 4, 1, 2, 2, 1, 3, 2>(a, st, what);
      case 2: return launch<EPI, HW, 4, 2, 2, 2, 1, 4, 2>(a, st, what);
      case 3: return launch<EPI, HW, 4, 2, 2, 4, 1, 4, 2>(a, st, what);
      default: return launch<EPI, HW, 4, 2, 4, 4, 1, 3, 2>(a, st, what);
    }
  }
}

}  // namespace gemm_small
}  // namespace qh

// Four-wave 256 x 256 bf16 GEMM with a hand-scheduled K-loop (K1, large M):
//
//   C[M, N] = A[M, K] . B[N, K]^T        (A: activations row-major, B: weights [out, in])
//
// One workgroup = 4 waves = one SIMD each, 128 x 128 outputs per wave held in all 256
// AGPRs (8 x 8 v_mfma_f32_16x16x32_bf16 accumulators).  Both operands stream global -> LDS
// by LDS-DMA (buffer_load_dwordx4 ... lds) into two 64 KiB buffers; the K-loop is ONE
// inline-asm statement generated by ops/gen_gemm_w4.py (csrc/gemm_w4_asm.h) so that every
// MFMA is followed by at most one LDS read or DMA issue and the two barriers per K-tile sit
// between MFMAs: with one wave per SIMD the interleave is the only latency hiding, and hipcc
// re-orders a HIP-source version of it (profiles/r03_gemm_fourwave.md: 126-137 us at 4096^3).
// The DMA for K-tile t+2 goes into the buffer of tile t as soon as every wave has its
// fragments of tile t in registers, so one buffer pair keeps a whole tile in flight.
// BMT = 128 is the half-height tile (planner variant 6): 64 x 128
// outputs per wave (a[0:127]), 12 DMA pieces per K-tile, its own generated loop
// (MLOP_W4H_KLOOP_*, 64 MFMAs per K-tile), every epilogue shared with the full tile.  BMT = 160, 192 and 224
// (80, 96 and 112 output rows per wave, loops MLOP_W4_160_* / _192_* / _224_*) stand between them for grids that both
// fill badly: whole rounds take 0.70, 0.805 and 0.90 of the full tile's (gemm.hip big_plan has the choice and its
// figures).
//
// HIP handles the rest: tile placement (XCD-contiguous bands, as gemm_pp_kernel), per-lane
// DMA source offsets (rows clamped to the last valid row, XOR swizzle in the source), the
// accumulator read-out (v_accvgpr_read statements) and the epilogues, all straight from the
// accumulators (the loop computes C^T, so each lane owns 4 consecutive columns): plain store,
// SiLU-mul (gate / up interleaved in groups of 16 columns), RoPE + paged K / V (both pages
// token-major; a wave's 128 columns are one head; rotate-half partners sit in the same lane).  Requirements: K % 64 == 0, K >= 192, lda / ldb % 8 == 0.
#include "common.h"
#include "launch.h"
#include "gemm_w4_asm.h"

#include <type_traits>
#include <utility>

namespace mlop {

namespace {
// epilogue = base (bits 0-1) | flags: W4_ADD_SS (plain base only) C += A.B^T in place with the
// per-row sum-of-squares partials of the new C; W4_RS rows scaled by the RMSNorm factor from
// re.ss_in (launch.h RopeEpi; the norm chain of launch_w4_chain).  W4_SLAB: K in ranges, fp32 slabs [range][M][N] in C
// (run_w4_slab; one item per workgroup, nothing prefetched behind it)
enum { W4_NONE = 0, W4_SILU_MUL = 1, W4_SLAB = 2, W4_ROPE = 3, W4_ADD_SS = 4, W4_RS = 8 };
using i32x4 = __attribute__((ext_vector_type(4))) int;
typedef __attribute__((address_space(3))) uint16_t lds_u16;

__device__ __forceinline__ i32x4 make_srd(const void* p) {
  const uint64_t a = (uint64_t)p;
  i32x4 r;
  r.x = __builtin_amdgcn_readfirstlane((int)(uint32_t)a);
  r.y = __builtin_amdgcn_readfirstlane((int)(uint32_t)(a >> 32));
  r.z = 0x7fffffff;  // num_records: offsets stay < 2^31, but for those of A rows past the last (dma_offsets)
  r.w = 0x00020000;
  return r;
}

// accumulator row-block I (acc(I, 0..7), 32 AGPRs) -> v[0..31]; v[4j + r] = acc(I, j)[r]
template <int I>
__device__ __forceinline__ void read_block(float (&v)[32]) {
#define MLOP_W4_OUTS                                                                                   \
  "=v"(v[0]), "=v"(v[1]), "=v"(v[2]), "=v"(v[3]), "=v"(v[4]), "=v"(v[5]), "=v"(v[6]), "=v"(v[7]),     \
      "=v"(v[8]), "=v"(v[9]), "=v"(v[10]), "=v"(v[11]), "=v"(v[12]), "=v"(v[13]), "=v"(v[14]),         \
      "=v"(v[15]), "=v"(v[16]), "=v"(v[17]), "=v"(v[18]), "=v"(v[19]), "=v"(v[20]), "=v"(v[21]),       \
      "=v"(v[22]), "=v"(v[23]), "=v"(v[24]), "=v"(v[25]), "=v"(v[26]), "=v"(v[27]), "=v"(v[28]),       \
      "=v"(v[29]), "=v"(v[30]), "=v"(v[31])
  if constexpr (I == 0) asm volatile(MLOP_W4_READ0_ASM : MLOP_W4_OUTS);
  else if constexpr (I == 1) asm volatile(MLOP_W4_READ1_ASM : MLOP_W4_OUTS);
  else if constexpr (I == 2) asm volatile(MLOP_W4_READ2_ASM : MLOP_W4_OUTS);
  else if constexpr (I == 3) asm volatile(MLOP_W4_READ3_ASM : MLOP_W4_OUTS);
  else if constexpr (I == 4) asm volatile(MLOP_W4_READ4_ASM : MLOP_W4_OUTS);
  else if constexpr (I == 5) asm volatile(MLOP_W4_READ5_ASM : MLOP_W4_OUTS);
  else if constexpr (I == 6) asm volatile(MLOP_W4_READ6_ASM : MLOP_W4_OUTS);
  else asm volatile(MLOP_W4_READ7_ASM : MLOP_W4_OUTS);
#undef MLOP_W4_OUTS
}

// f(integral_constant<int, I>) for I = 0 .. N-1 (static row-block indices)
template <typename F, int... I>
__device__ __forceinline__ void unroll_impl(F& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void unroll(F&& f) {
  unroll_impl(f, std::make_integer_sequence<int, N>{});
}
}  // namespace

// GROUPED (the experts' products): A rows sorted by expert, rows offsets[e] .. offsets[e + 1] - 1 against B + e N ldb;
// A row r is re.a_rows[r] where given.  The routed tiles are counted here, from the offsets, as is their tail split.
template <int EPI, int BMT, bool GROUPED>
__device__ __forceinline__ void gemm_w4_tiles(
    const uint16_t* __restrict__ A, int lda, const uint16_t* __restrict__ B, int ldb,
    uint16_t* __restrict__ C, int ldc, int M, int N, int K, int n_tiles_x, int m_tiles, int group_m,
    const RopeEpi& re, int n_dp, int n_items, float* __restrict__ ws, int* __restrict__ cnt,
    const int* __restrict__ offsets, int n_groups) {
  static_assert(!GROUPED || EPI == W4_NONE || EPI == W4_SILU_MUL, "grouped epilogues");
  // BMT = 256: 128 x 128 outputs per wave; BMT = 128 (the half-height tile, twice the tiles for
  // the mid-M and QKV grids): 64 x 128 per wave, 4 x 8 accumulators, 12 DMA pieces per K-tile
  constexpr int BM = BMT, BN = 256;
  static_assert(BMT == 256 || BMT == 224 || BMT == 192 || BMT == 160 || BMT == 128, "tile heights of the generated K-loops");
  constexpr int NI = BMT / 32;      // 16-row accumulator blocks per wave
  constexpr int NPC = NI + 8;       // DMA pieces per wave and K-tile (NI of A, 8 of B)
  // epilogue store instructions per wave and tile (the next tile's K-loop waits for its
  // prefetched K-tile 0 with vmcnt(16 + NS): the count must be exact, so every store is
  // issued, rows >= M dropped by the buffer range check instead of a branch -- and a store that
  // is dropped whole may leave the count before the older DMAs, so a tile with rows >= M waits for
  // them at its end)
  // (RoPE: a wave with rows < M loads its rows' slots or positions first, and the compiler's wait
  // for those loads retires the older prefetch DMAs anyway)
  // (ADD_SS: the 32 stores come after its residual loads, which retire the DMAs anyway; RS: the
  // ss loads likewise)
  constexpr int BASE = EPI & 3;
  constexpr bool ADD = (EPI & W4_ADD_SS) != 0, RS = (EPI & W4_RS) != 0;
  static_assert(!ADD || BASE == W4_NONE, "residual add on the plain epilogue only");
  constexpr int NS = BASE == W4_SILU_MUL ? 2 * NI : 4 * NI;
  extern __shared__ __attribute__((aligned(16))) uint16_t smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wid >> 1, wn = wid & 1;
  const int nk = K / 64;

  // Work items: i < n_dp is tile i over the whole K; the r = T - n_dp tail tiles (r <= CUs / 2,
  // run_w4_t) are cut into K-halves, items n_dp + 2j + h (h = 0, 1) of tail tile n_dp + j, so the
  // last round fills the chip (QKV at M = 4088: 384 tiles = 256 + 2 x 128 half-tiles).
  // XCD-aware remap (T1, bijective): the grid is dealt round-robin over the 8 XCDs, so XCD x
  // gets a contiguous range of lids (a tail tile's two halves land on one XCD); a workgroup walks
  // items lid, lid + G, ... (persistent for the plain / SiLU epilogues; RoPE launches one
  // workgroup per item).  Tiles are ordered in bands of group_m m-tiles (a B panel is reused by
  // group_m consecutive tiles in one L2).
  const int G = gridDim.x, Lb = blockIdx.x;
  const int q = G >> 3, rr = G & 7, xcd = Lb & 7, slot = Lb >> 3;
  const int lid = (xcd < rr ? xcd * (q + 1) : rr * (q + 1) + (xcd - rr) * q) + slot;
  // GROUPED tables past the K-tile buffers: [0, 65) the offsets, [65, 129) the row tiles up to and with each expert,
  // then per wave three items' A rows
  int* tab = reinterpret_cast<int*>(smem + 65536);
  int* rows_lds = tab + 192 + wid * 192;
  if constexpr (GROUPED) {
    int o0 = 0, o1 = 0;
    if (lane < n_groups) o0 = offsets[lane], o1 = offsets[lane + 1];
    int c = (o1 - o0 + BM - 1) / BM;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int x = __shfl_up(c, d);
      if (lane >= d) c += x;
    }
    const int T = __builtin_amdgcn_readfirstlane(__shfl(c, 63)) * n_tiles_x, r = T % G;
    if (wid == 0) {
      if (lane < n_groups) tab[lane] = o0;
      if (lane == n_groups - 1) tab[n_groups] = o1;
      tab[65 + lane] = lane < n_groups ? c : 0x7fffffff;
    }
    __syncthreads();
    const bool halves = ws != nullptr && r > 0 && 2 * r <= G && nk % 2 == 0 && nk / 2 >= 3;  // gemm_w4_split_ok
    n_dp = halves ? T - r : T;
    n_items = halves ? T + r : T;
  }
  // (GROUPED: an expert's tiles are consecutive, its row tiles fastest: they share a B panel, and the next column
  // tile reuses their A rows.  B offsets carry the expert, the rows end at m_end.)
  auto origin = [&](int t, int& m0, int& n0, int& m_end, uint32_t& b0) {
    m_end = M;
    b0 = 0;
    if constexpr (GROUPED) {
      const int e = __popcll(__ballot(tab[65 + lane] <= t / n_tiles_x));  // the first expert whose tiles end past t
      const int base = e > 0 ? __builtin_amdgcn_readfirstlane(tab[64 + e]) : 0;
      const int c = __builtin_amdgcn_readfirstlane(tab[65 + e]) - base, ti = t - base * n_tiles_x;
      const int r0 = __builtin_amdgcn_readfirstlane(tab[e]);
      m_end = __builtin_amdgcn_readfirstlane(tab[e + 1]);
      m0 = r0 + ti % c * BM;
      n0 = ti / c * BN;
      b0 = (uint32_t)e * (uint32_t)N * (uint32_t)(ldb * 2);
      return;
    }
    const int band = t / (group_m * n_tiles_x), in_band = t % (group_m * n_tiles_x);
    const int gm_here = min(group_m, m_tiles - band * group_m);
    m0 = (band * group_m + in_band % gm_here) * BM;
    n0 = (in_band / gm_here) * BN;
    // RoPE epilogue: the V-head tiles first (as gemm_pp_kernel)
    if constexpr (BASE == W4_ROPE) n0 = (n_tiles_x - 1) * BN - n0;
  };
  // DMA piece i (0..NPC-1) of this wave: p = wid + 4 i, 8 rows x 128 B at LDS byte 1024 p;
  // i < NI A rows 8p.., else B rows 8(p - 4 NI).. (B starts at LDS byte 128 BMT); lane -> row
  // 8p + lane / 8, LDS slot lane % 8 holds source chunk (lane % 8) ^ swz(row)
  auto item = [&](int i, int& m0, int& n0, int& m_end, uint32_t& b0, int& kb, int& nkl) {
    if constexpr (BASE == W4_SLAB) {  // range by range: an XCD's items share their panels' columns
      const int sp = i / n_dp, ns = n_items / n_dp;
      origin(i % n_dp, m0, n0, m_end, b0);
      kb = sp * nk / ns;
      nkl = (sp + 1) * nk / ns - kb;
      return;
    }
    const bool tail = i >= n_dp;
    origin(tail ? n_dp + ((i - n_dp) >> 1) : i, m0, n0, m_end, b0);
    kb = tail ? ((i - n_dp) & 1) * (nk >> 1) : 0;
    nkl = tail ? nk >> 1 : nk;
  };
  auto dma_offsets = [&](int m0, int n0, int m_end, uint32_t b0, int kb, const int* rows, uint32_t (&vo)[NPC]) {
#pragma unroll
    for (int i = 0; i < NPC; ++i) {
      const int p = wid + 4 * i;
      const int r = (i < NI ? p : p - 4 * NI) * 8 + (lane >> 3);
      const uint32_t ch = (uint32_t)(((lane & 7) ^ ((r >> 1) & 7)) << 4);
      if (i < NI) {
        // A rows past the last load nothing: past num_records an LDS-DMA is dropped, and counted by vmcnt in its turn (of 5e8 words
        // that a DMA brought from HBM, waited for with a count over eight dropped or half-dropped ones behind it, none was read too early).
        // What the LDS then holds reaches accumulators that are never stored, and multiplying it costs less power than the last row again and
        // again (three Mixtral layers at 1628 tokens, a tenth of whose tiles is such rows: 1.2 % of 3.7 ms in two sessions, in which two runs
        // of one side differ by 1 - 2; no other step beyond what two runs differ).
        const int row = GROUPED && re.a_rows != nullptr ? rows[8 * i + (lane >> 3)] : m0 + r;
        vo[i] = m0 + r < m_end ? (uint32_t)row * (uint32_t)(lda * 2) + ch + kb * 128 : 0x80000000u;
      } else {
        vo[i] = b0 + (uint32_t)min(n0 + r, N - 1) * (uint32_t)(ldb * 2) + ch + kb * 128;
      }
    }
  };
  const i32x4 srdA = make_srd(A), srdB = make_srd(B);
  const uint32_t lbase = (uint32_t)(uintptr_t)((lds_u16*)smem);
  // GROUPED: lane l holds the row of piece l / 8's row l % 8 (l / 8 < NI)
  auto row_of = [&](int l) { return (wid + 4 * (l >> 3)) * 8 + (l & 7); };
  int slot_i = 0;
  if constexpr (GROUPED) {
    if (re.a_rows != nullptr && lid < n_items) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        int m, n, e, kb, nkl;
        uint32_t b;
        item(lid + j * G < n_items ? lid + j * G : lid, m, n, e, b, kb, nkl);
        rows_lds[j * 64 + lane] = re.a_rows[min(m + row_of(lane), e - 1)];
      }
    }
  }
  // fragment read addresses (buffer 0): row = wm*BMT/2 + (lane & 15) (+16 per fragment via the
  // offset field), chunk (k-half h) = (4h + lane / 16) ^ swz(row); swz depends on lane only
  const uint32_t sw = ((lane & 15) >> 1) & 7;
  const uint32_t c0 = (((uint32_t)(lane >> 4)) ^ sw) << 4, c1 = (((uint32_t)(lane >> 4) + 4) ^ sw) << 4;
  const uint32_t a_row = lbase + (uint32_t)(wm * (BMT / 2) + (lane & 15)) * 128;
  const uint32_t b_row = lbase + BMT * 128 + (uint32_t)(wn * 128 + (lane & 15)) * 128;
  const uint32_t dbase0 = __builtin_amdgcn_readfirstlane(lbase + wid * 1024);
  // W4_RS: per-wave row sums of squares after the two 64 KiB K-tile buffers; W4_ADD_SS: the
  // band ticket's flag after them (run_w4_t sizes the LDS)
  float* rinv_lds = reinterpret_cast<float*>(smem + 65536);
  int* band_flag = reinterpret_cast<int*>(smem + 65536 + 1024);

  for (int it = lid, first = 1; it < n_items; it += G, first = 0) {
    // offsets of this item (recomputed, not carried from the previous iteration: nothing but
    // the item index stays live across the epilogue) and of the next one (prefetched at the
    // end of the K-loop statement)
    int m0, n0, m_end, kb, nkl;
    uint32_t b0;
    item(it, m0, n0, m_end, b0, kb, nkl);
    uint32_t vo[NPC], vn[NPC];
    dma_offsets(m0, n0, m_end, b0, kb, rows_lds + slot_i * 64, vo);
    const bool next = it + G < n_items;
    // the K walk starts at another eighth per XCD (w4_k_walk): tiles in step would otherwise all read the columns of the
    // same few memory channels
    auto k_at = [&](int len, int j) {
      const int k = ((re.k_walk * xcd) & 7) * len / 8 + j;
      return (uint32_t)__builtin_amdgcn_readfirstlane((k >= len ? k - len : k) * 128);
    };
    const uint32_t k0 = k_at(nkl, 0), k1 = k_at(nkl, 1), kend = __builtin_amdgcn_readfirstlane(nkl * 128);
    uint32_t kn0, kn1;
    {
      int m1 = m0, n1 = n0, e1 = m_end, kb1 = kb, nkl1 = nkl;
      uint32_t b1 = b0;
      if (next) item(it + G, m1, n1, e1, b1, kb1, nkl1);
      dma_offsets(m1, n1, e1, b1, kb1, rows_lds + (slot_i == 2 ? 0 : slot_i + 1) * 64, vn);
      kn0 = k_at(nkl1, 0), kn1 = k_at(nkl1, 1);
    }
    if constexpr (GROUPED) {
      // the A rows of the item after the next into the third slot, by LDS-DMA like W4_RS's below and for its reason
      int m2 = m0, n2, e2 = m_end, kb2, nkl2;
      uint32_t b2;
      if (it + 2 * G < n_items) item(it + 2 * G, m2, n2, e2, b2, kb2, nkl2);
      const auto rs_rows = __builtin_amdgcn_make_buffer_rsrc((void*)re.a_rows, 0, re.a_rows != nullptr ? (int)((uint32_t)M * 4u) : 0,
                                                             0x00020000);
      const uint32_t voff = (uint32_t)min(m2 + row_of(lane), e2 - 1) * 4u;
      const uint32_t lds_dst =
          __builtin_amdgcn_readfirstlane(lbase + 131072u + (uint32_t)(192 + wid * 192 + (slot_i == 0 ? 2 : slot_i - 1) * 64) * 4u);
      uint32_t msave;
      asm volatile(
          "s_mov_b32 %[ms], m0\n"
          "s_mov_b32 m0, %[dst]\n"
          "s_nop 4\n"  // (the descriptor may come straight from v_readfirstlane / v_readlane)
          "buffer_load_dword %[vo], %[srd], 0 offen lds\n"
          "buffer_load_dword %[vo], %[srd], 0 offen lds\n"  // (twice: the built K-loops count two)
          "s_mov_b32 m0, %[ms]\n"
          : [ms] "=&s"(msave)
          : [dst] "s"(lds_dst), [vo] "v"(voff), [srd] "s"(rs_rows)
          : "memory", "scc");
      slot_i = slot_i == 2 ? 0 : slot_i + 1;
    }
    // C rows >= m_end fall outside num_records: their stores are dropped, never branched around
    const auto srdC = __builtin_amdgcn_make_buffer_rsrc((void*)C, 0, (int)((uint32_t)m_end * (uint32_t)ldc * 2u), 0x00020000);
    // W4_RS: the sums of squares of the wave's BMT / 2 rows (BMT = 128: the second load reads
    // rows past them, unused, so both tile heights count two VMEM ops) go to its LDS slot past the two K-tile
    // buffers by LDS-DMA, issued BEFORE the K-loop and invisible to the compiler: a load it
    // knew of would be waited for after the K-loop, and vmcnt retires in order, so the wait
    // would also cover the next tile's prefetch DMAs (gate_up +3 % per call measured so).  The
    // K-loop's nodma body waits vmcnt(0), which retires these two; its first wait counts them
    // (the S18 / S34 loops: vmcnt(16 + NS + 2) still retires exactly K-tile 0).
    if constexpr (RS) {
      const auto rs_ss = __builtin_amdgcn_make_buffer_rsrc((void*)re.ss_in, 0, (int)((uint32_t)M * 4u), 0x00020000);
      const uint32_t voff = (uint32_t)(m0 + wm * (BMT / 2) + lane) * 4u;
      const uint32_t lds_dst = __builtin_amdgcn_readfirstlane(lbase + 131072u + (uint32_t)wid * 512u);
      uint32_t msave;
      asm volatile(
          "s_mov_b32 %[ms], m0\n"
          "s_mov_b32 m0, %[dst]\n"
          "s_nop 4\n"  // (the descriptor may come straight from v_readfirstlane / v_readlane)
          "buffer_load_dword %[vo], %[srd], 0 offen lds\n"
          "s_add_u32 m0, m0, 0x100\n"
          "s_nop 0\n"
          "buffer_load_dword %[vo2], %[srd], 0 offen lds\n"
          "s_mov_b32 m0, %[ms]\n"
          : [ms] "=&s"(msave)
          : [dst] "s"(lds_dst), [vo] "v"(voff), [vo2] "v"(voff + 256u), [srd] "s"(rs_ss)
          : "memory", "scc");
    }
    uint32_t rA0 = a_row + c0, rA1 = a_row + c1, rB0 = b_row + c0, rB1 = b_row + c1;
    uint32_t dbase = dbase0, koff = k_at(nkl, 2), m0save;
    uint32_t iter = __builtin_amdgcn_readfirstlane(nkl - 3);
    const uint32_t s_first = __builtin_amdgcn_readfirstlane(first), s_next = __builtin_amdgcn_readfirstlane((int)next);
    bf16x8 fa0_0, fa0_1, fa0_2, fa0_3, fa0_4, fa0_5, fa0_6, fa0_7;
    bf16x8 fb0_0, fb0_1, fb0_2, fb0_3, fb0_4, fb0_5, fb0_6, fb0_7;
    bf16x8 fa1_0, fa1_1, fa1_2, fa1_3, fa1_4, fa1_5, fa1_6, fa1_7;
    bf16x8 fb1_0, fb1_1, fb1_2, fb1_3, fb1_4, fb1_5, fb1_6, fb1_7;
    // one generated K-loop per count of VMEM ops between the prefetched K-tiles and the loop: the
    // previous epilogue's NS stores (+ the two row-sum DMAs of W4_RS, issued above)
    constexpr int NQ = NS + (RS || GROUPED ? 2 : 0);
    if constexpr (BMT == 256) {
      static_assert(NQ == 32 || NQ == 16 || NQ == 34 || NQ == 18, "one generated K-loop per VMEM count");
      if constexpr (NQ == 32) asm volatile(MLOP_W4_KLOOP_S32_P0_ASM MLOP_W4_256_OPERANDS);
      else if constexpr (NQ == 16) asm volatile(MLOP_W4_KLOOP_S16_P0_ASM MLOP_W4_256_OPERANDS);
      else if constexpr (NQ == 34) asm volatile(MLOP_W4_KLOOP_S34_P0_ASM MLOP_W4_256_OPERANDS);
      else asm volatile(MLOP_W4_KLOOP_S18_P0_ASM MLOP_W4_256_OPERANDS);
    } else if constexpr (BMT == 224) {
      static_assert(NQ == 28 || NQ == 14 || NQ == 30 || NQ == 16, "one generated K-loop per VMEM count");
      if constexpr (NQ == 28) asm volatile(MLOP_W4_224_KLOOP_S28_ASM MLOP_W4_224_OPERANDS);
      else if constexpr (NQ == 14) asm volatile(MLOP_W4_224_KLOOP_S14_ASM MLOP_W4_224_OPERANDS);
      else if constexpr (NQ == 30) asm volatile(MLOP_W4_224_KLOOP_S30_ASM MLOP_W4_224_OPERANDS);
      else asm volatile(MLOP_W4_224_KLOOP_S16_ASM MLOP_W4_224_OPERANDS);
    } else if constexpr (BMT == 192) {
      static_assert(NQ == 24 || NQ == 12 || NQ == 26 || NQ == 14, "one generated K-loop per VMEM count");
      if constexpr (NQ == 24) asm volatile(MLOP_W4_192_KLOOP_S24_ASM MLOP_W4_192_OPERANDS);
      else if constexpr (NQ == 12) asm volatile(MLOP_W4_192_KLOOP_S12_ASM MLOP_W4_192_OPERANDS);
      else if constexpr (NQ == 26) asm volatile(MLOP_W4_192_KLOOP_S26_ASM MLOP_W4_192_OPERANDS);
      else asm volatile(MLOP_W4_192_KLOOP_S14_ASM MLOP_W4_192_OPERANDS);
    } else if constexpr (BMT == 160) {
      static_assert(NQ == 20 || NQ == 10 || NQ == 22 || NQ == 12, "one generated K-loop per VMEM count");
      if constexpr (NQ == 20) asm volatile(MLOP_W4_160_KLOOP_S20_ASM MLOP_W4_160_OPERANDS);
      else if constexpr (NQ == 10) asm volatile(MLOP_W4_160_KLOOP_S10_ASM MLOP_W4_160_OPERANDS);
      else if constexpr (NQ == 22) asm volatile(MLOP_W4_160_KLOOP_S22_ASM MLOP_W4_160_OPERANDS);
      else asm volatile(MLOP_W4_160_KLOOP_S12_ASM MLOP_W4_160_OPERANDS);
    } else {
      static_assert(NQ == 16 || NQ == 8 || NQ == 18 || NQ == 10, "one generated K-loop per VMEM count");
      if constexpr (NQ == 16) asm volatile(MLOP_W4H_KLOOP_S16_ASM MLOP_W4_128_OPERANDS);
      else if constexpr (NQ == 8) asm volatile(MLOP_W4H_KLOOP_S8_ASM MLOP_W4_128_OPERANDS);
      else if constexpr (NQ == 18) asm volatile(MLOP_W4H_KLOOP_S18_ASM MLOP_W4_128_OPERANDS);
      else asm volatile(MLOP_W4H_KLOOP_S10_ASM MLOP_W4_128_OPERANDS);
    }

    // read-out: the K-loop accumulates C^T, so acc(i, j)[r] of lane l is
    //   C[m0 + wm*BMT/2 + 16i + (l & 15)][n0 + wn*128 + 16j + 4(l >> 4) + r]
    // -- four consecutive columns per lane; a permlane16 swap between the accumulators of
    // column blocks j and j+1 gives each lane 8 consecutive columns of one of them: one 16-B
    // buffer store per lane and pair (plain: 4 pairs x NI row blocks = NS per wave;
    // SiLU-mul: the 4 outputs of the (gate, up) pairs jp, jp+1 swapped the same way, NS / 2)
    const int lr = wm * (BMT / 2) + (lane & 15), qd = lane >> 4;
    // tail half-tile: both halves store their fp32 partial (accumulator layout, 16-B sc1 =
    // write-through stores), every wave drains (vmcnt(0)), a barrier, then ONE lane's agent-scope
    // ticket; the half whose ticket came last adds the other slot (16-B sc1 loads) and runs the
    // epilogue (MI355X_MICROARCH.md "Valid forms"; the gemm_pp_kernel stream-K hand-off).  A
    // tail item is its workgroup's last, so no prefetch is in flight and the LDS is free for
    // the flag.  own + other is commutative: bit-identical whichever half arrives last.
    const bool part = BASE != W4_SLAB && it >= n_dp;
    const int sidx = part ? it - n_dp : 0;
    const auto rs_other = __builtin_amdgcn_make_buffer_rsrc(part ? ws + (size_t)(sidx ^ 1) * 65536 : (float*)C, 0,
                                                           65536 * 4, 0x00020000);
    if (part) {
      const int tt = sidx >> 1;
      const auto rs_own = __builtin_amdgcn_make_buffer_rsrc(ws + (size_t)sidx * 65536, 0, 65536 * 4, 0x00020000);
      auto put = [&](auto I_) {
        constexpr int I = decltype(I_)::value;
        float v[32];
        read_block<I>(v);
#pragma unroll
        for (int q4 = 0; q4 < 8; ++q4)
          __builtin_amdgcn_raw_buffer_store_b128(
              u32x4{__float_as_uint(v[4 * q4]), __float_as_uint(v[4 * q4 + 1]), __float_as_uint(v[4 * q4 + 2]),
                    __float_as_uint(v[4 * q4 + 3])},
              rs_own, (uint32_t)(((I * 8 + q4) * 256 + tid) * 16), 0, 16 /* sc1 */);
      };
      unroll<NI>(put);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      int* flag = reinterpret_cast<int*>(smem);
      if (tid == 0) {
        const int tk = __hip_atomic_fetch_add(cnt + tt, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (tk == 1) __hip_atomic_store(cnt + tt, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        flag[0] = tk == 1;
      }
      __syncthreads();
      const int last = flag[0];
      __syncthreads();  // flag read everywhere before the epilogue may reuse the LDS
      if (!last) break;  // the other half finishes the tile (a tail item is the last item)
    }
    // accumulator row block I (+ the other half's partial for a tail tile; x the row's RMSNorm
    // factor under W4_RS)
    auto fetch = [&](auto I_, float (&v)[32]) {
      constexpr int I = decltype(I_)::value;
      read_block<I>(v);
      if (part) {
#pragma unroll
        for (int b4 = 0; b4 < 8; b4 += 4) {
          u32x4 o[4];
#pragma unroll
          for (int q4 = 0; q4 < 4; ++q4)
            o[q4] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                                  rs_other, (uint32_t)(((I * 8 + b4 + q4) * 256 + tid) * 16), 0, 16 /* sc1 */));
#pragma unroll
          for (int q4 = 0; q4 < 4; ++q4)
#pragma unroll
            for (int e = 0; e < 4; ++e) v[4 * (b4 + q4) + e] += __uint_as_float(o[q4][e]);
        }
      }
      if constexpr (RS) {
        const float f = rsqrtf(rinv_lds[wid * 128 + 16 * I + (lane & 15)] * re.ss_inv_k + re.ss_eps);
#pragma unroll
        for (int e = 0; e < 32; ++e) v[e] *= f;
      }
    };
    // lane quad qd after the swap of (x = block j, y = block j+1): qd even holds x, odd y;
    // columns 8 (qd >> 1) .. +7 of that block
    const int odd = qd & 1, half = qd >> 1;
    auto swap_f = [&](const float* x, const float* y, float (&lo)[4], float (&hi)[4]) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const auto sw2 = __builtin_amdgcn_permlane16_swap(__float_as_uint(x[r]), __float_as_uint(y[r]), false, false);
        lo[r] = __uint_as_float(sw2[0]);
        hi[r] = __uint_as_float(sw2[1]);
      }
    };
    auto swap_pair = [&](const float* x, const float* y, u32x4& out) {
      float lo[4], hi[4];
      swap_f(x, y, lo, hi);
      // even quads: lo = own x (cols 0-3), hi = partner's x (cols 4-7); odd quads: lo =
      // partner's y (cols 0-3), hi = own y (cols 4-7)
      out = u32x4{pack2(lo[0], lo[1]), pack2(lo[2], lo[3]), pack2(hi[0], hi[1]), pack2(hi[2], hi[3])};
    };
    if constexpr (BASE == W4_SLAB) {
      const auto rs_ws = __builtin_amdgcn_make_buffer_rsrc((float*)C + (size_t)(it / n_dp) * M * N, 0, (int)((uint32_t)M * (uint32_t)N * 4u),
                                                           0x00020000);
      unroll<NI>([&](auto I_) {
        constexpr int I = decltype(I_)::value;
        float v[32];
        read_block<I>(v);
        const uint32_t off = ((uint32_t)(m0 + lr + I * 16) * (uint32_t)N + (uint32_t)(n0 + wn * 128 + 4 * qd)) * 4u;
#pragma unroll
        for (int j = 0; j < 8; ++j)
          __builtin_amdgcn_raw_buffer_store_b128(u32x4{__float_as_uint(v[4 * j]), __float_as_uint(v[4 * j + 1]), __float_as_uint(v[4 * j + 2]),
                                                       __float_as_uint(v[4 * j + 3])}, rs_ws, off + 64u * j, 0, 0);
      });
    } else if constexpr (BASE == W4_ROPE) {
      // RoPE + paged cache from the accumulators: a wave's 128 columns are ONE head, and a
      // lane's rotate-half partners (c, c + 64) sit in acc(i, j) / acc(i, j + 4) element r of the
      // same lane, so nothing is staged in LDS (which stays free for the next tile's prefetch).
      // Values are bf16-rounded first (rope_cache_kernel's math on the projection's bf16 output).
      constexpr int D = 128, HALF = 64;
      const bool r_nt = (re.ws_nt & 8) != 0;  // q / K / V stores non-temporal (gemm_slab_nt bit 3)
      auto put16 = [&](uint16_t* p, const u32x4& v) {
        if (r_nt) __builtin_nontemporal_store(v, reinterpret_cast<u32x4*>(p));
        else *reinterpret_cast<u32x4*>(p) = v;
      };
      const int head = (n0 + wn * 128) / D;
      const int n_rope = re.Hq + re.Hkv, n_all = re.Hq + 2 * re.Hkv;
      if (head >= n_all) {
        // padding columns: nothing to store
      } else if (head >= n_rope) {
        // V head: its token-major page rows [NB, Hkv, BS, 128] (attention.hip reads V
        // transposed out of LDS), 4 x 16-B stores per row block as the K rows below.  The slot
        // loads come first: their wait retires the prefetched DMAs, so the store count after
        // them need not be exact.
        const int kh = head - n_rope;
        int sl[NI];
#pragma unroll
        for (int I = 0; I < NI; ++I) {
          const int m = m0 + lr + I * 16;
          sl[I] = m < M ? re.slots[m] : -1;
        }
        auto vstore = [&](auto I_) {
          constexpr int I = decltype(I_)::value;
          float v[32];
          fetch(I_, v);
          u32x4 d[4];
#pragma unroll
          for (int pr = 0; pr < 4; ++pr) swap_pair(v + 8 * pr, v + 8 * pr + 4, d[pr]);
          const int slot = sl[I];
          if (slot < 0) return;
          uint16_t* dst = re.v_cache + (((size_t)(slot / re.BS) * re.Hkv + kh) * re.BS + slot % re.BS) * D;
#pragma unroll
          for (int pr = 0; pr < 4; ++pr)
            put16(dst + (2 * pr + odd) * 16 + 8 * half, d[pr]);
        };
        unroll<NI>(vstore);
      } else {
        // q / k head: positions (and slots) of the lane's 8 rows first, one batch; the waits
        // for them also retire the prefetched DMAs (older in the vmcnt order)
        const bool is_k = head >= re.Hq;
        int pp[NI], sl[NI];
#pragma unroll
        for (int I = 0; I < NI; ++I) {
          const int m = m0 + lr + I * 16;
          const bool ok = m < M;
          pp[I] = ok ? re.pos[m] : 0;
          sl[I] = ok && is_k ? re.slots[m] : -1;
        }
        const int c0 = 4 * qd;
        // cos / sin of row block I+1 are loaded while block I is rotated and stored (two
        // register sets, named so every index is static)
        auto load_cs = [&](int I, float4 (&cs)[8]) {
          const float4* cr = reinterpret_cast<const float4*>(re.cos_sin + (size_t)pp[I] * D);
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            cs[j] = cr[(j * 16 + c0) / 4];
            cs[4 + j] = cr[(HALF + j * 16 + c0) / 4];
          }
        };
        auto rstore = [&](auto I_, const float4 (&cs)[8], float4 (&nxt)[8]) {
          constexpr int I = decltype(I_)::value;
          if constexpr (I < NI - 1) load_cs(I + 1, nxt);
          float v[32];
          fetch(I_, v);
          float xo[4][4], yo[4][4];
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const float cv[4] = {cs[j].x, cs[j].y, cs[j].z, cs[j].w};
            const float sv[4] = {cs[4 + j].x, cs[4 + j].y, cs[4 + j].z, cs[4 + j].w};
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const float x = bf2f(f2bf(v[4 * j + r])), y = bf2f(f2bf(v[4 * (j + 4) + r]));
              xo[j][r] = x * cv[r] - y * sv[r];
              yo[j][r] = y * cv[r] + x * sv[r];
            }
          }
          u32x4 d[4];
          swap_pair(xo[0], xo[1], d[0]);
          swap_pair(xo[2], xo[3], d[1]);
          swap_pair(yo[0], yo[1], d[2]);
          swap_pair(yo[2], yo[3], d[3]);
          const int m = m0 + lr + I * 16;
          if (m >= M) return;
          uint16_t* dst;
          if (!is_k) {
            dst = re.q_out + ((size_t)m * re.Hq + head) * D;
          } else {
            const int slot = sl[I];
            if (slot < 0) return;
            dst = re.k_cache + (((size_t)(slot / re.BS) * re.Hkv + (head - re.Hq)) * re.BS + slot % re.BS) * D;
          }
#pragma unroll
          for (int b = 0; b < 4; ++b)
            put16(dst + (b >> 1) * HALF + ((b & 1) * 2 + odd) * 16 + 8 * half, d[b]);
        };
        float4 csa[8], csb[8];
        load_cs(0, csa);
        unroll<NI>([&](auto I_) {
          if constexpr (decltype(I_)::value % 2 == 0) rstore(I_, csa, csb);
          else rstore(I_, csb, csa);
        });
      }
    } else {
      const int col_w = BASE == W4_NONE ? n0 + wn * 128 : (n0 + wn * 128) / 2;
      const bool c_nt = (re.ws_nt & 2) != 0;  // C stores non-temporal (gemm_slab_nt bit 1, A/B)
      // W4_ADD_SS: partial sum of squares of this wave's 128 columns of each row -> ss_out[row][g]
      const int n_groups = N >> 7, g_out = (n0 + wn * 128) >> 7;
      const auto rs_sso = __builtin_amdgcn_make_buffer_rsrc((void*)re.ss_out, 0, ADD ? (int)((uint32_t)M * n_groups * 4u) : 0,
                                                            0x00020000);
      auto store = [&](auto I_) {
        constexpr int I = decltype(I_)::value;
        float v[32];
        fetch(I_, v);
        const uint32_t row_off = (uint32_t)(m0 + lr + I * 16) * (uint32_t)ldc * 2u;
        if constexpr (GROUPED && BASE == W4_SILU_MUL) {
          if (re.row_scale != nullptr) {
            const float f = re.row_scale[min(m0 + lr + I * 16, m_end - 1)];
#pragma unroll
            for (int e = 0; e < 32; ++e) v[e] *= f;
          }
        }
        if constexpr (BASE == W4_SILU_MUL) {
          float o[16];
          if (BASE == W4_SILU_MUL && re.p0 > 0.f) {
#pragma unroll
            for (int jp = 0; jp < 4; ++jp)
#pragma unroll
              for (int r = 0; r < 4; ++r)
                o[4 * jp + r] = clamp_glu_f(v[8 * jp + r], v[8 * jp + 4 + r], re.p0, re.p1);
          } else {
#pragma unroll
            for (int jp = 0; jp < 4; ++jp)
#pragma unroll
              for (int r = 0; r < 4; ++r) o[4 * jp + r] = silu_bf(v[8 * jp + r]) * bf2f(f2bf(v[8 * jp + 4 + r]));
          }
#pragma unroll
          for (int pr = 0; pr < 2; ++pr) {
            u32x4 d;
            swap_pair(o + 8 * pr, o + 8 * pr + 4, d);
            const int col = col_w + (2 * pr + odd) * 16 + 8 * half;
            if (c_nt) __builtin_amdgcn_raw_buffer_store_b128(d, srdC, row_off + col * 2, 0, 2 /* nt */);
            else __builtin_amdgcn_raw_buffer_store_b128(d, srdC, row_off + col * 2, 0, 0);
          }
        } else {
          if constexpr (BASE == W4_NONE) act_outs(re, v, col_w);
#pragma unroll
          for (int pr = 0; pr < 4; ++pr) {
            u32x4 d;
            swap_pair(v + 8 * pr, v + 8 * pr + 4, d);
            const int col = col_w + (2 * pr + odd) * 16 + 8 * half;
            if (c_nt) __builtin_amdgcn_raw_buffer_store_b128(d, srdC, row_off + col * 2, 0, 2 /* nt */);
            else __builtin_amdgcn_raw_buffer_store_b128(d, srdC, row_off + col * 2, 0, 0);
          }
        }
      };
      // residual (C) += acc: the lane's 8 columns of each pair are loaded, added in fp32, rounded,
      // squared into the row's partial and stored back (rows >= M: loads read 0, stores dropped by
      // the range check).  Row block I+1's residual loads are issued before block I is processed
      // (two register sets, named so every index is static), one memory latency per tile, not 8.
      auto load_res = [&](int I, u32x4 (&rv)[4]) {
        const uint32_t row_off = (uint32_t)(m0 + lr + I * 16) * (uint32_t)ldc * 2u;
#pragma unroll
        for (int pr = 0; pr < 4; ++pr) {
          const int col = col_w + (2 * pr + odd) * 16 + 8 * half;
          rv[pr] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(srdC, row_off + col * 2, 0, 0));
        }
      };
      auto store_add = [&](auto I_, const u32x4 (&rv)[4], u32x4 (&nxt)[4]) {
        constexpr int I = decltype(I_)::value;
        if constexpr (I < NI - 1) load_res(I + 1, nxt);
        float v[32];
        fetch(I_, v);
        const uint32_t row_off = (uint32_t)(m0 + lr + I * 16) * (uint32_t)ldc * 2u;
        float ssq = 0.f;
#pragma unroll
        for (int pr = 0; pr < 4; ++pr) {
          float lo[4], hi[4];
          swap_f(v + 8 * pr, v + 8 * pr + 4, lo, hi);
          float h[8];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            h[e] = bf2f(f2bf(lo[e] + bf2f((uint16_t)(rv[pr][e >> 1] >> (16 * (e & 1))))));
            h[4 + e] = bf2f(f2bf(hi[e] + bf2f((uint16_t)(rv[pr][2 + (e >> 1)] >> (16 * (e & 1))))));
          }
#pragma unroll
          for (int e = 0; e < 8; ++e) ssq += h[e] * h[e];
          const int col = col_w + (2 * pr + odd) * 16 + 8 * half;
          const u32x4 hv{pack2(h[0], h[1]), pack2(h[2], h[3]), pack2(h[4], h[5]), pack2(h[6], h[7])};
          if (c_nt) __builtin_amdgcn_raw_buffer_store_b128(hv, srdC, row_off + col * 2, 0, 2 /* nt */);
          else __builtin_amdgcn_raw_buffer_store_b128(hv, srdC, row_off + col * 2, 0, 0);
        }
        ssq += __shfl_xor(ssq, 16);
        ssq += __shfl_xor(ssq, 32);
        if (qd == 0)
          __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(ssq), rs_sso,
                                                ((uint32_t)(m0 + lr + I * 16) * n_groups + g_out) * 4u, 0, 16 /* sc1 */);
      };
      if constexpr (ADD) {
        u32x4 ra[4], rb[4];
        load_res(0, ra);
        unroll<NI>([&](auto I_) {
          if constexpr (decltype(I_)::value % 2 == 0) store_add(I_, ra, rb);
          else store_add(I_, rb, ra);
        });
      } else {
        unroll<NI>(store);
      }
      if constexpr (ADD) {
        // band ticket: the last of the band's n_tiles_x tiles adds every row's partials in a fixed
        // order into ss_tot (sc1 partial stores, vmcnt(0), barrier, one agent-scope ticket: the
        // K-half hand-off above).  The flag lives past the K-tile buffers, which the next tile's
        // prefetch may be filling.
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        const int band = m0 / BM;
        if (tid == 0) {
          const int tk = __hip_atomic_fetch_add(re.ss_cnt + band, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          const int lastb = tk == n_tiles_x - 1;
          if (lastb) __hip_atomic_store(re.ss_cnt + band, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          band_flag[0] = lastb;
        }
        __syncthreads();
        if (band_flag[0]) {
          const int r = m0 + tid;
          if (tid < BM && r < M) {
            float sum = 0.f;
            int c = 0;
            for (; c + 4 <= n_groups; c += 4) {
              const u32x4 x = __builtin_bit_cast(
                  u32x4, __builtin_amdgcn_raw_buffer_load_b128(rs_sso, (uint32_t)(r * n_groups + c) * 4u, 0, 16 /* sc1 */));
              sum += __uint_as_float(x[0]) + __uint_as_float(x[1]) + __uint_as_float(x[2]) + __uint_as_float(x[3]);
            }
            if (c < n_groups) {  // N = 256 mod 512: the row's last 2 groups (N % 256 == 0 keeps n_groups even)
              const u32x2 x = __builtin_bit_cast(
                  u32x2, __builtin_amdgcn_raw_buffer_load_b64(rs_sso, (uint32_t)(r * n_groups + c) * 4u, 0, 16 /* sc1 */));
              sum += __uint_as_float(x[0]) + __uint_as_float(x[1]);
            }
            re.ss_tot[r] = sum;
          }
        }
      }
    }
    // rows past M (stores dropped or, RoPE, not issued), or a RoPE wave of padding columns: the counted wait at the next
    // tile's start does not cover the prefetched DMAs (K = 192, M = 643: a few blocks of the next tile read its K-tile 0
    // too early)
    if (m0 + BM > m_end || (BASE == W4_ROPE && (n0 + wn * 128) / 128 >= re.Hq + 2 * re.Hkv))
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }
}

template <int EPI, int BMT>
__global__ void __launch_bounds__(256, 1) gemm_w4_kernel(
    const uint16_t* __restrict__ A, int lda, const uint16_t* __restrict__ B, int ldb,
    uint16_t* __restrict__ C, int ldc, int M, int N, int K, int n_tiles_x, int m_tiles, int group_m,
    RopeEpi re, int n_dp, int n_items, float* __restrict__ ws, int* __restrict__ cnt) {
  gemm_w4_tiles<EPI, BMT, false>(A, lda, B, ldb, C, ldc, M, N, K, n_tiles_x, m_tiles, group_m, re, n_dp, n_items, ws, cnt,
                                 nullptr, 0);
}

// Tile height of the experts' products, by estimated time in rounds of 256-row tiles (a round of the lower ones .89 / .79 /
// .69, K-halves .59; W: the weights' rounds at one tile per expert, which bound the lower tiles).  tNNN: row tiles of that height
// over all experts, experts: those with rows, G: workgroups.
__host__ __device__ __forceinline__ int w4_grouped_height(int t256, int t224, int t192, int t160, int experts, int n_tiles_x, int G,
                                                          int nk, bool halves) {
  auto rounds = [&](int t) {
    const int T = t * n_tiles_x, r = T % G;
    return (float)(T / G) + (r == 0 ? 0.f : 2 * r <= G && nk % 2 == 0 && halves ? .59f : 1.f);
  };
  const float W = (float)(experts * n_tiles_x) / (float)G;
  const float e256 = rounds(t256), e224 = fmaxf(.89f * rounds(t224), .94f * W);
  const float e192 = fmaxf(.79f * rounds(t192), .88f * W), e160 = fmaxf(.69f * rounds(t160), .81f * W);
  const float upper = fminf(e256, e224), lower = fminf(e192, e160);
  return upper <= lower ? (e256 <= e224 ? 256 : 224) : e192 <= e160 ? 192 : 160;
}

// The same for given counts of rows (tests).
int gemm_grouped_height(const int64_t* rows, int n_groups, int N, int K, int cus) {
  int t[4] = {}, experts = 0, total = 0;
  for (int g = 0; g < n_groups; ++g) {
    const int r = (int)rows[g];
    t[0] += (r + 255) / 256, t[1] += (r + 223) / 224, t[2] += (r + 191) / 192, t[3] += (r + 159) / 160;
    experts += r > 0, total += r;
  }
  const int G = (int)std::min<long>((long)(N / 256) * ((total + 159) / 160 + n_groups), cus);  // run_w4_grouped_t's grid
  return w4_grouped_height(t[0], t[1], t[2], t[3], experts, N / 256, G, K / 64, true);
}

// The experts' products of a prompt.  What the grid loses is rows of partial tiles and the last round, and both hang on
// the routing, which only the device knows: the height is chosen here (w4_grouped_height).  gate_up of 8 experts, 256 / 192 / 160 rows: 300 rows each 738 / 619 / 532 us, 350 747 / 595 / 691, 500 779 /
// 836 / 911, 550 1021 / 836 / 941, 1024 1497 / 1561 / 1598 (1.29 PFLOP/s); over 22 sizes, even and with the experts
// 0.6 - 1.4 of the mean, the choice is within 1 % of the best of these three on average (all
// measured before the MFMAs had their present order, which the heights share).  With 224 rows 407 each take 663
// us where the ping-pong kernel took 735 and the three heights 714 - 745.  One XCD's workgroups share
// panels and stay in step; each XCD's K walk starts at another eighth, and nothing is loaded between tiles that the
// stores and the next tile's DMAs would be waited for with (offsets in LDS, gathered rows two tiles ahead): 1661 / 1577
// / 1501 us before at 1024 rows, 800 before and 745 after at 450.
template <int EPI>
__global__ void __launch_bounds__(256, 1) gemm_w4_grouped_kernel(
    const uint16_t* __restrict__ A, int lda, const uint16_t* __restrict__ B, int ldb, uint16_t* __restrict__ C, int ldc,
    int M, int N, int K, int n_tiles_x, RopeEpi re, float* __restrict__ ws, int* __restrict__ cnt,
    const int* __restrict__ offsets, int n_groups) {
  const int lane = threadIdx.x & 63, G = gridDim.x, nk = K / 64;
  const int rows = lane < n_groups ? offsets[lane + 1] - offsets[lane] : 0;
  // (16 bits each: M K < 2^30 and K >= 192 keep every count below 2^16)
  uint32_t a = (uint32_t)((rows + 255) / 256) | (uint32_t)((rows + 191) / 192) << 16, b = (uint32_t)((rows + 159) / 160) | (uint32_t)((rows + 223) / 224) << 16;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    a += __shfl_xor(a, d);
    b += __shfl_xor(b, d);
  }
  a = __builtin_amdgcn_readfirstlane(a);
  b = __builtin_amdgcn_readfirstlane(b);
  const int h = __builtin_amdgcn_readfirstlane(w4_grouped_height(a & 0xffff, b >> 16, a >> 16, b & 0xffff,
                                                                 __popcll(__ballot(rows > 0)), n_tiles_x, G, nk, ws != nullptr));
#define MLOP_W4_GROUPED(h_)                                                                                           \
  gemm_w4_tiles<EPI, h_, true>(A, lda, B, ldb, C, ldc, M, N, K, n_tiles_x, 0, 1, re, 0, 0, ws, cnt, offsets, n_groups)
  if (h == 256) MLOP_W4_GROUPED(256);
  else if (h == 224) MLOP_W4_GROUPED(224);
  else if (h == 192) MLOP_W4_GROUPED(192);
  else MLOP_W4_GROUPED(160);
#undef MLOP_W4_GROUPED
}

// the r = T % CUs tail tiles are cut into K-halves (one extra round of half-length items)
bool gemm_w4_split_ok(int T, int nk) {
  int cus = 0;
  if (!gemm_sk_available(&cus) || cus <= 0) return false;
  const int r = T % cus;
  return r > 0 && 2 * r <= cus && nk % 2 == 0 && nk / 2 >= 3;
}

// true when the four-wave kernel can run this shape (the planner's variant 5)
bool gemm_w4_ok(int M, int N, int K, int lda, int ldb, int ldc) {
  return M > 0 && K % 64 == 0 && K >= 192 && lda % 8 == 0 && ldb % 8 == 0 && N % 256 == 0 &&
         (long)M * lda * 2 < (1l << 31) && (long)N * ldb * 2 < (1l << 31) && (long)M * (ldc > 0 ? ldc : N) * 2 < (1l << 31);
}

// Each XCD's K walk from another eighth on (XCD x from eighth k_walk x mod 8; 0: all in step): where rows are a multiple of
// 4 KB apart, tiles in step ask for the same few memory channels.  Not where XCDs share weights (several bands of tiles a
// round) that the 256 MB cache behind the L2s does not hold: out of step each of them reads HBM.  Cold weights, 21 shapes at
// 640 - 7000 rows: where the rule walks apart 0.992 of the time in step (0.91 - 1.03; 16384 x 16384 0.94 - 0.97, 8192 x 14336
// at 1500 - 2300 rows 0.92, 12288 x 4096 at 1500 and 8192 x 8192 at 1500 the worst); the shapes that the first condition
// leaves out 0.998 (0.97 - 1.04), those of the second 0.92 - 1.0 at up to 2300 rows and 1.02 - 1.03 above (8192 x 28672 and
// x 20480; one line, since few steps have such weights at few rows).  In a step (Llama-3-8B widths) o and down together 105 ->
// 99 us each at 1500 rows, 415 -> 402 at 8000.  Neighbours five eighths apart: 0.5 - 1.5 % of a step better than one apart
// at 1500 rows and in mixed steps, level elsewhere and in products alone.
static int w4_k_walk(int N, int K, int band_tiles, int cus) {
  return K % 2048 == 0 && ((long)N * K * 2 <= (256l << 20) || band_tiles >= cus) ? 5 : 0;
}

// whether a product's tiles walk K in step: rounds of few_rows_w4's estimate
bool gemm_w4_in_step(int M, int N, int K, int bm) {
  return w4_k_walk(N, K, std::max(1, std::min(1024 / bm, (M + bm - 1) / bm)) * ((N + 255) / 256), kCus) == 0;
}

template <int EPI, int BMT>
static bool run_w4_t(const uint16_t* A, int lda, const uint16_t* B, int ldb, uint16_t* C, int ldc, int M, int N,
                     int K, hipStream_t st, const RopeEpi& re) {
  constexpr size_t ring = 2ull * 65536 + ((EPI & (W4_RS | W4_ADD_SS)) ? 4 * 128 * 4 + 16 : 0);
  constexpr size_t stg = 0;  // every epilogue works from the accumulators
  constexpr size_t lds = ring > stg ? ring : stg;
  static_assert(lds <= 163840, "LDS budget");
  auto kern = gemm_w4_kernel<EPI, BMT>;
  static bool attr = false;
  if (!attr) {
    (void)hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    attr = true;
  }
  const int gx = (N + 255) / 256, gy = (M + BMT - 1) / BMT;
  // m-tiles per band: a B panel is reused by 1024 rows of tiles while L2-resident
  constexpr int group_m = 1024 / BMT;
  const int gm = std::max(1, std::min(group_m, gy));
  // tail split: the r = T % CUs last tiles cut into K-halves when 2r <= CUs (one round)
  const int T = gx * gy;
  int n_dp = T, n_items = T;
  float* ws = nullptr;
  int* cnt = nullptr;
  int cus = 256;
  if (gemm_w4_split_ok(T, K / 64)) {
    int c2 = 0;
    if (gemm_sk_scratch(&ws, &cnt, &c2)) {
      n_dp = T - T % c2;
      n_items = n_dp + 2 * (T % c2);
    }
  }
  // one persistent workgroup per CU walks items lid, lid + G, ...
  int grid = n_items;
  if (!gemm_sk_available(&cus) || cus <= 0) {
    static int cu_count[16] = {};
    int dev = 0;
    (void)hipGetDevice(&dev);
    if (dev >= 0 && dev < 16 && cu_count[dev] == 0)
      (void)hipDeviceGetAttribute(&cu_count[dev], hipDeviceAttributeMultiprocessorCount, dev);
    cus = (dev >= 0 && dev < 16 && cu_count[dev] > 0) ? cu_count[dev] : 256;
  }
  grid = std::min(grid, cus);
  RopeEpi re2 = re;
  re2.ws_nt = gemm_slab_nt(-1);
  re2.k_walk = w4_k_walk(N, K, gm * gx, cus);
  if constexpr ((EPI & W4_ADD_SS) != 0) {  // one band ticket per BMT-row band (launch_w4_chain checks gy)
    float* w2 = nullptr;
    int c3 = 0;
    if (!gemm_sk_scratch(&w2, &re2.ss_cnt, &c3)) return false;  // nothing launched: the caller must know
  }
  kern<<<grid, 256, lds, st>>>(A, lda, B, ldb, C, ldc, M, N, K, gx, gy, gm, re2, n_dp, n_items, ws, cnt);
  return true;
}

// K in `splits` ranges, one workgroup per (tile, range): fp32 slabs ws[range][M][N].  At most one item per CU, three K-tiles or more each.
template <int BMT>
static void run_w4_slab_t(const uint16_t* A, int lda, const uint16_t* B, int ldb, float* ws, int M, int N, int K, int splits, hipStream_t st) {
  constexpr size_t lds = 2ull * 65536;
  auto kern = gemm_w4_kernel<W4_SLAB, BMT>;
  static const bool attr =
      hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) == hipSuccess;
  (void)attr;
  const int gx = N / 256, gy = (M + BMT - 1) / BMT, T = gx * gy, gm = std::max(1, std::min(1024 / BMT, gy));
  RopeEpi re{};
  re.k_walk = w4_k_walk(N, K, gm * gx, kCus);
  kern<<<T * splits, 256, lds, st>>>(A, lda, B, ldb, (uint16_t*)ws, N, M, N, K, gx, gy, gm, re, T, T * splits, nullptr, nullptr);
}

void run_w4_slab(const uint16_t* A, int lda, const uint16_t* B, int ldb, float* ws, int M, int N, int K, int splits, int bm, hipStream_t st) {
  if (bm == 128) run_w4_slab_t<128>(A, lda, B, ldb, ws, M, N, K, splits, st);
  else if (bm == 160) run_w4_slab_t<160>(A, lda, B, ldb, ws, M, N, K, splits, st);
  else if (bm == 192) run_w4_slab_t<192>(A, lda, B, ldb, ws, M, N, K, splits, st);
  else if (bm == 224) run_w4_slab_t<224>(A, lda, B, ldb, ws, M, N, K, splits, st);
  else run_w4_slab_t<256>(A, lda, B, ldb, ws, M, N, K, splits, st);
}

// (a_n: A's rows where a_rows picks them; the kernel's offsets are 32 bits and its tables hold 64 experts)
bool gemm_w4_grouped_ok(int M, int N, int K, int n_groups, int a_n) {
  return M > 0 && n_groups <= 64 && K % 64 == 0 && K >= 192 && N % 256 == 0 && (long)std::max(M, a_n) * K * 2 < (1l << 31) &&
         (long)M * N * 2 < (1l << 31) && (long)n_groups * N * K * 2 < (1l << 31);
}

template <int EPI>
static void run_w4_grouped_t(const uint16_t* A, int lda, const uint16_t* B, int ldb, uint16_t* C, int ldc, int M, int N,
                             int K, hipStream_t st, const RopeEpi& re, const int* offsets, int n_groups) {
  constexpr size_t lds = 2ull * 65536 + 4096;
  auto kern = gemm_w4_grouped_kernel<EPI>;
  static const bool attr =
      hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) == hipSuccess;
  (void)attr;
  float* ws = nullptr;
  int *cnt = nullptr, cus = 256;
  gemm_sk_scratch(&ws, &cnt, &cus);  // without it: no K-halves
  const long most = (long)(N / 256) * ((M + 159) / 160 + n_groups);  // every expert's last tile partial
  RopeEpi re2 = re;
  re2.ws_nt = gemm_slab_nt(-1);
  // (an expert's column tiles are walked by one XCD: no condition as in w4_k_walk.  Seven shapes of 4 - 32 experts, 260 - 500 rows
  // each, equal and random: neighbours five eighths apart take 0.98 of the time of one eighth apart (0.92 - 1.02), 560 - 1500
  // rows 0.995 (0.96 - 1.016).  Steps of three Mixtral layers: 1500 / 1800 tokens, 375 / 450 rows per expert, 3761 -> 3674,
  // 4144 -> 4076 us, two prompts of 900 3769 -> 3690; at 900 - 1500 rows 7576 -> 7624, 12059 -> 12156, so one apart there.)
  re2.k_walk = M <= 512l * n_groups ? 5 : 1;
  kern<<<(int)std::min<long>(most, cus), 256, lds, st>>>(A, lda, B, ldb, C, ldc, M, N, K, N / 256, re2, ws, cnt, offsets,
                                                          n_groups);
}

void run_w4_grouped(int epi, const uint16_t* A, int lda, const uint16_t* B, int ldb, uint16_t* C, int ldc, int M, int N,
                    int K, hipStream_t st, const RopeEpi& re, const int* offsets, int n_groups) {
  if (epi == W4_NONE) run_w4_grouped_t<W4_NONE>(A, lda, B, ldb, C, ldc, M, N, K, st, re, offsets, n_groups);
  else run_w4_grouped_t<W4_SILU_MUL>(A, lda, B, ldb, C, ldc, M, N, K, st, re, offsets, n_groups);
}

template <int BMT>
static bool run_w4_h(int epi, const uint16_t* A, int lda, const uint16_t* B, int ldb, uint16_t* C, int ldc, int M,
                     int N, int K, hipStream_t st, const RopeEpi& re) {
  switch (epi) {
    case W4_NONE: return run_w4_t<W4_NONE, BMT>(A, lda, B, ldb, C, ldc, M, N, K, st, re);
    case W4_SILU_MUL: return run_w4_t<W4_SILU_MUL, BMT>(A, lda, B, ldb, C, ldc, M, N, K, st, re);
    case W4_ROPE: return run_w4_t<W4_ROPE, BMT>(A, lda, B, ldb, C, ldc, M, N, K, st, re);
    case W4_ADD_SS: return run_w4_t<W4_ADD_SS, BMT>(A, lda, B, ldb, C, ldc, M, N, K, st, re);
    case W4_NONE | W4_RS: return run_w4_t<W4_NONE | W4_RS, BMT>(A, lda, B, ldb, C, ldc, M, N, K, st, re);
    case W4_SILU_MUL | W4_RS: return run_w4_t<W4_SILU_MUL | W4_RS, BMT>(A, lda, B, ldb, C, ldc, M, N, K, st, re);
    case W4_ROPE | W4_RS: return run_w4_t<W4_ROPE | W4_RS, BMT>(A, lda, B, ldb, C, ldc, M, N, K, st, re);
    default: return false;
  }
}

bool run_w4(int epi, const uint16_t* A, int lda, const uint16_t* B, int ldb, uint16_t* C, int ldc, int M, int N,
            int K, hipStream_t st, const RopeEpi& re, int bm) {
  if (bm == 128) return run_w4_h<128>(epi, A, lda, B, ldb, C, ldc, M, N, K, st, re);
  if (bm == 160) return run_w4_h<160>(epi, A, lda, B, ldb, C, ldc, M, N, K, st, re);
  if (bm == 224) return run_w4_h<224>(epi, A, lda, B, ldb, C, ldc, M, N, K, st, re);
  if (bm == 192) return run_w4_h<192>(epi, A, lda, B, ldb, C, ldc, M, N, K, st, re);
  if (bm == 256) return run_w4_h<256>(epi, A, lda, B, ldb, C, ldc, M, N, K, st, re);
  return false;
}

}  // namespace mlop

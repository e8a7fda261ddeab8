// bf16 GEMM on MFMA for gfx950 (K1 prefill / K2 decode / K13 MoE grouped).
//
//   C[M, N] = A[M, K] . B[N, K]^T        (A: activations row-major, B: weights [out, in])
//
// Structure (cdna_hip_programming.md §5 "glds vs register staging", "Pipelining
// across barriers"):
//   * a workgroup owns a BM x BN tile; K is walked in BK = 64 steps;
//   * BOTH operands stream global -> LDS with global_load_lds_dwordx4 (LDS-DMA,
//     no VGPR staging) into a 3-deep ring: two k-steps stay in flight while the
//     MFMAs consume the third;
//   * one raw s_barrier per k-step, preceded by a COUNTED vmcnt (never 0 in the
//     steady state) — __syncthreads() would drain the DMA queue (its fence emits
//     vmcnt(0));
//   * the LDS image is lane-linear per 1 KiB piece (8 rows x 128 B), XOR-swizzled
//     through the SOURCE address: 16-B chunk c of row r sits at slot c ^ ((r>>1)&7),
//     so the 16 rows a ds_read_b128 lane group reads hit 16 different bank slots
//     (T2, rule 21: swizzle the source and the read, never the LDS destination);
//   * all LDS lives in ONE extern __shared__ array (a second object can make hipcc
//     emit vmcnt(0) before every ds_read: §5 item 4(a));
//   * waves WM x WN, each owning (BM/WM) x (BN/WN) as 16x16 accumulators fed by
//     v_mfma_f32_16x16x32_bf16.
//
// Decode (M <= 256) is weight-streaming: BM covers the batch so each weight byte
// is fetched from HBM once; when the N tiles cannot fill 256 CUs, K is split over
// blockIdx.z and fp32 slabs are combined by a reduce kernel that also applies
// the epilogue — optionally fused with the decoder's residual add + RMSNorm
// (launch-boundary reduce, §5 "Projection GEMM at M = 256" item 2).
//
// Epilogues (fp32 LDS copy of the tile, 16-B coalesced stores):
//   EPI_NONE      C = bf16(acc), or an activation of acc (RopeEpi::act, act_n0)
//   EPI_SILU_MUL  B rows gate/up interleaved in groups of 16, C[:, j] = silu(g_j) * u_j (N/2 cols)
//   EPI_ROPE      QKV projection: RoPE on q/k heads + q_out / paged K,V cache stores from the
//                 staged tile (RopeEpi, launch.h); needs whole 128-wide heads per staged chunk
// Grouped mode (MoE K13): A rows sorted by expert, offsets[e]..offsets[e+1];
// B = W[e] ([E, N, K]); blockIdx.y enumerates (expert, m-tile) pairs on device.
#include "common.h"
#include "launch.h"
#include "rope_epi.h"

namespace mlop {

enum { EPI_NONE = 0, EPI_SILU_MUL = 1, EPI_ROPE = 3 };
constexpr int kBK = 64;
constexpr int kStages = 3;
constexpr int kMaxSplits = 8;  // plan(): split-K factors are at most 8

// 16-B slot of chunk c in image row r is c ^ swz(r).  Two 128-B rows share one
// 256-B bank row, so (r>>1)&7 (not r&7) makes the 16 rows of a ds_read_b128 lane
// group land on 16 distinct slots: (r&1) picks the half, swz the slot in it.
__device__ __forceinline__ int swz(int r) { return (r >> 1) & 7; }



// Mid-M norm chain (above the decode form's rows, up to 64; launch_mid_res_ss): the O / down projection's split-K GEMM
// finishes itself.  Every split stored its fp32 partial write-through (sc1), waited for it,
// met its workgroup at a barrier, and one lane draws a relaxed agent-scope ticket on the
// tile's counter; the split that draws the last ticket reads the partials with sc1 loads only
// (re.mid_acq 0: MI355X_MICROARCH.md "Valid forms", sc1 stores, every storing wave's vmcnt(0)
// and the workgroup barrier before the ONE lane's ticket, sc1 loads of every handed-off byte),
// or with plain loads behind one agent acquire (re.mid_acq 1: attention.hip's split-KV combine
// protocol, for kernels with several workgroups per CU), and
//   * sums the tile's slabs in split order (splitk_add_rmsnorm's order and rounding: the
//     residual comes out bit-identical to the unfused path), residual = bf16(res + bf16(y));
//   * stores each row's sum of squares over the tile's BN columns (sc1) to the partials
//     [M][gx] past the slabs, then draws the row band's ticket;
// the band's last tile sums every row's partials in tile order into ss_tot[M], which the
// consumers (gate_up / QKV) turn into their rows' RMSNorm factors.  Counters: [gx * gy) tiles,
// then gy bands, re-armed by their last arriver.
// buffer loads with a fixed cache policy (AUX 16: sc1)
template <int AUX>
__device__ __forceinline__ u32x4 ld_b128(__amdgpu_buffer_rsrc_t rs, uint32_t off) {
  return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, off, 0, AUX));
}
template <int AUX>
__device__ __forceinline__ float ld_f32(__amdgpu_buffer_rsrc_t rs, uint32_t off) {
  return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, off, 0, AUX));
}

template <int BM, int BN, int T>
__device__ __forceinline__ void mid_chain_finish(uint16_t* __restrict__ C, int ldc, float* __restrict__ ws, int M,
                                                 int N, int m0, int n0, int rows_here, int bx, int by, int gx, int gy,
                                                 int n_splits, const RopeEpi& re, int* flag) {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();  // every wave's partial stored (and its LDS ring reads retired: flag reuses it)
  const int tid = threadIdx.x;
  int* tcnt = re.ss_cnt + by * gx + bx;
  if (tid == 0) flag[0] = __hip_atomic_fetch_add(tcnt, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == n_splits - 1;
  __syncthreads();
  if (!flag[0]) return;
  const bool acq = re.mid_acq != 0;
  if (tid == 0) {
    if (acq) {
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    __hip_atomic_store(tcnt, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  if (acq) __syncthreads();
  constexpr int VPR = BN / 8;  // 8-column vectors per tile row
  constexpr int RPP = T / VPR;  // rows per pass
  static_assert(T % VPR == 0 && VPR <= 64 && (VPR & (VPR - 1)) == 0, "row lanes");
  float* ssp = ws + (size_t)n_splits * M * N;  // [M][gx] row partials
  const auto rsS = __builtin_amdgcn_make_buffer_rsrc(ssp, 0, 0x7fffffff, 0x00020000);
  const auto rsW = __builtin_amdgcn_make_buffer_rsrc(ws, 0, 0x7fffffff, 0x00020000);
  for (int r0 = 0; r0 < BM; r0 += RPP) {
    const int r = r0 + tid / VPR, c = (tid % VPR) * 8;
    const int m = m0 + r, n = n0 + c;
    const bool ok = r < rows_here && n < N;
    float ssq = 0.f;
    if (ok) {
      // every slab's two loads in flight together (a runtime-bound loop waits out one memory
      // round trip per split), then summed in split order
      u32x4 x[kMaxSplits], y[kMaxSplits];
#pragma unroll
      for (int sp = 0; sp < kMaxSplits; ++sp)
        if (sp < n_splits) {
          const uint32_t off = (uint32_t)((((size_t)sp * M + m) * N + n) * 4);
          x[sp] = acq ? ld_b128<0>(rsW, off) : ld_b128<16>(rsW, off);
          y[sp] = acq ? ld_b128<0>(rsW, off + 16u) : ld_b128<16>(rsW, off + 16u);
        }
      float a[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int sp = 0; sp < kMaxSplits; ++sp)
        if (sp < n_splits) {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            a[e] += __uint_as_float(x[sp][e]);
            a[4 + e] += __uint_as_float(y[sp][e]);
          }
        }
      uint16_t* rp = C + (size_t)m * ldc + n;
      const u32x4 res = *reinterpret_cast<const u32x4*>(rp);
      u32x4 o;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        o[j] = pack2(bf2f(f2bf(a[2 * j])) + lo_bf(res[j]), bf2f(f2bf(a[2 * j + 1])) + hi_bf(res[j]));
        const float h0 = lo_bf(o[j]), h1 = hi_bf(o[j]);
        ssq += h0 * h0 + h1 * h1;
      }
      *reinterpret_cast<u32x4*>(rp) = o;
    }
#pragma unroll
    for (int o2 = VPR / 2; o2 > 0; o2 >>= 1) ssq += __shfl_xor(ssq, o2);
    if (ok && (tid % VPR) == 0)
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(ssq), rsS, (uint32_t)(((size_t)m * gx + bx) * 4), 0,
                                            16 /* sc1 */);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  int* bcnt = re.ss_cnt + gx * gy + by;
  if (tid == 0) flag[1] = __hip_atomic_fetch_add(bcnt, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == gx - 1;
  __syncthreads();
  if (!flag[1]) return;
  if (tid == 0) {
    if (acq) {
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    __hip_atomic_store(bcnt, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  if (acq) __syncthreads();
  // row totals: L = T / BM lanes per row, each summing the partials b = l, l + L, ... (loads
  // batched 8 at a time), then a fixed shuffle tree over the L lanes: deterministic, and no
  // chain of gx dependent memory round trips
  constexpr int L = T / BM >= 64 ? 64 : T / BM;
  static_assert(L >= 1 && (L & (L - 1)) == 0, "lanes per row");
  for (int r0 = 0; r0 < BM; r0 += T / L) {
    const int r = r0 + tid / L, l = tid % L;
    float sum = 0.f;
    if (r < rows_here) {
      const uint32_t row_off = (uint32_t)((size_t)(m0 + r) * gx * 4);
      for (int b0 = l; b0 < gx; b0 += 8 * L) {
        float v[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          const int b = b0 + k * L;
          v[k] = b >= gx ? 0.f : acq ? ld_f32<0>(rsS, row_off + (uint32_t)b * 4u) : ld_f32<16>(rsS, row_off + (uint32_t)b * 4u);
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) sum += v[k];
      }
    }
#pragma unroll
    for (int o2 = L / 2; o2 > 0; o2 >>= 1) sum += __shfl_xor(sum, o2);
    if (r < rows_here && l == 0) re.ss_tot[m0 + r] = sum;
  }
}

template <int BM, int BN, int WM, int WN, int EPI, bool GROUPED, int STAGES = 3, bool SETPRIO = false>
__global__ void __launch_bounds__(WM * WN * 64) gemm_kernel(
    const uint16_t* __restrict__ A, int lda, const uint16_t* __restrict__ B, int ldb,
    uint16_t* __restrict__ C, int ldc, float* __restrict__ ws, int M, int N, int K, int k_chunk,
    const int* __restrict__ offsets, int n_groups, int n_tiles_x, int m_tiles_y, int n_splits,
    RopeEpi re) {
  constexpr int NW = WM * WN, T = NW * 64;
  constexpr int WTM = BM / WM, WTN = BN / WN;
  constexpr int TM = WTM / 16, TN = WTN / 16;
  constexpr int NP = (BM + BN) / 8;  // 1-KiB pieces (8 rows x 128 B) per stage
  static_assert(NP % NW == 0, "pieces must divide the waves");
  constexpr int PPW = NP / NW;        // LDS-DMA instructions per wave per stage
  constexpr int STAGE = (BM + BN) * kBK;  // bf16 elements per stage
  extern __shared__ __attribute__((aligned(16))) uint16_t smem[];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wid / WN, wn = wid % WN;
  // XCD-aware remap (T1, bijective form): the 1-D grid is dealt round-robin over
  // the 8 XCDs, so give each XCD a CONTIGUOUS range of logical tiles ordered
  // (split, m-tile, n-tile): tiles sharing an A panel / K-chunk share an L2.
  // Speed only — correctness never depends on placement.
  const int G = gridDim.x, L = blockIdx.x;
  const int q = G >> 3, rr = G & 7, xcd = L & 7, slot = L >> 3;
  const int lid = (xcd < rr ? xcd * (q + 1) : rr * (q + 1) + (xcd - rr) * q) + slot;
  const int gx = n_tiles_x;
  // grouped: the (expert, m-tile) slot is the FAST index, so the slots left empty by a
  // routing (the grid is sized for the worst case, m_tiles + n_groups) are spread over
  // every XCD's contiguous range instead of idling the XCDs that drew the tail slots
  const int bx = GROUPED ? (lid / m_tiles_y) % gx : lid % gx;
  const int by = GROUPED ? lid % m_tiles_y : (lid / gx) % m_tiles_y;
  const int bz = lid / (gx * m_tiles_y);
  const int n0 = bx * BN;
  int m0 = by * BM, m_end = M;
  const uint16_t* Bg = B;
  if constexpr (GROUPED) {
    int t = by, e = 0;
    for (; e < n_groups; ++e) {
      const int rows = offsets[e + 1] - offsets[e];
      const int tiles = (rows + BM - 1) / BM;
      if (t < tiles) break;
      t -= tiles;
    }
    if (e >= n_groups) return;
    m0 = offsets[e] + t * BM;
    m_end = offsets[e + 1];
    Bg = B + (size_t)e * N * ldb;
  }
  const int kbeg = bz * k_chunk;
  const int kend = min(K, kbeg + k_chunk);
  const int nk = (kend - kbeg) / kBK;
  const bool split = n_splits > 1;

  // per-lane source row / chunk of each piece this wave issues (k advances by kBK)
  const int prow = lane >> 3;                  // row inside the 8-row piece
  const uint16_t* src[PPW];
#pragma unroll
  for (int i = 0; i < PPW; ++i) {
    const int p = wid + i * NW;
    const int r = p * 8 + prow;
    const int pchunk = (lane & 7) ^ swz(r);     // source chunk for LDS slot (lane & 7)
    if (r < BM) {
      int gr = min(m0 + r, m_end - 1);
      if (GROUPED && re.a_rows != nullptr) gr = re.a_rows[gr];
      src[i] = A + (size_t)gr * lda + kbeg + pchunk * 8;
    } else {
      const int gn = min(n0 + r - BM, N - 1);
      src[i] = Bg + (size_t)gn * ldb + kbeg + pchunk * 8;
    }
  }
  // weight pieces non-temporal when re.b_nt (wave-uniform: a piece is A or B by its index)
  const bool b_nt = re.b_nt != 0;
  // experts: column tile bx walks K from step bx % nk on (the channels of tiles in step: gemm_mid.hip; down of eight
  // experts at 20 rows 145 -> 140 us).  Dense split-K ranges are too short for it (qkv 17.5 -> 17.8)
  const int rot = GROUPED && nk > 0 ? bx % nk : 0;
  auto issue = [&](int buf, int kt) {
    kt = kt + rot >= nk ? kt + rot - nk : kt + rot;
    uint16_t* base = smem + buf * STAGE;
#pragma unroll
    for (int i = 0; i < PPW; ++i) {
      const int p = wid + i * NW;
      if (b_nt && p >= BM / 8)
        __builtin_amdgcn_global_load_lds((const void*)(src[i] + kt * kBK),
                                         (lds_void_t*)(base + p * 512), 16, 0, 2 /* nt */);
      else
        __builtin_amdgcn_global_load_lds((const void*)(src[i] + kt * kBK),
                                         (lds_void_t*)(base + p * 512), 16, 0, 0);
    }
  };

  f32x4 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

#pragma unroll
  for (int s = 0; s < STAGES - 1; ++s)
    if (s < nk) issue(s, s);
  for (int kt = 0; kt < nk; ++kt) {
    // stage kt must have landed; the STAGES-2 younger stages may stay in flight
    // the STAGES-2 younger stages may stay in flight (fewer near the end: drain)
    if (STAGES >= 3 && kt + STAGES - 2 < nk) wait_vmcnt<(STAGES >= 3 ? (STAGES - 2) * PPW : 0)>();
    else wait_vmcnt<0>();
    raw_barrier();  // stage kt visible to all waves; stage kt-1's buffer free
    if (kt + STAGES - 1 < nk) issue((kt + STAGES - 1) % STAGES, kt + STAGES - 1);
    const uint16_t* sA = smem + (kt % STAGES) * STAGE;
    const uint16_t* sB = sA + BM * kBK;
    if constexpr (SETPRIO) __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      const int ch = kk * 4 + (lane >> 4);
      bf16x8 af[TM], bfr[TN];
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const int r = wm * WTM + i * 16 + (lane & 15);
        af[i] = *reinterpret_cast<const bf16x8*>(sA + r * kBK + ((ch ^ swz(r)) << 3));
      }
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int r = wn * WTN + j * 16 + (lane & 15);
        bfr[j] = *reinterpret_cast<const bf16x8*>(sB + r * kBK + ((ch ^ swz(r)) << 3));
      }
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = mfma16(af[i], bfr[j], acc[i][j]);
    }
    if constexpr (SETPRIO) __builtin_amdgcn_s_setprio(0);
  }

  const int rows_here = min(BM, m_end - m0);
  if (split) {
    // split-K: fp32 partial slab [kz][M][N] (plain stores; reduce kernel in the next launch).
    // Mid norm chain (re.ss_cnt set, launch_mid_res_ss): write-through (sc1) stores, then the
    // last split of the tile finishes it in this launch (mid_chain_finish).
    float* P = ws + (size_t)bz * M * N;
    const bool fix = !GROUPED && re.ss_cnt != nullptr;
    const auto rsP = __builtin_amdgcn_make_buffer_rsrc(P, 0, 0x7fffffff, 0x00020000);
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int n = n0 + wn * WTN + j * 16 + (lane & 15);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int ml = wm * WTM + i * 16 + 4 * (lane >> 4) + r;
          if (ml < rows_here && n < N) {
            if (fix)
              __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(acc[i][j][r]), rsP,
                                                    (uint32_t)(((size_t)(m0 + ml) * N + n) * 4), 0, 16 /* sc1 */);
            else if (re.ws_nt & 1) __builtin_nontemporal_store(acc[i][j][r], P + (size_t)(m0 + ml) * N + n);
            else P[(size_t)(m0 + ml) * N + n] = acc[i][j][r];
          }
        }
      }
    if constexpr (!GROUPED) {
      if (fix) mid_chain_finish<BM, BN, T>(C, ldc, ws, M, N, m0, n0, rows_here, bx, by, gx, m_tiles_y, n_splits, re,
                                           reinterpret_cast<int*>(smem));
    }
    return;
  }
  raw_barrier();  // every wave is done reading the ring before it becomes the C tile
  // the C tile goes through LDS in column chunks of <= 128 (fp32 [BM][EW + 4])
  float* sC = reinterpret_cast<float*>(smem);
  constexpr int EW = BN < 128 ? BN : 128;
  constexpr int LDC = EW + 4;
#pragma unroll
  for (int c0 = 0; c0 < BN; c0 += EW) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int n = wn * WTN + j * 16 + (lane & 15) - c0;
        if (n >= 0 && n < EW) {
#pragma unroll
          for (int r = 0; r < 4; ++r) sC[(wm * WTM + i * 16 + 4 * (lane >> 4) + r) * LDC + n] = acc[i][j][r];
        }
      }
    __syncthreads();
    if constexpr (EPI == EPI_ROPE) {
      static_assert(EW == 128, "EPI_ROPE stages one whole head per chunk");
      static_assert(BM == 256, "EPI_ROPE tiles are 256 rows");
      auto at = [&](int r, int c) { return bf2f(f2bf(sC[r * LDC + c])); };
      rope_tile_store<T>(at, (n0 + c0) / 128, 1, m0, rows_here, re, tid);
    } else if constexpr (EPI == EPI_NONE) {
      constexpr int VPR = EW / 8;
      for (int v = tid; v < BM * VPR; v += T) {
        const int r = v / VPR, c = (v % VPR) * 8;
        if (r >= rows_here || n0 + c0 + c >= N) continue;
        float s[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) s[j] = sC[r * LDC + c + j];
        act_outs(re, s, n0 + c0 + c);
        u32x4 o;
#pragma unroll
        for (int j = 0; j < 4; ++j) o[j] = pack2(s[2 * j], s[2 * j + 1]);
        *reinterpret_cast<u32x4*>(C + (size_t)(m0 + r) * ldc + n0 + c0 + c) = o;
      }
    } else {
      constexpr int OUTW = EW / 2, VPR = OUTW / 8;
      for (int v = tid; v < BM * VPR; v += T) {
        const int r = v / VPR, j0 = (v % VPR) * 8;
        const int gcol = (j0 / 16) * 32 + (j0 % 16);
        if (r >= rows_here || n0 + c0 + gcol >= N) continue;
        const float* g = sC + r * LDC + gcol;
        const float* u = g + 16;
        // mid norm chain (re.ss_in: the producer's row totals): the row's RMSNorm factor scales
        // the accumulators first (W4_RS's order)
        float f = re.ss_in != nullptr ? rsqrtf(re.ss_in[m0 + r] * re.ss_inv_k + re.ss_eps) : 1.f;
        if constexpr (GROUPED) f = re.row_scale != nullptr ? re.row_scale[m0 + r] : 1.f;
        u32x4 o;
#pragma unroll
        for (int j = 0; j < 4; ++j)
          o[j] = pack2(glu_out(re, g[2 * j] * f, u[2 * j] * f), glu_out(re, g[2 * j + 1] * f, u[2 * j + 1] * f));
        *reinterpret_cast<u32x4*>(C + (size_t)(m0 + r) * ldc + (n0 + c0) / 2 + j0) = o;
      }
    }
    if (c0 + EW < BN) __syncthreads();
  }
}

// sum the split-K slabs and apply the epilogue; one thread per 8 outputs
template <int EPI>
__global__ void __launch_bounds__(256) splitk_reduce_kernel(uint16_t* __restrict__ C, int ldc,
                                                           const float* __restrict__ ws, int M,
                                                           int N, int splits, RopeEpi re = RopeEpi{}) {
  const int outw = EPI == EPI_NONE ? N : N / 2;
  const int vpr = outw / 8;
  const long total = (long)M * vpr;
  for (long v = blockIdx.x * (long)blockDim.x + threadIdx.x; v < total;
       v += (long)gridDim.x * blockDim.x) {
    const int r = (int)(v / vpr), j0 = (int)(v % vpr) * 8;
    const int col = EPI == EPI_NONE ? j0 : (j0 / 16) * 32 + (j0 % 16);
    float a[8] = {0, 0, 0, 0, 0, 0, 0, 0}, b[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    for (int s = 0; s < splits; ++s) {
      const float4* p = reinterpret_cast<const float4*>(ws + ((size_t)s * M + r) * N + col);
      float4 x = p[0], y = p[1];
      a[0] += x.x; a[1] += x.y; a[2] += x.z; a[3] += x.w;
      a[4] += y.x; a[5] += y.y; a[6] += y.z; a[7] += y.w;
      if (EPI == EPI_SILU_MUL) {
        const float4* q = p + 4;  // +16 floats: the matching up columns
        float4 z = q[0], w = q[1];
        b[0] += z.x; b[1] += z.y; b[2] += z.z; b[3] += z.w;
        b[4] += w.x; b[5] += w.y; b[6] += w.z; b[7] += w.w;
      }
    }
    if (EPI == EPI_SILU_MUL && re.row_scale != nullptr) {
      const float f = re.row_scale[r];
#pragma unroll
      for (int j = 0; j < 8; ++j) a[j] *= f, b[j] *= f;
    }
    if (EPI == EPI_NONE) act_outs(re, a, j0);
    u32x4 o;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (EPI == EPI_NONE)
        o[j] = pack2(a[2 * j], a[2 * j + 1]);
      else
        o[j] = pack2(glu_out(re, a[2 * j], b[2 * j]), glu_out(re, a[2 * j + 1], b[2 * j + 1]));
    }
    *reinterpret_cast<u32x4*>(C + (size_t)r * ldc + j0) = o;
  }
}

// split-K reduce fused with the decoder's residual add + RMSNorm (one row per block):
//   y = bf16(sum_s slab[s][r]);  residual[r] = bf16(residual[r] + y);  out[r] = rmsnorm(residual[r]) * w
template <int VPT>
__global__ void __launch_bounds__(512) splitk_add_rmsnorm_kernel(
    uint16_t* __restrict__ out, uint16_t* __restrict__ residual, const float* __restrict__ ws,
    const uint16_t* __restrict__ w, float eps, int M, int N, int splits) {
  __shared__ float scratch[16];
  const int r = blockIdx.x;
  const int nvec = N >> 3;
  float v[VPT][8];
  float ss = 0.f;
  // the norm weights load with the slabs (one memory latency on the chain, not two)
  u32x4 wpre[VPT];
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    const int vi = threadIdx.x + i * blockDim.x;
    if (vi < nvec) wpre[i] = *reinterpret_cast<const u32x4*>(w + vi * 8);
  }
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    const int vi = threadIdx.x + i * blockDim.x;
    if (vi < nvec) {
      // every slab's two loads (and the residual's) in flight together: a runtime-bound loop
      // waited out one L2 round trip per split (~5 us per call at batch 8-64, twice per layer)
      float4 x[kMaxSplits], y[kMaxSplits];
#pragma unroll
      for (int s = 0; s < kMaxSplits; ++s)
        if (s < splits) {
          const float4* p = reinterpret_cast<const float4*>(ws + ((size_t)s * M + r) * N + vi * 8);
          x[s] = p[0];
          y[s] = p[1];
        }
      const u32x4 res = *reinterpret_cast<const u32x4*>(residual + (size_t)r * N + vi * 8);
      float a[8] = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
      for (int s = 0; s < kMaxSplits; ++s)
        if (s < splits) {
          a[0] += x[s].x; a[1] += x[s].y; a[2] += x[s].z; a[3] += x[s].w;
          a[4] += y[s].x; a[5] += y[s].y; a[6] += y[s].z; a[7] += y[s].w;
        }
      u32x4 o;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float s0 = bf2f(f2bf(a[2 * j])) + lo_bf(res[j]);
        const float s1 = bf2f(f2bf(a[2 * j + 1])) + hi_bf(res[j]);
        o[j] = pack2(s0, s1);
        v[i][2 * j] = lo_bf(o[j]);
        v[i][2 * j + 1] = hi_bf(o[j]);
      }
      *reinterpret_cast<u32x4*>(residual + (size_t)r * N + vi * 8) = o;
#pragma unroll
      for (int j = 0; j < 8; ++j) ss += v[i][j] * v[i][j];
    }
  }
  ss = block_sum(ss, scratch);
  const float inv = rsqrtf(ss / (float)N + eps);
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    const int vi = threadIdx.x + i * blockDim.x;
    if (vi < nvec) {
      const u32x4 wv = wpre[i];
      u32x4 o;
#pragma unroll
      for (int j = 0; j < 4; ++j)
        o[j] = pack2(bf2f(f2bf(v[i][2 * j] * inv)) * lo_bf(wv[j]),
                     bf2f(f2bf(v[i][2 * j + 1] * inv)) * hi_bf(wv[j]));
      *reinterpret_cast<u32x4*>(out + (size_t)r * N + vi * 8) = o;
    }
  }
}

template <int BM, int BN, int STAGES>
constexpr size_t lds_bytes() {
  constexpr size_t ring = (size_t)STAGES * (BM + BN) * kBK * 2;
  constexpr int EW = BN < 128 ? BN : 128;
  constexpr size_t epi = (size_t)BM * (EW + 4) * 4;
  return ring > epi ? ring : epi;
}

// non-temporal weight stream of the decode-shaped GEMMs (gemm_small_nt op; MI355X_MICROARCH.md
// "nt-weights": serving streams 16 GB of other weights between two reads of one matrix, so the
// default policy's L2 / MALL fills are pure cost).  Interleaved on one box: Llama batch 16 +4.4 %,
// batch 64 +2.6 %, Mixtral batch 64 +6.3 % (gate_up at M = 16 / 64 46.1 -> 41.3 / 52.1 -> 47.7 us);
// bit 0 dense one-m-tile launches, bit 1 grouped small tiles, bit 2 grouped ping-pong
static int g_small_nt_flags = 7;
int gemm_small_nt(int set) {
  if (set >= 0) g_small_nt_flags = set;
  return g_small_nt_flags;
}

// non-temporal stores of GEMM outputs the next launch reads (gemm_slab_nt op; not left dirty in
// L2 for the kernel boundary's write-back, MI355X_MICROARCH.md "boundary"): bit 0 gemm_kernel's split-K
// slabs (batch 256 +0.6 %, batch 64 neutral), bit 1 the four-wave kernel's C (headline +1.2 %),
// bit 2 the ping-pong kernel's C (Mixtral batch 256 / 1024 and Llama batch 512 +0.3-0.4 %),
// bit 3 the four-wave RoPE epilogue's q / K / V (with attn_kv_nt 3: headline +0.5 % over 5 pairs)
static int g_slab_nt = 15;
static int g_split_target = 512;  // gemm_split_target op: workgroups the split-K of the 16-row tiles aims at
int gemm_split_target(int set) {
  if (set >= 1) g_split_target = set;
  return g_split_target;
}
int gemm_slab_nt(int set) {
  if (set >= 0) g_slab_nt = set;
  return g_slab_nt;
}
// weights of the dense weight-streaming launches (gemm_kernel, gemm_mid.hip) non-temporal: where one workgroup streams
// each of them
bool gemm_weights_nt(int m_tiles) { return (g_small_nt_flags & 1) != 0 && m_tiles == 1; }

template <int BM, int BN, int WM, int WN, int EPI, bool GROUPED, int STAGES, bool SETPRIO>
static void run_cfg(const uint16_t* A, int lda, const uint16_t* B, int ldb, uint16_t* C, int ldc,
                    float* ws, int M, int N, int K, int splits, int k_chunk, const int* offsets,
                    int n_groups, int m_tiles, hipStream_t st, const RopeEpi& re) {
  constexpr int T = WM * WN * 64;
  constexpr size_t lds = lds_bytes<BM, BN, STAGES>();
  static_assert(lds <= 163840, "LDS budget");
  auto kern = gemm_kernel<BM, BN, WM, WN, EPI, GROUPED, STAGES, SETPRIO>;
  static bool attr = false;
  if (!attr) {
    hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    attr = true;
  }
  const int gx = (N + BN - 1) / BN;
  const int blocks = gx * m_tiles * splits;
  // non-temporal weights where each weight byte is streamed by ONE workgroup: one m-tile
  // (dense), or the grouped decode tiles (an expert's few routed rows)
  RopeEpi r = re;
  r.b_nt = GROUPED ? (g_small_nt_flags & 2) != 0 && BM <= 64 : gemm_weights_nt(m_tiles);
  r.ws_nt = g_slab_nt;
  kern<<<blocks, T, lds, st>>>(A, lda, B, ldb, C, ldc, ws, M, N, K, k_chunk, offsets, n_groups, gx,
                               m_tiles, splits, r);
}

static int g_small_stages = 3;
int gemm_small_stages(int set) {
  if (set >= 0) g_small_stages = set;
  return g_small_stages;
}

// Row-fitted narrow tiles for M <= 64 (plan()): 0 = the 64 x 64 tile; 32 / 64 = BN with BM the
// batch rounded up to 16 / 32 / 64; 1 (default) = BM fitted, BN and ring depth per shape (no padding rows streamed through the A ring: the 16-row
// tile's 4-stage ring is 10 KB instead of 16, so more workgroups stay resident per CU).
// Default 64: M <= 32 cold projections 6-17 % faster than the 64 x 64 tile (qkv 18.3 -> 15.3 us,
// o+norm 14.9 -> 12.9, gate_up 47.1 -> 45.6, down+norm 32.9 -> 27.3 at M = 16; BN 32 loses:
// profiles/r02_midbatch_decode.md, scripts/run131.sh).  Run-time settable for A/B.
static int g_small_tile = 1;  // 1 = per-shape (plan); 64 x 64 for M 33-64
// ring depth of the grouped (MoE) 64-row tiles on narrow N (the down projection): 6 measured
// neutral on Mixtral batch 32 / 64 (1,651 vs 1,655, 3,142 vs 3,134 tok/s, scripts/run141.sh)
constexpr int g_grouped_small_stages = 3;
int gemm_small_tile(int set) {
  if (set >= 0) g_small_tile = set;
  return g_small_tile;
}

// grouped-plan override (scripts/bench_moe_decode.py compares MoE decode tilings in one process):
// BM, BN, ring stages, K splits; -1 = the planner's own choice.  Only tile shapes launch_plan has
// a grouped config for are accepted.
static int g_gp[4] = {-1, -1, -1, -1};
void gemm_grouped_plan(int bm, int bn, int stages, int splits) {
  if (bm > 0) {
    static const int ok[][2] = {{16, 32}, {16, 64}, {32, 32}, {32, 64}, {64, 32}, {64, 64},
                                {128, 64}, {256, 64}, {256, 128}, {256, 256}};
    bool found = false;
    for (const auto& t : ok) found = found || (t[0] == bm && t[1] == bn);
    if (!found) throw std::runtime_error("gemm_grouped_plan: no grouped config for this tile");
  }
  g_gp[0] = bm, g_gp[1] = bn, g_gp[2] = stages, g_gp[3] = splits;
}

// dense-plan override (scripts/bench_mid_m.py sweeps the mid-M projection tilings in one
// process): variant (0 = gemm_kernel BM x BN, 1 = 256x256 two-stage, 3 = ping-pong, 5 =
// four-wave, 6 = four-wave of BM 160, 192 or 224 rows, else half height, 8 = four-wave of BM rows over K ranges, behind
// gemm_add_rmsnorm only; one range: no such form), BM, BN, K splits (0 and 8 only), LDS
// ring depth of the small tiles (0 = the default); -1 = the planner's own choice
static int g_dp[5] = {-1, -1, -1, -1, 0};
static int g_slab[2] = {0, 0};  // variant 8's tile height (0: slab_plan's choice) and ranges
void gemm_dense_plan(int variant, int bm, int bn, int splits, int stages) {
  if (variant >= 0 && variant != 0 && variant != 1 && variant != 3 && variant != 5 && variant != 6 && variant != 8)
    throw std::runtime_error("gemm_dense_plan: variant must be 0, 1, 3, 5, 6 or 8");
  if (variant == 0) {
    static const int ok[][2] = {{16, 32}, {16, 64}, {32, 32}, {32, 64}, {64, 32}, {64, 64}, {96, 64}, {128, 64}, {192, 64}, {256, 64}, {256, 128}};
    bool found = false;
    for (const auto& t : ok) found = found || (t[0] == bm && t[1] == bn);
    if (!found) throw std::runtime_error("gemm_dense_plan: no dense config for this tile");
  }
  g_slab[0] = variant == 8 ? bm : 0, g_slab[1] = splits;
  if (variant == 8) variant = -1;  // (the plain plans keep their choice)
  g_dp[0] = variant, g_dp[1] = bm, g_dp[2] = bn, g_dp[3] = splits, g_dp[4] = stages > 0 ? stages : 0;
}

// large-M kernel choice (plan() variants below), settable at run time (gemm_big_variant op) so
// A/B microbenches run in one process
static int g_big_variant = 5;
int gemm_big_variant(int set) {
  if (set >= 0) g_big_variant = set;
  return g_big_variant;
}
// the grouped <= 32-rows-per-expert rule (plan() below) on / off (gemm_grouped_narrow op)
static int g_grouped_narrow = 1;
int gemm_grouped_narrow(int set) {
  if (set >= 0) g_grouped_narrow = set;
  return g_grouped_narrow;
}
// the planner's half-height four-wave tile (variant 6) on / off (gemm_half_tile op, A/B runs)
static int g_half_tile = 1;
int gemm_half_tile(int set) {
  if (set >= 0) g_half_tile = set;
  return g_half_tile;
}

// ---------------------------------------------------------------------------
// Ping-pong 256x256 GEMM (after cdna_hip_programming.md "The 256^2 8-phase template"):
// 8 waves = 2 wave GROUPS (A halves) x 4 column strips, 128x64 outputs per wave.
// Each K-tile (BK = 64) is 2 phases, one 64x64 half of the wave's outputs x K=64 (32 MFMAs):
//     [ds_read the half's fragments | issue LDS-DMA | drain lgkmcnt]
//     s_barrier; setprio(1) 32 x MFMA setprio(0); s_barrier
// Group 1 executes one extra barrier up front, so it is always one half-phase
// behind group 0: while one group's waves issue LDS reads / DMA, the other
// group's waves (one per SIMD each) keep the matrix cores busy — the barrier
// and LDS latency that idles a single-group loop (27% SQ_WAIT_ANY in
// profiles/r01_gemm_pmc.md) is overlapped by the partner group instead.
// Two LDS buffers (K-tile parity, 2 x 64 KB); the DMA schedule and its vmcnt /
// barrier accounting are in the comment above the K-loop.
//
// GROUPED (MoE K13 at >= 512 rows per expert): the (expert, m-tile) slot is the fast
// tile index (empty slots of the worst-case grid spread over all XCDs), B = W[e] and
// rows stop at offsets[e+1]; everything else is the dense schedule.
// Stream-K tail (plain, non-grouped launches): the T tiles are T / C full rounds on the C
// CUs plus r = T % C tail tiles, and a tail of r < C whole tiles leaves C - r CUs idle for
// a whole tile time (gate_up at M = 2040: 896 tiles = 3.5 rounds, 12.5 % of the kernel).
// The first T - r tiles stay data-parallel (one per workgroup); the r tail tiles' K-tiles
// are dealt as contiguous ranges of `ipw` K-tiles to n_sk more workgroups.  A workgroup
// whose range covers only part of a tile writes its fp32 accumulators to its own slot
// (2 per workgroup: the piece its range starts in, the piece it ends in), releases at
// agent scope and takes a ticket on the tile's counter; the LAST contributor acquires,
// adds the other slots and runs the normal epilogue, then resets the counter for the next
// launch.  Nobody waits on anybody (placement-independent, MI355X_MICROARCH.md
// "Correctness boundaries": dispatch order and co-residency are not assumed).
struct SkArgs {
  int n_dp;     // data-parallel workgroups = tiles before the tail (blockIdx < n_dp)
  int t0;       // first tail tile (logical tile index)
  int ipw;      // K-tiles per stream-K workgroup
  int n_iters;  // r * nk: K-tiles of the whole tail
  float* ws;    // 2 slots x 256 x 256 fp32 per stream-K workgroup
  int* cnt;     // one ticket counter per tail tile, zero between launches
  int n_base;   // first stream-K block (grouped: the worst-case tile count of the grid)
  int cus;      // CUs the split was planned for
  int min_half; // shortest K-range (K-tiles) the planner may cut
  int skip_dead;  // 1: quadrants past the last row issue no MFMAs (MLOP_GEMM_SKIP_DEAD=0: A/B)
  int balance;    // grouped: an expert over c > 1 m-tiles gets c EQUAL row ranges (gemm_grouped_balance)
  int order;      // grouped: 0 = (expert, m-tile) slot fastest, 1 = expert-major (gemm_grouped_order)
};

// d for the r = T % cus tail tiles of a T-tile launch: each is cut into d equal K-ranges
// (d | nk, so no range straddles two tiles), one per extra workgroup, d <= cus / r, when the
// cost model (in K-tile times, calibrated on scripts/bench_proj.py) beats the tail round's nk:
//   nk / d                   the range itself
//   max(2, 0.04 * r * d)     256 KB fp32 partial per workgroup, HBM-bound when all write
//   2 * (d - 1, or d)        the last contributor's slot reads (one CU, ~3 us per slot)
//   1                        a second pipeline fill + ticket
// 0: keep the data-parallel grid.  Host (plain launches) and device (grouped launches, whose
// tile count depends on the routing) evaluate the same function.
__host__ __device__ inline float sk_tail_cost(int r, int nk, int d) {
  const float w = 0.04f * r * d;
  return nk / d + (w > 2.f ? w : 2.f) + 2.f * (d >= 3 ? d : d - 1) + 1.f;
}

__host__ __device__ inline int sk_choose_d(int T, int nk, int cus, int min_half) {
  const int r = T % cus;
  if (r == 0) return 0;
  float best = 0.9f * nk;  // require a 10 % gain on the tail round
  int best_d = 0;
  const int dmax = cus / r < 32 ? cus / r : 32;
  for (int d = 2; d <= dmax; ++d) {
    if (nk % d || nk / d < min_half) continue;
    const float cost = sk_tail_cost(r, nk, d);
    if (cost < best) {
      best = cost;
      best_d = d;
    }
  }
  return best_d;
}

// Stream-K workgroup Lb (of n_sk starting at block n0) -> its range index, XCD-contiguous:
// blocks are dealt to the 8 XCDs round-robin (block & 7), so consecutive ranges -- which walk
// consecutive tiles and share their A / B panels -- must sit on ONE XCD's L2.  Dealing them
// round-robin made every XCD fetch nearly all of A and B (QKV at M = 2304: 2x slower).
__device__ __forceinline__ int sk_index(int Lb, int n0, int n_sk) {
  const int x = Lb & 7;
  int before = 0;
  for (int y = 0; y < x; ++y) {
    const int first = (y - n0) & 7;  // offset of XCD y's first block in the region
    before += first < n_sk ? (n_sk - first + 7) / 8 : 0;
  }
  return before + (Lb - n0) / 8;
}

template <int EPI, bool GROUPED = false, bool SK = false>
__global__ void __launch_bounds__(512, 1) gemm_pp_kernel(
    const uint16_t* __restrict__ A, int lda, const uint16_t* __restrict__ B, int ldb,
    uint16_t* __restrict__ C, int ldc, int M, int N, int K, int n_tiles_x, int m_tiles, int group_m,
    RopeEpi re, const int* __restrict__ offsets, int n_groups, SkArgs sk) {
  constexpr int BM = 256, BN = 256;
  constexpr int BUF = (BM + BN) * kBK;  // bf16 per K-tile buffer (64 KB)
  extern __shared__ __attribute__((aligned(16))) uint16_t smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int grp = wid >> 2, wc = wid & 3;
  const int Lb = blockIdx.x;
  const int nk = K / kBK;
  // launch geometry: data-parallel tiles [0, n_dp) on blocks [0, n_base), stream-K ranges
  // over the tail tiles [t0, T) on blocks [n_base, n_base + n_sk)
  int n_dp = sk.n_dp, t0 = sk.t0, ipw = sk.ipw, n_iters = sk.n_iters, n_sk = (int)gridDim.x - sk.n_base;
  int S = 0;  // grouped: (expert, m-tile) slots the routing actually filled
  bool expert_major = false;
  if constexpr (GROUPED) {
    int busy = 0;
    for (int e = 0; e < n_groups; ++e) {
      const int c = (offsets[e + 1] - offsets[e] + BM - 1) / BM;
      S += c;
      busy += c > 0;
    }
    // gemm_grouped_order 2 (auto): expert-major from 3 m-tiles per routed expert on average
    // (Mixtral at 765 rows per expert: gate_up -6 %, down -3.5 %; at 256 rows it lost 3.5 %)
    expert_major = sk.order == 1 || (sk.order == 2 && S >= 3 * busy);
    const int T = S * n_tiles_x;
    n_dp = T;
    t0 = T;
    ipw = 1;
    n_iters = 0;
    n_sk = 0;
    if constexpr (SK) {
      const int d = sk_choose_d(T, nk, sk.cus, sk.min_half);
      if (d) {
        const int r = T % sk.cus;
        n_dp = t0 = T - r;
        ipw = nk / d;
        n_iters = r * nk;
        n_sk = r * d;
      }
    }
  }
  const bool dp = !SK || Lb < sk.n_base;
  if (dp ? Lb >= n_dp : Lb - sk.n_base >= n_sk) return;  // whole workgroup, before any barrier

  // tile (logical index) -> origin.  Plain: bands of group_m m-tiles, m fastest within a band
  // (a B panel is reused by group_m consecutive tiles while L2-resident).  Grouped: the
  // routed (expert, m-tile) slot is the fast index, rows stop at offsets[e + 1], B = W[e].
  int m_end = M;
  const uint16_t* Bg = B;
  bool b_once = false;  // grouped: the expert fits one m-tile, its weights are streamed once
  auto tile_origin = [&](int lid, int& m0, int& n0) {
    if constexpr (GROUPED) {
      int e = 0, k = 0, nt = 0;
      if (expert_major) {
        // expert-major (gemm_grouped_order 1): expert e's c_e x n_tiles_x tiles are consecutive
        // lids, its m-tiles fastest, then its n-tiles.  The XCD-contiguous remap then gives each
        // XCD a run of n-tiles of one or two experts: the c_e m-tiles of an n-tile share its B
        // slice, and consecutive n-tiles reuse the same A rows from L2.  (Slot-fastest order put
        // every expert's m-tiles of an n-tile on the XCD at once: each A slice was read once per
        // n-tile from beyond L2.)
        int base = 0;
        for (; e < n_groups; ++e) {
          const int c = (offsets[e + 1] - offsets[e] + BM - 1) / BM;
          if (lid < base + c * n_tiles_x) break;
          base += c * n_tiles_x;
        }
        const int c = (offsets[e + 1] - offsets[e] + BM - 1) / BM;
        k = (lid - base) % c;
        nt = (lid - base) / c;
      } else {
        const int slot = lid % S;
        int before = 0;
        for (; e < n_groups; ++e) {
          const int c = (offsets[e + 1] - offsets[e] + BM - 1) / BM;
          if (slot < before + c) break;
          before += c;
        }
        k = slot - before;
        nt = lid / S;
      }
      const int rows_e = offsets[e + 1] - offsets[e], c = (rows_e + BM - 1) / BM;
      if (sk.balance && c > 1) {
        // c near-equal row ranges instead of c - 1 full tiles + a spill tile: the tiles of one
        // (expert, n-tile) then do near-equal work, stay in step on one XCD (adjacent lids) and
        // share each B K-tile through L2; a 257-row expert was 256 + 1 rows, the spill tile a
        // whole second walk of the B panel at HBM rate (profiles/r06_moe_spill.md).  Inner
        // boundaries sit on 64-row quadrants (the fewest MFMA quadrants, ceil(rows / 64)), each
        // tile at most BM rows.
        auto bnd = [&](int kk) {
          if (kk >= c) return rows_e;
          int b = 64 * (int)(((long)kk * rows_e + 32L * c) / (64L * c));
          b = min(b, BM * kk);
          return max(b, rows_e - BM * (c - kk));
        };
        m0 = offsets[e] + (k > 0 ? bnd(k) : 0);
        m_end = offsets[e] + bnd(k + 1);
      } else {
        m0 = offsets[e] + k * BM;
        m_end = offsets[e + 1];
      }
      n0 = nt * BN;
      Bg = B + (size_t)e * N * ldb;
      b_once = rows_e <= BM;
    } else {
      const int band = lid / (group_m * n_tiles_x), in_band = lid % (group_m * n_tiles_x);
      const int gm_here = min(group_m, m_tiles - band * group_m);
      m0 = (band * group_m + in_band % gm_here) * BM;
      n0 = (in_band / gm_here) * BN;
      // RoPE epilogue: walk each band's n-tiles backwards (the V heads, last columns, first;
      // they were the slow tiles while V pages were dim-major, and the order costs nothing)
      if constexpr (EPI == EPI_ROPE) n0 = (n_tiles_x - 1) * BN - n0;
    }
  };
  // iteration range of this workgroup in K-tiles of the logical tile space
  int it, it_end, m0g = 0, n0g = 0;
  const int s_idx = dp ? 0 : sk_index(Lb, sk.n_base, n_sk);
  if (dp) {
    // XCD-aware remap of the data-parallel part: each XCD a contiguous range of tiles
    const int G = n_dp;
    const int q = G >> 3, rr = G & 7, xcd = Lb & 7, slot = Lb >> 3;
    const int lid = (xcd < rr ? xcd * (q + 1) : rr * (q + 1) + (xcd - rr) * q) + slot;
    tile_origin(lid, m0g, n0g);
    it = lid * nk;
    it_end = it + nk;
  } else {
    it = t0 * nk + s_idx * ipw;
    it_end = t0 * nk + min((s_idx + 1) * ipw, n_iters);
  }

  f32x4 acc[8][4];
  const int prow = lane >> 3;
  bool first_piece = true;
  do {
    const int tile = SK ? it / nk : 0;
    const int k0 = SK ? it - tile * nk : 0, k1 = SK ? min(nk, k0 + (it_end - it)) : nk;
    it += k1 - k0;
    int m0 = m0g, n0 = n0g;
    if (SK && !dp) tile_origin(tile, m0, n0);
    if (SK && !first_piece) __syncthreads();  // the previous piece's epilogue is done with the LDS
    first_piece = false;
    const int nkp = k1 - k0;

    // DMA sources: half-tile h (0 A rows mi 0 = 0-63 and 128-191, 1 A rows mi 1, 2 B rows
    // 0-127, 3 B rows 128-255) = 16 pieces of 8 rows x 128 B; wave w moves pieces w, w+8.
    // Buffer-form LDS loads (buffer_load_dwordx4 ... lds): the per-lane byte offset into the
    // operand is fixed per tile and the K-tile advance rides in the scalar soffset, so an issue
    // is M0 + one VMEM instruction -- the global form needed a 64-bit VALU address add per
    // issue, serialised through one reused register pair.
    const auto rsA = __builtin_amdgcn_make_buffer_rsrc((void*)A, 0, 0x7fffffff, 0x00020000);
    const auto rsB = __builtin_amdgcn_make_buffer_rsrc((void*)Bg, 0, 0x7fffffff, 0x00020000);
    uint32_t voff[4][2];
#pragma unroll
    for (int h = 0; h < 4; ++h)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int r = h < 2 ? i * 128 + h * 64 + wid * 8 + prow : (h & 1) * 128 + (wid + 8 * i) * 8 + prow;
        const int ch = (lane & 7) ^ swz(r);
        // A rows past the tile's last row (the ragged / grouped tail: a spill m-tile of an expert
        // with 256 + a few rows is almost all such rows) load nothing: an offset past the
        // resource's num_records makes the LDS-DMA a dropped out-of-range access, still counted
        // by vmcnt (the counted waits stay exact) but fetching no line.  Their LDS rows hold
        // don't-care values that only ever reach accumulator rows that are never stored.
        const int arow = (GROUPED && re.a_rows != nullptr && m0 + r < m_end) ? re.a_rows[m0 + r] : m0 + r;
        voff[h][i] = h < 2 ? (m0 + r < m_end ? (uint32_t)((size_t)arow * lda * 2) + ch * 16 : 0x80000000u)
                           : (uint32_t)((size_t)min(n0 + r, N - 1) * ldb * 2) + ch * 16;
      }
    auto issue_half = [&](int buf, int h, int kt) {
      const uint32_t soff = (uint32_t)(k0 + kt) * kBK * 2;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int r0 = h < 2 ? i * 128 + h * 64 + wid * 8 : (h & 1) * 128 + (wid + 8 * i) * 8;
        uint16_t* dst = smem + buf * BUF + (h >= 2 ? BM * kBK : 0) + r0 * kBK;
        if (GROUPED && h >= 2 && re.b_nt && b_once)  // an expert's weights streamed once
          __builtin_amdgcn_raw_ptr_buffer_load_lds(rsB, (lds_void_t*)dst, 16, voff[h][i], soff, 0, 2 /* nt */);
        else
          __builtin_amdgcn_raw_ptr_buffer_load_lds(h < 2 ? rsA : rsB, (lds_void_t*)dst, 16, voff[h][i], soff, 0, 0);
      }
    };
    auto read_a = [&](int buf, int mi, bf16x8 (&fa)[4][2]) {
      const uint16_t* sA = smem + buf * BUF;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = grp * 128 + mi * 64 + i * 16 + (lane & 15);
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
          const int ch = kk * 4 + (lane >> 4);
          fa[i][kk] = *reinterpret_cast<const bf16x8*>(sA + r * kBK + ((ch ^ swz(r)) << 3));
        }
      }
    };
    auto read_b = [&](int buf, int nj, bf16x8 (&fb)[2][2]) {
      const uint16_t* sB = smem + buf * BUF + BM * kBK;
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int r = wc * 64 + nj * 32 + j * 16 + (lane & 15);
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
          const int ch = kk * 4 + (lane >> 4);
          fb[j][kk] = *reinterpret_cast<const bf16x8*>(sB + r * kBK + ((ch ^ swz(r)) << 3));
        }
      }
    };

#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    // a 64-row quadrant wholly past the tile's last row issues no MFMAs (wave-uniform): the
    // partner group's MFMAs then run alone on the SIMD.  Ragged M, and above all the last
    // m-tile of every expert in the grouped (MoE) GEMM, half empty on average.
    const int rows_here = sk.skip_dead ? m_end - m0 : BM;
    // K-loop: two phases per K-tile, 32 MFMAs each.
    //   X(t): read A(mi 0) + B(nj 0, 1) of t | DMA A(mi 1) of t+1 -> buffer (t+1)&1
    //   Y(t): read A(mi 1) of t             | DMA A(mi 0) + B of t+2 -> buffer t&1
    // Group 1 runs one barrier behind group 0, so each SIMD's two waves alternate: one issues
    // its phase's LDS reads and DMAs while the other runs 32 MFMAs.  (The guide's 4 x 16-MFMA
    // template hands the matrix core over twice as often: 2-9 % slower on every Llama-3-8B
    // projection, profiles/r03_gemm_fourwave.md.)  Every phase drains its LDS reads before its
    // first barrier, so a buffer region can be restaged in the phase after its last read; every
    // wait (counted vmcnt) precedes the first barrier of the phase before the reads (RAW across
    // the staggered groups):
    //   X(t) wait: A(mi 1, t) retired; 8 younger DMAs (A0+B of t+1, A1 of t+1) stay in flight
    //   Y(t) wait: A(mi 0) + B of t+1 retired; A1(t+1) and A0+B(t+2) stay in flight
    bf16x8 fa[4][2], fb0[2][2], fb1[2][2];
    auto seg_mma = [&](int mi) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // drain before the barrier
      raw_barrier();
      __builtin_amdgcn_sched_barrier(0);
      // a 64-row quadrant wholly past the tile's last row issues no MFMAs (wave-uniform)
      if (grp * 128 + mi * 64 < rows_here) {
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          // balance 2: 16-row blocks past the last row skipped too (wave-uniform; a 257-row
          // expert's balanced tiles then do 8 and 9 blocks, near-equal, and stay in step)
          if (i > 0 && sk.balance == 2 && grp * 128 + mi * 64 + i * 16 >= rows_here) continue;
#pragma unroll
          for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int kk = 0; kk < 2; ++kk) {
              acc[mi * 4 + i][j] = mfma16(fa[i][kk], fb0[j][kk], acc[mi * 4 + i][j]);
              acc[mi * 4 + i][2 + j] = mfma16(fa[i][kk], fb1[j][kk], acc[mi * 4 + i][2 + j]);
            }
        }
        __builtin_amdgcn_s_setprio(0);
      }
      __builtin_amdgcn_sched_barrier(0);
      raw_barrier();
    };
    issue_half(0, 0, 0);
    issue_half(0, 1, 0);
    issue_half(0, 2, 0);
    issue_half(0, 3, 0);
    if (nkp > 1) { issue_half(1, 0, 1); issue_half(1, 2, 1); issue_half(1, 3, 1); }
    if (nkp > 1) wait_vmcnt<6>(); else wait_vmcnt<0>();
    raw_barrier();
    if (grp == 1) raw_barrier();  // stagger: group 1 runs one barrier behind group 0
    for (int t = 0; t < nkp; ++t) {
      const int cur = t & 1, nxt = cur ^ 1;
      const bool m1 = t + 1 < nkp, m2 = t + 2 < nkp;
      read_a(cur, 0, fa);  // X(t)
      read_b(cur, 0, fb0);
      read_b(cur, 1, fb1);
      if (m1) {
        issue_half(nxt, 1, t + 1);
        wait_vmcnt<8>();
      } else {
        wait_vmcnt<0>();
      }
      seg_mma(0);
      read_a(cur, 1, fa);  // Y(t)
      if (m2) {
        issue_half(cur, 0, t + 2);
        issue_half(cur, 2, t + 2);
        issue_half(cur, 3, t + 2);
        wait_vmcnt<8>();
      } else if (m1) {
        wait_vmcnt<2>();
      }
      seg_mma(1);
    }
    if (grp == 0) raw_barrier();  // barrier counts of the two groups must match
    __syncthreads();              // all LDS reads retired everywhere: the ring becomes C staging

    if (SK && k1 - k0 != nk) {
      // stream-K partial tile: slot, ticket, and (last contributor only) the fixup
      const int s = s_idx, base = t0 * nk;
      auto slot_of = [&](int w) { return 2 * w + (tile == (base + w * ipw) / nk ? 0 : 1); };
      const int first_w = (tile * nk - base) / ipw, last_w = (tile * nk + nk - 1 - base) / ipw;
      // hand-off (MI355X_MICROARCH.md "Valid forms", first table row): 16-B sc1 (write-through)
      // stores, every storing wave's vmcnt(0), a barrier, ONE lane's agent-scope ticket add;
      // the workgroup whose add came last loads the other slots with 16-B sc1 loads after a
      // barrier.  No L2 write-back / invalidate: an agent release here (buffer_wbl2) writes
      // back every dirty line of the XCD's L2 -- the C tiles of the other workgroups too.
      constexpr int kSlotBytes = BM * BN * 4;
      auto slot_rsrc = [&](int w) {
        return __builtin_amdgcn_make_buffer_rsrc(sk.ws + (size_t)slot_of(w) * (BM * BN), 0, kSlotBytes, 0x00020000);
      };
      {
        const auto rs = slot_rsrc(s);
#pragma unroll
        for (int i = 0; i < 8; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j)
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, acc[i][j]), rs, tid * 16,
                                                   (i * 4 + j) * 512 * 16, 16 /* sc1 */);
      }
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      int* flag = reinterpret_cast<int*>(smem);
      if (tid == 0) {
        const int t = __hip_atomic_fetch_add(sk.cnt + (tile - t0), 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const bool last = t == last_w - first_w;
        if (last) __hip_atomic_store(sk.cnt + (tile - t0), 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        flag[0] = last;
      }
      __syncthreads();
      const int last = flag[0];
      __syncthreads();  // flag read everywhere before the epilogue reuses the LDS
      if (!last) continue;
      // deterministic sum: with 2 contributors own + other is exact whichever arrives last;
      // with 3+ the last one re-reads its own slot and sums every slot in contributor order
      const bool reload = last_w - first_w >= 2;
      if (reload) {
#pragma unroll
        for (int i = 0; i < 8; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
      for (int w = first_w; w <= last_w; ++w) {
        if (w == s && !reload) continue;
        const auto rs = slot_rsrc(w);
        // 16 loads in flight per batch: one load -> wait -> add at a time is ~1.5 us per
        // round trip, 48 us per slot (the compiler keeps these loads in program order)
#pragma unroll
        for (int g = 0; g < 2; ++g) {
          f32x4 v[16];
#pragma unroll
          for (int q = 0; q < 16; ++q)
            v[q] = __builtin_bit_cast(
                f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, tid * 16, (g * 16 + q) * 512 * 16, 16 /* sc1 */));
#pragma unroll
          for (int q = 0; q < 16; ++q) acc[(g * 16 + q) / 4][q % 4] += v[q];
        }
      }
    }

    if constexpr (EPI == EPI_ROPE) {
      // stage the whole 256 x 256 bf16 tile (two heads), then rotate / scatter per head
      constexpr int LDR = BN + 8;
#pragma unroll
      for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int row = grp * 128 + i * 16 + 4 * (lane >> 4) + r;
#pragma unroll
          for (int j = 0; j < 4; ++j) smem[row * LDR + wc * 64 + j * 16 + (lane & 15)] = f2bf(acc[i][j][r]);
        }
      __syncthreads();
      const int rows = min(BM, m_end - m0);
      auto at = [&](int r, int c) { return bf2f(smem[r * LDR + c]); };
      rope_tile_store<512>(at, n0 / 128, 2, m0, rows, re, tid);
      continue;
    }
    // epilogue: each wave stages its 128 x 64 (or 128 x 32 after SiLU.mul) bf16 tile
    constexpr int OW = EPI == EPI_NONE ? 64 : 32;
    constexpr int LD = OW + 8;
    uint16_t* sC = smem + wid * 128 * LD;
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = i * 16 + 4 * (lane >> 4) + r;
        if constexpr (EPI == EPI_NONE) {
          float v[4] = {acc[i][0][r], acc[i][1][r], acc[i][2][r], acc[i][3][r]};
          act_outs(re, v, n0 + wc * 64);
#pragma unroll
          for (int j = 0; j < 4; ++j) sC[row * LD + j * 16 + (lane & 15)] = f2bf(v[j]);
        } else {
          float f = 1.f;
          if constexpr (GROUPED)
            if (re.row_scale != nullptr) f = re.row_scale[min(m0 + grp * 128 + row, m_end - 1)];
#pragma unroll
          for (int jp = 0; jp < 2; ++jp) {
            const float g = acc[i][2 * jp][r] * f, u = acc[i][2 * jp + 1][r] * f;
            sC[row * LD + jp * 16 + (lane & 15)] = f2bf(glu_out(re, g, u));
          }
        }
      }
    __syncthreads();
    constexpr int CPR = OW / 8;  // 16-B chunks per staged row
    const int out_col0 = EPI == EPI_NONE ? n0 + wc * 64 : (n0 + wc * 64) / 2;
    const int out_n = EPI == EPI_NONE ? N : N / 2;
#pragma unroll
    for (int i2 = 0; i2 < 128 * CPR / 64; ++i2) {
      const int c = i2 * 64 + lane;
      const int row = c / CPR, cc = (c % CPR) * 8;
      const int gm = m0 + grp * 128 + row, gn = out_col0 + cc;
      if (gm < m_end && gn < out_n) {
        const u32x4 v = *reinterpret_cast<const u32x4*>(sC + row * LD + cc);
        if (re.ws_nt & 4) __builtin_nontemporal_store(v, reinterpret_cast<u32x4*>(C + (size_t)gm * ldc + gn));
        else *reinterpret_cast<u32x4*>(C + (size_t)gm * ldc + gn) = v;
      }
    }
  } while (SK && it < it_end);
}

// Stream-K buffers (per device, allocated once outside graph capture by gemm_sk_reserve):
// 2 partial slots per stream-K workgroup and kCntRegions rotating sets of tail-tile counters,
// so back-to-back launches never share a counter set while one may still be resetting.
constexpr int kSkMaxWg = 256, kCntRegions = 64;
struct SkBuf {
  float* ws = nullptr;
  int* cnt = nullptr;
  int next = 0, cus = 0;
};
static SkBuf g_sk[16];
static int g_sk_mode = 1;
static const int g_sk_min_iters = 16;
static const int g_skip_dead = 1;
// gemm_grouped_balance op: 1 = quadrant-aligned equal row ranges for an expert over several
// m-tiles (8 x 257 rows gate_up 677 -> 639 us, down 353 -> 308; Mixtral batch 1024 +0.75 %);
// 2 (default) = that + 16-row blocks past the tile's last row skip their MFMAs, so the two
// tiles of a 257-row expert do 8 and 9 blocks (gate_up 597 us; batch 1024 +0.3-0.5 % over 1)
// (profiles/r06_moe_spill.md)
static int g_grouped_balance = 2;
int gemm_grouped_balance(int set) {
  if (set >= 0) g_grouped_balance = set;
  return g_grouped_balance;
}
static int g_grouped_order = 2;  // 0 slot fastest, 1 expert-major, 2 expert-major from 3 m-tiles / expert
int gemm_grouped_order(int set) {
  if (set >= 0) g_grouped_order = set;
  return g_grouped_order;
}

int gemm_sk_mode(int set) {
  if (set >= 0) g_sk_mode = set;
  return g_sk_mode;
}

bool gemm_sk_reserve() {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 16) return false;
  SkBuf& b = g_sk[dev];
  if (b.ws) return true;
  int cus = 0;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0) return false;
  b.cus = std::min(cus, kSkMaxWg);
  float* ws = nullptr;
  int* cnt = nullptr;
  if (hipMalloc((void**)&ws, (size_t)2 * kSkMaxWg * 256 * 256 * sizeof(float)) != hipSuccess) return false;
  if (hipMalloc((void**)&cnt, (size_t)kCntRegions * kSkMaxWg * sizeof(int)) != hipSuccess) {
    (void)hipFree(ws);
    return false;
  }
  if (hipMemset(cnt, 0, (size_t)kCntRegions * kSkMaxWg * sizeof(int)) != hipSuccess ||
      hipDeviceSynchronize() != hipSuccess) {
    (void)hipFree(ws);
    (void)hipFree(cnt);
    return false;
  }
  b.ws = ws;
  b.cnt = cnt;
  return true;
}

// Split of a plain launch's T tiles: n_dp data-parallel workgroups + a stream-K tail
// (n_sk = 0: no tail).  The r = T % C tail tiles are each cut into d equal K-ranges (d | nk,
// so no range straddles two tiles), one per extra workgroup, d <= C / r, when the cost model
// (in K-tile times, calibrated on scripts/bench_proj.py) beats the tail round's nk:
//   ipw                      the range itself
//   max(2, w * 0.04)         256 KB fp32 partial per workgroup, HBM-bound when all write
//   (d - 1 or d) * 2         the last contributor's slot reads (one CU, ~3 us per slot)
//   1                        a second pipeline fill + ticket
// Ranges that straddle tiles (general stream-K) were measured slower than the data-parallel
// grid whenever the tail exceeds half the chip: twice the partial traffic, two fills.
static int sk_min_half() { return std::max(1, g_sk_min_iters / 2); }

static SkBuf* sk_buf() {
  int dev = 0;
  if (!g_sk_mode || hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 16) return nullptr;
  SkBuf& b = g_sk[dev];
  return b.ws && b.cus > 0 ? &b : nullptr;
}

// partial-tile scratch for the four-wave kernel's split tail (gemm_w4.hip): the same per-device
// slot buffer and a rotated ticket-counter region; false when the buffers are not reserved
bool gemm_sk_scratch(float** ws, int** cnt, int* cus) {
  SkBuf* b = sk_buf();
  if (!b) return false;
  *ws = b->ws;
  *cnt = b->cnt + (size_t)(b->next++ % kCntRegions) * kSkMaxWg;
  *cus = b->cus;
  return true;
}

bool gemm_sk_available(int* cus) {
  SkBuf* b = sk_buf();
  if (b && cus) *cus = b->cus;
  return b != nullptr;
}

static SkArgs sk_plan(int T, int nk, int& n_sk) {
  SkArgs a{T, T, 1, 0, nullptr, nullptr, T, 256, sk_min_half(), g_skip_dead};
  n_sk = 0;
  SkBuf* b = sk_buf();
  if (!b) return a;
  const int d = sk_choose_d(T, nk, b->cus, sk_min_half());
  if (!d) return a;
  const int r = T % b->cus;
  a.n_dp = T - r;
  a.t0 = T - r;
  a.ipw = nk / d;
  a.n_iters = r * nk;
  a.ws = b->ws;
  a.cnt = b->cnt + (size_t)(b->next++ % kCntRegions) * kSkMaxWg;
  a.n_base = a.n_dp;
  a.cus = b->cus;
  n_sk = r * d;
  return a;
}

template <int EPI, bool GROUPED = false>
static void run_pp(const uint16_t* A, int lda, const uint16_t* B, int ldb, uint16_t* C, int ldc, int M,
                   int N, int K, hipStream_t st, const RopeEpi& re, const int* offsets = nullptr,
                   int n_groups = 0) {
  constexpr size_t ring = 2ull * (256 + 256) * kBK * 2;
  constexpr size_t epi = EPI == EPI_ROPE ? 256ull * (256 + 8) * 2
                                         : 8ull * 128 * ((EPI == EPI_NONE ? 64 : 32) + 8) * 2;
  constexpr size_t lds = ring > epi ? ring : epi;
  static_assert(lds <= 163840, "LDS budget");
  auto kern = gemm_pp_kernel<EPI, GROUPED>;
  static bool attr = false;
  if (!attr) {
    hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    attr = true;
  }
  const int gx = (N + 255) / 256, gy = (M + 255) / 256 + (GROUPED ? n_groups : 0);
  constexpr int group_m = 4;
  const int gm = std::max(1, std::min(group_m, gy));
  int n_sk = 0;
  SkArgs sk = sk_plan(gx * gy, K / kBK, n_sk);
  // expert weights non-temporal where the expert fits one 256-row m-tile (decided per tile on
  // device): Mixtral batch 256 (64 rows per expert on average) +3.9 %; nt on every expert lost
  // 1.5 % at batch 1024, where the spill m-tiles of the > 256-row experts re-read the weights
  RopeEpi r = re;
  r.b_nt = GROUPED && (g_small_nt_flags & 4) != 0;
  r.ws_nt = g_slab_nt;
  if constexpr (GROUPED) {
    // the routed tile count is only known on device: the grid is the worst case (every
    // expert's last m-tile partial) plus one stream-K block per CU; the kernel plans the
    // split from offsets[] with the same sk_choose_d and idles the blocks it does not need
    SkBuf* b = sk_buf();
    const int T_max = gx * gy;
    sk = SkArgs{T_max, T_max, 1, 0, nullptr, nullptr, T_max, 256, sk_min_half(), g_skip_dead, g_grouped_balance, g_grouped_order};
    if (b) {
      sk.ws = b->ws;
      sk.cnt = b->cnt + (size_t)(b->next++ % kCntRegions) * kSkMaxWg;
      sk.cus = b->cus;
      n_sk = b->cus;
    }
  }
  if (n_sk > 0) {
    auto ksk = gemm_pp_kernel<EPI, GROUPED, true>;
    static bool attr_sk = false;
    if (!attr_sk) {
      hipFuncSetAttribute((const void*)ksk, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
      attr_sk = true;
    }
    ksk<<<sk.n_base + n_sk, 512, lds, st>>>(A, lda, B, ldb, C, ldc, M, N, K, gx, gy, gm, r, offsets, n_groups, sk);
    return;
  }
  kern<<<gx * gy, 512, lds, st>>>(A, lda, B, ldb, C, ldc, M, N, K, gx, gy, gm, r, offsets, n_groups, sk);
}

struct Plan {
  int BM, BN, splits, k_chunk, m_tiles, variant;
  int stages;  // LDS-DMA ring depth of the small-M tiles (0: g_small_stages)
  bool nosplit;  // grouped: one K range (the mid-size MoE split-K below is skipped)
};


// Tile choice by the (per-group) row count:
//   M <= 64 / 128: narrow tiles, many WGs (weight streaming);  M <= 256: the whole
//   batch in one tile (weights read once), BN by how many N tiles fill the chip;
//   large M: variant 0 = 256x128 (3-stage ring), 1 = 256x256 (2-stage, 128x64 per
//   wave: half the LDS + L2 bytes per FLOP), 2 = 256x256 + setprio around MFMAs,
//   3 = 256x256 two-group ping-pong (gemm_pp_kernel), 5 (default) = the four-wave kernel with
//   the hand-scheduled asm K-loop (gemm_w4.hip), 256 rows, 6 = its tiles of 128 - 224 rows (big_plan
//   chooses between 3, 5 and 6; without its scratch 5 where the grid fills the chip, else 3), 7 = the weight
//   stream of gemm_mid.hip (mid_plan, up to 384 rows, before all others).  (A four-wave 128x128-per-wave
//   variant was measured 10-20% slower: profiles/r02_gemm_fourwave_rejected.md.)
// true when the stream-K tail is available here and splits ALL T (<= C / 2) tiles
static bool sk_halves_ok(long T, int nk) {
  const SkBuf* b = sk_buf();
  return b && T * 2 <= b->cus && sk_choose_d((int)T, nk, b->cus, sk_min_half()) >= 2;
}

// Variant 7, the weight stream of gemm_mid.hip, for up to 384 rows: where its tasks take at least three
// quarters of the CUs, in one K range with 256 or 128 columns, or (65 rows and more) with K in up to 8 ranges of
// at least 12 K-steps.  Below that, and for split K at 64 rows and fewer, the small tiles are as fast or faster
// (o 4096 x 4096 at 100 rows 17.5 us against 18.6 in six ranges; down 4096 x 14336 at 16 / 64 rows 24.2 / 29.2
// against 26.6 / 29.5).
static bool mid_plan(int M, int N, int K, Plan& p) {
  constexpr int max_m = 384, fill = kCus * 3 / 4;
  if (M > max_m || K < kBK || K % kBK || N % 8) return false;  // (no K-step: gemm_kernel writes the empty sums)
  if (M <= 64 && g_small_tile != 1) return false;              // one of gemm_kernel's tiles is asked for
  const int m_tiles = M <= 256 ? 1 : 2, rows = (M + m_tiles - 1) / m_tiles;
  const int t256 = (N + 255) / 256 * m_tiles, t128 = (N + 127) / 128 * m_tiles, nk = K / kBK;
  // 32-row tiles up to one round of the CUs and again where a quarter of them has a second one; between, where few have, 64 rows
  // (33280 columns at 17 - 32 rows 2.3 % faster, 36864 1.6 %, 40960 level, 45056 2.6 % slower; 24576 - 32768 6 - 9 % slower)
  const bool second = t256 < fill && t128 > kCus && t128 < kCus * 5 / 4;
  const int bm = rows <= 32 && second ? 64 : (rows + 31) / 32 * 32;
  int s = 1;
  if (t256 < fill && t128 < fill) {
    s = std::min({kMaxSplits, kCus / t128, nk / 12});
    if (M <= 64 || t128 * s < fill) return false;
    const int t64 = (N + 63) / 64;
    // where the 64-column tiles need no K ranges, the slabs have to be small beside the weights (12544 x 2048 in two
    // ranges at 100 / 200 rows: 22 / 31 us against 20 / 24; 10240 x 8192 in three: 42 against 65); less so where those
    // tiles fill the CUs with K in a few ranges (8192 x 3584 in four at 80 / 112 / 128 rows 23 / 26.0 / 26.5 us against 24 /
    // 24.2 / 24.5, at 160 / 192 / 256 rows 28.5 / 31.6 / 36.4 against 29.6 / 30.2 / 32.2)
    if (t64 >= 160 && 4l * s * M > K * 3l / 10) return false;
    if (m_tiles == 1 && t64 < 160 && t64 * std::max(1, kCus / t64) >= 250 && 400l * s * M > K * (M <= 128 ? 43l : 80l)) return false;
  }
  // Two row tiles read the weights twice (the second from L2).  Where the four-wave kernel's lower tiles have a grid, they
  // are faster without K ranges, and with them above 320 rows (257 / 384 rows of gate_up 28672 x 4096 80 / 92 us ->
  // 71 / 73, lm_head 128256 x 4096 340 / 432 -> 272 / 332, 12288 x 4096 53 / 62 -> 43 / 49; down of Llama-3-70B at 350 rows
  // 255 -> 229, its quarter 8192 x 7168 at 384 66 -> 61)
  if (m_tiles == 2 && (s == 1 || M > 320) && (M + 127) / 128 * (N / 256) >= 64 && sk_buf() != nullptr && gemm_w4_ok(M, N, K, K, K))
    return false;
  p.variant = 7;
  p.BM = bm;
  p.BN = t256 >= fill ? 256 : 128;
  p.k_chunk = (nk + s - 1) / s * kBK;
  p.splits = (K + p.k_chunk - 1) / p.k_chunk;
  return true;
}

// Above the weight stream's rows: the four-wave kernel's tile height, or the ping-pong kernel with its stream-K tail,
// by estimated time in us.  A round of 256-row tiles takes 6 + 0.0207 K; lower tiles cost more per row (224 rows 0.90
// of it, 192 0.805, 160 0.70, 128 0.632: fewer MFMAs per fragment read), and an only round that fills a share f of the CUs runs
// faster.  A tail of at most half the CUs is cut into K-halves: half a round and the hand-off of the partials,
// 15 us.  A round of the ping-pong kernel takes 13.5 + 0.0206 K, its tail 1.1 of
// what sk_tail_cost says (1.0 fits as well; where the two are level the four-wave kernel is the better choice, since a
// layer whose four projections all run there needs no add + RMSNorm passes: 1024 rows of Llama-3-8B 2855 -> 2811 us).
// Constants of the ping-pong kernel and of 256, 192, 160 and 128 rows fitted to 39 weight shapes (the projections of
// Llama-3-8B and 70B, whole and in 2 - 8 shards, Mixtral's, a 1B model's and shapes of no model here: N 1024 - 128256, K
// 1024 - 28672) at 39 row counts from 385 to 8192, every variant measured in one process, two to four times: the choice was
// 0.13 % slower than the best of those five on average, more than 5 % at 8 of 1370 points, 12 % at worst; fitted to half of
// the shapes, 0.3 % on the others.  (Constants fitted to Llama-3-8B's matrices alone: 1.4 %, 110 of 1147 points and 38 %, and
// at 46 of them slower than the rule by tile counts that was here before: 70B qkv at 640 rows 113 us against 102, o at 1000
// 116 against 107, down at 2300 839 against 785.  The rule by tile counts, heights 256 and 128 only, was 8.4 % slower than
// the best on average: gate_up of Llama-3-8B at 400 / 700 / 1152 rows 138 -> 92, 158 -> 147, 245 -> 219 us, o at 1152 / 2300 /
// 2600 55 -> 43, 79 -> 62, 83 -> 68.)
// With the 224-row tile, 15 shapes at up to 30 row counts from 400 to 8000: it is the best at 62 of 352 points, by more than
// 2 % at 46 and 0.9 % on average (gate_up of Llama-3-8B at 400 / 892 rows 92 -> 84, 178 -> 165 us, 8192 x 8192 at 5200 495 -> 459);
// the choice is 0.48 % slower than the best of all six, more than 5 % at 11 points (8192 x 28672 at 400 - 512 rows up to 13 %,
// 10240 x 8192 at 6600 10 %).  All that was before the four-wave kernel's MFMAs had their present order, which made its rounds 2 - 4 %
// shorter and the ping-pong kernel's not.  Measured since, 18 shapes at 191 points of 390 - 8192 rows: the choice is 0.12 % slower than
// the best of all six, more than 5 % at 7 points (5120 x 13824 at 423 rows 23 %, 8192 x 28672 at 417 - 466 7 - 11 %, 6144 x 16384 at
// 418 - 506 8 %, all on the ping-pong kernel then; 2560 x 8192 at 777, 5120 x 5120 at 793 6 %).
struct W4Tile { int rows; float round, slope; };
constexpr W4Tile kW4Tiles[] = {{256, 1.f, .3f}, {224, .90f, .28f}, {192, .805f, .25f}, {160, .70f, .1f}, {128, .632f, 0.f}};
static bool big_plan(int M, int N, int K, bool pp_ok, Plan& p, float* us_out = nullptr) {
  const SkBuf* b = sk_buf();
  if (!b || !gemm_w4_ok(M, N, K, K, K)) return false;
  const float full = 6.f + 0.0207f * (float)K, C = (float)b->cus;
  const int nk = K / kBK;
  float best = 1e30f;
  p.variant = 3;
  p.BM = p.BN = 256;
  if (pp_ok) {
    const int T = (M + 255) / 256 * (N / 256), q = T / b->cus, r = T % b->cus, d = sk_choose_d(T, nk, b->cus, sk_min_half());
    // a grid of tails alone skips the last row tiles' empty 64-row quadrants
    const float live = q > 0 ? 1.f : .7f + .3f * (float)((M + 63) / 64) / (float)((M + 255) / 256 * 4);
    const float tail = d ? 1.1f * live * sk_tail_cost(r, nk, d) / (float)nk : r > 0 ? 1.f : 0.f;
    best = (13.5f + 0.0206f * (float)K) * ((float)q + tail);
  }
  for (const W4Tile& t : kW4Tiles) {
    if (t.rows < 256 && !g_half_tile) break;
    const long T = (long)((M + t.rows - 1) / t.rows) * (N / 256), q = T / b->cus, r = T % b->cus;
    // (From five whole rounds on the 224-row tile counts more.  By itself it does not need to: over 56 products of five
    // rounds and more the choice is 0.18 % slower than the best height with .90 throughout, 0.23 % with .925.  It is for steps: a
    // prompt of 3700 tokens of Llama-3-8B, seven rounds, took 8417 us with that tile in gate_up and 8336 with 256 rows, gate_up
    // itself 671 and 665, the kernels beside it 2.5 % longer; why was not measured.)
    const float one = full * (t.rows == 224 && q >= 5 ? .925f : t.round);
    float us = (float)q * one;
    const bool halves = r > 0 && gemm_w4_split_ok((int)T, nk);
    const float fill = (halves ? 2.f : 1.f) * (float)r / C, slope = q > 0 ? 0.f : t.slope;
    if (r > 0) us += (halves ? .5f : 1.f) * one * (1.f - slope * (1.f - fill));
    if (halves) us += q > 0 ? 15.f : 15.5f;
    if (us < best) {
      best = us;
      p.variant = t.rows == 256 ? 5 : 6;
      p.BM = t.rows;
    }
  }
  if (us_out) *us_out = best;
  return true;
}

static Plan plan(int M, int N, int K, bool grouped, int n_groups, int rows_per_group, bool stream = true) {
  Plan p{};
  p.variant = 0;
  const int mrows = grouped ? rows_per_group : M;
  // grouped (MoE): the ping-pong kernel from ~56 routed rows per expert.  Its 256 x 256 tile
  // streams each expert's weight panel once per n-tile and skips the MFMAs of empty 64-row
  // quadrants, so a half-empty expert tile costs less than the extra m-tiles (each a second walk
  // of the expert's weights) of the narrower kernels: Mixtral gate_up / down at 512 routed rows
  // 474 -> 370 / 266 -> 200 us, 1024 rows 692 -> 389 / 375 -> 208 us; 48 rows per expert equal
  // (scripts/bench_moe_decode.py, profiles/r05_moe_decode.md)
  constexpr int pp_group_min_rows = 56;
  if (!grouped && stream && g_dp[0] < 0 && mid_plan(M, N, K, p)) {
  } else if (grouped && mrows >= pp_group_min_rows && K % kBK == 0 && N % 256 == 0) {
    p.BM = 256; p.BN = 256; p.variant = 3;  // grouped ping-pong
  } else if (mrows <= 64 && !grouped && g_small_tile == 1) {
    // per shape (scripts/run137.sh, cold us at M = 16): wide N (gate_up) 64 columns with a
    // 6-deep ring (47.0 -> 44.8); narrow N 32 columns with an 8-deep ring at BM 16 (qkv
    // 15.3 -> 13.5, o / down unchanged): more weight bytes in flight per CU
    p.BM = mrows <= 16 ? 16 : mrows <= 32 ? 32 : 64;
    p.BN = 64;
    // (M 17-32 narrow projections on the 32-column 8-deep tiles of M <= 16: 1-2 % slower end to
    // end at batch 24 / 32, scripts/history INDEX run140)
    if (p.BM == 16) {
      const bool wide = N >= 16384;
      p.BN = wide ? 64 : 32;
      p.stages = wide ? (p.BM == 16 ? 6 : 0) : 8;
    } else if (p.BM == 64) {
      // M 33-64: narrow N on the 6-deep ring (run133: qkv 19.8 -> 18.4, down+norm 35.9 -> 32.0 us),
      // gate_up on a 4-deep one (run145: 48.2 -> 47.1 at M = 64, 6 stages lose: 50.4)
      p.stages = N < 16384 ? 6 : 4;
    }
  } else if (mrows <= 64 && !grouped && (g_small_tile == 32 || g_small_tile == 64)) {
    p.BM = mrows <= 16 ? 16 : mrows <= 32 ? 32 : 64;
    p.BN = g_small_tile;
  } else if (mrows <= 64) {
    p.BM = 64;
    p.BN = 64;
    // grouped (MoE at a few dozen rows per expert), narrow down projection: ring depth knob
    if (grouped && N < 16384) p.stages = g_grouped_small_stages;
    // grouped at <= 32 rows per expert (Mixtral batch 16-64): down on 32 x 64 tiles with a
    // 6-deep ring and ONE K range, gate_up on a 4-deep ring (scripts/bench_moe_decode.py, cold
    // expert weights, profiles/r05_moe_decode.md: down at 128 routed rows 172.4 -> 160.4 us,
    // 5.45 -> 5.86 TB/s; gate_up 318.2 -> 315.9)
    if (grouped && g_grouped_narrow && mrows <= 32) {
      if (N < 16384) { p.BM = 32; p.stages = 6; p.nosplit = true; }
      else p.stages = 4;
    }
  }
  else if (mrows <= 128) {
    // (96 and, below, 192 rows where the batch fits: a CU takes in less of A for the same weights; cold, 4096 x 4096 at 80 /
    // 176 rows 17.9 -> 16.7, 22.3 -> 21.1 us, 15 shapes of 1024 - 12544 columns and K 2048 - 8192 at 66 - 96 and 129 - 192 rows
    // 0.95 of the time on average, 0.91 - 1.001.  160 rows in four waves gained 1 %, 224 lost 10 %.)
    p.BM = !grouped && mrows <= 96 ? 96 : 128;
    p.BN = 64;
  }
  else if (mrows <= 256) {
    // 128 columns as soon as 64-column tiles would need a second round of the 256 CUs: 130-168 tiles
    // of 128 (N = 16640-21504) at M = 129-256 run 25-30 % faster than on 64-column tiles, 98 tiles
    // (N = 12544) 30 % slower
    constexpr int bn_min_tiles = 129;
    p.BM = 256;
    p.BN = ((N + 127) / 128 >= bn_min_tiles) ? 128 : 64;
    if (!grouped && p.BN == 64 && mrows <= 192) p.BM = 192;
  } else {
    const int big = g_big_variant;
    constexpr int big_min_m = 1024;
    p.BM = 256;
    p.BN = 128;
    // 128: o / down at 2049-2816 rows (the mixed steps of batch ~512: 144-176 tiles, no K-half
    // tail for the four-wave kernel) ran on the 256 x 128 kernel at 0.55x hipBLASLt; the
    // ping-pong kernel's stream-K tail takes them (o at M = 2560: 122 -> 88 us, down 394 -> 269;
    // scripts/history/r4_m2560.sh)
    constexpr int pp_min_tiles = 128;
    const long t256 = (long)((M + 255) / 256) * ((N + 255) / 256);
    // below pp_min_tiles the 256x256 grid leaves CUs idle, unless the stream-K tail can cut
    // every tile in two (T <= C / 2): o / down at M = 2040 (128 tiles)
    const bool pp_ok = K % kBK == 0 && (t256 >= pp_min_tiles || sk_halves_ok(t256, K / kBK));
    // variant 5: the four-wave kernel where its grid fills the chip: >= w4_min_tiles tiles, or
    // a tail it can cut in K-halves (o / down at M = 2048: 128 tiles -> 256 half-tiles); else
    // the ping-pong kernel with its general stream-K tail
    constexpr int w4_min_tiles = 192;
    const bool w4_fills = t256 >= w4_min_tiles || gemm_w4_split_ok((int)t256, K / kBK);
    // Wide projections take the large-M kernels from 512 rows: gate_up / lm_head at M = 512 /
    // 768 ran 127 -> 87 / 191 -> 153 us (8B) and 511 -> 404 us (70B gate_up), batch-512 serving
    // +5.3 %; narrow ones lose there (o / down at M = 512: 31 -> 48 / 66 -> 124 us) and keep the
    // 256 x 128 kernel (scripts/history/r4_bigminm.sh, r4_bigminm2.sh, r4_widemin.sh).
    // Below ~72 tiles of 256 x 256 (o / down at M = 512 - 1024: 32 - 64 tiles) the 256 x 128
    // kernel beats them at every M measured short of 2048 (o at M = 1024: 44.7 vs 48.6 us, down
    // 114.7 vs 129.5); from 72 tiles (qkv at M = 768, 70B qkv at 512) the large-M kernels win.
    constexpr int wide_min_m = 512;
    constexpr int mid_tiles = 72;
    // Fewer than 64 half-height tiles leave most CUs idle whatever the tile: the split-K tiles (variant 0).  So does
    // long K on a narrow N: fewer than 40 tiles of 256 rows (2048 x 8192 at M = 960 / 1000 47.3 us, the best of
    // big_plan's 59.3), and at up to 512 rows fewer than 72 (down at M = 400 / 512 70.9 / 72.8, the best 72.5 / 80).
    const bool narrow = K >= 8192 && (t256 < 40 || (M <= 512 && t256 < mid_tiles));
    const bool by_time = !grouped && big == 5 && (long)((M + 127) / 128) * (N / 256) >= 64 && !narrow && big_plan(M, N, K, pp_ok, p);
    const int big_from = t256 >= mid_tiles ? std::min(big_min_m, wide_min_m) : std::max(big_min_m, 2048);
    if (by_time) {
    } else if (big == 5 && !(mrows >= big_from && !grouped && w4_fills && gemm_w4_ok(M, N, K, K, K))) {
      if (mrows >= big_from && !grouped && pp_ok) { p.BN = 256; p.variant = 3; }
    } else if (big && mrows >= big_from && !grouped && (big < 3 || pp_ok)) {
      p.BN = 256;
      p.variant = big;
    }
    if (!grouped && big == 5 && !by_time) {
      // long-K narrow projections (down, K = 14336) at 40-71 tiles of 256 x 256 (M 640-1279):
      // the ping-pong kernel's stream-K tail spreads the few tiles' K over every CU (down at
      // M = 768: 105 -> 90 us, 1024: 118 -> 108; hipBLASLt 90 / 111)
      if (p.variant == 0 && K >= 8192 && t256 >= 40 && t256 < mid_tiles && K % kBK == 0 &&
          sk_halves_ok(t256, K / kBK)) {
        p.BN = 256;
        p.variant = 3;
      }
      // the half-height four-wave tile with its own K-half tail (t128 <= CUs / 2); below ~80 tiles the 256 x 128
      // split-K kernel wins (down at M = 512: 83.1 vs 67.6)
      const SkBuf* b = sk_buf();
      const long t128 = (long)((M + 127) / 128) * ((N + 255) / 256);
      if (g_half_tile && b && mrows >= 384 && K >= 8192 && t128 >= 80 && 2 * t128 <= b->cus &&
          (p.variant == 0 || p.variant == 3 || p.variant == 5) && gemm_w4_ok(M, N, K, K, K)) {
        p.BM = 128;
        p.BN = 256;
        p.variant = 6;
      }
    }
  }
  if (!grouped && g_dp[0] >= 0) {  // bench override (gemm_dense_plan)
    p.variant = g_dp[0];
    p.BM = p.variant == 0 || (p.variant == 6 && (g_dp[1] == 160 || g_dp[1] == 192 || g_dp[1] == 224)) ? g_dp[1] : p.variant == 6 ? 128 : 256;
    p.BN = p.variant == 0 ? g_dp[2] : 256;
    p.stages = g_dp[4];
  }
  if (grouped && g_gp[0] > 0) {  // bench override (gemm_grouped_plan)
    p.BM = g_gp[0];
    p.BN = g_gp[1];
    p.variant = (p.BM == 256 && p.BN == 256) ? 3 : 0;
    p.stages = g_gp[2] > 0 ? g_gp[2] : 0;
  }
  const int n_tiles = (N + p.BN - 1) / p.BN;
  const int real_m_tiles = (M + p.BM - 1) / p.BM;
  p.m_tiles = grouped ? real_m_tiles + n_groups : real_m_tiles;
  if (p.variant == 7) return p;
  p.splits = 1;
  p.k_chunk = K;
  const long tiles = (long)n_tiles * real_m_tiles;
  // run49: down -5..-15% at M 8-64.  The 16-row tiles (M 9-16) aim at 512 workgroups: batch 16
  // +5.6 / +6.0 % interleaved (scripts/r5_splittarget.sh, r5_splittarget2.sh), while 512 lost
  // 1.4-1.6 % at batch 24 / 32 (32-row tiles), 5 % at batch 64 and 4 % at 256
  const int split_target = p.BM <= 16 ? g_split_target : 256;
  constexpr int split_max_tiles = 160;
  if (!grouped && tiles < split_max_tiles && K >= 1024 && p.variant != 3 && p.variant < 5) {
    int s = (int)std::min<long>(8, std::max<long>(1, split_target / tiles));
    int kc = ((K / s + kBK - 1) / kBK) * kBK;
    p.splits = (K + kc - 1) / kc;
    p.k_chunk = kc;
  }
  if (!grouped && g_dp[0] == 0 && g_dp[3] >= 1) {
    const int kc = ((K / g_dp[3] + kBK - 1) / kBK) * kBK;
    p.splits = (K + kc - 1) / kc;
    p.k_chunk = kc;
  }
  return p;
}

template <int EPI, bool GROUPED>
static void launch_plan(const Plan& p, const uint16_t* A, int lda, const uint16_t* B, int ldb,
                        uint16_t* C, int ldc, float* ws, int M, int N, int K, const int* offsets,
                        int n_groups, hipStream_t st, const RopeEpi& re = RopeEpi{}) {
#define MLOP_GEMM(bm, bn, wm, wn, stages, prio)                                                   \
  run_cfg<bm, bn, wm, wn, EPI, GROUPED, stages, prio>(A, lda, B, ldb, C, ldc, ws, M, N, K,        \
                                                      p.splits, p.k_chunk, offsets, n_groups,     \
                                                      p.m_tiles, st, re)
  if constexpr (EPI == EPI_ROPE) {  // whole heads per staged chunk, no split-K (launch_gemm_rope)
    if (p.BN == 128) MLOP_GEMM(256, 128, 4, 2, 3, false);
    else if (!GROUPED && p.variant >= 5 && gemm_w4_ok(M, N, K, lda, ldb, ldc))
      run_w4(EPI, A, lda, B, ldb, C, ldc, M, N, K, st, re, p.BM);
    else if (!GROUPED && (p.variant == 3 || p.variant >= 5)) run_pp<EPI>(A, lda, B, ldb, C, ldc, M, N, K, st, re);
    else if (!GROUPED && p.variant == 2) MLOP_GEMM(256, 256, 2, 4, 2, true);
    else if (!GROUPED) MLOP_GEMM(256, 256, 2, 4, 2, false);
  } else {
    // weight-streaming tiles (M <= 128): a deeper LDS-DMA ring keeps more weight bytes in
    // flight per CU (3 stages x 16 KB per workgroup streamed gate_up at 4.7 TB/s at M = 64)
    const int sst = p.stages ? p.stages : g_small_stages;
    if (!GROUPED && p.variant == 7)
      launch_mid(EPI, p.BM, p.BN, A, lda, B, ldb, C, ldc, ws, M, N, K, p.splits, p.k_chunk, st, re);
    else if (!GROUPED && p.variant == 6 && p.splits == 1 && gemm_w4_ok(M, N, K, lda, ldb, ldc))
      run_w4(EPI, A, lda, B, ldb, C, ldc, M, N, K, st, re, p.BM);
    else if (!GROUPED && p.variant == 6) run_pp<EPI>(A, lda, B, ldb, C, ldc, M, N, K, st, re);
    else if (p.BM == 16 && p.BN == 32 && sst >= 8) MLOP_GEMM(16, 32, 1, 2, 8, false);
    else if (p.BM == 16 && p.BN == 32 && sst >= 6) MLOP_GEMM(16, 32, 1, 2, 6, false);
    else if (p.BM == 16 && p.BN == 32) MLOP_GEMM(16, 32, 1, 2, 4, false);
    else if (p.BM == 16 && p.BN == 64 && sst >= 8) MLOP_GEMM(16, 64, 1, 2, 8, false);
    else if (p.BM == 16 && p.BN == 64 && sst >= 6) MLOP_GEMM(16, 64, 1, 2, 6, false);
    else if (p.BM == 16 && p.BN == 64) MLOP_GEMM(16, 64, 1, 2, 4, false);
    else if (p.BM == 32 && p.BN == 32 && sst >= 8) MLOP_GEMM(32, 32, 1, 2, 8, false);
    else if (p.BM == 32 && p.BN == 32) MLOP_GEMM(32, 32, 1, 2, 4, false);
    else if (p.BM == 32 && p.BN == 64 && sst >= 6) MLOP_GEMM(32, 64, 1, 4, 6, false);
    else if (p.BM == 32 && p.BN == 64) MLOP_GEMM(32, 64, 1, 4, 4, false);
    else if (p.BM == 64 && p.BN == 32) MLOP_GEMM(64, 32, 1, 2, 4, false);
    else if (p.BM == 64 && p.BN == 64 && sst >= 6) MLOP_GEMM(64, 64, 1, 4, 6, false);
    else if (p.BM == 64 && p.BN == 64 && sst == 4) MLOP_GEMM(64, 64, 1, 4, 4, false);
    else if (p.BM == 64) MLOP_GEMM(64, 64, 1, 4, 3, false);
    else if (!GROUPED && p.BM == 96) MLOP_GEMM(96, 64, 2, 2, 3, false);
    else if (!GROUPED && p.BM == 192 && p.BN == 64) MLOP_GEMM(192, 64, 4, 2, 3, false);
    else if (p.BM == 128 && g_small_stages >= 5) MLOP_GEMM(128, 64, 2, 2, 5, false);
    else if (p.BM == 128) MLOP_GEMM(128, 64, 2, 2, 3, false);
    else if (p.BN == 64) MLOP_GEMM(256, 64, 4, 2, 3, false);
    else if (p.BN == 128) MLOP_GEMM(256, 128, 4, 2, 3, false);
    else if (GROUPED && p.variant == 5)
      run_w4_grouped(EPI, A, lda, B, ldb, C, ldc, M, N, K, st, re, offsets, n_groups);
    else if (GROUPED && p.variant == 3)
      run_pp<EPI, true>(A, lda, B, ldb, C, ldc, M, N, K, st, re, offsets, n_groups);
    else if (!GROUPED && p.variant == 5 && p.splits == 1 && gemm_w4_ok(M, N, K, lda, ldb, ldc))
      run_w4(EPI, A, lda, B, ldb, C, ldc, M, N, K, st, re);
    else if (!GROUPED && (p.variant == 3 || p.variant == 5) && p.splits == 1)
      run_pp<EPI>(A, lda, B, ldb, C, ldc, M, N, K, st, re);
    else if (!GROUPED && p.variant == 2) MLOP_GEMM(256, 256, 2, 4, 2, true);
    else if (!GROUPED) MLOP_GEMM(256, 256, 2, 4, 2, false);
  }
#undef MLOP_GEMM
}

// stream-K workgroups a plain launch of this shape would add (0: data-parallel grid only)
int gemm_sk_workgroups(int M, int N, int K) {
  if (M <= 0 || gemv_takes(M, N, K, EPI_NONE)) return 0;
  const Plan p = plan(M, N, K, false, 0, 0);
  if (p.variant != 3 || p.BN != 256 || p.splits != 1) return 0;
  int n_sk = 0;
  sk_plan(((M + 255) / 256) * ((N + 255) / 256), K / kBK, n_sk);
  return n_sk;
}

// EPI_ROPE: the plain (no split-K) plan must stage whole heads: BN >= 128, i.e. M > 256.
// Small M whose plan splits K: the slabs go to the stream-K scratch and the split-K reduce is
// fused into the RoPE + cache kernel (one launch instead of reduce + rope_cache).
static bool rope_slabs_ok(const Plan& p, int M, int N) {
  const SkBuf* b = sk_buf();
  return p.splits > 1 && (p.variant == 7 || (p.variant != 3 && p.variant < 5)) && b != nullptr &&
         (size_t)p.splits * M * N <= (size_t)2 * kSkMaxWg * 256 * 256;
}

// Small-M QKV: K split even where the plain plan keeps one K range (M <= 16: 192 tiles of 16 x
// 32): the slabs' reduce rides in the RoPE + cache kernel that runs anyway, so a second K range
// costs one fp32 slab and doubles the workgroups streaming the weights (gemm_rope_split op:
// the K ranges, 1 = the plain plan).  Interleaved, scripts/r5_ropesplitk.sh: batch 16 +1.9 %,
// batch 12 +3.0 % (4 ranges: +2.2 / +2.6 %)
static int g_rope_split_k = 2;
int gemm_rope_split(int set) {
  if (set >= 1) g_rope_split_k = set;
  return g_rope_split_k;
}

// The weight stream of gemm_mid.hip has all tasks of this product in flight at once, each over the whole K.
static bool mid_one_round(int M, int N, int K) {
  Plan p{};
  return mid_plan(M, N, K, p) && p.splits == 1 && (N + p.BN - 1) / p.BN <= kCus;
}

// The weight-streaming kernel (gemm_ws.hip) has this product: where its rule says so, and above the GEMV's rows no switch
// asks for a plan or one of the small tiles.  From 9 rows on not where the weight stream's tasks make one round and its own
// workgroups (of 32 rows there) leave one unfilled: 28672 x 4096 / 8192 at 16 rows 39.7 / 76.7 us against 37.3 / 73.7, 30016 x
// 5120 54.1 / 48.4, 50304 x 4096 67.7 / 64.6; 24576 and 65536 columns, whole rounds, 0.92 - 1.02 of the weight stream.
bool gemm_on_ws(int M, int N, int K, int epi) {
  if (g_dp[0] >= 0 || (M > gemv_chain_max_m() && g_small_tile != 1)) return false;
  if (M > 8 && N % (32 * kCus) && mid_one_round(M, N, K)) return false;
  return ws_prefer(M, N, K, epi);
}

static Plan rope_plan(int M, int N, int K) {
  Plan p = plan(M, N, K, false, 0, 0);
  if (p.variant == 7 && p.splits == 1) p = plan(M, N, K, false, 0, 0, false);  // no slabs, and no RoPE epilogue
  if (g_rope_split_k > 1 && p.splits == 1 && p.variant == 0 && p.BM <= 64 && K >= 2048) {
    const int kc = ((K / g_rope_split_k + kBK - 1) / kBK) * kBK;
    p.splits = (K + kc - 1) / kc;
    p.k_chunk = kc;
  }
  return p;
}

// plans whose kernel has the RoPE epilogue (whole heads per tile)
static bool rope_tiles(const Plan& p) { return p.variant != 7 && (p.BM == 256 || p.variant == 6) && p.BN >= 128; }

bool gemm_rope_supported(int M, int N, int K) {
  if (M <= 0 || N % 128 || K % kBK) return false;
  if (gemv_takes(M, N, K, EPI_ROPE) || gemm_on_ws(M, N, K, EPI_ROPE)) return true;  // decode: gemv.hip, gemm_ws.hip
  const Plan p = rope_plan(M, N, K);
  return rope_tiles(p) || rope_slabs_ok(p, M, N);
}

bool launch_gemm_rope(const void* A, int lda, const void* B, int M, int N, int K, const RopeEpi& re,
                      hipStream_t st) {
  if (M == 0) return true;
  if (!gemm_rope_supported(M, N, K)) return false;
  if (gemm_on_ws(M, N, K, EPI_ROPE) && ws_rows_ok(A, lda, M, K)) {  // up to 32 rows: the weight-streaming MFMA kernel
    launch_ws(A, lda, B, K, nullptr, 0, M, N, K, EPI_ROPE, false, re, 0.f, st);
    return true;
  }
  if (gemv_takes(M, N, K, EPI_ROPE) && lda % 8 == 0) {
    launch_gemv_rope(A, lda, B, M, N, K, re, st);
    return true;
  }
  Plan p = rope_plan(M, N, K);
  if (!rope_tiles(p)) {  // small M: split-K slabs + fused reduce / RoPE / cache
    if (!rope_slabs_ok(p, M, N)) return false;  // (supported for the weight-streaming kernel's sake)
    float* ws = sk_buf()->ws;
    launch_plan<EPI_NONE, false>(p, (const uint16_t*)A, lda, (const uint16_t*)B, K, nullptr, N, ws,
                                 M, N, K, nullptr, 0, st);
    launch_rope_cache_slabs(re, ws, p.splits, M, N, st);
    return true;
  }
  p.splits = 1;
  p.k_chunk = K;
  launch_plan<EPI_ROPE, false>(p, (const uint16_t*)A, lda, (const uint16_t*)B, K, nullptr, 0, nullptr,
                               M, N, K, nullptr, 0, st, re);
  return true;
}

// The large-M decoder's norm chain: O / down add into the residual and leave per-row sums of
// squares (W4_ADD_SS), gate_up / QKV scale their rows by the RMSNorm factor (W4_RS), so the
// add + RMSNorm passes over [M, H] disappear (norm weights folded into the consumer weights).
// Everything launch_w4_chain needs, so the caller decides the chain ONCE per forward (before the
// first in-place residual update) and never meets a refusal mid-layer: the shape on the
// four-wave kernel, the stream-K scratch that holds the band tickets reserved, and one ticket
// per band of BM rows.
// ``any``: also where another kernel is the faster choice for the product, on the best four-wave height.  A decode graph
// that stands in for one of more rows keeps that one's chain so (ops.norm_chain_ok ``like``).  Llama-3-8B widths, 6 layers:
// 700 sequences 4143 -> 4172 us and 0.0250 -> 0.0234 from 64 bits, 600 / 760 / 850 / 900 3773 -> 3800, 4045 -> 4065, 4489 ->
// 4490, 4440 -> 4434 (the norm passes that go pay for the slower down); three layers of the 70B at 300 rows 2653 -> 2708.
static bool w4_chain_plan(int M, int N, int K, bool any, Plan& p) {
  if (M <= 0 || gemv_takes(M, N, K, EPI_NONE) || gemv_takes(M, N, K, EPI_ROPE)) return false;
  int cus = 0;
  if (!gemm_sk_available(&cus) || cus <= 0) return false;
  p = plan(M, N, K, false, 0, 0);
  if (any && p.variant != 5 && p.variant != 6) {
    p = Plan{};
    p.splits = 1;
    if (!big_plan(M, N, K, false, p)) return false;
  }
  return (p.variant == 5 || p.variant == 6) && p.splits == 1 && p.BN == 256 && (M + p.BM - 1) / p.BM <= kSkMaxWg &&
         gemm_w4_ok(M, N, K, K, K, N);
}

bool w4_chain_ok(int M, int N, int K, bool any) {
  Plan p{};
  return w4_chain_plan(M, N, K, any, p);
}

bool launch_w4_chain(int epi, const void* A, int lda, const void* B, void* C, int ldc, int M, int N, int K,
                     const RopeEpi& re, hipStream_t st, bool any) {
  if (M == 0) return true;
  Plan p{};
  if (!w4_chain_plan(M, N, K, any, p) || !gemm_w4_ok(M, N, K, lda, K, ldc)) return false;
  if (!run_w4(epi, (const uint16_t*)A, lda, (const uint16_t*)B, K, (uint16_t*)C, ldc, M, N, K, st, re, p.BM)) return false;
  return true;
}

// Mid-M norm chain (rows in (decode_chain_max_m, 64], TP = 1): the decoder layer's two add +
// RMSNorm launches (splitk_add_rmsnorm) fold into the planner's small-tile GEMMs.  O / down
// (epi 0) split K and the tile's last split adds into the residual and leaves the row sums of
// squares (mid_chain_finish); gate_up (epi 1, one K range) scales its accumulator rows by the
// RMSNorm factor in its SiLU epilogue; QKV + RoPE (epi 3) takes the factor in the split-K slab
// reduce of the RoPE + cache kernel, or in the weight-streaming kernel's row-scale prologue at up
// to 32 rows (which computes it from the rows it streams).
// gemm_mid_chain op: 0 off (default), 1 on (sc1 hand-off), 2 on (acquire hand-off).  Off by
// default: the in-kernel finish adds ~3.5 us to each O / down call (two ticket round trips,
// write-through partials, the band's row totals) against the ~5 us splitk_add_rmsnorm launch it
// replaces, and the row scale costs gate_up ~0.8 us; interleaved on one box, batch 16 -1 % /
// -3 % and batch 64 -2.6 % / -3.7 % (sc1 / acquire); without the band step (a timing probe,
// numerics off) batch 16 +2-3 % and batch 64 -0.6 % (profiles/r06_mid_chain.md).
static int g_mid_chain = 0;
int gemm_mid_chain(int set) {
  if (set >= 0) g_mid_chain = set;
  return g_mid_chain;
}

bool mid_chain_ok(int M, int N, int K, int epi) {
  if (!g_mid_chain || M <= decode_chain_max_m() || M > 64 || K % kBK || N % 128) return false;
  int cus = 0;
  if (!gemm_sk_available(&cus)) return false;
  if (epi == EPI_ROPE) {
    if (gemm_on_ws(M, N, K, EPI_ROPE)) return true;  // (whole steps of 128 k are part of its rule)
    const Plan p = rope_plan(M, N, K);
    return !rope_tiles(p) && rope_slabs_ok(p, M, N);
  }
  const Plan p = plan(M, N, K, false, 0, 0);
  if (epi == EPI_SILU_MUL && p.variant == 7) return p.splits == 1;
  if (p.variant != 0 || p.BM > 64 || N % p.BN) return false;
  if (epi == EPI_SILU_MUL) return p.splits == 1;
  if (epi != EPI_NONE || p.splits < 2) return false;
  const long gx = N / p.BN, gy = (M + p.BM - 1) / p.BM;
  return gx * gy + gy <= kSkMaxWg &&
         (size_t)p.splits * M * N + (size_t)M * gx <= (size_t)2 * kSkMaxWg * 256 * 256;
}

// residual [M, N] += A . B^T in place and ss_tot [M] <- the new rows' sums of squares (epi 0)
bool launch_mid_res_ss(const void* A, int lda, const void* B, void* residual, int ldr, int M, int N, int K,
                       float* ss_tot, hipStream_t st) {
  if (M == 0) return true;
  if (!mid_chain_ok(M, N, K, EPI_NONE)) return false;
  float* ws = nullptr;
  int* cnt = nullptr;
  int cus = 0;
  if (!gemm_sk_scratch(&ws, &cnt, &cus)) return false;
  const Plan p = plan(M, N, K, false, 0, 0);
  RopeEpi re{};
  re.ss_cnt = cnt;
  re.ss_tot = ss_tot;
  re.mid_acq = g_mid_chain == 2;
  launch_plan<EPI_NONE, false>(p, (const uint16_t*)A, lda, (const uint16_t*)B, K, (uint16_t*)residual, ldr, ws, M,
                               N, K, nullptr, 0, st, re);
  return true;
}

// out = SiLU-mul(diag(rsqrt(ss_tot / K + eps)) . A . B^T) (epi 1, gate_up)
bool launch_mid_rs(const void* A, int lda, const void* B, void* out, int ldo, int M, int N, int K,
                   const float* ss_tot, float eps, hipStream_t st) {
  if (M == 0) return true;
  if (!mid_chain_ok(M, N, K, EPI_SILU_MUL)) return false;
  const Plan p = plan(M, N, K, false, 0, 0);
  RopeEpi re{};
  re.ss_in = ss_tot;
  re.ss_inv_k = 1.f / (float)K;
  re.ss_eps = eps;
  launch_plan<EPI_SILU_MUL, false>(p, (const uint16_t*)A, lda, (const uint16_t*)B, K, (uint16_t*)out, ldo, nullptr,
                                   M, N, K, nullptr, 0, st, re);
  return true;
}

// gate_up of the decode norm chain on the weight stream: out = SiLU-mul(diag(rsqrt(mean(a^2) + eps)) . A . B^T), the rows'
// factors from the rows themselves
bool mid_self_ok(int M, int N, int K) {
  Plan p{};
  return N % 32 == 0 && M <= 64 && g_dp[0] < 0 && mid_plan(M, N, K, p) && p.splits == 1;
}

void launch_mid_self(const void* A, int lda, const void* B, void* out, int ldo, int M, int N, int K, float eps, hipStream_t st) {
  Plan p{};
  mid_plan(M, N, K, p);
  RopeEpi re{};
  re.ss_inv_k = 1.f / (float)K;
  re.ss_eps = eps;
  launch_mid(2, p.BM, p.BN, (const uint16_t*)A, lda, (const uint16_t*)B, K, (uint16_t*)out, ldo, nullptr, M, N, K, 1, K, st, re);
}

static void few_rows_w4(int M, int N, int K, int epi, Plan& p);

void gemm_plan(int M, int N, int K, int epi, int out[5]) {
  if (epi_act(epi)) epi = EPI_NONE;
  if (gemm_on_ws(M, N, K, epi)) {
    out[0] = -2, out[1] = out[2] = 0, out[3] = 1, out[4] = gemm_weights_nt(1);
    return;
  }
  if (gemv_takes(M, N, K, epi)) {
    out[0] = -1, out[1] = out[2] = out[4] = 0, out[3] = 1;
    return;
  }
  Plan p = plan(M, N, K, false, 0, 0);
  few_rows_w4(M, N, K, epi, p);
  out[0] = p.variant, out[1] = p.BM, out[2] = p.BN, out[3] = p.splits;
  out[4] = (p.variant == 0 || p.variant == 7) && gemm_weights_nt((M + p.BM - 1) / p.BM);
}

// Products of 129 - 256 rows in one K range, gate_up and output heads (the plain ones of more than 32768 columns): the four-wave
// kernel where it is estimated to be 3 % faster than the weight stream, or than the 256 x 128 tiles that have 130 - 168 tiles of 128
// columns.  The weight stream's workgroup takes in the whole batch beside its 128 or 256 columns, and a grid of 1.1 rounds takes
// two; the four-wave kernel has 128-row tiles, two for a column, or one of the batch's height.  Not where it would cut the last tiles into
// K-halves (0.82 - 0.87 of the time at 18432 - 20480 and 65536 - 69888 columns): up to 256 rows no product but those with RoPE uses the
// scratch of the hand-over, so one may run beside another stream's that does (captured decode steps of Dibedra: a layer's experts beside
// its dense products).  us, cold weights, stream -> four-wave: gate_up 28672 x 4096, which changes over at 225 rows, at 225 / 240 / 256 72 -> 62,
// 74 -> 63, 74 -> 64; 57344 x 8192 at the same 235 -> 220, 234 -> 227, 233 -> 227, head 128256 x 4096 252 -> 215, 261 -> 225, 259 -> 229; 36864 x
// 4096 at 150 / 200 93 -> 76, 115 -> 82, 20480 x 4096 63 -> 54, 64 -> 57.  Steps of six Llama-3-8B layers: a prompt of 250
// tokens 1273 -> 1257, eight of 30 1225 -> 1202.
// Estimates in us fitted to 720 points (15 widths of 8192 - 128256, K 2048 - 8192, 135 - 256 rows, cold weights), 5 and 6 % off in the
// mean.  Weight stream of bm rows, g the share of the CUs in a round: 10.1 + a K-step's .117 + .00189 bm + .00121 bm g + .081 g with 128
// columns, 11.6 + -.261 + .00447 bm + .00168 bm g + .588 g with 256; the 256 x 128 tiles 8 + .0137 K.  Four-wave: 2.5 + rounds of .0227 K, .0262 where
// its tiles walk K in step, times the height's share, the last one less by .16 of its empty part, or 5.5 + the weights at 5 TB/s: the sixth
// root of the sum of their sixth powers, a maximum that is 12 % over where the two are level, as it is where a product waits for both.
// Of 325 products, these and drawn ones of 16384 - 160000 columns, the 153 chosen take 0.857 of the time, 4 of them 1.03 - 1.10 (88832 x 1280 at
// 224 rows 79 -> 87, 97024 x 2560 at 223 135 -> 148, 57344 x 4096 at 256 123 -> 126).  Left on the stream though the other is faster: heads at 193 - 224
// rows (128256 x 4096 at 197 / 224 in another session 241 / 249 and 210 / 218; the estimates say 230 and 223), and plain products up to 32768 columns,
// which the rule was not drawn for (32768 x 4096 at 256 rows 78 and 65).
static void few_rows_w4(int M, int N, int K, int epi, Plan& p) {
  if (M <= 128 || M > 256 || K < 1024 || g_dp[0] >= 0 || p.splits > 1 || (epi != EPI_SILU_MUL && N <= 32768) || !gemm_w4_ok(M, N, K, K, K)) return;
  const int nk = K / kBK;
  const float C = (float)kCus, k = (float)K, bm = (float)((M + 31) / 32 * 32);
  float now;
  if (p.variant == 7) {
    const int t = (N + p.BN - 1) / p.BN, rounds = (t + kCus - 1) / kCus;
    const float g = std::min((float)t / C, 1.f);
    const float step = p.BN == 128 ? .117f + .00189f * bm + .00121f * bm * g + .081f * g : -.261f + .00447f * bm + .00168f * bm * g + .588f * g;
    now = (p.BN == 128 ? 10.1f : 11.6f) + (float)(nk * rounds) * step;
  } else if (p.variant == 0 && p.BN == 128) {
    now = 8.f + .0137f * k;
  } else {
    return;
  }
  float best = now / 1.03f;
  int rows = 0;
  for (const W4Tile& t : kW4Tiles) {
    if (t.rows < 256 && !g_half_tile) break;
    if (t.rows != 128 && (t.rows < M || t.rows >= M + 32)) continue;
    const int T = (M + t.rows - 1) / t.rows * (N / 256), q = T / kCus, r = T % kCus;
    if ((r > 0 && 2 * r <= kCus && nk % 2 == 0) || gemm_w4_split_ok(T, nk)) continue;
    const float one = (gemm_w4_in_step(M, N, K, t.rows) ? .0262f : .0227f) * k * t.round;
    float us = 2.5f + (float)q * one;
    if (r > 0) us += one * (1.f - .16f * (1.f - (float)r / C));
    const float weights = 5.5f + (float)N * k * 2e-6f / 5.f;
    us = std::pow(std::pow(us, 6.f) + std::pow(weights, 6.f), 1.f / 6.f);
    if (us < best) best = us, rows = t.rows;
  }
  if (rows == 0) return;
  p = Plan{};
  p.BM = rows, p.BN = 256, p.splits = 1, p.k_chunk = K, p.variant = rows == 256 ? 5 : 6, p.m_tiles = (M + rows - 1) / rows;
}

// GEMM + residual add + RMSNorm above 256 rows: the four-wave kernel over K in 2 - 8 ranges, one workgroup per (tile, range), its
// fp32 slabs summed by the pass that adds and norms anyway.  A grid of few tiles fills the CUs with whole tiles so: what the
// K-half hand-over and the stream-K tail send through one workgroup of a tile (a CU takes in 50 GB/s of what is not in its L2) is read by
// all CUs, and the 128-row tiles, which halves need to fill the chip and whose loop waits for its loads (48 KB a K-tile in
// 0.73 us, of its 0.78), give way to taller ones.  us, GEMM + add + norm as it was -> so: 4096 x 14336 at 390 / 600 / 892 rows 71 -> 57, 100 -> 72,
// 113 -> 91, 4096 x 4096 at 390 / 640 38.4 -> 31, 42 -> 36, 8192 x 8192 at 330 80 -> 62, 8192 x 28672 at 390 217 -> 176.  (Slabs stored
// non-temporal: 101 instead of 91.)
// By estimated time: a range takes what big_plan says of its K, 4.5 us for 4-byte stores; the pass 3.1 us and its bytes at 8.3
// TB/s, the plain pass 3 and 6.  14 shapes and 250 drawn ones at 257 - 3000 rows: the choice of tile and ranges is 1 % off the best.
// Up to 320 rows the weight stream is the faster of small matrices (257 x 4096 x 7168 33.1 us, slabs 36.1; 270 x 5120 x 13824
// 68.8 and 60.9), so it is of narrow ones with K in 8 ranges (334 x 1536 x
// 19008, 144 workgroups, 41.5 and 45.6); K below 1536 is too short to cut (266 x 1024 x 1088 14.9 and 19.1), as are grids of less
// than 96 workgroups (335 x 768 x 1984 16.7 and 19.3).
static bool slab_plan(int M, int N, int K, int& bm, int& splits) {
  if (g_slab[0] > 0) {  // bench override (gemm_dense_plan)
    bm = g_slab[0];
    splits = g_slab[1];
    return splits > 1;
  }
  const SkBuf* b = sk_buf();
  if (!b || g_dp[0] >= 0 || M <= 256 || K < 1536 || !gemm_w4_ok(M, N, K, K, K) || (long)M * N * 4 >= (1l << 31)) return false;
  if (M < 320 && (long)N * K < 60l << 20) return false;
  const int nk = K / kBK;
  const float C = (float)b->cus, mn = (float)M * (float)N * 1e-6f;
  float best = 1e30f;
  int wgs = 0;
  for (const W4Tile& t : kW4Tiles) {
    const int T = (M + t.rows - 1) / t.rows * (N / 256);
    for (int s = 2; s <= kMaxSplits && s * T <= b->cus && nk / s >= 6; ++s) {
      if (s * T < 96) continue;
      const float one = (6.f + 0.0207f * (float)((nk + s - 1) / s * kBK)) * t.round;
      const float us = one * (1.f - t.slope * (1.f - (float)(T * s) / C)) + 4.5f + 3.1f + mn * (4.f * (float)s + 6.f) / 8.3f;
      if (us < best) best = us, bm = t.rows, splits = s, wgs = s * T;
    }
  }
  if (wgs == 0) return false;
  Plan p = plan(M, N, K, false, 0, 0);
  if (p.variant == 7) return wgs >= 160;
  if (p.splits > 1) return true;
  float us = 0.f;
  return big_plan(M, N, K, true, p, &us) && best * 1.03f + (K < 2600 ? 2.f : 0.f) < us + 3.f + mn * 8.f / 6.f;
}

// fp32 slabs of the K ranges: of a plain product, and (add_norm) of one with the residual add + RMSNorm behind it, for which 0
// also says that there is no such form; the weight-streaming kernel's has none, but A's rows may not suit it
long gemm_workspace_floats(int M, int N, int K, int epi, bool add_norm) {
  if (epi_act(epi)) epi = EPI_NONE;
  if (int bm, s; add_norm && slab_plan(M, N, K, bm, s)) return (long)s * M * N;
  if (gemv_takes(M, N, K, epi) || (!add_norm && gemm_on_ws(M, N, K, epi))) return 0;
  const Plan p = plan(M, N, K, false, 0, 0);
  return p.splits > 1 ? (long)p.splits * M * N : 0;
}

void launch_gemm(const void* A, int lda, const void* B, int ldb, void* C, int ldc, float* ws,
                 long ws_floats, int M, int N, int K, int epi, hipStream_t st, float p0, float p1, int act_n0) {
  if (M == 0) return;
  RopeEpi re{};
  re.act_n0 = act_n0;
  re.p0 = p0;
  re.p1 = p1;
  re.act = epi_act(epi);
  const int epi0 = epi;
  if (re.act) epi = EPI_NONE;
  if (gemm_on_ws(M, N, K, epi) && ws_rows_ok(A, lda, M, K) && ldb % 8 == 0) {
    launch_ws(A, lda, B, ldb, C, ldc, M, N, K, epi, false, re, 0.f, st);
    return;
  }
  if (gemv_takes(M, N, K, epi) && lda % 8 == 0 && ldb % 8 == 0) {
    launch_gemv(A, lda, B, ldb, C, ldc, M, N, K, epi0, st, p0, p1, act_n0);
    return;
  }
  Plan p = plan(M, N, K, false, 0, 0);
  if (gemm_w4_ok(M, N, K, lda, ldb, ldc) && ldc % 8 == 0 && (uintptr_t)C % 16 == 0) few_rows_w4(M, N, K, epi, p);
  if (p.splits > 1 && (long)p.splits * M * N > ws_floats) { p.splits = 1; p.k_chunk = K; }
  if (epi == EPI_NONE)
    launch_plan<EPI_NONE, false>(p, (const uint16_t*)A, lda, (const uint16_t*)B, ldb, (uint16_t*)C,
                                 ldc, ws, M, N, K, nullptr, 0, st, re);
  else
    launch_plan<EPI_SILU_MUL, false>(p, (const uint16_t*)A, lda, (const uint16_t*)B, ldb,
                                     (uint16_t*)C, ldc, ws, M, N, K, nullptr, 0, st, re);
  if (p.splits > 1) {
    const int outw = epi == EPI_NONE ? N : N / 2;
    const long total = (long)M * (outw / 8);
    const int g = (int)std::min<long>((total + 255) / 256, 4096);
    if (epi == EPI_NONE)
      splitk_reduce_kernel<EPI_NONE><<<g, 256, 0, st>>>((uint16_t*)C, ldc, ws, M, N, p.splits, re);
    else
      splitk_reduce_kernel<EPI_SILU_MUL><<<g, 256, 0, st>>>((uint16_t*)C, ldc, ws, M, N, p.splits, re);
  }
}

// y = A.B^T; residual += y; out = rmsnorm(residual) * w.  Returns false (nothing
// launched) when the shape does not take the split-K path: the caller then runs
// gemm + add_rmsnorm.
bool launch_gemm_add_rmsnorm(const void* A, int lda, const void* B, void* out, void* residual,
                             const void* w, float eps, float* ws, long ws_floats, int M, int N,
                             int K, hipStream_t st) {
  if (M == 0) return true;
  if (gemv_takes(M, N, K, EPI_NONE)) return false;  // decode sizes: GEMV + add_rmsnorm (or the norm chain)
  if (gemm_on_ws(M, N, K, 5) && ws_rows_ok(A, lda, M, K)) {
    // up to 16 rows: the weight-streaming MFMA kernel adds into the residual
    // in place (bf16(res + bf16(y)), norm.hip's rounding), then one RMSNorm pass
    launch_ws(A, lda, B, K, residual, N, M, N, K, 5, false, RopeEpi{}, 0.f, st);
    launch_rmsnorm(out, residual, w, eps, M, N, st);
    return true;
  }
  int splits, bm;
  if (slab_plan(M, N, K, bm, splits) && (long)splits * M * N <= ws_floats && gemm_w4_ok(M, N, K, lda, K) &&
      K / kBK / splits >= 3 && (long)M * N * 4 < (1l << 31)) {
    run_w4_slab((const uint16_t*)A, lda, (const uint16_t*)B, K, ws, M, N, K, splits, bm, st);
  } else {
    const Plan p = plan(M, N, K, false, 0, 0);
    if (p.splits <= 1 || p.splits > kMaxSplits || (long)p.splits * M * N > ws_floats || N % 8) return false;
    launch_plan<EPI_NONE, false>(p, (const uint16_t*)A, lda, (const uint16_t*)B, K, nullptr, N, ws,
                                 M, N, K, nullptr, 0, st);
    splits = p.splits;
  }
  const int nvec = N / 8;
  int vpt = 1;
  while (vpt < 8 && nvec / vpt > 512) vpt <<= 1;
  const int threads = ((nvec / vpt + 63) / 64) * 64;
  auto* o = (uint16_t*)out;
  auto* r = (uint16_t*)residual;
  auto* wv = (const uint16_t*)w;
  switch (vpt) {
    case 1: splitk_add_rmsnorm_kernel<1><<<M, threads, 0, st>>>(o, r, ws, wv, eps, M, N, splits); break;
    case 2: splitk_add_rmsnorm_kernel<2><<<M, threads, 0, st>>>(o, r, ws, wv, eps, M, N, splits); break;
    case 4: splitk_add_rmsnorm_kernel<4><<<M, threads, 0, st>>>(o, r, ws, wv, eps, M, N, splits); break;
    default: splitk_add_rmsnorm_kernel<8><<<M, threads, 0, st>>>(o, r, ws, wv, eps, M, N, splits); break;
  }
  return true;
}

// The experts' products: gemm_kernel's tiles, the ping-pong kernel (variant 3) or the four-wave kernel (5).  The latter
// where tiles of 224 rows (one per expert up to 256) make two and a half rounds or more; with fewer, stream-K's even split of the tail wins (down of 8
// experts at 200 / 407 / 700 rows each on average 200 / 341 / 547 us against 222 / 361 / 586; at 1024 805 against 770).
// gate_up of 8 experts, random tokens, ping-pong -> four-wave: 300 / 368 / 407 / 440 / 512 / 700 / 1024 rows each 651 -> 537,
// 681 -> 573, 755 -> 684, 782 -> 733, 921 -> 813, 1130 -> 1000, 1640 -> 1435 us; of 8 experts of half the width at 256 / 300 /
// 407 rows 295 -> 267, 345 -> 280, 380 -> 345, of 4 at 512 479 -> 417.  (Without the 224-row tile the ping-pong kernel had 368
// - 440 rows: two 256-row tiles of which a fifth is empty, and three lower ones.)  Not at 160 - 240 rows of up to 8 experts,
// one tile each: there the weights' latency bounds both, and the ping-pong kernel skips a tile's empty 64-row quadrants (200
// rows 394 us against 420; 16 x 12800 x 4096 378 against 355, 32 x 8192 x 2048 290 against 254); at 64 - 140 rows they are level.
// Measured in one process on six shapes (those, 8 experts of half the width, 4 of the same, 64 x 2816 x 2048), 16 row counts,
// equal experts, random tokens, experts 0.6 - 1.4 of the mean and one with two fifths: where the four-wave kernel is chosen it
// is 19 % faster than the ping-pong kernel on average, slower at 7 of 320 points and by 8 % at worst (8 x 28672 x 4096 at 240 -
// 256 equal rows by 3 - 4 % there, by 11 % in a run before).
static Plan grouped_plan(int M, int N, int K, int n_groups, int max_rows, int a_n) {
  Plan p = plan(M, N, K, true, n_groups, max_rows);
  const bool quadrants = max_rows >= 160 && max_rows < 240 && n_groups <= 8;
  const int tiles = max_rows <= 256 ? 1 : (max_rows + 223) / 224;
  if (p.variant == 3 && g_gp[0] <= 0 && !quadrants) {
    const SkBuf* b = sk_buf();
    if (b && 2l * n_groups * tiles * (N / 256) >= 5l * b->cus && gemm_w4_grouped_ok(M, N, K, n_groups, a_n))
      p.variant = 5;
  }
  return p;
}

int gemm_grouped_variant(int M, int N, int K, int n_groups, int max_rows, int a_n) {
  return grouped_plan(M, N, K, n_groups, max_rows, a_n).variant;
}

void launch_grouped_gemm(const void* A, const void* B, void* C, const int* offsets, int n_groups,
                         int M, int N, int K, int max_rows, int epi, hipStream_t st, const int* a_rows,
                         float** defer_ws, int* defer_splits, const float* row_scale, float p0, float p1, int a_n) {
  if (defer_splits) *defer_splits = 1;
  if (M == 0) return;
  if (a_rows == nullptr && row_scale == nullptr && defer_splits == nullptr && gemv_grouped_takes(M, N, K, epi)) {  // MoE decode: stream only the routed experts' weights
    launch_gemv_grouped(A, B, C, offsets, n_groups, M, N, K, epi, st, p0, p1);
    return;
  }
  Plan p = grouped_plan(M, N, K, n_groups, max_rows, a_n);
  float* ws = nullptr;
  if (p.variant == 0 && K >= 2048 && g_gp[3] != 1 && !(p.nosplit && g_gp[0] <= 0)) {
    const SkBuf* b = sk_buf();
    const long t_est = (long)((N + p.BN - 1) / p.BN) * std::max(1, std::min(n_groups, (M + p.BM - 1) / p.BM + n_groups));
    constexpr int target = 1024;
    int s = (int)std::min<long>(8, std::max<long>(1, target / std::max<long>(1, t_est)));
    if (g_gp[3] > 1) s = g_gp[3];
    while (s > 1 && (K / s) % kBK) --s;
    if (b && s > 1 && (size_t)s * M * N * 4 <= (size_t)2 * kSkMaxWg * 256 * 256 * 4) {
      p.splits = s;
      p.k_chunk = K / s;
      ws = b->ws;
    }
  }
  RopeEpi re{};
  re.a_rows = a_rows;
  re.row_scale = row_scale;
  re.p0 = p0;
  re.p1 = p1;
  if (epi == EPI_NONE)
    launch_plan<EPI_NONE, true>(p, (const uint16_t*)A, K, (const uint16_t*)B, K, (uint16_t*)C, N,
                                ws, M, N, K, offsets, n_groups, st, re);
  else
    launch_plan<EPI_SILU_MUL, true>(p, (const uint16_t*)A, K, (const uint16_t*)B, K, (uint16_t*)C,
                                    N / 2, ws, M, N, K, offsets, n_groups, st, re);
  if (p.splits > 1 && defer_splits != nullptr && epi == EPI_NONE) {  // the caller sums the slabs
    *defer_ws = ws;
    *defer_splits = p.splits;
  } else if (p.splits > 1) {
    const int outw = epi == EPI_NONE ? N : N / 2;
    const long total = (long)M * (outw / 8);
    const int g = (int)std::min<long>((total + 255) / 256, 4096);
    if (epi == EPI_NONE)
      splitk_reduce_kernel<EPI_NONE><<<g, 256, 0, st>>>((uint16_t*)C, N, ws, M, N, p.splits);
    else
      splitk_reduce_kernel<EPI_SILU_MUL><<<g, 256, 0, st>>>((uint16_t*)C, N / 2, ws, M, N, p.splits, re);
  }
}

}  // namespace mlop

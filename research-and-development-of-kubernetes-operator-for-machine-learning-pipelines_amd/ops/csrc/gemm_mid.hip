// K1 / K2 at 5-384 rows: a weight stream that feeds the matrix cores.
//
//   C[M, N] = A[M, K] . B[N, K]^T      (A activations, B weights [out, in], both bf16)
//
// What bounds it: reading B once (every weight byte from HBM, ~6.5 TB/s at best); A is small and comes
// from L2, once per workgroup.  The LDS-ring tiles of gemm.hip keep one ring for both operands: at 128
// rows two thirds of what is in flight is A, and the loop waits out the HBM latency of the rest.  Here
//   * the operands have rings of their own: half of the waves load A two to five K-steps ahead (L2), the
//     other half load B as many steps ahead as the 160 KB of LDS hold.  vmcnt retires in order, so one
//     wave cannot run two depths;
//   * column tile bx starts its walk of K at step bx % nk and wraps around.  Weight rows are a multiple of
//     4 KB apart: tiles that walk K in step ask for the same offset of every row, that is for the same
//     few memory channels (B alone, gate_up of Llama-3-8B: 43.8 -> 36.8 us);
//   * the next half K-step's fragments are read while this half multiplies (kBehind below);
//   * a workgroup walks its tiles without draining the rings: the next tile's first K-steps load under
//     this one's last (lm_head: four tiles per workgroup).
// Tiles are 256 columns where such tiles fill the chip (A is read half as often), else 128; rows are the
// batch in steps of 32, two row tiles above 256 rows (side by side on one XCD, so that the second reads
// the weights from L2); K is split over workgroups where the columns alone are too few.  C^T accumulators
// (the weights are the MFMA's first operand): a lane holds four neighbouring columns, gate and up of an
// output sit in one lane, and nothing is staged for the epilogue.
// Measured (cold weights, us, the LDS-ring tiles -> this kernel): gate_up 28672 x 4096 at 16 / 64 / 100 /
// 150 rows 42 -> 37, 49 -> 39, 59 -> 45, 68 -> 51 (24 rows, 32-row tiles: 39.5 -> 36.7); lm_head 128256 x 4096 at 64 / 100 /
// 150 / 256 rows 211 -> 168, 247 -> 175, 280 -> 181, 297 -> 251; down 4096 x 14336 with
// its reduce at 100 / 150 / 300 rows 37 -> 34, 46 -> 39, 68 -> 56.
#include "common.h"
#include "launch.h"

#include <stdexcept>
#include <type_traits>

namespace mlop {

namespace {

__device__ __forceinline__ int mid_swz(int r) { return (r >> 1) & 7; }

// c + the squares of eight bf16
__device__ __forceinline__ float mid_sq8(const bf16x8& v, float c) {
  typedef __attribute__((ext_vector_type(2))) __bf16 bf2;
  const u32x4 w = __builtin_bit_cast(u32x4, v);
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const uint32_t x = w[e];  // (bit_cast of the element itself reads the vector's first)
    const bf2 p = __builtin_bit_cast(bf2, x);
    c = __builtin_amdgcn_fdot2_f32_bf16(p, p, c, false);
  }
  return c;
}

// s_waitcnt vmcnt(min(n, MAX) * PER) for a wave-uniform n
template <int MAX, int PER>
__device__ __forceinline__ void wait_stages(int n) {
  if constexpr (MAX <= 0) {
    wait_vmcnt<0>();
  } else {
    if (n >= MAX) wait_vmcnt<MAX * PER>();
    else wait_stages<MAX - 1, PER>(n);
  }
}

// Tasks (column tile, row tile, K range), row tile fastest; a workgroup takes lid, lid + G, ...  SA / SB: ring
// depths in K-steps of 64.  EPI 0: plain (with an activation, RopeEpi::act), 1: gate / up, 2: gate / up of A's rows scaled by
// their RMSNorm factors, whose sums of squares a wave adds up from its own fragments (one K range: it sees whole rows); several
// K ranges leave fp32 slabs [range][M][N] in ws instead, non-temporal always (a second form of the stores cost 3 % at 200 rows).
template <int BM, int BN, int WM, int WN, int SA, int SB, int EPI, bool BEHIND>
__global__ void __launch_bounds__(WM * WN * 64) gemm_mid_kernel(
    const uint16_t* __restrict__ A, int lda, const uint16_t* __restrict__ B, int ldb, uint16_t* __restrict__ C, int ldc,
    float* __restrict__ ws, int M, int N, int K, int k_chunk, int m_tiles, int n_splits, int n_tasks, RopeEpi re) {
  constexpr int NW = WM * WN, HW = NW / 2;   // half of the waves issue A, half B
  constexpr int WTM = BM / WM, WTN = BN / WN, TM = WTM / 16, TN = WTN / 16;
  // Each half's reads stand behind the first MFMA of the half before: the compiler waits for every LDS read in flight before
  // a fragment's first use, so reads that stand before it overlap with nothing.  Not where two workgroups of 64 rows
  // share a CU and overlap each other, and 256 x 256, which would spill.  (Cold weights, us, reads before -> behind with the
  // rings as deep for A as for B: gate_up 28672 x 4096 at 100 / 150 / 192 rows 50 -> 47, 56 -> 51.5, 62 -> 59, down of
  // Llama-3-70B 8192 x 28672 at 150 / 300 107 -> 100, 191 -> 182, its gate_up at 100 / 224 153 -> 148, 220 -> 213.)
  constexpr bool kBehind = BEHIND;
  constexpr int PA = BM / 8 / HW, PB = BN / 8 / HW;  // 1-KiB pieces per issuing wave and K-step
  static_assert(BM % (8 * HW) == 0 && BN % (8 * HW) == 0 && WTM % 16 == 0 && WTN % 16 == 0, "tile");
  static_assert((SA - 1) * PA < 64 && (SB - 1) * PB < 64, "vmcnt");
  extern __shared__ __attribute__((aligned(16))) uint16_t smem[];
  uint16_t* const ringA = smem;
  uint16_t* const ringB = smem + SA * BM * 64;
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wid / WN, wn = wid % WN;
  const int G = gridDim.x, L = blockIdx.x;
  const int q = G >> 3, rr = G & 7, xcd = L & 7, slot = L >> 3;
  const int lid = (xcd < rr ? xcd * (q + 1) : rr * (q + 1) + (xcd - rr) * q) + slot;
  const int gx = (N + BN - 1) / BN;
  const int nk_all = K / 64, nk_c = k_chunk / 64;
  auto place = [&](int t, int& bx, int& by, int& bz, int& nk) {
    by = t % m_tiles;
    bx = (t / m_tiles) % gx;
    bz = t / (m_tiles * gx);
    nk = min(nk_c, nk_all - bz * nk_c);
  };
  const bool is_b = wid >= HW;
  const int iw = is_b ? wid - HW : wid;
  const bool nt = re.b_nt != 0;

  // load side: K-step i_kt of task i_task is the next to load
  constexpr int PMAX = PA > PB ? PA : PB;
  const uint16_t* src[PMAX];
  int i_task = lid, i_kt = 0, i_nk = 0, i_rot = 0, i_buf = 0;
  auto set_src = [&]() {
    int bx, by, bz;
    place(i_task, bx, by, bz, i_nk);
    i_rot = bx % i_nk;
#pragma unroll
    for (int i = 0; i < PMAX; ++i) {
      const int r = (iw + HW * i) * 8 + (lane >> 3);
      const int ch = (lane & 7) ^ mid_swz(r);
      src[i] = (is_b ? B + (size_t)min(bx * BN + r, N - 1) * ldb : A + (size_t)min(by * BM + r, M - 1) * lda) +
               bz * k_chunk + ch * 8;
    }
  };
  int total = 0;
  for (int t = lid; t < n_tasks; t += G) {
    int bx, by, bz, nk;
    place(t, bx, by, bz, nk);
    total += nk;
  }
  int issued = 0;
  auto issue = [&]() {
    if (issued >= total) return;
    if (i_kt == i_nk) {
      i_task += G;
      i_kt = 0;
      set_src();
    }
    int k = i_kt + i_rot;
    k = (k >= i_nk ? k - i_nk : k) * 64;
    if (is_b) {
      uint16_t* base = ringB + i_buf * (BN * 64);
      i_buf = i_buf == SB - 1 ? 0 : i_buf + 1;
#define MLOP_LOAD_B(aux) \
  __builtin_amdgcn_global_load_lds((const void*)(src[i] + k), (lds_void_t*)(base + (iw + HW * i) * 512), 16, 0, aux)
      if (kBehind && nt) {
#pragma unroll
        for (int i = 0; i < PB; ++i) MLOP_LOAD_B(2);
      } else {
#pragma unroll
        for (int i = 0; i < PB; ++i) {  // (64 rows: a branch per load is 1 - 3 % faster than one for all, above that 1 - 4 % slower)
          if (!kBehind && nt) MLOP_LOAD_B(2);
          else MLOP_LOAD_B(0);
        }
      }
#undef MLOP_LOAD_B
    } else {
      uint16_t* base = ringA + i_buf * (BM * 64);
      i_buf = i_buf == SA - 1 ? 0 : i_buf + 1;
#pragma unroll
      for (int i = 0; i < PA; ++i)
        __builtin_amdgcn_global_load_lds((const void*)(src[i] + k), (lds_void_t*)(base + (iw + HW * i) * 512), 16, 0, 0);
    }
    ++i_kt;
    ++issued;
  };
  set_src();
  const int depth = is_b ? SB : SA;
  for (int s = 0; s < depth; ++s) issue();

  float ss[TM];
#pragma unroll
  for (int i = 0; i < TM; ++i) ss[i] = 0.f;
  f32x4 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int arow = (wm * WTM + (lane & 15)) * 64, brow = (wn * WTN + (lane & 15)) * 64;
  const int sw = mid_swz(lane & 15), g4 = lane >> 4;
  const int off0 = (g4 ^ sw) << 3, off1 = ((4 + g4) ^ sw) << 3;
  bf16x8 fa[2][TM], fb[2][TN];  // fragments of the K-step's two halves
  int rbufA = 0, rbufB = 0;
  auto read = [&](auto kk_) {
    constexpr int kk = decltype(kk_)::value;
    const uint16_t* sA = ringA + rbufA * (BM * 64) + arow + (kk ? off1 : off0);
    const uint16_t* sB = ringB + rbufB * (BN * 64) + brow + (kk ? off1 : off0);
#pragma unroll
    for (int j = 0; j < TN; ++j) fb[kk][j] = *reinterpret_cast<const bf16x8*>(sB + j * 1024);
#pragma unroll
    for (int i = 0; i < TM; ++i) fa[kk][i] = *reinterpret_cast<const bf16x8*>(sA + i * 1024);
  };
  auto multiply = [&](auto kk_, auto&& behind) {
    constexpr int kk = decltype(kk_)::value;
    acc[0][0] = mfma16(fb[kk][0], fa[kk][0], acc[0][0]);
    behind();
#pragma unroll
    for (int i = 0; i < TM; ++i) {
#pragma unroll
      for (int j = i == 0; j < TN; ++j) acc[i][j] = mfma16(fb[kk][j], fa[kk][i], acc[i][j]);
      if constexpr (EPI == 2) ss[i] = mid_sq8(fa[kk][i], ss[i]);
    }
  };
  auto read_behind = [&](auto kk_, bool more) {
    if constexpr (kBehind) {
      __builtin_amdgcn_sched_barrier(0);
      if (more) read(kk_);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  using H0 = std::integral_constant<int, 0>;
  using H1 = std::integral_constant<int, 1>;
  int c_task = lid, c_kt = 0, c_bx, c_by, c_bz, c_nk;
  place(c_task, c_bx, c_by, c_bz, c_nk);

  auto epilogue = [&]() {
    // C^T accumulators: lane holds row i * 16 + (lane & 15), columns j * 16 + 4 g4 + 0..3
    const int mr = c_by * BM + wm * WTM + (lane & 15), nc = c_bx * BN + wn * WTN + 4 * g4;
    if (n_splits > 1) {
      float* P = ws + (size_t)c_bz * M * N;
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const int m = mr + i * 16;
        if (m < M) {
#pragma unroll
          for (int j = 0; j < TN; ++j) {
            const int n = nc + j * 16;
            if (n < N) __builtin_nontemporal_store(acc[i][j], reinterpret_cast<f32x4*>(P + (size_t)m * N + n));
          }
        }
      }
      return;
    }
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int m = mr + i * 16;
      if (m >= M) continue;
      if constexpr (EPI == 0) {
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          const int n = nc + j * 16;
          if (n >= N) continue;
          float v[4] = {acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]};
          act_outs(re, v, n);
          *reinterpret_cast<u32x2*>(C + (size_t)m * ldc + n) = u32x2{pack2(v[0], v[1]), pack2(v[2], v[3])};
        }
      } else {
        static_assert(EPI == 0 || TN % 2 == 0, "gate / up pairs");
        // (launch_mid_rs: the row's RMSNorm factor first)
        float f;
        if constexpr (EPI == 2) f = rsqrtf(sum_x16_x32(ss[i]) * re.ss_inv_k + re.ss_eps);
        else f = re.ss_in != nullptr ? rsqrtf(re.ss_in[m] * re.ss_inv_k + re.ss_eps) : 1.f;
#pragma unroll
        for (int j = 0; j < TN; j += 2) {
          const int n = nc + j * 16;
          if (n >= N) continue;
          const f32x4 g = acc[i][j] * f, u = acc[i][j + 1] * f;
          const int o = (c_bx * BN + wn * WTN + j * 16) / 2 + 4 * g4;
          *reinterpret_cast<u32x2*>(C + (size_t)m * ldc + o) =
              u32x2{pack2(glu_out(re, g[0], u[0]), glu_out(re, g[1], u[1])),
                    pack2(glu_out(re, g[2], u[2]), glu_out(re, g[3], u[3]))};
        }
      }
    }
  };

  if (is_b) wait_stages<SB - 1, PB>(total - 1);
  else wait_stages<SA - 1, PA>(total - 1);
  raw_barrier();
  read(H0{});
  for (int s = 0; s < total; ++s) {
    if constexpr (!kBehind) read(H1{});
    multiply(H0{}, [&]() { read_behind(H1{}, true); });
    if (s + 1 < total) {
      if (s + (SA > SB ? SA : SB) <= total) {
        if (is_b) wait_vmcnt<(SB - 2) * PB>();
        else wait_vmcnt<(SA - 2) * PA>();
      } else if (is_b) {
        wait_stages<SB - 2, PB>(total - 2 - s);
      } else {
        wait_stages<SA - 2, PA>(total - 2 - s);
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // this wave has step s in registers
      raw_barrier();                                      // step s + 1 landed; step s's buffers are free
      issue();
      rbufA = rbufA == SA - 1 ? 0 : rbufA + 1;
      rbufB = rbufB == SB - 1 ? 0 : rbufB + 1;
      if constexpr (!kBehind) read(H0{});
    }
    multiply(H1{}, [&]() { read_behind(H0{}, s + 1 < total); });
    if (++c_kt == c_nk) {
      epilogue();
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        ss[i] = 0.f;
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
      c_kt = 0;
      c_task += G;
      if (c_task < n_tasks) place(c_task, c_bx, c_by, c_bz, c_nk);
    }
  }
}

template <int BM, int BN, int WM, int WN, int SA, int SB, int EPI, bool BEHIND>
static void run_mid(const uint16_t* A, int lda, const uint16_t* B, int ldb, uint16_t* C, int ldc, float* ws, int M, int N,
                    int K, int splits, int k_chunk, hipStream_t st, const RopeEpi& re) {
  constexpr size_t lds = (size_t)(SA * BM + SB * BN) * 128;
  static_assert(lds <= 163840, "LDS budget");
  auto kern = gemm_mid_kernel<BM, BN, WM, WN, SA, SB, EPI, BEHIND>;
  static const bool attr =
      hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) == hipSuccess;
  (void)attr;
  const int m_tiles = (M + BM - 1) / BM, gx = (N + BN - 1) / BN;
  const int tasks = gx * m_tiles * splits;
  constexpr int per_cu = (int)(163840 / lds) >= 2 ? 2 : 1;
  RopeEpi r = re;
  r.b_nt = gemm_weights_nt(m_tiles);
  kern<<<std::min(tasks, kCus * per_cu), WM * WN * 64, lds, st>>>(A, lda, B, ldb, C, ldc, ws, M, N, K, k_chunk, m_tiles,
                                                                 splits, tasks, r);
}
}  // namespace

void launch_mid(int epi, int bm, int bn, const uint16_t* A, int lda, const uint16_t* B, int ldb, uint16_t* C, int ldc,
                float* ws, int M, int N, int K, int splits, int k_chunk, hipStream_t st, const RopeEpi& re) {
#define MLOP_MID_(m, n, wm, wn, sa, sb, e, behind) \
  return run_mid<m, n, wm, wn, sa, sb, e, behind>(A, lda, B, ldb, C, ldc, ws, M, N, K, splits, k_chunk, st, re)
#define MLOP_MID(m, n, wm, wn, sa, sb, behind)               \
  if (bm == m && bn == n) {                                  \
    if (epi == 0) MLOP_MID_(m, n, wm, wn, sa, sb, 0, behind); \
    if (epi == 1) MLOP_MID_(m, n, wm, wn, sa, sb, 1, behind); \
    if constexpr (m <= 64) MLOP_MID_(m, n, wm, wn, sa, sb, 2, behind); \
  }
  // ring depths: what fits 160 KB (half of it where two workgroups share a CU).  With 128 columns as deep for A as for B: with
  // A two or three deep and the rest for B 0 - 4 % slower (qkv, gate_up and down at 100 - 160 rows; 8192 x 28672 at 112 - 128 rows 2 %
  // faster); not 224 rows, where it made no difference.  64 x 128: the whole of it for grids of one workgroup per CU (28672 x 4096
  // at 33 / 64 rows 39.9 -> 37.7, 40.9 -> 39.3 us, 24576 x 3072 at 33 33.9 -> 30.3), half for larger ones (40960 x 4096 at 33 66
  // against 72).  32 rows: half (28672 x 4096 at 24 rows 39.5 -> 36.7 us, with the whole 38.4).
  const long tasks = (long)((N + bn - 1) / bn) * ((M + bm - 1) / bm) * splits;
  MLOP_MID(32, 128, 2, 4, 3, 4, true)
  if (tasks <= kCus) {
    MLOP_MID(64, 128, 2, 4, 4, 6, true)
  }
  MLOP_MID(64, 128, 2, 4, 2, 4, false)
  MLOP_MID(96, 128, 2, 4, 5, 6, true)
  MLOP_MID(128, 128, 2, 4, 5, 5, true)
  MLOP_MID(160, 128, 2, 4, 4, 5, true)
  MLOP_MID(192, 128, 2, 4, 4, 4, true)
  MLOP_MID(224, 128, 2, 4, 2, 6, true)
  MLOP_MID(256, 128, 4, 2, 3, 4, true)
  MLOP_MID(32, 256, 2, 4, 2, 4, true)
  MLOP_MID(64, 256, 2, 4, 3, 4, false)
  MLOP_MID(96, 256, 2, 4, 2, 4, true)
  MLOP_MID(128, 256, 2, 4, 3, 3, true)
  MLOP_MID(160, 256, 2, 4, 3, 3, true)
  MLOP_MID(192, 256, 2, 4, 2, 3, true)
  MLOP_MID(224, 256, 2, 4, 2, 3, true)
  MLOP_MID(256, 256, 2, 4, 2, 3, false)
#undef MLOP_MID
#undef MLOP_MID_
  throw std::runtime_error("gemm_mid: no such tile");
}

}  // namespace mlop

// K2 at 1-16 rows (decode of up to 16 sequences, the head of a prompt): the weight-streaming MFMA GEMM.
//
//   C[M, N] = A[M, K] . B[N, K]^T      (A activations, B weights [out, in], both bf16)
//
// What bounds it: every weight byte comes from HBM once, at 6.8 TB/s at best; at 4 rows a CU also takes in A once for every
// 16 weight rows.  Between the GEMV (gemv.hip: a quarter of its time at 4 rows is dot products) and the LDS-ring tiles (gemm.hip:
// K ranges whose fp32 sums a second launch adds) this kernel keeps the GEMV's way of loading and multiplies on the matrix cores:
//   * a workgroup has 16 (or 32) weight rows over the WHOLE K; its 8 waves take steps of 128 k in turn and meet in LDS once,
//     at the end: no slabs, no second launch, and the epilogue has whole sums;
//   * weights go straight to registers, non-temporal, one load instruction 8 rows x 128 B (whole lines).  The MFMA wants
//     16 rows from it: its row v holds the chunks 2 g + (v & 1) of weight row v / 2, is multiplied with the even and with the odd
//     chunks of A, and the halves that belong together are added at the end.  Twice the MFMAs, of which a CU has ten times what the
//     stream needs; 16 rows x 64 B per instruction, each line in two halves, ran at 6.3 TB/s instead of 6.8 (gate_up of
//     Llama-3-8B, weights alone: 37.3 -> 34.7 us), and needed the cached path;
//   * A comes as a wave-private LDS image per step, by LDS-DMA of 4 rows x 256 B.  As MFMA fragments straight from memory its
//     16-B pieces of 16 rows cost a lookup each: 28672 x 4096 at 16 rows 55.8 -> 41.9 us, 4096 x 14336 28.8 -> 24.3 (then);
//   * workgroups start their walk of K at steps that differ.  Rows are a multiple of 4 KB apart: in step they ask the same few
//     channels (28672 x 4096, 32 rows per workgroup, 50.6 -> 38.7 us; 16 rows 37.6 -> 36.3).
// What is left: 4096 x 14336 takes 20.1 / 20.9 / 22.2 / 23.4 us at 4 / 8 / 13 / 16 rows (into a residual the same), at 16 with half of A's image 19.8: weights and A share what a CU can have in
// flight.  The epilogue is 0.8 us of a launch of one workgroup per CU.  Tried and slower: A kept in registers for all tiles of a
// workgroup (28672 x 4096 39.5 us), four steps in flight (VGPRs for one workgroup fewer), 4 or 16 waves.
// Epilogues (the decode norm chain, so that a layer has no add + RMSNorm launch):
//   WS_NONE      bf16 store (with an activation, RopeEpi::act);
//   WS_RES       residual (C) += y in place, bf16(res + bf16(y)) (norm.hip's add rounding);
//   WS_SILU_MUL  gate rows 32b.. and their up rows 32b+16.. of the 16-interleaved gate_up;
//   WS_ROPE      a q / k head's rotate-half rows (d, d + 64), rotated and stored to q_out / the paged K cache; V rows straight
//                into their page rows;
// prologue RS (QKV / gate_up of the chain, norm weights folded into B): A is the raw residual; each row's sum of squares
// accumulates from the fragments the MFMAs read and rsqrt(mean + eps) scales the finished sums.
#include "common.h"
#include "launch.h"

#include <type_traits>

namespace mlop {

namespace {

enum { WS_NONE = 0, WS_SILU_MUL = 1, WS_ROPE = 3, WS_RES = 5 };

typedef __attribute__((ext_vector_type(2))) __bf16 ws_bf16x2;

__device__ __forceinline__ float ws_dot2(uint32_t a, uint32_t b, float c) {
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(ws_bf16x2, a), __builtin_bit_cast(ws_bf16x2, b), c,
                                        false);
}

__device__ __forceinline__ float ws_sq8(const u32x4& w, float c) {
  c = ws_dot2(w.x, w.x, c);
  c = ws_dot2(w.y, w.y, c);
  c = ws_dot2(w.z, w.z, c);
  return ws_dot2(w.w, w.w, c);
}

// A fragments of one 16-row tile and step (256 B of every row): f[2 h + x] = chunk 8 h + 2 (lane >> 4) + x of row m, in the
// image [row][16 x 16 B] with chunk c of row r at slot c ^ (r & 15).  `N`: vector memory operations younger than the image's.
template <int N>
__device__ __forceinline__ void ws_frags(uint32_t row, uint32_t x0, uint32_t x1, uint32_t x2, uint32_t x3, u32x4 (&f)[4]) {
  asm volatile(
      "s_waitcnt vmcnt(%8)\n"
      "ds_read_b128 %0, %4\n"
      "ds_read_b128 %1, %5\n"
      "ds_read_b128 %2, %6\n"
      "ds_read_b128 %3, %7\n"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(f[0]), "=&v"(f[1]), "=&v"(f[2]), "=&v"(f[3])
      : "v"(row + x0), "v"(row + x1), "v"(row + x2), "v"(row + x3), "n"(N)
      : "memory");
}

template <int AR, int G, int NW, int U, int EPI, bool RS, bool NT>
__global__ void __launch_bounds__(NW * 64) gemm_ws_kernel(const uint16_t* __restrict__ A, int lda,
                                                          const uint16_t* __restrict__ B, int ldb,
                                                          uint16_t* __restrict__ C, int ldc, int M, int K,
                                                          RopeEpi re, float eps) {
  static_assert(G % 2 == 0, "gate / up and rotate-half pairs of row groups");
  static_assert(AR == 4 || AR == 8 || AR % 16 == 0, "rows of A staged");
  constexpr int MT = (AR + 15) / 16, H2 = G / 2, T = NW * 64, D = 128;
  constexpr int AI = AR / 4;            // LDS-DMA instructions (4 rows x 256 B) per step
  constexpr int IMG = AR * 256;         // bytes of a step's A image
  extern __shared__ __attribute__((aligned(256))) uint8_t ws_lds[];
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int blk = blockIdx.x;
  // first weight row of the workgroup, and row group g's distance from it
  int row0, far;  // groups 0 .. H2 - 1: row0 + 8 g; H2 .. G - 1: row0 + far + 8 (g - H2)
  bool rope_blk = false;
  if constexpr (EPI == WS_SILU_MUL) {  // gate rows, and their up rows 16 further
    row0 = H2 == 2 ? 32 * blk : 32 * (blk >> 1) + 8 * (blk & 1);
    far = 16;
  } else if constexpr (EPI == WS_ROPE) {  // a q / k head's dims d .. and d + 64 ..; plain v rows
    constexpr int BPH = 8 / H2;  // workgroups per head
    const int rope_blocks = (re.Hq + re.Hkv) * BPH;
    rope_blk = blk < rope_blocks;
    row0 = rope_blk ? (blk / BPH) * D + (blk % BPH) * 8 * H2 : (re.Hq + re.Hkv) * D + (blk - rope_blocks) * 8 * G;
    far = rope_blk ? D / 2 : 8 * H2;
  } else {
    row0 = blk * 8 * G;
    far = 8 * H2;
  }

  // outputs of this thread: with one row tile, at most one (or one pair), whose old residual value, slot and position
  // load ahead of the weights
  constexpr int PAIR = EPI == WS_SILU_MUL || EPI == WS_ROPE, GO = PAIR ? H2 : G, OUTS = MT * 16 * GO * 8;
  const int ot = threadIdx.x;
  const int oj = ot & 7, og = (ot >> 3) % GO, om = ot / (8 * GO);
  uint16_t res_pf = 0;
  int pos_pf = 0, slot_pf = -1;
  float cos_pf = 0.f, sin_pf = 0.f;
  const bool out_pf = OUTS <= T && ot < OUTS && om < M;
  if constexpr (EPI == WS_RES) {
    if (out_pf) res_pf = C[(size_t)om * ldc + row0 + 8 * og + oj];
  }
  if constexpr (EPI == WS_ROPE) {
    if (out_pf) {
      slot_pf = re.slots[om];
      pos_pf = re.pos[om];
    }
  }

  // Weight loads cover 8 rows x 128 B: MFMA row v = lane & 15 holds chunks 2 g4 + (v & 1) of row v >> 1, so two neighbouring
  // lanes read 32 B, and a product with the even chunks of A counts for even v, one with the odd chunks for odd v.
  const int v = lane & 15, g4 = lane >> 4;
  const char* const Bw = reinterpret_cast<const char*>(B + (size_t)row0 * ldb);
  uint32_t bo[G], ao[AI];
#pragma unroll
  for (int g = 0; g < G; ++g) bo[g] = (uint32_t)((g < H2 ? 8 * g : far + 8 * (g - H2)) + (v >> 1)) * ldb * 2 + g4 * 32 + (v & 1) * 16;
#pragma unroll
  for (int i = 0; i < AI; ++i) {  // (rows past M: the last one again, never stored)
    const int r = 4 * i + g4;
    ao[i] = (uint32_t)min(r, M - 1) * lda * 2 + ((v ^ (r & 15)) << 4);
  }
  // steps of 128 k (256 B of a row): the waves take them in turn, from one that differs by workgroup on
  const int n_steps = K >> 7, rounds = n_steps / NW, rot = (blk >> 3) * 5 % n_steps;
  // (a generic pointer's low 32 bits are the LDS offset)
  const uint32_t img = (uint32_t)(uintptr_t)ws_lds + wv * (U * IMG);
  const int mr16 = AR < 16 ? lane & (AR - 1) : v;
  const uint32_t arow = img + mr16 * 256;
  const uint32_t x0 = ((2 * g4) ^ mr16) << 4, x1 = ((2 * g4 + 1) ^ mr16) << 4, x2 = ((8 + 2 * g4) ^ mr16) << 4, x3 = ((9 + 2 * g4) ^ mr16) << 4;

  f32x4 acc[MT][G][2];
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int g = 0; g < G; ++g) acc[t][g][0] = acc[t][g][1] = f32x4{0.f, 0.f, 0.f, 0.f};
  float ss[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) ss[t] = 0.f;

  u32x4 bq[U][2][G];
  const auto rsA = __builtin_amdgcn_make_buffer_rsrc((void*)A, 0, ((M - 1) * lda + K) * 2, 0x00020000);
  constexpr int OPS = AI + 2 * G;  // vector memory operations of a step
  auto load = [&](int u, int s) {
    int p = s * NW + wv + rot;
    p -= p >= n_steps ? n_steps : 0;
    const uint32_t k = (uint32_t)p * 256;
#pragma unroll
    for (int i = 0; i < AI; ++i)
      lds_dma16(rsA, img + u * IMG + i * 1024, ao[i] + k, 0);
    asm volatile("" ::: "memory");
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int g = 0; g < G; ++g) {
        const u32x4* p = reinterpret_cast<const u32x4*>(Bw + (bo[g] + k + h * 128));
        bq[u][h][g] = NT ? __builtin_nontemporal_load(p) : *p;
      }
    asm volatile("" ::: "memory");
  };
  // `younger`: steps loaded after this one
  auto consume = [&](auto younger, int u) {
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      u32x4 f[4];
      ws_frags<decltype(younger)::value * OPS + 2 * G>(arow + u * IMG + t * 4096, x0, x1, x2, x3, f);
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int x = 0; x < 2; ++x) {
#pragma unroll
          for (int g = 0; g < G; ++g)
            acc[t][g][x] = mfma16(__builtin_bit_cast(bf16x8, bq[u][h][g]), __builtin_bit_cast(bf16x8, f[2 * h + x]), acc[t][g][x]);
          if constexpr (RS) ss[t] = ws_sq8(f[2 * h + x], ss[t]);
        }
    }
  };
  using Y0 = std::integral_constant<int, 0>;
  auto load_cs = [&]() {
    if constexpr (EPI == WS_ROPE) {
      if (out_pf && rope_blk) {
        const float* cs = re.cos_sin + (size_t)pos_pf * D + (row0 % D) + 8 * og + oj;
        cos_pf = cs[0];
        sin_pf = cs[D / 2];
      }
    }
  };
  int s0 = 0;
  if (rounds >= U) {
    // whole passes of the ring without a branch (behind a guarded load the compiler waits for all that are in flight)
#pragma unroll
    for (int u = 0; u < U; ++u) load(u, u);
    load_cs();
    for (; s0 + 2 * U <= rounds; s0 += U) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        consume(std::integral_constant<int, U - 1>{}, u);
        load(u, s0 + U + u);
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) consume(Y0{}, u);
    s0 += U;
  } else {
    load_cs();
  }
  for (; s0 < rounds; ++s0) {
    load(0, s0);
    consume(Y0{}, 0);
  }
  if (wv < n_steps - rounds * NW) {
    load(0, rounds);
    consume(Y0{}, 0);
  }
  wait_vmcnt<0>();
  __syncthreads();  // the images' space now takes the waves' sums

  float (*red)[MT][G][16][8] = reinterpret_cast<float (*)[MT][G][16][8]>(ws_lds);
  float (*red_ss)[MT][16] = reinterpret_cast<float (*)[MT][16]>(ws_lds + NW * MT * G * 512);
#pragma unroll
  for (int t = 0; t < MT; ++t) {
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const float2 y = {acc[t][g][0][0] + acc[t][g][1][1], acc[t][g][0][2] + acc[t][g][1][3]};
      *reinterpret_cast<float2*>(&red[wv][t][g][v][2 * g4]) = y;
    }
    if constexpr (RS) {
      const float sum = sum_x16_x32(ss[t]);
      if (lane < 16) red_ss[wv][t][lane] = sum;
    }
  }
  __syncthreads();

#pragma unroll 1
  for (int o = ot; o < OUTS; o += T) {
    const int j = o & 7, g = (o >> 3) % GO, m = o / (8 * GO), t = m >> 4, mr = m & 15;
    if (m >= M) return;
    float y = 0.f, z = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      y += red[w][t][g][mr][j];
      if constexpr (PAIR) z += red[w][t][g + H2][mr][j];
    }
    if constexpr (RS) {
      float tot = 0.f;
#pragma unroll
      for (int w = 0; w < NW; ++w) tot += red_ss[w][t][mr];
      const float inv = rsqrtf(tot / (float)K + eps);
      y *= inv;
      z *= inv;
    }
    if constexpr (EPI == WS_SILU_MUL) {
      C[(size_t)m * ldc + blk * 8 * H2 + 8 * g + j] = f2bf(glu_out(re, y, z));
    } else if constexpr (EPI == WS_ROPE) {
      const int slot = OUTS <= T ? slot_pf : re.slots[m];
      const int pblk = slot >= 0 ? slot / re.BS : 0, poff = slot >= 0 ? slot % re.BS : 0;
      if (rope_blk) {
        const int hd = row0 / D, d = row0 % D + 8 * g + j;
        float c = cos_pf, s = sin_pf;
        if constexpr (OUTS > T) {
          const float* cs = re.cos_sin + (size_t)re.pos[m] * D + d;
          c = cs[0];
          s = cs[D / 2];
        }
        const float x = bf2f(f2bf(y)), w = bf2f(f2bf(z));
        const uint16_t oa = f2bf(x * c - w * s), ob = f2bf(w * c + x * s);
        uint16_t* dst;
        if (hd < re.Hq) {
          dst = re.q_out + ((size_t)m * re.Hq + hd) * D;
        } else {
          if (slot < 0) continue;
          dst = re.k_cache + (((size_t)pblk * re.Hkv + (hd - re.Hq)) * re.BS + poff) * D;
        }
        dst[d] = oa;
        dst[D / 2 + d] = ob;
      } else if (slot >= 0) {
        const int vr = row0 - (re.Hq + re.Hkv) * D + 8 * g + j;  // v row 0 .. Hkv * 128, and the one far from it
        uint16_t* v0 = re.v_cache + (((size_t)pblk * re.Hkv + vr / D) * re.BS + poff) * D + vr % D;
        const int vz = vr + far;
        v0[0] = f2bf(y);
        re.v_cache[(((size_t)pblk * re.Hkv + vz / D) * re.BS + poff) * D + vz % D] = f2bf(z);
      }
    } else {
      uint16_t* p = C + (size_t)m * ldc + row0 + 8 * g + j;  // (plain rows: far = 8 H2)
      if constexpr (EPI == WS_RES) *p = f2bf(bf2f(OUTS <= T ? res_pf : *p) + bf2f(f2bf(y)));
      else *p = f2bf(act_out(re, y, row0 + 8 * g + j));
    }
  }
}

// rows up to which this kernel is taken, in the decode chain and outside (gemm_ws_max_m op; 0: never)
int g_ws_max_m = 16;

// A / B plan (gemm_ws_plan op, 0 = by shape): 16-row blocks per workgroup (1 / 2) and K-steps in flight per wave (1; 2 up to 16
// rows of A)
int g_ws_rb = 0, g_ws_u = 0;

template <int AR, int G, int U, int EPI, bool RS, bool NT = true>
void run_ws_k(const uint16_t* A, int lda, const uint16_t* B, int ldb, uint16_t* C, int ldc, int M, int N, int K,
              const RopeEpi& re, float eps, hipStream_t st) {
  constexpr int MT = (AR + 15) / 16, NW = 8;
  constexpr size_t ring = (size_t)NW * U * AR * 256, red = (size_t)NW * MT * (G * 512 + 64), lds = ring > red ? ring : red;
  static_assert(lds <= 163840, "LDS");
  auto kern = gemm_ws_kernel<AR, G, NW, U, EPI, RS, NT>;
  static const bool attr =
      hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) == hipSuccess;
  (void)attr;
  kern<<<N / (8 * G), NW * 64, lds, st>>>(A, lda, B, ldb, C, ldc, M, K, re, eps);
}

template <int AR, int EPI, bool RS>
void run_ws_ar(const uint16_t* A, int lda, const uint16_t* B, int ldb, uint16_t* C, int ldc, int M, int N, int K,
               const RopeEpi& re, float eps, hipStream_t st) {
  // 32 weight rows take in half as much of A as 16 do, on half as many workgroups: where 16 make a second round of the CUs
  // and 32 do not (6144 x 4096 at 4 rows 10.6 -> 10.3 us, at 16 13.4 -> 11.8; 5120 x 5120 at 8 14.5 -> 13.2), and from 9 rows on
  // where 16 make more than three (28672 x 4096 at 16 rows 42 -> 39, lm_head 128256 x 4096 184 -> 158; 13824 x 4096 24.0 -> 21.7,
  // x 5120 31.8 -> 28.3; but 12288 x 4096, 768 workgroups of 16, 19.7 -> 21.2, 10240 x 8192 33.6 -> 36.8).  Up to 8 rows A costs
  // little: 28672 x 4096 at 8 36.2 against 38.2.
  const int w32 = N / 32;
  const bool wide = N % 32 == 0 && (g_ws_rb ? g_ws_rb == 2 : N / 16 > kCus && (w32 <= kCus || (M > 8 && N / 16 > 3 * kCus)));
  // two steps per wave in flight where there are as many and the images leave a second workgroup its LDS (lm_head at 4 rows
  // 152.2 -> 148.8 us; 16384 x 512 at 4, one step per wave, 5.3 -> 7.0; at 16 rows down 4096 x 14336 23.4 -> 24.0)
  const bool two = g_ws_u ? g_ws_u == 2 : AR <= 8 && K >= 2048;
#define MLOP_WS(G, U, ...) return run_ws_k<AR, G, U, EPI, RS __VA_ARGS__>(A, lda, B, ldb, C, ldc, M, N, K, re, eps, st)
  if constexpr (AR <= 32) {  // weights through the caches (gemm_small_nt op); the same sums, whatever is in flight
    if (!gemm_weights_nt(1)) {
      if (wide) MLOP_WS(4, 1, , false);
      MLOP_WS(2, 1, , false);
    }
  }
  if constexpr (AR <= 16) {  // (32 rows and two steps: 28 - 41 registers over)
    if (wide && two) MLOP_WS(4, 2);
    if (two) MLOP_WS(2, 2);
  }
  if (wide) MLOP_WS(4, 1);
  MLOP_WS(2, 1);
#undef MLOP_WS
}

template <int EPI, bool RS>
void run_ws(const uint16_t* A, int lda, const uint16_t* B, int ldb, uint16_t* C, int ldc, int M, int N, int K,
            const RopeEpi& re, float eps, hipStream_t st) {
  if (M <= 4) run_ws_ar<4, EPI, RS>(A, lda, B, ldb, C, ldc, M, N, K, re, eps, st);
  else if (M <= 8) run_ws_ar<8, EPI, RS>(A, lda, B, ldb, C, ldc, M, N, K, re, eps, st);
  else if (M <= 16) run_ws_ar<16, EPI, RS>(A, lda, B, ldb, C, ldc, M, N, K, re, eps, st);
  else if (M <= 32) run_ws_ar<32, EPI, RS>(A, lda, B, ldb, C, ldc, M, N, K, re, eps, st);
  else if (M <= 48) run_ws_ar<48, EPI, RS>(A, lda, B, ldb, C, ldc, M, N, K, re, eps, st);
  else run_ws_ar<64, EPI, RS>(A, lda, B, ldb, C, ldc, M, N, K, re, eps, st);
}

}  // namespace

int gemm_ws_max_m(int set) {
  if (set >= 0) g_ws_max_m = set > 64 ? 64 : set;
  return g_ws_max_m;
}

// and outside the chain: gemm_ws_small_m op, QKV + RoPE gemm_ws_rope_m.  The latter to 32 rows: its RoPE + cache epilogue
// spares the launch that sums the planner's K ranges (6144 x 4096 at 20 / 32 rows 16.1 + 4 -> 13.0, 16.4 + 4 -> 14.2 us; 10240 x
// 8192 at 24 / 32 43.8 + 4 -> 41.2, 44.2 + 4 -> 46.1; 3072 x 2048 at 32 9.3 + 3 -> 6.5)
int g_ws_small_m = 16, g_ws_rope_m = 32;

int gemm_ws_small_m(int set) {
  if (set >= 0) g_ws_small_m = set > 64 ? 64 : set;
  return g_ws_small_m;
}

int gemm_ws_rope_m(int set) {
  if (set >= 0) g_ws_rope_m = set > 64 ? 64 : set;
  return g_ws_rope_m;
}

// shapes this kernel can take: whole steps of 128 k, whole 16-row blocks (gate / up: 32-row groups; RoPE: 128-wide heads)
static bool ws_shape(int M, int N, int K, int epi) {
  if (M < 1 || M > 64 || K % 128 || K < 128 || K > (1 << 18) || N < 16) return false;
  if (epi == WS_SILU_MUL) return N % 32 == 0;
  if (epi == WS_ROPE) return N % 128 == 0;
  return (epi == WS_NONE || epi == WS_RES) && N % 16 == 0;
}

// Where it is the faster choice.  Against the GEMV (one to four rows): from 3 rows on, two where the matrix is not narrow, one
// where it is large (us, GEMV -> here: 6144 x 4096 at 2 / 4 rows 11.3 -> 10.5, 15.1 -> 10.5; 28672 x 4096 at 1 / 2 / 4 36.6 -> 37.2,
// 36.0 -> 36.5, 43.3 -> 36; 4096 x 14336 at 4 24.4 -> 19.9; 128256 x 4096 at 1 / 4 160 -> 155, 171 -> 150; 128256 x 8192 at 1 336 ->
// 307; 2048 x 4096 at 2 / 4 6.0 -> 6.6, 7.2 -> 6.2; 1024 x 4096 at 4 5.4 -> 5.8).  At two
// rows not where the last of a few rounds of workgroups is nearly empty, short K aside (4256 x 4736 9.8 -> 10.6, 8480 x 11136 32.8
// -> 36.0, 12704 x 8192 33.6 -> 37.0).
//   Against the planner's tiles and their K ranges' sums (5 to 16 rows), where a workgroup's walk of the whole K is no longer
// than those: it takes in 16 weight rows and A, and few workgroups cannot make up for it.  Measured at 5 - 16 rows on 120 shapes,
// here over there: narrow ones (128 - 1024 columns) at K 6144 0.80 - 0.98, at 8192 0.82 / 0.92 / 0.99 / 1.05 at 5 / 9 / 12 / 16 rows, at 9216
// 0.94 / 1.02 / 1.10 / 1.17; 1280 - 2048 columns at 8192 0.80 - 0.98, at 9216 0.90 / 0.95 / 1.02 / 1.07; 3072 x 14336 0.88 / 0.95 / 1.01 /
// 1.06, 3072 x 28672 0.96 / 1.05 / 1.11 / 1.17, 4096 x 28672 0.91 / 0.94 / 0.99 / 1.03; 5120 - 22016 columns 0.46 - 0.98, but 4112 -
// 5104, a second round for a few workgroups, 0.98 / 1.06 / 1.1 at K 9000 / 10000 / 14000 and 5 - 8 rows, 1.02 / 1.06 / 1.16 at 7300 / 9000 /
// 11000 and 11.  Short K under many columns are launches of thousands of short workgroups: 16384 x 256 / 512 / 1024 1.10 / 1.12 / 1.0, 65536 x 256 / 512 / 768 /
// 1024 1.30 / 1.15 / 1.04 / 0.9.  At 24 and 32 rows A is what a CU takes in: 28672 x 4096 40.4 -> 48.5, 4096 x 14336 25 -> 28.
//   With the residual add and a norm behind it, the planner's K ranges have the norm in the launch that sums them and this kernel a
// launch of its own: 512 x 2048 / 4096 / 8192 at 16 rows 0.97 / 1.17 / 1.38 (at 5 0.89 / 1.01 / 1.13), 1024 x 4096 1.14 (1.01), 2048 x 4096 /
// 8192 1.0 / 1.16 (0.89 / 0.98), 3072 x 8192 / 9216 1.0 / 1.09 (0.87 / 0.96), 3584 and 4096 x 14336 1.03 (0.93), 4352 x 3328 /
// 5120 / 14336 1.0 / 1.05 / 1.19, 5120 and more columns 0.54 - 0.86.
//   QKV + RoPE at 17 - 32 rows, where A is most of what a CU takes in, against K ranges and the launch that sums, rotates and stores them
// (34 numbers of heads, K 512 - 8192): K up to 4096 0.5 - 1.0; 768 - 2048 columns at 17 / 24 / 32 rows with K 5120 0.95 / 1.0 / 1.05, 6144
// 0.97 / 1.04 / 1.1, 8192 1.03 / 1.12 / 1.2; 3072 0.9 / 0.94 / 1.03 with 8192; 4352 - 5376 columns, a second round for few, 1.0 - 1.1 from
// 5120 on; 5632 - 8192 0.8 - 0.98; more at K 5120 - 7168 0.92 / 0.97 / 1.05, at 8192 0.88 / 0.94 / 1.0.
// Those are with K of whole 2048, mostly, where the K ranges are slower (3328 x 8192 at 19 rows 0.82); with others 2048 - 3583 columns are
// level at M K / N = 56 (3072 x 7808 at 25 rows, 63: 1.11), 3584 - 4096 at 48 (4096 x 8064 at 32, 63: 1.11).
static bool ws_fast(int M, int N, int K, int epi) {
  const long nk = (long)N * K, mk = (long)M * K;
  const int w = N / 16;  // workgroups of 16 rows
  if (M == 1) return nk >= 200L * 1000 * 1000;
  if (M == 2) return N >= 3072 && (K <= 2560 || w % kCus == 0 || w < kCus || w > 4 * kCus || w % kCus >= (w < 2 * kCus ? 64 : 128));
  if (M <= 4) return N >= 2048;
  // (launches, whichever the kernel; here one less, or an add less: 1280 x 512 with its norm at 6 rows 6.7 -> 5.2 us)
  if (nk < 1 << 20) return (epi == WS_ROPE || epi == WS_RES) && M <= 8 && K % 512 == 0;
  const bool second = w > kCus && w < kCus + 64;  // (workgroups of a second round that leave most CUs idle)
  if (epi == WS_RES) {
    if (second) return K <= 3072;
    if (N >= 3072) return N >= 5120 || (N >= 3584 ? mk <= 45L * N : mk < 36L * N);
    return K <= 2048 || (K <= 9216 && mk <= (N <= 1536 ? 24L : 28L) * N);
  }
  if (epi == WS_ROPE && M > 16)
    return K <= 4096 || (N <= 4096 ? K <= 8192 && mk <= (K % 2048 ? (N < 2048 ? 60L : N < 3584 ? 56L : 48L) : N < 3072 ? 60L : 64L) * N
                                   : N >= 5632 && (N <= 8192 || K % 4096 == 0 || mk <= 150000));
  if (epi == WS_ROPE && N <= 1280) return K <= 9216 && mk <= 100000;
  if (N >= 16384 && K < 1024) return false;
  if (second) return K <= (M > 8 ? 7168 : 9216);
  if (N >= 3072) return mk <= 190L * (N - 2100);
  return K <= 9216 && 1024L * M + 5L * K <= (N < 1280 ? 53760 : 57500);
}

bool ws_prefer(int M, int N, int K, int epi) {
  const int bound = epi == WS_ROPE ? (g_ws_max_m ? g_ws_rope_m : 0) : std::min(g_ws_max_m, g_ws_small_m);
  return M <= bound && ws_shape(M, N, K, epi) && ws_fast(M, N, K, epi);
}

// (the third argument chose a form of the weight loads: gemm_small_nt does)
void gemm_ws_plan(int rb, int u, int) {
  g_ws_rb = rb == 1 ? 1 : rb == 2 || rb == 4 ? 2 : 0;
  g_ws_u = u == 1 ? 1 : u > 1 ? 2 : 0;
}

bool ws_takes(int M, int N, int K, int epi) { return M <= g_ws_max_m && ws_shape(M, N, K, epi); }

int decode_chain_max_m() { return g_ws_max_m > gemv_chain_max_m() ? g_ws_max_m : gemv_chain_max_m(); }

// the chain's product of this shape on this kernel rather than the GEMV
bool chain_on_ws(int M, int N, int K, int epi) {
  return ws_takes(M, N, K, epi) && (M > gemv_chain_max_m() || ws_fast(M, N, K, epi));
}

// and gate_up on gemm_mid.hip's stream, where that takes it: above 8 rows A is what a CU of this kernel takes in (28672 x
// 4096 at 16 rows 42.3 -> 37.1 us, at 9 39.6 -> 37.0; at 8 35.8 here, 36.8 there)
bool chain_on_mid(int M, int N, int K) { return M > 8 && M <= g_ws_max_m && mid_self_ok(M, N, K); }

bool decode_chain_takes(int M, int N, int K, int epi) {
  return gemv_chain_takes(M, N, K, epi) || (ws_takes(M, N, K, epi) && ((long)N * K >= 1 << 20));
}

void launch_ws(const void* A, int lda, const void* B, int ldb, void* C, int ldc, int M, int N, int K, int epi,
               bool rs, const RopeEpi& re, float eps, hipStream_t st) {
  auto* a = (const uint16_t*)A;
  auto* b = (const uint16_t*)B;
  auto* c = (uint16_t*)C;
  if (epi == WS_SILU_MUL) {
    if (rs) run_ws<WS_SILU_MUL, true>(a, lda, b, ldb, c, ldc, M, N, K, re, eps, st);
    else run_ws<WS_SILU_MUL, false>(a, lda, b, ldb, c, ldc, M, N, K, re, eps, st);
  } else if (epi == WS_ROPE) {
    if (rs) run_ws<WS_ROPE, true>(a, lda, b, ldb, c, ldc, M, N, K, re, eps, st);
    else run_ws<WS_ROPE, false>(a, lda, b, ldb, c, ldc, M, N, K, re, eps, st);
  } else if (epi == WS_RES) {
    run_ws<WS_RES, false>(a, lda, b, ldb, c, ldc, M, N, K, re, eps, st);
  } else {
    if (rs) run_ws<WS_NONE, true>(a, lda, b, ldb, c, ldc, M, N, K, re, eps, st);
    else run_ws<WS_NONE, false>(a, lda, b, ldb, c, ldc, M, N, K, re, eps, st);
  }
}

}  // namespace mlop

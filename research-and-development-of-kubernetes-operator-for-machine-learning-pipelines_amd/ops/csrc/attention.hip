// Paged attention over the block-table KV cache (K6 decode, and the ragged /
// chunked-prefill path of K7) with MFMA 16x16x32 bf16 on gfx950.
//
// Layouts (written by rope_cache.hip and the fused QKV GEMM epilogues):
//   k_cache[page, Hkv, 16, 128]  token-major  -> A operand of  S^T = K . Q^T
//   v_cache[page, Hkv, 16, 128]  token-major  -> staged in LDS, read back transposed
//                                                (ds_read_b64_tr_b16) as the A operand of
//                                                O^T = V^T . P^T
// A token's V row is one contiguous 256-B store for its writer (a decode token used to scatter
// 128 2-B stores over a dim-major page; scripts/bench_vt.py measured the two layouts).
// Both products keep the q-row on the lane (col = lane&15), so the online
// softmax (max, exp2, rescale of O) is entirely lane-local except the two
// cross-lane max steps (xor 16, xor 32), and P^T feeds the second MFMA straight
// from the first one's accumulator registers (cdna_hip_programming.md §3
// "An accumulator tile as the next MFMA's operand", with a permuted k order).
// Decode kernel token order of a page pair (A, B; pair token t = 16*page + offset):
// lane group g = lane>>4 owns the 8 CONSECUTIVE pair tokens 8g..8g+7 (K rows are
// loaded in a row order that makes it so: load_k) - so each lane's V^T fragment is two transposed
// 4-row reads of the pair's LDS image and P^T comes from the S registers as before.
//
// MFMA rows: 16 q-rows per tile = (16/G query tokens) x (G heads of one kv head).
// A workgroup = 4 waves = one (tile, kv head, kv partition); the waves split
// the partition's page pairs round-robin and merge (m, l, O) through LDS.
// Partitions > 1 (long context, small batch: fill 256 CUs) write fp32 partials
// that attn_reduce_kernel combines.
//
// Memory-bound: each K byte is loaded once per tile straight into VGPRs, 8 token rows x 128 B an instruction; each V
// byte once into the wave's LDS image by LDS-DMA (the transpose needs it in LDS).
//
// REQUIREMENT: the cache is zero-initialised at allocation (masked lanes multiply
// p = 0 with whatever the unused slots hold; NaN garbage would poison O).
#include <type_traits>
#include <algorithm>

#include "common.h"
#include "launch.h"

namespace mlop {

// exp2 as the bare v_exp_f32: exp2f() wraps it in a denormal-range rescale (v_cmp +
// v_cndmask + v_ldexp per call, a fifth of the flash loop's VALU).  Softmax arguments are
// <= 0, so results below 2^-126 flushing to 0 changes nothing that survives bf16 P / f32 l.
__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

constexpr int kD = 128;
constexpr int kBS = 16;
constexpr float kNegBig = -1.0e30f;

// token-major V image in LDS: [rows][256 B], 16-B chunk c of row t at slot c ^ vswz(t)
// (cdna_hip_programming.md T10 image (b)); filled by LDS-DMA through the source address and
// read back transposed with ds_read_b64_tr_b16: a half-wave's two 4-row blocks 8 rows apart in
// the same columns are conflict-free
__device__ __forceinline__ int vswz(int t) { return ((t & 3) << 2) | ((t >> 2) & 3); }
typedef short v4s16 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) v4s16 lds_v4s16;

// V^T fragment (A operand of O^T = V^T . P^T, 16x16x32) for dims 16d .. 16d+15 and image rows
// 8 g4 .. 8 g4 + 7 of lane group g4 = lane >> 4 (two ds_read_b64_tr_b16: rows +0..3, +4..7).
// Lane 4q + p of a group addresses row t = 8 g4 + 4h + q, dims 16d + 4p .. +3, i.e. byte
//   256 t + 16 ((2d + (p >> 1)) ^ vswz(t)) + 8 (p & 1) = vt_base(lane) ^ 32 d          (h = 0)
// because 2d only moves bits 5-7, which the rest leaves 0 (the image is 256-B aligned); rows
// t + 4 flip bit 0 of vswz and nothing else the offset uses, so h = 1 is (that ^ 16) + 1024: ONE
// base VGPR, two v_xor and an immediate offset per fragment.
__device__ __forceinline__ uint32_t vt_base(int lane) {
  const int g4 = lane >> 4, q = (lane >> 2) & 3, p = lane & 3;
  const int row = 8 * g4 + q, sw = vswz(row & 15);
  return 256u * row + 16u * ((p >> 1) ^ (sw & 1)) + 8u * (p & 1) + 32u * (sw >> 1);
}
// the fragments of four dim blocks d..d+3 (b = vt_base ^ 32 d), read and waited for in one statement: the compiler
// orders LDS reads that it knows of behind every vector memory operation in flight, not only behind the image's DMA
__device__ __forceinline__ void vt_frag4(uint32_t b, bf16x8 (&f)[4]) {
  v4s16 r[8];
  const uint32_t a0 = b, a1 = b ^ 32u, a2 = b ^ 64u, a3 = b ^ 96u;
  asm volatile(
      "ds_read_b64_tr_b16 %0, %8\n"
      "ds_read_b64_tr_b16 %1, %9 offset:1024\n"
      "ds_read_b64_tr_b16 %2, %10\n"
      "ds_read_b64_tr_b16 %3, %11 offset:1024\n"
      "ds_read_b64_tr_b16 %4, %12\n"
      "ds_read_b64_tr_b16 %5, %13 offset:1024\n"
      "ds_read_b64_tr_b16 %6, %14\n"
      "ds_read_b64_tr_b16 %7, %15 offset:1024\n"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(r[0]), "=&v"(r[1]), "=&v"(r[2]), "=&v"(r[3]), "=&v"(r[4]), "=&v"(r[5]), "=&v"(r[6]), "=&v"(r[7])
      : "v"(a0), "v"(a0 ^ 16u), "v"(a1), "v"(a1 ^ 16u), "v"(a2), "v"(a2 ^ 16u), "v"(a3), "v"(a3 ^ 16u)
      : "memory");
#pragma unroll
  for (int d = 0; d < 4; ++d)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      f[d][e] = r[2 * d][e];
      f[d][4 + e] = r[2 * d + 1][e];
    }
}

__device__ __forceinline__ int wid_of(unsigned t) { return __builtin_amdgcn_readfirstlane((int)(t >> 6)); }

constexpr int kEnoughParts = 8;
// Keys per partition of one sequence: `even` shares of its own keys where a launch's lengths are alike.  (A captured
// decode step plans for the longest context the engine admits; a fixed length cut for that one leaves shorter
// sequences on a few workgroups: 13 sequences of 2500 keys under a limit of 4096 on 5 of 8 partitions.)
// A sequence of more than 1.6 times the launch's mean is what the launch would end on: it gets up to the nparts that
// were planned, of a 512th of the launch's keys or 512 keys each (8 kv heads, whole or in two -> so: 1 x 4000 keys beside
// 40 x 200 67 -> 28 us, 1 x 24000 beside 20 x 500 195 -> 102, 10 x 4000 beside 10 x 100 70 -> 43).  From kEnoughParts shares
// on, further slabs cost what shorter walks save (2 x 16000 beside 2 x 200 in 8 shares 38.7 us, in 31 45.5).  Every
// workgroup of the launch and the reduction sum the same integers.
__device__ __forceinline__ int seq_part(int kv_end, int part_tokens, int nparts, int even, int even_from, const int* load,
                                        const int* tile_seq, const int* ctx_len, int tiles, int Hkv) {
  constexpr int min_part = 128;  // attn_meta.MIN_PART
  constexpr int long_part = 512;
  if (nparts == 1) return part_tokens;
  // (by the mean where the host has summed them: a launch of which some sequences are cut is slower than either)
  if (even_from > 0 && (load != nullptr ? load[0] < (long)even_from * load[1] : kv_end < even_from)) even = 1;
  int n = even;
  if (even < nparts && kv_end > long_part * 3 / 2 * even) {  // (two long shares or more)
    float sum = 0.f;  // (below 2^24 exact, above the same everywhere)
    int live = 0;
    if (load != nullptr) {
      sum = threadIdx.x & 63 ? 0.f : (float)load[0];
      live = load[1];
      tiles = 0;
    }
    for (int i = 0; i < tiles; i += 256) {
      const int l = i + (threadIdx.x & 63);
      int c[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) c[u] = tile_seq[min(l + 64 * u, tiles - 1)];
#pragma unroll
      for (int u = 0; u < 4; ++u) c[u] = ctx_len[c[u]];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const bool in = l + 64 * u < tiles && c[u] > 0;
        sum += in ? (float)c[u] : 0.f;
        live += __popcll(__ballot(in));
      }
    }
    const int keys = __builtin_amdgcn_readfirstlane((int)wave_sum(sum));  // (uniform: page numbers hang on it)
    if (10l * kv_end * live > 16l * keys) {
      const int share = max(long_part, (int)((long)keys * Hkv / 512));
      n = max(even, min(nparts, (kv_end + share / 2) / share));
    }
  }
  return max(min_part, ((kv_end + n - 1) / n + 31) & ~31);
}

// Row rr, dims c..c+7 of a (tile, kv head)'s combined output from its partitions' slabs.  Four partitions' loads
// are in flight together: one at a time, 32 partitions were 64 round trips behind each other.
__device__ __forceinline__ void combine_parts(const float* part_o, const float* part_ml, size_t base, int nvalid, int rr,
                                              int c, u32x4& ov) {
  constexpr int U = 4;
  float M = kNegBig, L = 0.f, a[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  for (int p0 = 0; p0 < nvalid; p0 += U) {
    float2 ml[U];
    float4 x[U], y[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {  // past the end: the last partition again, weighted 0
      const size_t pb = (base + min(p0 + u, nvalid - 1)) * 16 + rr;
      ml[u] = *reinterpret_cast<const float2*>(part_ml + pb * 2);
      const float4* po = reinterpret_cast<const float4*>(part_o + pb * kD + c);
      x[u] = po[0];
      y[u] = po[1];
    }
    float mn = M;
#pragma unroll
    for (int u = 0; u < U; ++u) mn = fmaxf(mn, ml[u].x);
    const float alpha = exp2f(M - mn);
    M = mn;
    L *= alpha;
#pragma unroll
    for (int j = 0; j < 8; ++j) a[j] *= alpha;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const float f = p0 + u < nvalid ? exp2f(ml[u].x - mn) : 0.f;
      L += f * ml[u].y;
      a[0] += f * x[u].x; a[1] += f * x[u].y; a[2] += f * x[u].z; a[3] += f * x[u].w;
      a[4] += f * y[u].x; a[5] += f * y[u].y; a[6] += f * y[u].z; a[7] += f * y[u].w;
    }
  }
  const float inv = L > 0.f ? 1.f / L : 0.f;
#pragma unroll
  for (int j = 0; j < 4; ++j) ov[j] = pack2(a[2 * j] * inv, a[2 * j + 1] * inv);
}

template <int G, int NT, bool BY_HEAD>  // NT bit 0: K / V loads non-temporal, bit 1: the output stores
__global__ void __launch_bounds__(256, 3) paged_attn_kernel(
    uint16_t* __restrict__ out, float* __restrict__ part_o, float* __restrict__ part_ml,
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ kc,
    const uint16_t* __restrict__ vc, const int* __restrict__ block_tables, int bt_stride,
    const int* __restrict__ tile_seq, const int* __restrict__ tile_q0,
    const int* __restrict__ q_start, const int* __restrict__ q_len,
    const int* __restrict__ ctx_len, int Hq, int Hkv, float scale_log2, int part_tokens,
    int nparts, int even, int even_from, int num_blocks, int* __restrict__ sem, const int* __restrict__ load) {
  constexpr int QT = 16 / G;
  // (3 waves per SIMD: 154 VGPRs; asked for two fewer the compiler keeps O in AGPRs and copies it for every rescale)
  // wave w stages its page pair's V image (2 x 16 token rows x 256 B = 8 KB) inside sm_o[w]
  // (8448 B, 256-B aligned: vt_frag), which it alone writes after its loop.  (A second image per
  // wave, prefetching the next pair, measured 1-4 % SLOWER on every decode shape: r04 profile.)
  __shared__ __attribute__((aligned(256))) float sm_o[4][16][kD + 4];
  __shared__ float sm_m[4][16];
  __shared__ float sm_l[4][16];
  __shared__ int sm_last;

  const int tile = BY_HEAD ? blockIdx.y : blockIdx.x, kvh = BY_HEAD ? blockIdx.x : blockIdx.y, part = blockIdx.z;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int s = tile_seq[tile], q0 = tile_q0[tile];
  const int* bt = block_tables + (size_t)s * bt_stride;
  const int ql = q_len[s], ctx = ctx_len[s], qs = q_start[s];
  const int last_q = min(q0 + QT, ql) - 1;           // last valid query of the tile
  const int kv_end = last_q >= 0 ? ctx - ql + last_q + 1 : 0;
  part_tokens = seq_part(kv_end, part_tokens, nparts, even, even_from, load, tile_seq, ctx_len, BY_HEAD ? gridDim.y : gridDim.x, Hkv);
  const int p_begin = part * part_tokens;
  const int p_end = min(kv_end, p_begin + part_tokens);
  if (p_begin >= p_end) {                            // reducer skips empty partitions
    // kv_end == 0 (graph-bucket padding rows, ctx 0): no partition draws the last ticket of
    // the in-launch combine, so partition 0 writes the zero row attn_reduce_kernel would
    if ((sem != nullptr || nparts == 1) && part == 0 && kv_end <= 0) {
      const int rr = threadIdx.x >> 4, c = (threadIdx.x & 15) * 8;
      const int qi2 = q0 + rr / G;
      if (qi2 < ql)
        *reinterpret_cast<u32x4*>(out + ((size_t)(qs + qi2) * Hq + kvh * G + (rr % G)) * kD + c) =
            u32x4{0u, 0u, 0u, 0u};
    }
    return;
  }

  // this lane's q-row (B operand column) and its causal limit
  const int r = lane & 15, g4 = lane >> 4;
  const int qi = q0 + r / G;
  const bool row_ok = qi < ql;
  const int head = kvh * G + (r % G);
  const int pos_r = row_ok ? ctx - ql + qi : -1;

  bf16x8 qf[2][2];  // [half of the head's dims][even / odd 16-B chunks]
  {
    const uint16_t* qrow = q + ((size_t)(qs + (row_ok ? qi : 0)) * Hq + head) * kD;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        bf16x8 v = *reinterpret_cast<const bf16x8*>(qrow + h * 64 + g4 * 16 + x * 8);
        qf[h][x] = row_ok ? v : bf16x8{0, 0, 0, 0, 0, 0, 0, 0};
      }
  }

  f32x4 o[8];
#pragma unroll
  for (int d = 0; d < 8; ++d) o[d] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = kNegBig, l = 0.f;

  const int pp_begin = p_begin >> 5;
  const int pp_end = (p_end + 31) >> 5;
  const int n_pages = (p_end + kBS - 1) / kBS;
  const size_t page_stride = (size_t)Hkv * kBS * kD;

  // (a generic pointer's low 32 bits are the LDS offset)
  const uint32_t vimg = (uint32_t)(uintptr_t)&sm_o[0][0][0] + wid * 8448u;
  // clamp: a corrupt block table must not become an out-of-bounds fault
  auto page_of = [&](int raw) { return min(max(raw, 0), num_blocks - 1); };
  // the pair's 32 token rows of this kv head by LDS-DMA into this wave's V image
  uint32_t vo[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) vo[i] = (4 * i + g4) * (2 * kD) + ((r ^ vswz(4 * i + g4)) << 4);
  auto issue_v = [&](int pa, int pb) {
    const uint16_t* vh = vc + (size_t)kvh * kBS * kD;
    const auto rA = __builtin_amdgcn_make_buffer_rsrc((void*)(vh + pa * page_stride), 0, kBS * kD * 2, 0x00020000);
    const auto rB = __builtin_amdgcn_make_buffer_rsrc((void*)(vh + pb * page_stride), 0, kBS * kD * 2, 0x00020000);
#pragma unroll
    for (int i = 0; i < 4; ++i) lds_dma16(rA, vimg + 1024u * i, vo[i], NT & 1);
#pragma unroll
    for (int i = 0; i < 4; ++i) lds_dma16(rB, vimg + 4096u + 1024u * i, vo[i], NT & 1);
  };
  // K: instruction (t, h) loads half h (128 B, a whole line) of 8 token rows.  MFMA row r holds the chunks 2 g4 + (r & 1) of
  // the half of pair token 8 (r >> 2) + 2 t + ((r >> 1) & 1); multiplied with Q's even chunks its even rows count, with the
  // odd ones its odd rows, and a lane's accumulators 0 and 2 of the one and 1 and 3 of the other make its tokens
  // 8 g4 + 2 t and + 1.  (Twice the MFMAs, of which there are plenty.)
  bf16x8 kf[4][2];
  auto load_k = [&](int pa, int pb) {
    const uint16_t* kP = kc + (r >> 3 ? pb : pa) * page_stride + (size_t)kvh * kBS * kD;
    const uint16_t* kR = kP + (8 * ((r >> 2) & 1) + ((r >> 1) & 1)) * kD + g4 * 16 + (r & 1) * 8;
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const bf16x8* p = reinterpret_cast<const bf16x8*>(kR + 2 * t * kD + h * 64);
        if constexpr ((NT & 1) != 0) kf[t][h] = __builtin_nontemporal_load(p);
        else kf[t][h] = *p;
      }
  };
  // A pair's K loads (registers) and V image (LDS) are issued a pair ahead: K(p + 4) as soon as the S MFMAs have
  // taken K(p), V(p + 4) as soon as the transposed reads have taken V(p).  The workgroups of a launch run in step, and
  // memory stood still while they all multiplied (100 sequences of 1000 keys 96.7 -> 90.2 us, 64 of 4000 217 -> 196).
  // Each is waited for alone, by count: with the global form of LDS-DMA the compiler waited for K and V together at the
  // loop's top, and with 16 rows x 64 B per K instruction (one MFMA each) every line was asked for twice.  Both together, us per
  // launch, 8 kv heads: 7 x 1000 keys 12.2 -> 10.4, 13 x 2500 34.8 -> 29.7, 20 x 800 22.2 -> 15.6, 100 x 1000 83.1 -> 74.5, 300 x
  // 600 130 -> 122, 700 x 500 243 -> 234 (6.1 TB/s).
  int pgA = 0, pgB = 0, rawA = 0, rawB = 0;  // page ids of the pair whose K is loading; the next pair's as read
  auto load_pages = [&](int pp) {  // (past the end: entries of the row, never used)
    rawA = bt[min(2 * pp, bt_stride - 1)];
    rawB = bt[min(2 * pp + 1, bt_stride - 1)];
  };
  auto take_pages = [&](int pp) {
    pgA = page_of(rawA);
    pgB = 2 * pp + 1 < n_pages ? page_of(rawB) : pgA;
  };
  int pp = pp_begin + wid_of(threadIdx.x);
  {
    // (a wave without a pair loads the last one and waits for it)
    const int first = min(pp, pp_end - 1);
    load_pages(first);
    take_pages(first);
    load_k(pgA, pgB);
    asm volatile("" ::: "memory");
    load_pages(pp + 4);
    asm volatile("" ::: "memory");
    issue_v(pgA, pgB);
  }
  auto pair = [&](auto more_) {
    constexpr bool more = decltype(more_)::value;
    // S^T[token][row]: lane holds row r, tokens 8 g4 + i of the pair
    float sc[8];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      f32x4 e = {0.f, 0.f, 0.f, 0.f}, d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        e = mfma16(kf[t][h], qf[h][0], e);
        d = mfma16(kf[t][h], qf[h][1], d);
      }
      sc[2 * t] = e[0] + d[1];
      sc[2 * t + 1] = e[2] + d[3];
    }
    // the next K loads stay behind the MFMAs that read this pair's
    asm volatile("" : "+v"(sc[0]), "+v"(sc[1]), "+v"(sc[2]), "+v"(sc[3]), "+v"(sc[4]), "+v"(sc[5]), "+v"(sc[6]), "+v"(sc[7])::"memory");
    if constexpr (more) {
      take_pages(pp + 4);
      load_k(pgA, pgB);
      asm volatile("" ::: "memory");
      load_pages(pp + 8);
      asm volatile("" ::: "memory");
    }
    const int tok = pp * 32 + g4 * 8;
    float mx = kNegBig;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      sc[i] = (tok + i < p_end && tok + i <= pos_r) ? sc[i] * scale_log2 : -INFINITY;
      mx = fmaxf(mx, sc[i]);
    }
    mx = max_x16_x32(mx);
    const float m_new = fmaxf(m, mx);
    const float alpha = fast_exp2(m - m_new);
    m = m_new;
    float rs = 0.f;
    bf16x8 pf;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      sc[i] = fast_exp2(sc[i] - m_new);
      rs += sc[i];
      pf[i] = (short)f2bf(sc[i]);
    }
    l = l * alpha + rs;
    // this wave's V image has landed: at least the eight K loads are younger
    if constexpr (more) asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    const uint32_t b0 = vimg + vt_base(lane);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      bf16x8 vf[4];
      vt_frag4(b0 ^ (128u * h), vf);
      if constexpr (more) {
        if (h == 1) issue_v(pgA, pgB);  // the image is in registers
      }
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        o[4 * h + d] *= alpha;
        o[4 * h + d] = mfma16(vf[d], pf, o[4 * h + d]);
      }
    }
  };
  for (; pp + 4 < pp_end; pp += 4) pair(std::true_type{});
  if (pp < pp_end) pair(std::false_type{});
  else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

  l = sum_x16_x32(l);
  // O^T[d][row]: lane holds row r, dims 16*dblk + 4*g4 + i
#pragma unroll
  for (int d = 0; d < 8; ++d)
#pragma unroll
    for (int i = 0; i < 4; ++i) sm_o[wid][r][d * 16 + g4 * 4 + i] = o[d][i];
  if (g4 == 0) {
    sm_m[wid][r] = m;
    sm_l[wid][r] = l;
  }
  __syncthreads();

  const int rr = threadIdx.x >> 4, c = (threadIdx.x & 15) * 8;
  float M = kNegBig;
#pragma unroll
  for (int w = 0; w < 4; ++w) M = fmaxf(M, sm_m[w][rr]);
  float L = 0.f, acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    const float f = exp2f(sm_m[w][rr] - M);
    L += f * sm_l[w][rr];
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[j] += f * sm_o[w][rr][c + j];
  }
  const int qi2 = q0 + rr / G;
  const bool row_valid = qi2 < ql;
  const int head2 = kvh * G + (rr % G);
  const int nvalid = min(nparts, (kv_end + part_tokens - 1) / part_tokens);
  if (nvalid == 1) {  // nothing to combine
    if (!row_valid) return;
    const float inv = L > 0.f ? 1.f / L : 0.f;
    u32x4 ov;
#pragma unroll
    for (int j = 0; j < 4; ++j) ov[j] = pack2(acc[2 * j] * inv, acc[2 * j + 1] * inv);
    u32x4* dst = reinterpret_cast<u32x4*>(out + ((size_t)(qs + qi2) * Hq + head2) * kD + c);
    if constexpr ((NT & 2) != 0) __builtin_nontemporal_store(ov, dst);
    else *dst = ov;
    return;
  }
  if (row_valid) {
    // The slab is stored sc1 (write-through to L2) so that the hand-off below needs no
    // agent release (MI355X_MICROARCH.md, hand-off producer rule (2)).  Buffer offsets
    // are relative to this (tile, kvh, part) slab: 16 rows x kD floats, 16 x 2 floats.
    const size_t slab = (((size_t)tile * Hkv + kvh) * nparts + part) * 16;
    const auto rs_o = __builtin_amdgcn_make_buffer_rsrc(part_o + slab * kD, 0, 16 * kD * 4, 0x00020000);
    const uint32_t oo = (uint32_t)(rr * kD + c) * 4u;
    u32x4 w0, w1;
    w0[0] = __float_as_uint(acc[0]); w0[1] = __float_as_uint(acc[1]);
    w0[2] = __float_as_uint(acc[2]); w0[3] = __float_as_uint(acc[3]);
    w1[0] = __float_as_uint(acc[4]); w1[1] = __float_as_uint(acc[5]);
    w1[2] = __float_as_uint(acc[6]); w1[3] = __float_as_uint(acc[7]);
    __builtin_amdgcn_raw_buffer_store_b128(w0, rs_o, oo, 0, 16 /* sc1 */);
    __builtin_amdgcn_raw_buffer_store_b128(w1, rs_o, oo + 16u, 0, 16 /* sc1 */);
    if ((threadIdx.x & 15) == 0) {
      const auto rs_ml = __builtin_amdgcn_make_buffer_rsrc(part_ml + slab * 2, 0, 16 * 2 * 4, 0x00020000);
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(M), rs_ml, (uint32_t)rr * 8u, 0, 16);
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(L), rs_ml, (uint32_t)rr * 8u + 4u, 0, 16);
    }
  }
  if (sem == nullptr) return;  // attn_reduce_kernel combines in a second launch
  // In-launch combine (cdna_hip_programming.md §5 split-K item 2, counter form of the
  // §6 Guideline 16 hand-off).  Producer: sc1 stores, every wave waits vmcnt(0), a
  // workgroup barrier, then one lane draws a relaxed agent-scope ticket -- no release
  // fence (it cost every partition an L2 writeback).  Consumer: the partition that draws
  // nvalid-1 keeps the agent acquire (this kernel runs two workgroups per CU, outside the
  // guide's fence-free table row) and reduces every slab, then re-arms the counter for
  // the next launch (the buffer is zero-initialised once).
  int* cnt = sem + (size_t)tile * Hkv + kvh;
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x == 0) {
    const int t = __hip_atomic_fetch_add(cnt, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    sm_last = (t == nvalid - 1);
  }
  __syncthreads();
  if (!sm_last) return;
  if (threadIdx.x == 0) {
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __hip_atomic_store(cnt, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  if (!row_valid) return;
  const size_t base = ((size_t)tile * Hkv + kvh) * nparts;
  u32x4 ov;
  combine_parts(part_o, part_ml, base, nvalid, rr, c, ov);
  *reinterpret_cast<u32x4*>(out + ((size_t)(qs + qi2) * Hq + head2) * kD + c) = ov;
}

template <int G>
__global__ void __launch_bounds__(256) attn_reduce_kernel(
    uint16_t* __restrict__ out, const float* __restrict__ part_o,
    const float* __restrict__ part_ml, const int* __restrict__ tile_seq,
    const int* __restrict__ tile_q0, const int* __restrict__ q_start,
    const int* __restrict__ q_len, const int* __restrict__ ctx_len, int Hq, int Hkv,
    int part_tokens, int nparts, int even, int even_from, const int* __restrict__ load) {
  constexpr int QT = 16 / G;
  const int tile = blockIdx.x, kvh = blockIdx.y;
  const int s = tile_seq[tile], q0 = tile_q0[tile];
  const int ql = q_len[s], ctx = ctx_len[s], qs = q_start[s];
  const int last_q = min(q0 + QT, ql) - 1;
  const int kv_end = last_q >= 0 ? ctx - ql + last_q + 1 : 0;
  part_tokens = seq_part(kv_end, part_tokens, nparts, even, even_from, load, tile_seq, ctx_len, gridDim.x, Hkv);
  const int nvalid = min(nparts, (kv_end + part_tokens - 1) / part_tokens);
  const int rr = threadIdx.x >> 4, c = (threadIdx.x & 15) * 8;
  const int qi = q0 + rr / G;
  if (qi >= ql || nvalid == 1) return;  // (one partition: written by the kernel before)
  const size_t base = ((size_t)tile * Hkv + kvh) * nparts;
  u32x4 ov;
  combine_parts(part_o, part_ml, base, nvalid, rr, c, ov);
  const int head = kvh * G + (rr % G);
  *reinterpret_cast<u32x4*>(out + ((size_t)(qs + qi) * Hq + head) * kD + c) = ov;
}

// K / V pages of the decode kernel non-temporal (read once per step by one workgroup; the
// headline step reads ~100 GB of them): headline +2.2 / +3.2 % interleaved (attn_kv_nt op, bit
// 0); bit 1 the output stores too (with gemm_slab_nt bit 3: +0.5 %)
static int g_attn_kv_nt = 3;
int attn_kv_nt(int set) {
  if (set >= 0) g_attn_kv_nt = set;
  return g_attn_kv_nt;
}

// Partitions of a sequence in a launch of `base` (tile, kv head) pairs of like lengths, and the keys from which on a sequence
// is cut into them.  A CU reads its pages at up to 35 GB/s however many workgroups it has, all of them together 6.3 TB/s.  So in
// units of the launch's bytes at that rate, w workgroups of equal shares take a 256 / w for the a = w / 256 that every CU has and
// max(180, w % 256) / w for the rest: 136 pairs whole 1.32, in 2 / 3 / 4 shares 1.60 / 1.07 / 1.27 (measured, 17 x 4000 keys 57.1, 64.0,
// 51.4, 56.2 us); 192 1.0, 1.14, 1.20, 1.0 (24 x 4000 68.2, 75.5, 76.0, 70.2); 264 1.65, 1.31, 1.20, 1.14 (33 x 4000 111, 103, 101, 98.9).
// A cut costs its slabs, tickets and combining, 2.6 - 4.2 us, which short contexts do not earn back: 16 x 300 keys whole 7.6
// us, in 2 shares 8.8, 16 x 1000 17.1 and 15.5; 24 x 300 8.5, 11.2; 20 x 1000 18.9, 19.2 in 3.
struct EvenParts {
  int n, from;
};
static EvenParts even_parts(int base, int nparts) {
  // few pairs: the CUs filled once (1 x 24000 keys 47 us in four workgroups per CU, 27.6 so; a share has 128 keys at least)
  if (base <= kCus / 4) return {std::min(nparts, kCus / base), 0};
  auto model = [&](int n) {
    const int w = n * base, a = w / kCus, r = w % kCus;
    return (float)(a * kCus + (r ? std::max(180, r) : 0)) / (float)w;
  };
  const int most = std::min(nparts, 4);
  int n = 1;
  float best = model(1);
  for (int i = 2; i <= most; ++i) {
    const float t = model(i) + .05f + .01f * (float)i;
    if (t < best - .01f * (n == 1)) best = t, n = i;
  }
  if (n == 1) return {1, 0};
  // a key of `base` pairs is base / 12300 us of the launch; above 256 pairs unequal lengths hide part of a whole launch's end
  const float gain = std::max(model(1) - model(n), .01f) * (base > kCus ? .6f : 1.f);
  return {n, (int)std::min(1e6f, (n == 4 ? 4.2f : 2.6f) * 12300.f / ((float)base * gain))};
}

template <int G>
static void launch_g(void* out, float* part_o, float* part_ml, const void* q, const void* kc,
                     const void* vc, const int* bt, int bt_stride, const int* tile_seq,
                     const int* tile_q0, const int* q_start, const int* q_len, const int* ctx_len,
                     int num_tiles, int Hq, int Hkv, float scale_log2, int part_tokens, int nparts,
                     int num_blocks, int* sem, const int* load, hipStream_t st) {
  const EvenParts ep = even_parts(num_tiles * Hkv, nparts);
  const int even = ep.n, even_from = ep.from;
  if (num_tiles == 1 || even >= kEnoughParts) {  // (seq_part: none needs more)
    if (even == 1 && nparts > 1) part_tokens = 1 << 30;  // the only partition has all keys, whatever was planned
    nparts = even;
  }
  // Above 32 tiles of 8 kv heads the heads are the grid's fastest index: a page holds the heads' 4-KB blocks one behind the
  // other, and whatever workgroups run at a time read them all.  With tiles fastest a launch ended on two heads, a quarter of
  // every page (a step of 40 x 8000 keys 2620 -> 2518 us, 48 x 7000 2472 -> 2408, 200 x 1500 2562 -> 2507, 700 x 500 4119 -> 4084).
  // 32 tiles of 8 heads are one workgroup per CU, no order to gain from (32 x 800 23.5 us, heads fastest 23.9).  Fewer heads are
  // less of a page than that anyhow, and one tile's heads end together: 2 and 4 heads (a tensor-parallel shard's) lose 1 -
  // 3 % at 24 - 200 tiles on average and 8 % at worst (4 heads, 36 tiles of 4000 keys 63.0 -> 67.0 us), and gain 1 - 5 % from 250 -
  // 300 on.  Kernel times by heads fastest over tiles fastest, contexts of 500 - 20000, means over 4 - 24 launches: 8 heads 1.00
  // at 24 tiles, 0.99 at 28, 1.01 / 0.97 / 0.98 / 0.96 / 0.94 / 0.96 at 32 / 36 / 40 / 64 / 80 / 150, 1.02 at 300 - 700 of equal lengths
  // and 0.99 of unequal ones; 16 and 32 heads 0.97 - 1.0 from 32 on; 4 heads 1.02 / 1.02 / 1.01 / 0.98 / 0.95 at 32 / 64 / 150 / 300 /
  // 700.  A kernel of its own for each order: chosen inside, by a division of the linear index, it cost every launch 0.2 us
  // (7 x 1000 keys 12.05 -> 12.3).
  const bool by_head = Hkv > 1 && num_tiles >= (Hkv >= 8 ? 33 : 256) && num_tiles <= 65535;  // (the grid's second dimension)
  const dim3 grid = by_head ? dim3(Hkv, num_tiles, nparts) : dim3(num_tiles, Hkv, nparts);
  // K / V pages non-temporal (attn_kv_nt op): each is read once per step by one workgroup (1 x 24000 keys 22.5 -> 20.8 us, 3 x
  // 24000 55.1 -> 51.0; while a line of K was read in two halves few tiles were faster cached)
  const int nt = g_attn_kv_nt;
  auto pick = [&](auto h) {
    constexpr bool H = decltype(h)::value;
    return nt == 3 ? paged_attn_kernel<G, 3, H> : nt ? paged_attn_kernel<G, 1, H> : paged_attn_kernel<G, 0, H>;
  };
  auto kern = by_head ? pick(std::true_type{}) : pick(std::false_type{});
  kern<<<grid, 256, 0, st>>>((uint16_t*)out, part_o, part_ml, (const uint16_t*)q, (const uint16_t*)kc,
                             (const uint16_t*)vc, bt, bt_stride, tile_seq, tile_q0, q_start, q_len, ctx_len,
                             Hq, Hkv, scale_log2, part_tokens, nparts, even, even_from, num_blocks, sem, load);
  if (nparts > 1 && sem == nullptr) {
    attn_reduce_kernel<G><<<dim3(num_tiles, Hkv), 256, 0, st>>>(
        (uint16_t*)out, part_o, part_ml, tile_seq, tile_q0, q_start, q_len, ctx_len, Hq, Hkv,
        part_tokens, nparts, even, even_from, load);
  }
}

void launch_paged_attention(void* out, float* part_o, float* part_ml, const void* q,
                            const void* kc, const void* vc, const int* bt, int bt_stride,
                            const int* tile_seq, const int* tile_q0, const int* q_start,
                            const int* q_len, const int* ctx_len, int num_tiles, int Hq, int Hkv,
                            float scale_log2, int part_tokens, int nparts, int num_blocks,
                            int* sem, const int* load, hipStream_t st) {
  if (num_tiles == 0) return;
  const int G = Hq / Hkv;
#define MLOP_ATTN_CASE(GG)                                                                        \
  case GG:                                                                                        \
    launch_g<GG>(out, part_o, part_ml, q, kc, vc, bt, bt_stride, tile_seq, tile_q0, q_start,     \
                 q_len, ctx_len, num_tiles, Hq, Hkv, scale_log2, part_tokens, nparts, num_blocks, sem, load, st);   \
    break;
  switch (G) {
    MLOP_ATTN_CASE(1)
    MLOP_ATTN_CASE(2)
    MLOP_ATTN_CASE(4)
    MLOP_ATTN_CASE(8)
    MLOP_ATTN_CASE(16)
    default: break;
  }
#undef MLOP_ATTN_CASE
}

// ---------------------------------------------------------------------------
// K7 flash prefill on the 16x16x32 MFMA (cdna_hip_programming.md "Fused attention prefill":
// swapped QK^T, an accumulator tile as the next MFMA's operand).  One workgroup = 128 MFMA
// q-rows (128/G query tokens x the G heads of one kv head) against EVERY key of its causal
// range, so every K/V byte fetched from L2 feeds all 128 q-rows.  Page pairs (32 keys, 8 KB of K, 8 of V)
// stream through LDS rings of four by LDS-DMA (buffer form, counted vmcnt, one raw barrier per pair),
// swizzled through the SOURCE address:
//   K pair [32 keys][16 x 16 B]: chunk c of key k at slot c ^ (4 (k >> 3) + (k & 3)) (ds_read_b128)
//   V pair [32 keys][16 x 16 B]: chunk c of key k at slot c ^ vswz(k & 15)           (ds_read_b64_tr_b16)
// both conflict-free for the fragment reads below.  Per wave 32 q-rows, two per lane column (qb):
//   S^T [2 x 16 keys][2 x 16 q] = K . Q^T: 16 MFMAs (A = K rows by ds_read_b128, B = Q^T in registers); the
//     rows of A are keys 8 (i >> 2) + (i & 3) and + 4, so lane group g4 holds keys 8 g4 + 0 .. 7 of q column
//     l & 15: the row max and sum are lane-local, the quarters meet where the max moves and in the epilogue;
//   O^T [128 d][2 x 16 q] += V^T . P^T: 16 MFMAs, P^T straight from the S registers (bf16, 32 keys = one MFMA),
//     V^T by two ds_read_b64_tr_b16 per fragment from the token-major image.
// What bounds it at long contexts: power (1.7 GHz).  With a pair's three phases one behind the other (32x32x16 MFMAs),
// matrix and vector work overlapped only between a SIMD's waves; now each wave has the softmax of one pair between
// the MFMAs of S of the next and O of the one before (step), with a quarter fewer vector instructions, and the
// 16x16x32 MFMA does the same FLOPs on less power (registers only, all CUs: 2020 TFLOP/s against 1795).  A wave in its
// MFMAs goes before the SIMD's other one, which then does its waiting in the shadow (2048 x 11048 586 -> 570, 2 x 900
// 30.6 -> 28.2, 1 x 2048 47.7 -> 49).  us, phases in turn -> software pipeline -> now: 2048 queries of 64 heads at 11048
// keys 670 -> 613 -> 565 (1190 TFLOP/s), 512 at 4000 94 -> 82 -> 77; 32 heads, 2048 at 8000 250 -> 224 -> 205, prompts of
// 1 x 8192 550 -> 525 -> 464, 1 x 2048 57 -> 50.7 -> 49, 2 x 900 33.4 -> 30 -> 28.2, 3 x 333 14.2 -> 13 -> 12.5; many
// short ones, where the start of a workgroup counts and two of 214 registers share a CU that had three of 168, 16 x
// 500 61 -> 62 -> 60.5, 64 x 100 36 -> 38.5 -> 37.5.
using f32x16 = __attribute__((ext_vector_type(16))) float;
constexpr int kFlashRing = 4;  // pairs in flash_item's rings
constexpr int kFlashSplits = 16, kFlashPart = 128 * 128 + 2 * 128;  // most key ranges of a tile; floats of one: O, (max, sum) by rows
constexpr float kRescaleLog2 = 8.f;  // flash prefill's deferred-rescale threshold (exp2 units)
// two floats -> one dword of two bf16 in ONE v_cvt_pk_bf16_f32 (pack2's two scalar casts
// become two cvt + shift + or)
__device__ __forceinline__ uint32_t cvt_pk_bf16(float lo, float hi) {
  uint32_t r;
  asm("v_cvt_pk_bf16_f32 %0, %1, %2" : "=v"(r) : "v"(lo), "v"(hi));
  return r;
}
__device__ __forceinline__ f32x16 mfma32(bf16x8 a, bf16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}
// byte offset (page 0, dim block 0, rows 4h + q) of lane l's first transposed V read: lane
// 4q + p of 16-lane group g addresses row t = 4h + q, chunk 2 (g & 1) + (p >> 1), half p & 1.
// Dim block dblk flips address bits 6-7 (^ 64 dblk: the chunk's high bits only meet q there),
// rows + 8 flip bit 5 and add 2048, page B adds 4096.
__device__ __forceinline__ uint32_t vt32_base(int lane) {
  const int g = lane >> 4, h = lane >> 5, q = (lane >> 2) & 3, p = lane & 3;
  const int t = 4 * h + q, c = 2 * (g & 1) + (p >> 1);
  return 256u * t + 16u * (c ^ vswz(t)) + 8u * (p & 1);
}

// s_waitcnt lgkmcnt(W) for the reads of a (and b), then c += a . b, or c = a . b, in place.  As builtins the compiler gives the
// results registers of their own, 64 of the output's beside the 64 they replace, and pads each MFMA behind an asm wait.  It
// does not know this asm for an MFMA: vector instructions that read c wait for mfma16_settle or stand behind eight more MFMAs,
// as does the next one on c.
template <int W, bool ZERO = false>
__device__ __forceinline__ void mfma16_into(f32x4& c, const bf16x8& a, const bf16x8& b) {
  if constexpr (ZERO) {
    if constexpr (W >= 0) asm volatile("s_waitcnt lgkmcnt(%3)\nv_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=&v"(c) : "v"(a), "v"(b), "n"(W));
    else asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=&v"(c) : "v"(a), "v"(b));
  } else {
    if constexpr (W >= 0) asm volatile("s_waitcnt lgkmcnt(%3)\nv_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(c) : "v"(a), "v"(b), "n"(W));
    else asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(c) : "v"(a), "v"(b));
  }
}
__device__ __forceinline__ void mfma16_settle(f32x4 (&c)[8][2]) {
  asm volatile("s_nop 15\ns_nop 3"
               : "+v"(c[0][0]), "+v"(c[0][1]), "+v"(c[1][0]), "+v"(c[1][1]), "+v"(c[2][0]), "+v"(c[2][1]), "+v"(c[3][0]), "+v"(c[3][1]),
                 "+v"(c[4][0]), "+v"(c[4][1]), "+v"(c[5][0]), "+v"(c[5][1]), "+v"(c[6][0]), "+v"(c[6][1]), "+v"(c[7][0]), "+v"(c[7][1]));
}

// one flash tile (128 q-rows of ONE kv head against its whole causal key range, or, SPLIT, pairs n split / n_splits .. of its n
// pairs: O unnormalised [128][128] and (max, sum) [128][2] of the rows to part)
template <int G, bool SPLIT>
__device__ __forceinline__ void flash_item(
    uint16_t* smem, int tile, int kvh, uint16_t* __restrict__ out, const uint16_t* __restrict__ q,
    const uint16_t* __restrict__ kc, const uint16_t* __restrict__ vc, const int* __restrict__ block_tables,
    int bt_stride, const int* __restrict__ ptile_seq, const int* __restrict__ ptile_q0,
    const int* __restrict__ q_start, const int* __restrict__ q_len, const int* __restrict__ ctx_len, int Hq,
    int Hkv, float scale_log2, int num_blocks, int split, int n_splits, float* __restrict__ part) {
  constexpr int QB = 128 / G;            // query tokens per workgroup
  constexpr int STAGES = kFlashRing;
  constexpr int STAGE = 4 * kBS * kD;    // bf16 per stage: K page A | K page B | V page A | V page B
  constexpr int PAGE = kBS * kD;
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int s = ptile_seq[tile], q0 = ptile_q0[tile];
  const int ql = q_len[s], ctx = ctx_len[s], qs = q_start[s];
  const int last_q = min(q0 + QB, ql) - 1;
  int kv_end = ctx - ql + last_q + 1, first_key = 0;
  if constexpr (SPLIT) {  // keys and positions from the range's first key on
    const int n = (kv_end + 31) >> 5, from = n * split / n_splits, to = n * (split + 1) / n_splits;
    if (from == to) {  // (no pair of a tile of few)
      if (threadIdx.x < 128) *reinterpret_cast<u32x2*>(part + 128 * 128 + 2 * threadIdx.x) = u32x2{0, 0};
      return;
    }
    first_key = 32 * from;
    kv_end = min(kv_end, 32 * to) - first_key;
  }
  const int n_pairs = (kv_end + 31) >> 5;
  const int n_pages = (kv_end + kBS - 1) / kBS;
  const int wg_min_pos = ctx - ql + q0 - first_key;
  const int r16 = lane & 15, g4 = lane >> 4;

  // this lane's two q rows (MFMA columns): R = 32 wid + 16 qb + r16
  int qi[2], pos_r[2];
  bool q_ok[2];
  bf16x8 qf[2][4];
  float m[2], l[2], mc[2], alpha[2];
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    const int R = 32 * wid + 16 * b + r16;
    qi[b] = q0 + R / G;
    q_ok[b] = qi[b] < ql;
    pos_r[b] = q_ok[b] ? ctx - ql + qi[b] - first_key : -1;  // (before the range: all of it masked, sums of 0)
    const uint16_t* qrow = q + ((size_t)(qs + (q_ok[b] ? qi[b] : 0)) * Hq + kvh * G + R % G) * kD + 8 * g4;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const bf16x8 v = *reinterpret_cast<const bf16x8*>(qrow + 32 * t);
      qf[b][t] = q_ok[b] ? v : bf16x8{0, 0, 0, 0, 0, 0, 0, 0};
    }
    m[b] = kNegBig, l[b] = 0.f, mc[b] = -kNegBig * scale_log2, alpha[b] = 1.f;
  }
  f32x4 o[8][2];
#pragma unroll
  for (int d = 0; d < 8; ++d)
#pragma unroll
    for (int b = 0; b < 2; ++b) o[d][b] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int* bt = block_tables + (size_t)s * bt_stride + first_key / kBS;
  const uint32_t page_bytes = (uint32_t)Hkv * (2 * PAGE);
  const int kkey = wid * 4 + (lane >> 4);
  const int ksw = (kkey >> 3) * 4 + (kkey & 3);  // (page B: + 8)
  const uint32_t k_off[2] = {2u * (uint32_t)(kkey * kD + ((r16 ^ ksw) << 3)), 2u * (uint32_t)(kkey * kD + ((r16 ^ ksw ^ 8) << 3))};
  const uint32_t v_off[1] = {2u * (uint32_t)(kkey * kD + ((r16 ^ vswz(kkey)) << 3))};
  const uint16_t* kh = kc + kvh * PAGE;
  const uint16_t* vh = vc + kvh * PAGE;
  struct Ids {
    int a, b;
  };
  struct Pages {
    uint64_t a, b;
  };
  // ids of pair pp (past the last page: the last), and their bytes from the first page (clamped: a corrupt block table must
  // not become an out-of-bounds fault)
  auto id_at = [&](uint32_t i) { return *reinterpret_cast<const int*>((const char*)bt + 4u * i); };
  auto ids_of = [&](int pp) {
    const uint32_t i = min(2 * pp, n_pages - 1);
    return Ids{id_at(i), id_at(min((int)i + 1, n_pages - 1))};
  };
  auto at = [&](int id) { return (uint64_t)(uint32_t)min(max(id, 0), num_blocks - 1) * page_bytes; };
  auto pages_of = [&](Ids i) { return Pages{at(i.a), at(i.b)}; };
  // a pair's two pages of K / of V into a slot of their ring
  const uint32_t ring = (uint32_t)(uintptr_t)smem + wid * 1024;
  auto issue = [&](const uint16_t* head, uint32_t off_a, uint32_t off_b, uint32_t slot, Pages pg) {
    auto page = [&](uint64_t at) { return __builtin_amdgcn_make_buffer_rsrc((void*)((const char*)head + at), 0, 2 * PAGE, 0x00020000); };
    lds_dma16(page(pg.a), ring + slot, off_a, 0);
    lds_dma16(page(pg.b), ring + slot + 2 * PAGE, off_b, 0);
  };
  constexpr uint32_t SLOT = 4 * PAGE, RING_V = STAGES * SLOT;  // bytes
  // K fragment (kb, t): key row 8 (r16 >> 2) + (r16 & 3) + 4 kb of the pair, chunk 4t + g4 at slot
  // (4t + g4) ^ r16: byte (k_b0 ^ 64 t) + 1024 kb
  const uint32_t k_b0 = (uint32_t)(uintptr_t)smem + (uint32_t)((8 * (r16 >> 2) + (r16 & 3)) * 256 + ((g4 ^ r16) << 4));
  const uint32_t v_b0 = (uint32_t)(uintptr_t)smem + RING_V + vt_base(lane);
  // The fragment reads are inline asm with counted waits: as plain loads the compiler reused one register set and waited
  // lgkmcnt(0) before every MFMA, and, for V, vmcnt(0) (it cannot tell them from the LDS-DMA in flight).  No scalar load may
  // be in flight beside them (it would be counted): page ids are loaded where a step's last read has landed.
  // (f = 2 t + kb)
#define MLOP_KREAD(f, r, so) \
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(r) : "v"(k_b0 ^ (64u * ((f) >> 1))), "n"((so) + 1024u * ((f) & 1)))
  // dims 16 d .. + 15 of keys 8 g4 + 0 .. 3 and + 4 .. 7; vx: a ring slot's bytes
#define MLOP_VREAD(d, r, vx, so)                                                                                        \
  asm volatile("ds_read_b64_tr_b16 %0, %2 offset:%4\nds_read_b64_tr_b16 %1, %3 offset:%5"                               \
               : "=&v"(r[0]), "=&v"(r[1])                                                                               \
               : "v"((v_b0 ^ (32u * (d))) + (vx)), "v"((v_b0 ^ (32u * (d)) ^ 16u) + (vx)), "n"(so), "n"((so) + 1024u))
  auto frag = [&](const v4s16 (&r)[2]) {
    bf16x8 f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      f[e] = r[0][e];
      f[4 + e] = r[1][e];
    }
    return f;
  };

  bool resc = false;
  using Sc = f32x4[2][2];  // S^T [kb][qb]: keys 8 g4 + 4 kb + 0 .. 3 of q row qb
  // Row max of a pair's scores (raw units; the scale folds into the exponent's FMA).  Deferred rescale: the running max
  // moves only when some row's new max exceeds it by more than 2^kRescaleLog2 in exp2 units (always on a row's first
  // keys: m starts at -1e30); otherwise P stays scaled against the old max, <= 2^8, which bf16 P and f32 O / l carry
  // exactly as well.  The quarters of a row's keys meet only when it does.  O takes the factor (resc) once the pair before
  // has been added to it.
  auto row_max = [&](Sc& sc, int pp) {
    if (pp * 32 + 31 > wg_min_pos) {  // a pair crossing the workgroup's causal diagonal
      // (a side effect keeps this a branch: if-converted, the 47 compare / select / add of the
      // mask ran on every pair, a third of the loop's VALU)
      asm volatile("");
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          const int tok = pp * 32 + 8 * g4 + k;
          sc[k >> 2][b][k & 3] = tok <= pos_r[b] ? sc[k >> 2][b][k & 3] : -INFINITY;
        }
    }
    float mx[2];
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const float x = fmaxf(fmaxf(sc[0][b][0], sc[0][b][1]), sc[0][b][2]), y = fmaxf(fmaxf(sc[0][b][3], sc[1][b][0]), sc[1][b][1]);
      mx[b] = fmaxf(fmaxf(x, y), fmaxf(sc[1][b][2], sc[1][b][3]));
    }
    if (__ballot(fmaf(mx[0], scale_log2, mc[0]) > kRescaleLog2) | __ballot(fmaf(mx[1], scale_log2, mc[1]) > kRescaleLog2)) {
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const float m_new = fmaxf(m[b], max_x16_x32(mx[b]));
        alpha[b] = fast_exp2((m[b] - m_new) * scale_log2);
        m[b] = m_new;
        mc[b] = -m_new * scale_log2;
        l[b] *= alpha[b];
      }
      resc = true;
    }
  };
  auto rescale = [&]() {
    if (resc) {
      mfma16_settle(o);
#pragma unroll
      for (int d = 0; d < 8; ++d)
#pragma unroll
        for (int b = 0; b < 2; ++b) o[d][b] *= alpha[b];
      resc = false;
    }
  };
  // P of element r of the lane's 2 x 8; every second makes a dword of the P^T fragments (r = 16: the last of them; a pair is
  // packed behind the next element's exponential, which a VALU instruction could not read at once)
  float rs, pe[2];
  auto soft = [&](int r, const Sc& sc, u32x4 (&w)[2]) {
    float p = 0.f;
    if (r < 16) p = fast_exp2(fmaf(sc[(r >> 2) & 1][r >> 3][r & 3], scale_log2, mc[r >> 3]));
    if (r > 0 && r % 2 == 0) {
      const int e = r - 2;
      rs = e % 8 == 0 ? pe[0] + pe[1] : rs + (pe[0] + pe[1]);
      asm volatile("v_cvt_pk_bf16_f32 %0, %2, %3" : "=v"(w[e >> 3][(e & 7) >> 1]), "+v"(rs) : "v"(pe[0]), "v"(pe[1]));
      if (e % 8 == 6) l[e >> 3] += rs;
    }
    if (r < 16) pe[r & 1] = p;
  };

#define MLOP_SLOT(t)                 \
  __builtin_amdgcn_sched_barrier(0); \
  soft(t, sc, wn);                   \
  __builtin_amdgcn_sched_barrier(0)
  // S += K . Q^T of fragment f (its wait, its two MFMAs with an element between, the next read), and O += V^T . P^T of d
#define MLOP_QK(f, n, t)                                                   \
  mfma16_into<n, ((f) < 2)>(sn[(f) & 1][0], kf[f], qf[0][(f) >> 1]);       \
  MLOP_SLOT(t);                                                            \
  mfma16_into<-1, ((f) < 2)>(sn[(f) & 1][1], kf[f], qf[1][(f) >> 1])
#define MLOP_PV(d, n, t)                        \
  mfma16_into<n>(o[d][0], frag(vf[d]), p0f);    \
  MLOP_SLOT(t);                                 \
  mfma16_into<-1>(o[d][1], frag(vf[d]), p1f)
  // Step pp: S(pp + 1) = K . Q^T and O += V^T . P(pp - 1)^T, 32 MFMAs, with an element of P(pp)'s softmax behind every
  // second, so that a wave's matrix and vector work overlap, and not only those of a SIMD's waves.  K is a pair ahead of the
  // softmax and V a pair behind it: rings of their own.  (pp = 0: no P before.)
  auto step = [&](auto p_, auto first_, int pp, Sc& sc, Sc& sn, const u32x4 (&wp)[2], u32x4 (&wn)[2], Pages p1, Ids i3, Pages& p3) {
    constexpr int P = decltype(p_)::value;
    constexpr bool FIRST = decltype(first_)::value;
    constexpr uint32_t ks = (P + 1) % STAGES * SLOT, vs = (P + STAGES - 1) % STAGES * SLOT;
    if (pp + 2 < n_pairs) wait_vmcnt<4>(); else wait_vmcnt<2>();
    raw_barrier();  // K of pp + 1 and V of pp - 1 visible to every wave; the slots of K pp and V pp - 2 free
    issue(vh, v_off[0], v_off[0], RING_V + ks, p1);
    p3 = pages_of(i3);
    if (pp + 3 < n_pairs) issue(kh, k_off[0], k_off[1], (P + 3) % STAGES * SLOT, p3);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the page ids
    bf16x8 kf[8];
    v4s16 vf[8][2];
#pragma unroll
    for (int f = 0; f < 8; ++f) MLOP_KREAD(f, kf[f], ks);
    row_max(sc, pp);
    __builtin_amdgcn_sched_barrier(0);
    // (reads in flight at each wait: the K behind this one, then V's by twos)
    __builtin_amdgcn_s_setprio(1);
    MLOP_QK(0, 7, 0);
    if constexpr (FIRST) {
      MLOP_QK(1, 6, 1); MLOP_SLOT(2);
      MLOP_QK(2, 5, 3); MLOP_SLOT(4);
      MLOP_QK(3, 4, 5); MLOP_SLOT(6);
      MLOP_QK(4, 3, 7); MLOP_SLOT(8);
      MLOP_QK(5, 2, 9); MLOP_SLOT(10);
      MLOP_QK(6, 1, 11); MLOP_SLOT(12);
      MLOP_QK(7, 0, 13); MLOP_SLOT(14); MLOP_SLOT(15);
    } else {
      MLOP_QK(1, 6, 1); MLOP_VREAD(0, vf[0], 0, vs);
      MLOP_QK(2, 7, 2); MLOP_VREAD(1, vf[1], 0, vs);
      MLOP_QK(3, 8, 3); MLOP_VREAD(2, vf[2], 0, vs);
      MLOP_QK(4, 9, 4); MLOP_VREAD(3, vf[3], 0, vs);
      MLOP_QK(5, 10, 5); MLOP_VREAD(4, vf[4], 0, vs);
      MLOP_QK(6, 11, 6); MLOP_VREAD(5, vf[5], 0, vs);
      MLOP_QK(7, 12, 7);
      const bf16x8 p0f = __builtin_bit_cast(bf16x8, wp[0]), p1f = __builtin_bit_cast(bf16x8, wp[1]);
      MLOP_PV(0, 10, 8); MLOP_VREAD(6, vf[6], 0, vs);
      MLOP_PV(1, 10, 9); MLOP_VREAD(7, vf[7], 0, vs);
      MLOP_PV(2, 10, 10);
      MLOP_PV(3, 8, 11);
      MLOP_PV(4, 6, 12);
      MLOP_PV(5, 4, 13);
      MLOP_PV(6, 2, 14);
      MLOP_PV(7, 0, 15);
    }
    __builtin_amdgcn_s_setprio(0);
    soft(16, sc, wn);
    rescale();
  };
  // The last pair: its softmax under O += V^T . P^T of the pair before, then its own
  auto finish = [&](Sc& sc, const u32x4 (&wp)[2]) {
    u32x4 wn[2];
    v4s16 vf[8][2];
    wait_vmcnt<0>();
    raw_barrier();
    const uint32_t v1 = (uint32_t)((n_pairs + STAGES - 2) % STAGES) * SLOT, v0 = (uint32_t)((n_pairs + STAGES - 1) % STAGES) * SLOT;
    row_max(sc, n_pairs - 1);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (n_pairs > 1) {
#pragma unroll
      for (int d = 0; d < 6; ++d) MLOP_VREAD(d, vf[d], v1, 0);
      const bf16x8 p0f = __builtin_bit_cast(bf16x8, wp[0]), p1f = __builtin_bit_cast(bf16x8, wp[1]);
      MLOP_PV(0, 10, 0); MLOP_VREAD(6, vf[6], v1, 0); MLOP_SLOT(1);
      MLOP_PV(1, 10, 2); MLOP_VREAD(7, vf[7], v1, 0); MLOP_SLOT(3);
      MLOP_PV(2, 10, 4); MLOP_SLOT(5);
      MLOP_PV(3, 8, 6); MLOP_SLOT(7);
      MLOP_PV(4, 6, 8); MLOP_SLOT(9);
      MLOP_PV(5, 4, 10); MLOP_SLOT(11);
      MLOP_PV(6, 2, 12); MLOP_SLOT(13);
      MLOP_PV(7, 0, 14); MLOP_SLOT(15);
    } else {
#pragma unroll
      for (int r = 0; r < 16; ++r) soft(r, sc, wn);
    }
    soft(16, sc, wn);
    rescale();
    const bf16x8 p0f = __builtin_bit_cast(bf16x8, wn[0]), p1f = __builtin_bit_cast(bf16x8, wn[1]);
#define MLOP_PV1(d, n)                       \
  mfma16_into<n>(o[d][0], frag(vf[d]), p0f); \
  mfma16_into<-1>(o[d][1], frag(vf[d]), p1f)
#pragma unroll
    for (int d = 0; d < 6; ++d) MLOP_VREAD(d, vf[d], v0, 0);
    MLOP_PV1(0, 10); MLOP_VREAD(6, vf[6], v0, 0);
    MLOP_PV1(1, 10); MLOP_VREAD(7, vf[7], v0, 0);
    MLOP_PV1(2, 10);
    MLOP_PV1(3, 8);
    MLOP_PV1(4, 6);
    MLOP_PV1(5, 4);
    MLOP_PV1(6, 2);
    MLOP_PV1(7, 0);
#undef MLOP_PV1
  };
#undef MLOP_SLOT
#undef MLOP_QK
#undef MLOP_PV
  // S of pair 0
  auto qk0 = [&](Sc& sc) {
    bf16x8 kf[8];
#pragma unroll
    for (int f = 0; f < 8; ++f) MLOP_KREAD(f, kf[f], 0);
#define MLOP_QK0(f, n)                                               \
  mfma16_into<n, ((f) < 2)>(sc[(f) & 1][0], kf[f], qf[0][(f) >> 1]); \
  mfma16_into<-1, ((f) < 2)>(sc[(f) & 1][1], kf[f], qf[1][(f) >> 1])
    MLOP_QK0(0, 7); MLOP_QK0(1, 6); MLOP_QK0(2, 5); MLOP_QK0(3, 4); MLOP_QK0(4, 3); MLOP_QK0(5, 2); MLOP_QK0(6, 1); MLOP_QK0(7, 0);
#undef MLOP_QK0
    asm volatile("s_nop 15" : "+v"(sc[0][0]), "+v"(sc[0][1]), "+v"(sc[1][0]), "+v"(sc[1][1]));
  };

  // pages of the pairs pp + 1 .. pp + 3, ids of pp + 3 and pp + 4 (pair p in g[p % 4], ids[p % 2])
  Pages g[4];
  Ids ids[2] = {ids_of(4), ids_of(3)};
#pragma unroll
  for (int i = 0; i < 3; ++i) g[i] = pages_of(ids_of(i));
  issue(kh, k_off[0], k_off[1], 0, g[0]);
  if (n_pairs > 1) issue(kh, k_off[0], k_off[1], SLOT, g[1]);
  issue(vh, v_off[0], v_off[0], RING_V, g[0]);
  if (n_pairs > 2) issue(kh, k_off[0], k_off[1], 2 * SLOT, g[2]);
  if (n_pairs > 2) wait_vmcnt<6>(); else if (n_pairs > 1) wait_vmcnt<4>(); else wait_vmcnt<2>();
  raw_barrier();
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the page ids
  Sc sa, sb;
  u32x4 wa[2], wb[2];
  qk0(sa);
  const int last = n_pairs - 1;
#define MLOP_STEP(P, FIRST, SC, SN, WP, WN)                                                                             \
  step(std::integral_constant<int, P>{}, std::bool_constant<FIRST>{}, pp, SC, SN, WP, WN, g[(P + 1) % 4], ids[(P + 1) % 2], \
       g[(P + 3) % 4]);                                                                                                 \
  ids[(P + 1) % 2] = ids_of(pp + 5);                                                                                    \
  ++pp
  if (last > 0) {
    int pp = 0;
    MLOP_STEP(0, true, sa, sb, wb, wa);
    while (pp + 4 <= last) {
      MLOP_STEP(1, false, sb, sa, wa, wb);
      MLOP_STEP(2, false, sa, sb, wb, wa);
      MLOP_STEP(3, false, sb, sa, wa, wb);
      MLOP_STEP(0, false, sa, sb, wb, wa);
    }
    if (pp < last) {
      MLOP_STEP(1, false, sb, sa, wa, wb);
      if (pp < last) {
        MLOP_STEP(2, false, sa, sb, wb, wa);
        if (pp < last) {
          MLOP_STEP(3, false, sb, sa, wa, wb);
        }
      }
    }
  }
#undef MLOP_STEP
  Sc sl;
  const bool odd = last & 1;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) sl[i >> 1][i & 1][e] = odd ? sb[i >> 1][i & 1][e] : sa[i >> 1][i & 1][e];
  const u32x4 wl[2] = {odd ? wa[0] : wb[0], odd ? wa[1] : wb[1]};
  finish(sl, wl);
#undef MLOP_KREAD
#undef MLOP_VREAD

  mfma16_settle(o);
  // the four lane groups' partial row sums; O^T element e of dim block d is dim 16 d + 4 g4 + e of q row b
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    const float sum = sum_x16_x32(l[b]);
    if (!q_ok[b]) continue;
    if constexpr (SPLIT) {
      const int R = 32 * wid + 16 * b + r16;
#pragma unroll
      for (int d = 0; d < 8; ++d) *reinterpret_cast<f32x4*>(part + R * 128 + 16 * d + 4 * g4) = o[d][b];
      if (g4 == 0) *reinterpret_cast<u32x2*>(part + 128 * 128 + 2 * R) = u32x2{__float_as_uint(m[b]), __float_as_uint(sum)};
      continue;
    }
    const float inv = sum > 0.f ? 1.f / sum : 0.f;
    uint16_t* orow = out + ((size_t)(qs + qi[b]) * Hq + kvh * G + (32 * wid + 16 * b + r16) % G) * kD + 4 * g4;
#pragma unroll
    for (int d = 0; d < 8; ++d) {
      const f32x4 y = o[d][b] * inv;
      *reinterpret_cast<u32x2*>(orow + 16 * d) = u32x2{pack2(y[0], y[1]), pack2(y[2], y[3])};
    }
  }
}

// The same tile with a pair's three phases (S, softmax, O) one behind the other, on the 32x32x16 MFMA, K and V pair in one ring
// of three: 160 registers and 48 KB, three workgroups per CU where flash_item has two, and half as much to run before the first
// score and after the last.  For short tiles (flash_in_turn).  Per wave 32 q-rows, one per lane column: S^T [32 keys x 32 q], lane
// l holds keys (r & 3) + 8 (r >> 2) + 4 h (h = l >> 5) of q column l & 31; O^T [128 d x 32 q], P^T from registers 8 s .. 8 s + 7 of
// S as the k-step s fragment, V^T keys 16 s + 4 h + 0 .. 3 and + 8, dims 32 dblk + (l & 31).
template <int G>
__device__ __forceinline__ void flash_item_in_turn(
    uint16_t* smem, int tile, int kvh, uint16_t* __restrict__ out, const uint16_t* __restrict__ q,
    const uint16_t* __restrict__ kc, const uint16_t* __restrict__ vc, const int* __restrict__ block_tables,
    int bt_stride, const int* __restrict__ ptile_seq, const int* __restrict__ ptile_q0,
    const int* __restrict__ q_start, const int* __restrict__ q_len, const int* __restrict__ ctx_len, int Hq,
    int Hkv, float scale_log2, int num_blocks) {
  constexpr int QB = 128 / G;            // query tokens per workgroup
  constexpr int STAGES = 3;
  constexpr int STAGE = 4 * kBS * kD;    // bf16 per stage: K page A | K page B | V page A | V page B
  constexpr int PAGE = kBS * kD;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int s = ptile_seq[tile], q0 = ptile_q0[tile];
  const int ql = q_len[s], ctx = ctx_len[s], qs = q_start[s];
  const int last_q = min(q0 + QB, ql) - 1;
  const int kv_end = ctx - ql + last_q + 1;
  const int n_pairs = (kv_end + 31) >> 5;
  const int n_pages = (kv_end + kBS - 1) / kBS;
  const int wg_min_pos = ctx - ql + q0;
  const int col = lane & 31, h = lane >> 5;

  // this lane's q row (MFMA column): R = 32 wid + col
  const int R = 32 * wid + col;
  const int qi = q0 + R / G;
  const bool q_ok = qi < ql;
  const int pos_r = q_ok ? ctx - ql + qi : -1;
  bf16x8 qf[8];
  {
    const uint16_t* qrow = q + ((size_t)(qs + (q_ok ? qi : 0)) * Hq + kvh * G + R % G) * kD + 8 * h;
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      const bf16x8 v = *reinterpret_cast<const bf16x8*>(qrow + 16 * t);
      qf[t] = q_ok ? v : bf16x8{0, 0, 0, 0, 0, 0, 0, 0};
    }
  }
  f32x16 o[4];
#pragma unroll
  for (int d = 0; d < 4; ++d)
#pragma unroll
    for (int e = 0; e < 16; ++e) o[d][e] = 0.f;
  float m = kNegBig, l = 0.f;

  const int* bt = block_tables + (size_t)s * bt_stride;
  const size_t page_stride = (size_t)Hkv * PAGE;
  const int kkey = wid * 4 + (lane >> 4);
  // K image: chunk c of key k at slot c ^ k on BOTH pages (the 32x32 A-operand reads take keys
  // {0-3, 12-15} of one page and {4-11} of the other per 16-lane group: 16 distinct slots)
  const int k_off = kvh * PAGE + kkey * kD + (((lane & 15) ^ (kkey & 15)) << 3);
  const int v_off = kvh * PAGE + kkey * kD + (((lane & 15) ^ vswz(kkey)) << 3);
  auto page_of = [&](int idx) { return idx < n_pages ? min(max(bt[idx], 0), num_blocks - 1) : -1; };
  auto issue_pages = [&](int buf, int pgA, int pgB) {
    if (pgB < 0) pgB = pgA;
    uint16_t* base = smem + buf * STAGE + wid * 512;
    __builtin_amdgcn_global_load_lds((const void*)(kc + pgA * page_stride + k_off), (lds_void_t*)(base), 16, 0, 0);
    __builtin_amdgcn_global_load_lds((const void*)(kc + pgB * page_stride + k_off), (lds_void_t*)(base + PAGE), 16, 0, 0);
    __builtin_amdgcn_global_load_lds((const void*)(vc + pgA * page_stride + v_off), (lds_void_t*)(base + 2 * PAGE), 16, 0, 0);
    __builtin_amdgcn_global_load_lds((const void*)(vc + pgB * page_stride + v_off), (lds_void_t*)(base + 3 * PAGE), 16, 0, 0);
  };
  // K fragment t of this lane: key col of the pair (page col >> 4, row col & 15), chunk 2t + h at
  // slot (2t + h) ^ (col & 15): byte k_b0 ^ 32 t
  const int k15 = col & 15;
  const uint32_t k_b0 = (uint32_t)(uintptr_t)smem + (uint32_t)((col >> 4) * PAGE * 2 + k15 * 256 + ((h ^ k15) << 4));
  const uint32_t v_b0 = (uint32_t)(uintptr_t)smem + 2 * PAGE * 2 + vt32_base(lane);

  // S^T of the pair in ring slot ST: K fragment t at k_b0 ^ 32 t, four reads in flight (inline
  // asm with counted waits: as plain loads the compiler reused one register set and waited
  // lgkmcnt(0) in front of every MFMA, one LDS latency per fragment)
  auto qk = [&](auto st_tag) {
    constexpr uint32_t so = (uint32_t)(decltype(st_tag)::value * STAGE * 2);
    uint32_t kb = k_b0;
    asm volatile("" : "+v"(kb));
    auto kread = [&](int t, bf16x8& f) {
      asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(f) : "v"(kb ^ (32u * t)), "n"(so));
    };
    f32x16 sc;
#pragma unroll
    for (int e = 0; e < 16; ++e) sc[e] = 0.f;
    bf16x8 kf[4];
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // nothing else (SMEM) in the counts below
#pragma unroll
    for (int t = 0; t < 4; ++t) kread(t, kf[t]);
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      bf16x8& f = kf[t & 3];
      if (t <= 4) asm volatile("s_waitcnt lgkmcnt(3)" : "+v"(f));
      else if (t == 5) asm volatile("s_waitcnt lgkmcnt(2)" : "+v"(f));
      else if (t == 6) asm volatile("s_waitcnt lgkmcnt(1)" : "+v"(f));
      else asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(f));
      sc = mfma32(f, qf[t], sc);
      if (t + 4 < 8) kread(t + 4, kf[t & 3]);
    }
    return sc;
  };
  // online softmax on the lane's 16 keys of its q column (raw score units; the scale folds into
  // the exponent's FMA) -> P^T fragments of the two k-steps; O and l rescaled when the max moved
  auto softmax = [&](f32x16 sc, int pp, bf16x8 (&pf)[2]) {
    if (pp * 32 + 31 > wg_min_pos) {  // a pair crossing the workgroup's causal diagonal
      // (a side effect keeps this a branch: if-converted, the 47 compare / select / add of the
      // mask ran on every pair, a third of the loop's VALU)
      asm volatile("");
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int tok = pp * 32 + (r & 3) + 8 * (r >> 2) + 4 * h;
        sc[r] = tok <= pos_r ? sc[r] : -INFINITY;
      }
    }
    float mx = fmaxf(fmaxf(sc[0], sc[1]), sc[2]);
#pragma unroll
    for (int r = 3; r < 15; r += 2) mx = fmaxf(fmaxf(mx, sc[r]), sc[r + 1]);
    mx = fmaxf(mx, sc[15]);
    {
      const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
      mx = fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1]));
    }
    // deferred rescale (cdna_hip_programming.md T13): the running max moves only when some row's
    // new max exceeds it by more than 2^kRescaleLog2 in exp2 units (always on a row's first
    // keys: m starts at -1e30); otherwise P stays scaled against the old max, <= 2^8, which
    // bf16 P and f32 O / l carry exactly as well.  The decision covers this pair's P and is
    // taken before it is exponentiated, with the previous pair's P.V complete, so O, l and P
    // all see the same factor.
    float alpha = 1.f;
    if (__ballot((mx - m) * scale_log2 > kRescaleLog2)) {
      const float m_new = fmaxf(m, mx);
      alpha = fast_exp2((m - m_new) * scale_log2);
      m = m_new;
#pragma unroll
      for (int d = 0; d < 4; ++d) o[d] *= alpha;
      l *= alpha;
    }
    const float mc = -m * scale_log2;
    float rs = 0.f;
    u32x4 w[2];
#pragma unroll
    for (int r = 0; r < 16; r += 2) {
      const float p0 = fast_exp2(fmaf(sc[r], scale_log2, mc)), p1 = fast_exp2(fmaf(sc[r + 1], scale_log2, mc));
      rs += p0 + p1;
      w[r >> 3][(r & 7) >> 1] = cvt_pk_bf16(p0, p1);
    }
    pf[0] = __builtin_bit_cast(bf16x8, w[0]);
    pf[1] = __builtin_bit_cast(bf16x8, w[1]);
    l += rs;
  };
  // O^T += V^T . P^T from ring slot ST; the V^T fragment of (dblk, page) = two transposed reads.
  // The reads are inline asm: as builtins the compiler put s_waitcnt vmcnt(0) in front of them
  // (it cannot tell them from the in-flight LDS-DMA of the next pairs), which exposed the
  // latency of the DMA just issued on every pair.  The ring protocol (vmcnt + barrier at the
  // top of the step) already covers this pair; the asm waits below count only these reads.
  auto pv = [&](auto st_tag, const bf16x8 (&pf)[2]) {
    constexpr uint32_t so = (uint32_t)(decltype(st_tag)::value * STAGE * 2);
    uint32_t vb = v_b0;
    asm volatile("" : "+v"(vb));
    // both pages' fragments of dim block dblk: 4 reads, results in (lo, hi) of f0 (page A), f1
    auto issue = [&](int dblk, v4s16 (&r)[4]) {
      const uint32_t a0 = vb ^ (64u * dblk), a1 = a0 ^ 32u;
      asm volatile(
          "ds_read_b64_tr_b16 %0, %4 offset:%6\n"
          "ds_read_b64_tr_b16 %1, %5 offset:%7\n"
          "ds_read_b64_tr_b16 %2, %4 offset:%8\n"
          "ds_read_b64_tr_b16 %3, %5 offset:%9\n"
          : "=&v"(r[0]), "=&v"(r[1]), "=&v"(r[2]), "=&v"(r[3])
          : "v"(a0), "v"(a1), "n"(so), "n"(so + 2048u), "n"(so + 4096u), "n"(so + 6144u));
    };
    auto frag = [&](const v4s16& lo, const v4s16& hi) {
      bf16x8 f;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        f[e] = lo[e];
        f[4 + e] = hi[e];
      }
      return f;
    };
    v4s16 ra[4], rb[4];
    issue(0, ra);
#pragma unroll
    for (int dblk = 0; dblk < 4; ++dblk) {
      v4s16 (&cur)[4] = (dblk & 1) ? rb : ra;
      v4s16 (&nxt)[4] = (dblk & 1) ? ra : rb;
      if (dblk < 3) {
        issue(dblk + 1, nxt);
        asm volatile("s_waitcnt lgkmcnt(4)" : "+v"(cur[0]), "+v"(cur[1]), "+v"(cur[2]), "+v"(cur[3]));
      } else {
        asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(cur[0]), "+v"(cur[1]), "+v"(cur[2]), "+v"(cur[3]));
      }
      o[dblk] = mfma32(frag(cur[0], cur[1]), pf[0], o[dblk]);
      o[dblk] = mfma32(frag(cur[2], cur[3]), pf[1], o[dblk]);
    }
  };

  issue_pages(0, page_of(0), page_of(1));
  if (n_pairs > 1) issue_pages(1, page_of(2), page_of(3));
  int nxtA = page_of(4), nxtB = page_of(5);
  auto pair_step = [&](auto st_tag, int pp) {
    constexpr int ST = decltype(st_tag)::value;
    if (pp + 1 < n_pairs) wait_vmcnt<4>(); else wait_vmcnt<0>();
    raw_barrier();  // pair pp visible to every wave; ring slot (pp - 1) % 3 free
    if (pp + 2 < n_pairs) {
      issue_pages((ST + 2) % STAGES, nxtA, nxtB);
      nxtA = page_of(2 * pp + 6);
      nxtB = page_of(2 * pp + 7);
    }
    bf16x8 pf[2];
    softmax(qk(st_tag), pp, pf);
    pv(st_tag, pf);
  };
  for (int pp = 0; pp < n_pairs; pp += STAGES) {
    pair_step(std::integral_constant<int, 0>{}, pp);
    if (pp + 1 < n_pairs) pair_step(std::integral_constant<int, 1>{}, pp + 1);
    if (pp + 2 < n_pairs) pair_step(std::integral_constant<int, 2>{}, pp + 2);
  }

  // the two lane halves' partial row sums; O^T element r of dim block d is dim
  // 32 d + 8 (r >> 2) + 4 h + (r & 3) of q row R
  {
    const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(l), __float_as_uint(l), false, false);
    l = __uint_as_float(sw[0]) + __uint_as_float(sw[1]);
  }
  if (!q_ok) return;
  const float inv = l > 0.f ? 1.f / l : 0.f;
  uint16_t* orow = out + ((size_t)(qs + qi) * Hq + kvh * G + R % G) * kD + 4 * h;
#pragma unroll
  for (int d = 0; d < 4; ++d)
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      u32x2 v;
      v[0] = pack2(o[d][4 * b] * inv, o[d][4 * b + 1] * inv);
      v[1] = pack2(o[d][4 * b + 2] * inv, o[d][4 * b + 3] * inv);
      *reinterpret_cast<u32x2*>(orow + 32 * d + 8 * b) = v;
    }
}

// STREAM (flash_stream op; off: with a pair's phases in turn, as flash_item_in_turn, with which it tied at two workgroups per CU): the
// persistent grid's tiles as ONE stream of K / V page pairs per
// workgroup, so a tile's fixed cost hides under the previous tile's pairs (the 29 us fixed term
// of profiles/r06_flash_persist.md):
//   * the 3-deep LDS ring runs across tiles: while the last pairs of tile i are consumed, the
//     first two pairs of tile i+1 (or i+2: one-pair tiles) are already being fetched;
//   * tile i+1's Q rows arrive by LDS-DMA into a wave-private 8 KB while tile i runs, and are
//     read into registers at tile i+1's start (80 KB of LDS: 2 workgroups per CU);
//   * the loop is unrolled by the ring depth, so every step's stage is a constant (LDS read
//     offsets in the instruction) and tile boundaries are a branch inside a step.
// On the 32x32x16 MFMA: per wave 32 q-rows, ONE per lane column; S^T [32 keys x 32 q]: lane l holds keys (r & 3) + 8 (r >> 2)
// + 4 h (h = l >> 5) of q column l & 31; O^T [128 d x 32 q], P^T from registers 8s .. 8s + 7 of S as the k-step s fragment,
// V^T keys 16 s + 4 h + 0..3 and + 8, dims 32 dblk + (l & 31).
// Every vector memory operation of a wave is counted (4 LDS-DMAs per pair, 8 Q DMAs per tile,
// 16 O stores per tile: buffer stores, rows past the prompt dropped by the range check, so the
// count never depends on the data), and a pair's wait is vmcnt(operations issued after its DMAs):
// vmcnt(4) in the steady state.
// Tiles per workgroup, boustrophedon order and the kv head per XCD as the PERSIST grid.
//
// s_waitcnt vmcnt(n) for a run-time n (a multiple of 4; rounded down, and capped at 60: waiting
// for MORE retired operations than needed is always safe); n = 4 on the first compare
__device__ __forceinline__ void wait_vmcnt_rt(int n) {
  if (__builtin_expect(n == 4, 1)) {
    asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
    return;
  }
  switch (n < 0 ? 0 : n > 60 ? 15 : n >> 2) {
    case 0: asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); break;
    case 1: asm volatile("s_waitcnt vmcnt(4)" ::: "memory"); break;
    case 2: asm volatile("s_waitcnt vmcnt(8)" ::: "memory"); break;
    case 3: asm volatile("s_waitcnt vmcnt(12)" ::: "memory"); break;
    case 4: asm volatile("s_waitcnt vmcnt(16)" ::: "memory"); break;
    case 5: asm volatile("s_waitcnt vmcnt(20)" ::: "memory"); break;
    case 6: asm volatile("s_waitcnt vmcnt(24)" ::: "memory"); break;
    case 7: asm volatile("s_waitcnt vmcnt(28)" ::: "memory"); break;
    case 8: asm volatile("s_waitcnt vmcnt(32)" ::: "memory"); break;
    case 9: asm volatile("s_waitcnt vmcnt(36)" ::: "memory"); break;
    case 10: asm volatile("s_waitcnt vmcnt(40)" ::: "memory"); break;
    case 11: asm volatile("s_waitcnt vmcnt(44)" ::: "memory"); break;
    case 12: asm volatile("s_waitcnt vmcnt(48)" ::: "memory"); break;
    case 13: asm volatile("s_waitcnt vmcnt(52)" ::: "memory"); break;
    case 14: asm volatile("s_waitcnt vmcnt(56)" ::: "memory"); break;
    default: asm volatile("s_waitcnt vmcnt(60)" ::: "memory"); break;
  }
}

// item k of a persistent slot (boustrophedon rounds of S tiles), its causal extent in pairs and
// pages; tile -1 past the end of the list
struct FlashTile {
  int tile, q0, ql, ctx, qs, n_pairs, n_pages, wg_min_pos, seq;
};
// metadata reads through the constant address space: scalar loads (the tables are not written
// during the launch; as global pointers the loads after the first O store became vector loads,
// each followed by a vmcnt(0) that drained the in-flight K / V ring)
using cint_p = const __attribute__((address_space(4))) int*;
__device__ __forceinline__ int ld_const(const int* p, int i) {
  return ((cint_p)p)[__builtin_amdgcn_readfirstlane(i)];
}
template <int QB>
__device__ __forceinline__ FlashTile flash_tile(int k, int slot, int S, int num_ptiles, const int* __restrict__ ptile_seq,
                                                const int* __restrict__ ptile_q0, const int* __restrict__ q_start,
                                                const int* __restrict__ q_len, const int* __restrict__ ctx_len) {
  FlashTile it;
  const int t = k * S + ((k & 1) ? S - 1 - slot : slot);
  const bool ok = t < num_ptiles;
  const int tt = ok ? t : num_ptiles - 1;  // loads stay in bounds; the fields are ignored past the end
  it.tile = ok ? t : -1;
  it.seq = ld_const(ptile_seq, tt);
  it.q0 = ld_const(ptile_q0, tt);
  it.ql = ld_const(q_len, it.seq);
  it.ctx = ld_const(ctx_len, it.seq);
  it.qs = ld_const(q_start, it.seq);
  const int kv_end = it.ctx - it.ql + min(it.q0 + QB, it.ql);
  it.n_pairs = (kv_end + 31) >> 5;
  it.n_pages = (kv_end + kBS - 1) / kBS;
  it.wg_min_pos = it.ctx - it.ql + it.q0;
  return it;
}

template <int G>
__global__ void __launch_bounds__(256, 2) flash32_stream_kernel(
    uint16_t* __restrict__ out, const uint16_t* __restrict__ q, const uint16_t* __restrict__ kc,
    const uint16_t* __restrict__ vc, const int* __restrict__ block_tables, int bt_stride,
    const int* __restrict__ ptile_seq, const int* __restrict__ ptile_q0,
    const int* __restrict__ q_start, const int* __restrict__ q_len,
    const int* __restrict__ ctx_len, int Hq, int Hkv, float scale_log2, int num_blocks, int num_ptiles) {
  constexpr int QB = 128 / G;
  constexpr int STAGE = 4 * kBS * kD;  // bf16 per stage: K page A | K page B | V page A | V page B
  constexpr int PAGE = kBS * kD;
  constexpr int QW = 32 * kD;  // bf16 of one wave's 32 Q rows
  __shared__ __attribute__((aligned(256))) uint16_t smem[3 * STAGE + 4 * QW];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int col = lane & 31, h = lane >> 5, R = 32 * wid + col;
  const int kvh = blockIdx.x % Hkv, slot = blockIdx.x / Hkv, S = gridDim.x / Hkv;
  const size_t page_stride = (size_t)Hkv * PAGE;
  const int kkey = wid * 4 + (lane >> 4);
  const int k_off = kvh * PAGE + kkey * kD + (((lane & 15) ^ (kkey & 15)) << 3);
  const int v_off = kvh * PAGE + kkey * kD + (((lane & 15) ^ vswz(kkey)) << 3);
#define MLOP_FT(k) flash_tile<QB>((k), slot, S, num_ptiles, ptile_seq, ptile_q0, q_start, q_len, ctx_len)

  FlashTile cur = MLOP_FT(0);
  if (cur.tile < 0) return;  // the whole workgroup, before any barrier

  // the issue pointer of the pair stream: item iss_k, its next pair iss_p, whose pages pA / pB
  // were looked up one issue ahead.  vm = vector memory operations this wave has issued; markS
  // = vm right after the DMAs of the pair in ring stage S.  Pair n goes to stage n % 3 and is
  // consumed by the loop's step n % 3.
  FlashTile iss = cur;
  int iss_k = 0, iss_p = 0, vm = 0, mark0 = 0, mark1 = 0, mark2 = 0;
  const int* iss_bt = block_tables + (size_t)iss.seq * bt_stride;
  int pA = min(max(ld_const(iss_bt, 0), 0), num_blocks - 1);
  int pB = iss.n_pages > 1 ? min(max(ld_const(iss_bt, 1), 0), num_blocks - 1) : pA;
  auto issue_next = [&](auto st_tag) __attribute__((always_inline)) {
    constexpr int ST = decltype(st_tag)::value;
    if (iss.tile < 0) return;
    uint16_t* base = smem + ST * STAGE + wid * 512;
    __builtin_amdgcn_global_load_lds((const void*)(kc + pA * page_stride + k_off), (lds_void_t*)(base), 16, 0, 0);
    __builtin_amdgcn_global_load_lds((const void*)(kc + pB * page_stride + k_off), (lds_void_t*)(base + PAGE), 16, 0, 0);
    __builtin_amdgcn_global_load_lds((const void*)(vc + pA * page_stride + v_off), (lds_void_t*)(base + 2 * PAGE), 16, 0, 0);
    __builtin_amdgcn_global_load_lds((const void*)(vc + pB * page_stride + v_off), (lds_void_t*)(base + 3 * PAGE), 16, 0, 0);
    vm += 4;
    if constexpr (ST == 0) mark0 = vm;
    else if constexpr (ST == 1) mark1 = vm;
    else mark2 = vm;
    if (++iss_p >= iss.n_pairs) {  // every item has >= 1 pair
      iss = MLOP_FT(++iss_k);
      iss_p = 0;
      iss_bt = block_tables + (size_t)iss.seq * bt_stride;
    }
    if (iss.tile >= 0) {
      const int a = 2 * iss_p, b = a + 1 < iss.n_pages ? a + 1 : a;
      pA = min(max(ld_const(iss_bt, a), 0), num_blocks - 1);
      pB = min(max(ld_const(iss_bt, b), 0), num_blocks - 1);
    }
  };
  // the next tile's Q rows by LDS-DMA into this wave's private 8 KB (the compiler neither
  // tracks nor copies them: as register loads its own wait for them became a vmcnt(0) that
  // drained the ring at every tile start).  DMA t writes 1 KB, lane L's 16 B at 16 L: row
  // 32 wid + (L & 31), dims 16 t + 8 (L >> 5) -- fragment t of lane L, read back linearly.
  uint16_t* const q_lds = smem + 3 * STAGE + wid * QW;
  int markQ = 0;
  auto q_issue = [&](const FlashTile& it) __attribute__((always_inline)) {
    const int qi = it.q0 + R / G;
    const uint16_t* qrow = q + ((size_t)(it.qs + (qi < it.ql ? qi : 0)) * Hq + kvh * G + R % G) * kD + 8 * h;
#pragma unroll
    for (int t = 0; t < 8; ++t)
      __builtin_amdgcn_global_load_lds((const void*)(qrow + 16 * t), (lds_void_t*)(q_lds + t * 512), 16, 0, 0);
    vm += 8;
    markQ = vm;
  };
  const uint32_t q_b0 = (uint32_t)(uintptr_t)q_lds + 16u * lane;
  const int k15 = col & 15;
  const uint32_t k_b0 = (uint32_t)(uintptr_t)smem + (uint32_t)((col >> 4) * PAGE * 2 + k15 * 256 + ((h ^ k15) << 4));
  const uint32_t v_b0 = (uint32_t)(uintptr_t)smem + 2 * PAGE * 2 + vt32_base(lane);
  // the O stores' range: every valid row below 2 GB (checked on the host), masked rows at 2 GB
  const auto rsO = __builtin_amdgcn_make_buffer_rsrc(out, 0, 0x7fffffff, 0x00020000);

  // per-tile state: this lane's q row, its Q fragments, the accumulators
  int qi = 0, pos_r = -1, pp = 0, k = 0;
  bool q_ok = false;
  bf16x8 qf[8];
  f32x16 o[4];
  float m = kNegBig, l = 0.f;
  auto tile_start = [&]() __attribute__((always_inline)) {
    qi = cur.q0 + R / G;
    q_ok = qi < cur.ql;
    pos_r = q_ok ? cur.ctx - cur.ql + qi : -1;
    wait_vmcnt_rt(vm - markQ);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    asm volatile(
        "ds_read_b128 %0, %8\n"
        "ds_read_b128 %1, %8 offset:1024\n"
        "ds_read_b128 %2, %8 offset:2048\n"
        "ds_read_b128 %3, %8 offset:3072\n"
        "ds_read_b128 %4, %8 offset:4096\n"
        "ds_read_b128 %5, %8 offset:5120\n"
        "ds_read_b128 %6, %8 offset:6144\n"
        "ds_read_b128 %7, %8 offset:7168\n"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(qf[0]), "=&v"(qf[1]), "=&v"(qf[2]), "=&v"(qf[3]), "=&v"(qf[4]), "=&v"(qf[5]), "=&v"(qf[6]),
          "=&v"(qf[7])
        : "v"(q_b0));
    if (!q_ok) {
#pragma unroll
      for (int t = 0; t < 8; ++t) qf[t] = bf16x8{0, 0, 0, 0, 0, 0, 0, 0};
    }
#pragma unroll
    for (int d = 0; d < 4; ++d)
#pragma unroll
      for (int e = 0; e < 16; ++e) o[d][e] = 0.f;
    m = kNegBig;
    l = 0.f;
    pp = 0;
  };
  // epilogue: 16 buffer stores per lane, always issued (masked rows go past the range)
  auto tile_end = [&]() __attribute__((always_inline)) {
    {
      const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(l), __float_as_uint(l), false, false);
      l = __uint_as_float(sw[0]) + __uint_as_float(sw[1]);
    }
    const float inv = l > 0.f ? 1.f / l : 0.f;
    const uint32_t obase =
        q_ok ? (uint32_t)((((size_t)(cur.qs + qi) * Hq + kvh * G + R % G) * kD + 4 * h) * 2) : 0x80000000u;
    asm volatile("" ::: "memory");
#pragma unroll
    for (int d = 0; d < 4; ++d)
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        u32x2 v;
        v[0] = pack2(o[d][4 * b] * inv, o[d][4 * b + 1] * inv);
        v[1] = pack2(o[d][4 * b + 2] * inv, o[d][4 * b + 3] * inv);
        __builtin_amdgcn_raw_buffer_store_b64(v, rsO, obase + (uint32_t)(32 * d + 8 * b) * 2u, 0, 0);
      }
    vm += 16;
    asm volatile("" ::: "memory");
  };

  // one stream step: consume the pair in ring stage ST (true: the stream has ended)
  FlashTile nxt;
  auto step = [&](auto st_tag) __attribute__((always_inline)) -> bool {
    constexpr int ST = decltype(st_tag)::value;
    constexpr uint32_t so = (uint32_t)(ST * STAGE * 2);
    wait_vmcnt_rt(vm - (ST == 0 ? mark0 : ST == 1 ? mark1 : mark2));
    raw_barrier();  // pair visible to every wave; the stage consumed one step ago is free
    issue_next(std::integral_constant<int, (ST + 2) % 3>{});
    if (pp == 0 && nxt.tile >= 0) q_issue(nxt);  // the next tile's Q under this tile's pairs
    // S^T = K . Q^T of this pair
    f32x16 sc;
    {
      uint32_t kb = k_b0;
      asm volatile("" : "+v"(kb));
#pragma unroll
      for (int e = 0; e < 16; ++e) sc[e] = 0.f;
      bf16x8 kf[4];
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
      for (int t = 0; t < 4; ++t)
        asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(kf[t]) : "v"(kb ^ (32u * t)), "n"(so));
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        bf16x8& f = kf[t & 3];
        if (t <= 4) asm volatile("s_waitcnt lgkmcnt(3)" : "+v"(f));
        else if (t == 5) asm volatile("s_waitcnt lgkmcnt(2)" : "+v"(f));
        else if (t == 6) asm volatile("s_waitcnt lgkmcnt(1)" : "+v"(f));
        else asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(f));
        sc = mfma32(f, qf[t], sc);
        if (t + 4 < 8)
          asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(kf[t & 3]) : "v"(kb ^ (32u * (t + 4))), "n"(so));
      }
    }
    // online softmax (deferred rescale)
    bf16x8 pf[2];
    {
      if (pp * 32 + 31 > cur.wg_min_pos) {
        asm volatile("");
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int tok = pp * 32 + (r & 3) + 8 * (r >> 2) + 4 * h;
          sc[r] = tok <= pos_r ? sc[r] : -INFINITY;
        }
      }
      float mx = fmaxf(fmaxf(sc[0], sc[1]), sc[2]);
#pragma unroll
      for (int r = 3; r < 15; r += 2) mx = fmaxf(fmaxf(mx, sc[r]), sc[r + 1]);
      mx = fmaxf(mx, sc[15]);
      {
        const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
        mx = fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1]));
      }
      if (__ballot((mx - m) * scale_log2 > kRescaleLog2)) {
        const float m_new = fmaxf(m, mx);
        const float alpha = fast_exp2((m - m_new) * scale_log2);
        m = m_new;
#pragma unroll
        for (int d = 0; d < 4; ++d) o[d] *= alpha;
        l *= alpha;
      }
      const float mc = -m * scale_log2;
      float rs = 0.f;
      u32x4 w[2];
#pragma unroll
      for (int r = 0; r < 16; r += 2) {
        const float p0 = fast_exp2(fmaf(sc[r], scale_log2, mc)), p1 = fast_exp2(fmaf(sc[r + 1], scale_log2, mc));
        rs += p0 + p1;
        w[r >> 3][(r & 7) >> 1] = cvt_pk_bf16(p0, p1);
      }
      pf[0] = __builtin_bit_cast(bf16x8, w[0]);
      pf[1] = __builtin_bit_cast(bf16x8, w[1]);
      l += rs;
    }
    // O^T += V^T . P^T
    {
      uint32_t vb = v_b0;
      asm volatile("" : "+v"(vb));
      v4s16 ra[4], rb[4];
#define MLOP_VT_ISSUE(dblk, r)                                                              \
  {                                                                                         \
    const uint32_t a0 = vb ^ (64u * (dblk)), a1 = a0 ^ 32u;                                 \
    asm volatile(                                                                           \
        "ds_read_b64_tr_b16 %0, %4 offset:%6\n"                                             \
        "ds_read_b64_tr_b16 %1, %5 offset:%7\n"                                             \
        "ds_read_b64_tr_b16 %2, %4 offset:%8\n"                                             \
        "ds_read_b64_tr_b16 %3, %5 offset:%9\n"                                             \
        : "=&v"(r[0]), "=&v"(r[1]), "=&v"(r[2]), "=&v"(r[3])                                \
        : "v"(a0), "v"(a1), "n"(so), "n"(so + 2048u), "n"(so + 4096u), "n"(so + 6144u));  \
  }
      MLOP_VT_ISSUE(0, ra)
#pragma unroll
      for (int dblk = 0; dblk < 4; ++dblk) {
        v4s16 (&cv)[4] = (dblk & 1) ? rb : ra;
        v4s16 (&nv)[4] = (dblk & 1) ? ra : rb;
        if (dblk < 3) {
          MLOP_VT_ISSUE(dblk + 1, nv)
          asm volatile("s_waitcnt lgkmcnt(4)" : "+v"(cv[0]), "+v"(cv[1]), "+v"(cv[2]), "+v"(cv[3]));
        } else {
          asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(cv[0]), "+v"(cv[1]), "+v"(cv[2]), "+v"(cv[3]));
        }
        bf16x8 f0, f1;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          f0[e] = cv[0][e];
          f0[4 + e] = cv[1][e];
          f1[e] = cv[2][e];
          f1[4 + e] = cv[3][e];
        }
        o[dblk] = mfma32(f0, pf[0], o[dblk]);
        o[dblk] = mfma32(f1, pf[1], o[dblk]);
      }
#undef MLOP_VT_ISSUE
    }
    if (++pp < cur.n_pairs) return false;
    tile_end();
    if (nxt.tile < 0) return true;
    cur = nxt;
    nxt = MLOP_FT(++k + 1);
    tile_start();
    return false;
  };

  q_issue(cur);
  issue_next(std::integral_constant<int, 0>{});
  issue_next(std::integral_constant<int, 1>{});
  nxt = MLOP_FT(1);
  tile_start();
  for (;;) {
    if (step(std::integral_constant<int, 0>{})) break;
    if (step(std::integral_constant<int, 1>{})) break;
    if (step(std::integral_constant<int, 2>{})) break;
  }
#undef MLOP_FT
}

// PERSIST: a persistent grid of S x Hkv workgroups (S slots per kv head; blockIdx % Hkv = kv
// head, so each head stays on one XCD as in the one-item grid) walks the tile list in rounds of
// S tiles, boustrophedon: slot j takes tile r S + j in even rounds and r S + S - 1 - j in odd
// ones.  The host's per-sequence latest-first tile order then pairs a heavy tile with its light
// mirror on every slot (16 x 512: positions p, 15 - p, p, 15 - p), and the launch holds whole
// rounds instead of ~2 k one-item workgroups.
template <int G, int WPC, bool PERSIST, bool IN_TURN>
__global__ void __launch_bounds__(256, WPC) flash_prefill_kernel(
    uint16_t* __restrict__ out, const uint16_t* __restrict__ q, const uint16_t* __restrict__ kc,
    const uint16_t* __restrict__ vc, const int* __restrict__ block_tables, int bt_stride,
    const int* __restrict__ ptile_seq, const int* __restrict__ ptile_q0,
    const int* __restrict__ q_start, const int* __restrict__ q_len,
    const int* __restrict__ ctx_len, int Hq, int Hkv, float scale_log2, int num_blocks, int num_ptiles) {
  constexpr int STAGES = IN_TURN ? 3 : kFlashRing;
  constexpr int STAGE = 4 * kBS * kD;    // bf16 per stage: K page A | K page B | V page A | V page B
  __shared__ __attribute__((aligned(256))) uint16_t smem[STAGES * STAGE];
  if constexpr (IN_TURN) {
    static_assert(!PERSIST, "one tile per workgroup");
    flash_item_in_turn<G>(smem, blockIdx.x / Hkv, blockIdx.x % Hkv, out, q, kc, vc, block_tables, bt_stride, ptile_seq,
                          ptile_q0, q_start, q_len, ctx_len, Hq, Hkv, scale_log2, num_blocks);
  } else if constexpr (!PERSIST) {
    flash_item<G, false>(smem, blockIdx.x / Hkv, blockIdx.x % Hkv, out, q, kc, vc, block_tables, bt_stride, ptile_seq,
                         ptile_q0, q_start, q_len, ctx_len, Hq, Hkv, scale_log2, num_blocks, 0, 1, nullptr);
  } else {
    const int kvh = blockIdx.x % Hkv, j = blockIdx.x / Hkv, S = gridDim.x / Hkv;
    for (int r = 0; r * S < num_ptiles; ++r) {
      const int t = r * S + ((r & 1) ? S - 1 - j : j);
      if (t >= num_ptiles) continue;  // a partial last round: every slot still leaves the loop
      if (r > 0) __syncthreads();      // the previous tile's last ring reads before this tile's DMAs
      flash_item<G, false>(smem, t, kvh, out, q, kc, vc, block_tables, bt_stride, ptile_seq, ptile_q0, q_start, q_len,
                           ctx_len, Hq, Hkv, scale_log2, num_blocks, 0, 1, nullptr);
    }
  }
}

// A tile's keys in n_splits ranges, one workgroup each (flash_splits): blockIdx.x = (range * tiles + tile) * Hkv + kv head, parts of
// kFlashPart floats in that order.
template <int G>
__global__ void __launch_bounds__(256, 2) flash_split_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ kc, const uint16_t* __restrict__ vc,
    const int* __restrict__ block_tables, int bt_stride, const int* __restrict__ ptile_seq, const int* __restrict__ ptile_q0,
    const int* __restrict__ q_start, const int* __restrict__ q_len, const int* __restrict__ ctx_len, int Hq, int Hkv,
    float scale_log2, int num_blocks, int num_ptiles, int n_splits, float* __restrict__ part) {
  __shared__ __attribute__((aligned(256))) uint16_t smem[kFlashRing * 4 * kBS * kD];
  const int i = blockIdx.x / Hkv;
  flash_item<G, true>(smem, i % num_ptiles, blockIdx.x % Hkv, nullptr, q, kc, vc, block_tables, bt_stride, ptile_seq, ptile_q0,
                      q_start, q_len, ctx_len, Hq, Hkv, scale_log2, num_blocks, i / num_ptiles, n_splits,
                      part + (size_t)blockIdx.x * kFlashPart);
}

// out = sum of the ranges' O, each by 2^(its max - the largest), over their sums so weighted: 32 lanes a row, 8 rows a workgroup
// (32 one behind the other took four trips to memory: 240 parts of 6 ranges 10.5 us, now 5.0)
// A range counts unless its sum is 0, and not only where it is above: NaN and infinite scores make the sum NaN, which O and so the
// output then are, as without ranges.  (By its bits: this file's comparisons need not see a NaN.)
template <int G>
__global__ void __launch_bounds__(256) flash_merge_kernel(
    uint16_t* __restrict__ out, const float* __restrict__ part, const int* __restrict__ ptile_seq, const int* __restrict__ ptile_q0,
    const int* __restrict__ q_start, const int* __restrict__ q_len, int Hq, int Hkv, float scale_log2, int num_ptiles, int n_splits) {
  const int tile = blockIdx.x / Hkv, kvh = blockIdx.x % Hkv, s = ptile_seq[tile], q0 = ptile_q0[tile];
  const int ql = q_len[s], qs = q_start[s], c = (threadIdx.x & 31) * 4;
  const size_t step = (size_t)num_ptiles * Hkv * kFlashPart;
  const int R = blockIdx.y * 8 + (threadIdx.x >> 5);
  const int qi = q0 + R / G;
  if (qi >= ql) return;
  const float* p = part + (size_t)blockIdx.x * kFlashPart;
  float2 ml[kFlashSplits];
  f32x4 o[kFlashSplits];
  float M = kNegBig;
#pragma unroll
  for (int i = 0; i < kFlashSplits; ++i)
    if (i < n_splits) {
      ml[i] = *reinterpret_cast<const float2*>(p + i * step + 128 * 128 + 2 * R);
      o[i] = *reinterpret_cast<const f32x4*>(p + i * step + R * 128 + c);  // (not written where the range had no pair)
    }
#pragma unroll
  for (int i = 0; i < kFlashSplits; ++i)
    if (i < n_splits && __float_as_uint(ml[i].y) != 0) M = fmaxf(M, ml[i].x);
  f32x4 y{0.f, 0.f, 0.f, 0.f};
  float l = 0.f;
#pragma unroll
  for (int i = 0; i < kFlashSplits; ++i)
    if (i < n_splits && __float_as_uint(ml[i].y) != 0) {
      const float f = fast_exp2((ml[i].x - M) * scale_log2);
      l += f * ml[i].y;
      y += f * o[i];
    }
  y *= l > 0.f ? 1.f / l : 0.f;
  *reinterpret_cast<u32x2*>(out + ((size_t)(qs + qi) * Hq + kvh * G + R % G) * kD + c) = u32x2{pack2(y[0], y[1]), pack2(y[2], y[3])};
}

// flash_persist op: 0 = one workgroup per (tile, kv head) item; n = the persistent grid of n
// workgroups per CU (flash_prefill_kernel PERSIST); n >= 64: exactly n / 64 slots per kv head
// (tests: several rounds on a few tiles).  Off by default: +3-5 % at 16 x 512 in the host's
// per-sequence order, nothing or -1-2 % at 1024+ tokens in the LPT order the engine uses there
// (profiles/r06_flash_persist.md).
static int g_flash_persist = 0;
int flash_persist(int set) {
  if (set >= 0) g_flash_persist = set;
  return g_flash_persist;
}

// flash_stream op: 1 = the persistent grid runs flash32_stream_kernel (cross-tile K / V ring and
// Q prefetch, 2 workgroups per CU) instead of flash_item per tile; 0 = off
static int g_flash_stream = 0;
int flash_stream(int set) {
  if (set >= 0) g_flash_stream = set;
  return g_flash_stream;
}

// flash_form op: 0 by flash_in_turn, 1 flash_item, 2 flash_item_in_turn
static int g_flash_form = 0;
int flash_form(int set) {
  if (set >= 0) g_flash_form = set;
  return g_flash_form;
}

// The form in turn: for launches of short tiles, by their workgroups w and the keys that a tile reads on average (keys: summed over
// the tiles, 0 where not known).  What the software pipeline gains per pair it has to earn back: a longer way to the first score
// and from the last, and two workgroups per CU instead of three.  2244 launches (whole prompts alike and unlike, chunks behind
// cached keys, 1 - 32 kv heads, groups of 1 - 8), time of the pipeline over the form in turn at 48 / 100 / 200 / 320 / 512 keys: up to
// 224 workgroups 1.04 / 1.01 / 0.95 / 0.91 / 0.87; 225 - 512, one round of either, below 1; 513 - 640 1.16 / 1.05 / 0.95 / 0.93 / 0.92; 641 -
// 768, one round of it and two of the pipeline, 1.09 / 1.08 / 1.1 / 0.99 / 0.93; 769 - 896 about 1.0 up to 256 keys; 897 - 1024, two rounds
// of the pipeline, 1.03 / 1.0 / 0.94 / 0.96 / 0.9; 1025 - 1280 1.06 / 1.03 / 1.01 / 0.99 / 1.0; 1281 - 1792 1.03 / 1.02 / 1.03 / 1.0 / 0.99;
// 1793 - 2560 1.03 / 1.06 / 1.06 / 1.03 / 1.01; more 1.05 / 1.08 / 1.06 / 1.05 / 1.02, 0.97 from 768 keys on.
static bool flash_in_turn(int num_ptiles, int Hkv, long keys) {
  const long w = (long)num_ptiles * Hkv, mean = keys / num_ptiles;
  if (keys <= 0) return false;
  if (w <= kCus * 7 / 8) return mean <= 80;
  if (w <= 2 * kCus) return false;
  if (w <= kCus * 5 / 2) return mean <= 180;
  if (w <= kCus * 7 / 2) return mean <= 256;
  if (w <= 4 * kCus) return false;
  return mean <= std::min(512L, 200 + (w - 4 * kCus) / 5);
}

// Key ranges of each tile, for launches of few workgroups over many keys (a chat's next turn behind its cached ones: 150 tokens of 8
// kv heads are 40 workgroups, each walking all keys, 0.57 us a pair of pages).  By estimated time in us, w workgroups of n pairs
// each on average: whole 6.9 + .57 n; in s ranges up to 256 of them 10.3 + .5 n / s + .02 s + .0063 w s + .15 w n / 256, up to 512, two on
// a CU, 11 + .57 n / s + .0103 w s + .215 w n / 256; the best, where it is 10 % faster.  240 launches of 1 - 32 kv heads
// (1 and 3 sequences of 17 - 800 tokens behind 0 - 12000 cached ones): 0.75 of the time whole on average, 1.2 % off the best
// number, slower than whole in 1 (1.04).  us, whole -> now, 8 kv heads, groups of 4: 150 tokens behind 1024 / 4096 / 12000 26.1 ->
// 15.4, 79.3 -> 25.3, 220 -> 46.5; 512 behind 2048 / 12000 50.8 -> 35.6, 227 -> 105.2.
int flash_splits(int num_ptiles, int Hkv, long keys) {
  if (num_ptiles <= 0 || keys <= 0 || g_flash_form || g_flash_persist) return 1;
  const float w = (float)num_ptiles * (float)Hkv, n = (float)keys / (float)num_ptiles / 32.f;
  float best = (6.9f + .57f * n) / 1.1f;
  int splits = 1;
  for (int s = 2; s <= kFlashSplits && w * s <= 2 * kCus && s <= n; ++s) {
    const float f = (float)s;
    const float us = w * f <= kCus ? 10.3f + .5f * n / f + .02f * f + .0063f * w * f + .15f * w * n / kCus
                                   : 11.f + .57f * n / f + .0103f * w * f + .215f * w * n / kCus;
    if (us < best) best = us, splits = s;
  }
  return splits;
}

long flash_part_floats(int num_ptiles, int Hkv, int n_splits) { return (long)num_ptiles * Hkv * n_splits * kFlashPart; }

static int device_cus() {
  static int cus[16] = {};
  int dev = 0;
  (void)hipGetDevice(&dev);
  if (dev < 0 || dev >= 16) return 256;
  if (cus[dev] == 0) (void)hipDeviceGetAttribute(&cus[dev], hipDeviceAttributeMultiprocessorCount, dev);
  return cus[dev] > 0 ? cus[dev] : 256;
}

void launch_flash_prefill(void* out, const void* q, const void* kc, const void* vc, const int* bt,
                          int bt_stride, const int* ptile_seq, const int* ptile_q0,
                          const int* q_start, const int* q_len, const int* ctx_len, int num_ptiles,
                          int Hq, int Hkv, float scale_log2, int num_blocks, long keys, int n_splits, float* part, hipStream_t st) {
  if (num_ptiles == 0) return;
  if (n_splits > 1) {
    auto run = [&](auto g) {
      constexpr int G = decltype(g)::value;
      flash_split_kernel<G><<<num_ptiles * Hkv * n_splits, 256, 0, st>>>(
          (const uint16_t*)q, (const uint16_t*)kc, (const uint16_t*)vc, bt, bt_stride, ptile_seq, ptile_q0, q_start, q_len, ctx_len, Hq,
          Hkv, scale_log2, num_blocks, num_ptiles, n_splits, part);
      flash_merge_kernel<G><<<dim3(num_ptiles * Hkv, 16), 256, 0, st>>>((uint16_t*)out, part, ptile_seq, ptile_q0, q_start, q_len, Hq, Hkv,
                                                                      scale_log2, num_ptiles, n_splits);
    };
    switch (Hq / Hkv) {
      case 1: return run(std::integral_constant<int, 1>{});
      case 2: return run(std::integral_constant<int, 2>{});
      case 4: return run(std::integral_constant<int, 4>{});
      case 8: return run(std::integral_constant<int, 8>{});
      default: return;
    }
  }
  const bool in_turn = g_flash_form ? g_flash_form == 2 : flash_in_turn(num_ptiles, Hkv, keys);
  const int slots = g_flash_persist >= 64 ? g_flash_persist / 64
                    : g_flash_persist > 0 ? std::max(1, g_flash_persist * device_cus() / Hkv) : 0;
  const bool persist = slots > 0 && num_ptiles > slots;
  dim3 grid((persist ? slots : num_ptiles) * Hkv);
  const bool stream = persist && g_flash_stream;
#define MLOP_FLASH_CASE(GG)                                                                              \
  case GG:                                                                                               \
    if (stream)                                                                                          \
      flash32_stream_kernel<GG><<<grid, 256, 0, st>>>(                                                   \
          (uint16_t*)out, (const uint16_t*)q, (const uint16_t*)kc, (const uint16_t*)vc, bt, bt_stride,   \
          ptile_seq, ptile_q0, q_start, q_len, ctx_len, Hq, Hkv, scale_log2, num_blocks, num_ptiles);    \
    else if (persist)                                                                                    \
      flash_prefill_kernel<GG, 2, true, false><<<grid, 256, 0, st>>>(                                  \
          (uint16_t*)out, (const uint16_t*)q, (const uint16_t*)kc, (const uint16_t*)vc, bt, bt_stride,   \
          ptile_seq, ptile_q0, q_start, q_len, ctx_len, Hq, Hkv, scale_log2, num_blocks, num_ptiles);    \
    else if (in_turn)                                                                                    \
      flash_prefill_kernel<GG, 2, false, true><<<grid, 256, 0, st>>>(                                  \
          (uint16_t*)out, (const uint16_t*)q, (const uint16_t*)kc, (const uint16_t*)vc, bt, bt_stride,   \
          ptile_seq, ptile_q0, q_start, q_len, ctx_len, Hq, Hkv, scale_log2, num_blocks, num_ptiles);    \
    else                                                                                                 \
      flash_prefill_kernel<GG, 2, false, false><<<grid, 256, 0, st>>>(                                 \
          (uint16_t*)out, (const uint16_t*)q, (const uint16_t*)kc, (const uint16_t*)vc, bt, bt_stride,   \
          ptile_seq, ptile_q0, q_start, q_len, ctx_len, Hq, Hkv, scale_log2, num_blocks, num_ptiles);    \
    break;
  switch (Hq / Hkv) {
    MLOP_FLASH_CASE(1)
    MLOP_FLASH_CASE(2)
    MLOP_FLASH_CASE(4)
    MLOP_FLASH_CASE(8)
    default: break;
  }
#undef MLOP_FLASH_CASE
}

}  // namespace mlop

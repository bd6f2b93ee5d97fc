// lt_attn_head.hip -- decode attention of one query head over one sequence's cache, unsplit (the
// single-pass order of k_attn_decode_masked): the decode step (RoPE, KV append, attention,
// quant) and batched decode, bit-identical to k_attn_w1 and k_attn_dec of lt_attn.hip (but for the sign
// of a zero that underflowed products left: lt_attn_mm.hip).
//
// The unsplit order leaves one serial chain per (head, dim) over all positions, so a head's
// latency is what counts: a workgroup of NW waves takes one head and shares out everything that
// is not that chain.
//   scores   rounds of 64 positions, a wave every NW-th: rows come in by whole 128-byte lines,
//            pass through the wave's own LDS (padded) and lane l runs position l's chain;
//   softmax  the exps over all threads, Z by one wave (64-lane fold and tree);
//   O        on the fp32 matrix cores, whose v_mfma_f32_16x16x4_f32 is a sequential fma chain
//            over its four products (lt_attn_mm.hip): 16 DT dims a wave, four positions an
//            instruction, the exps broadcast to all 16 columns.  One instruction per 32 cycles
//            for four positions beats four dependent vector fmas with their operand reads; the
//            operands are read from LDS a block ahead.
// Short contexts are all latency, and loads return in order.  So a step's inputs are requested before any
// cache row, only the first one or two K rounds before the length is known (a round by every wave, 512
// rows, costs 0.4 to 3 us where the length is 64), and all else through descriptors that end at the
// length: later rows read zeros and cost no traffic.
//
// k_attn_group below does the same with a workgroup per KV group for grids of more heads than CUs.
//
// The heads of a KV group run on one XCD (workgroups are dealt to the 8 XCDs round-robin), so a
// group's rows are fetched into one L2 once.
#include "lt_q8_device.h"

namespace {

using namespace lt;

// Position t's slot in the exps: a lane of group k reads its four steps' exps (t = 4 i + k, i =
// 0..3) of a 16-position tile as one 16-byte word.
__device__ __forceinline__ int e_slot(int t) { return (t & ~15) | ((t & 3) << 2) | ((t >> 2) & 3); }

// Where block j of row b's quantized output goes: row-major, or block-major over obm rows
// (q8_out_block, whose 64-bit division a short context would wait for).
__device__ __forceinline__ size_t out_block(const LtAttnHead& A, int hd, int b, int j) {
  return A.obm > 0 ? (size_t)j * A.obm + b : (size_t)b * (A.nh * hd / 32) + j;
}

template <bool kF16, int HD, int NW, bool kStep>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(NW / 4, NW / 2))) void k_attn_head(
    LtAttnHead A) {
  extern __shared__ __attribute__((aligned(16))) float lds[];
  constexpr int kEb = kF16 ? 2 : 4;
  constexpr int NL = HD * kEb / 128;                // 128-byte lines per cache row
  constexpr int R = NL == 1 ? 2 : 4;                // K lines (of 64 rows) in flight
  constexpr int kKRow = 144;                        // a line's pitch in LDS (lanes 36 banks apart)
  constexpr int NP = NW < HD / 16 ? NW : HD / 16;   // waves that fold O
  constexpr int DT = HD / 16 / NP;                  // adjacent dims per lane in O
  constexpr int kVB = DT * kEb;
  constexpr int SB = 16 * kVB;                      // a wave's bytes of one V row
  constexpr int RB = 1024 / SB;                     // V rows per block (one 16-byte load per lane)
  constexpr int D = 256 / RB;                       // V blocks in flight: 256 rows
  float* sq = lds;                                  // [HD] q (roped in a step)
  float* sk = sq + HD;                              // [HD] step: the new k in the cache's format
  float* sv = sk + HD;                              // [HD] step: the new v through the cache's type
  float* so = sv + HD;                              // [HD] the output
  float* sm = so + HD;                              // [NW] maxima, then [1] Z
  uint8_t* vbuf = (uint8_t*)(sm + 12);              // [NP][2][1024]
  uint8_t* kbuf = vbuf + NP * 2048;                 // [NW][64][kKRow] K lines
  float* P = (float*)(kbuf + NW * 64 * kKRow);      // [cap] exps by e_slot
  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63;
  const int n16 = l & 15, g4 = l >> 4;

  // grid (8, heads per group, octets of (sequence, KV group) pairs)
  const int pair = (int)(8 * blockIdx.z + blockIdx.x);
  if (pair >= A.batch * A.nkv) return;
  const int b = kStep ? 0 : (int)((uint32_t)pair * A.rnkv >> 22), g = pair - b * A.nkv;
  const int rep = (int)gridDim.y, r0 = (int)blockIdx.y, h = g * rep + r0;

  const int len0 = A.len[kStep ? 0 : b];
  const uint32_t pitch = (uint32_t)A.nkv * HD * kEb;
  const uint32_t seq = (uint32_t)b * (uint32_t)A.maxt * pitch;
  const uint32_t gb = seq + (uint32_t)g * HD * kEb;
  auto rows_of = [&](void* c, int rows) {           // the cache up to row `rows`; later rows read zeros
    return __builtin_amdgcn_make_buffer_rsrc(c, 0, (int)(seq + (uint32_t)rows * pitch), 0x00020000);
  };

  // K line u (line u % NL of round w + NW (u / NL)): row 8 i + l / 8, bytes 16 (l % 8) of the line;
  // rows past the cache read zeros
  const uint32_t kb0 = gb + (uint32_t)(l >> 3) * pitch + (uint32_t)(l & 7) * 16u;
  auto load_k = [&](__amdgpu_buffer_rsrc_t krsrc, int u, u32x4 (&k)[8]) {
    const uint32_t off = kb0 + (uint32_t)((w + NW * (u / NL)) * 64) * pitch + (uint32_t)(u % NL) * 128u;
#pragma unroll
    for (int i = 0; i < 8; i++)
      k[i] = __builtin_amdgcn_raw_buffer_load_b128(krsrc, (int)(off + (uint32_t)(8 * i) * pitch), 0, 0);
  };
  // a step's inputs
  float x1 = 0.0f, x2 = 0.0f, fr = 0.0f, vn[HD / 64];
  if (kStep) {
    if (w < 2 && l < HD / 2) {
      const float* src = w == 0 ? A.qkv + (size_t)h * HD : A.qkv + (size_t)A.nh * HD + (size_t)g * HD;
      x1 = src[l];
      x2 = src[l + HD / 2];
      fr = A.freqs[l];
    } else if (w == 2) {
#pragma unroll
      for (int i = 0; i < HD / 64; i++) vn[i] = A.qkv[(size_t)(A.nh + A.nkv) * HD + (size_t)g * HD + l + 64 * i];
    }
  }
  u32x4 kr[R][8];
  // the first rounds, before the length (of a step of 32 heads of 128 fp32 at 64 rows 6.5 us with one
  // round, 7.0 with two; 14 heads of 64 fp16 at 300 rows 7.3 with one, 7.0 with two)
  constexpr int kEarly = HD == 64 ? 2 : 1;
  if (w < kEarly) {
    const __amdgpu_buffer_rsrc_t all = rows_of(A.kc, A.maxt);
#pragma unroll
    for (int u = 0; u < NL; u++) load_k(all, u, kr[u]);
  }
  int Lnew = -1, n;
  bool valid = true;
  if (kStep) {
    valid = len0 >= 0 && len0 < A.maxt;
    Lnew = valid ? len0 : -1;
    n = valid ? len0 + 1 : 0;
  } else {
    n = len0 < 0 ? 0 : (len0 > A.maxt ? A.maxt : len0);
  }
  const int nv = kStep && valid ? len0 : n;         // rows that come from the cache
  const int nr = (n + 63) >> 6;
  const int nu = w < nr ? (nr - w + NW - 1) / NW * NL : 0;   // this wave's K lines
  const __amdgpu_buffer_rsrc_t krsrc = rows_of(A.kc, n), vrsrc = rows_of(A.vc, nv);
  if (w >= kEarly && nu > 0) {
#pragma unroll
    for (int u = 0; u < NL; u++) load_k(krsrc, u, kr[u]);
  }
#pragma unroll
  for (int u = NL; u < R; u++)
    if (u < nu) load_k(krsrc, u, kr[u]);
  // V block at row p: 16 bytes of row p + l / (SB / 16) per lane
  const int db = w * 16 * DT;
  const int vrow = l / (SB / 16);
  const uint32_t vb = gb + (uint32_t)db * kEb + (uint32_t)(l % (SB / 16)) * 16u;
  auto load_v = [&](int p) {
    return __builtin_amdgcn_raw_buffer_load_b128(vrsrc, (int)((uint32_t)(p + vrow) * pitch + vb), 0, 0);
  };

  if (kStep) {
    // RoPE (the arithmetic of k_rope, rope_from_facts.pl:40-69) of q on wave 0 and of the group's
    // k on wave 1; v on wave 2; k and v through the cache's type
    auto round_kv = [&](float x) { return kF16 ? lt_half_to_float_bits(lt_float_to_half_bits(x)) : x; };
    if (w < 2) {
      if (l < HD / 2) {
        float sn, cs;
        lt_sincosf((float)(valid ? len0 : 0) * fr, &sn, &cs);
        const float o1 = fmaf(x1, cs, -(x2 * sn)), o2 = fmaf(x1, sn, x2 * cs);
        if (w == 1 && kF16) {
          ((uint16_t*)sk)[l] = lt_float_to_half_bits(o1);
          ((uint16_t*)sk)[l + HD / 2] = lt_float_to_half_bits(o2);
        } else {
          float* dst = w == 0 ? sq : sk;
          dst[l] = o1;
          dst[l + HD / 2] = o2;
        }
      }
    } else if (w == 2) {
#pragma unroll
      for (int i = 0; i < HD / 64; i++)
        sv[l + 64 * i] = round_kv(vn[i]);
    }
  } else if (tid < HD) {
    sq[tid] = A.q[(size_t)b * A.q_stride + (size_t)h * HD + tid];
  }
  __syncthreads();
  if (kStep && valid && r0 == 0 && w == NW - 1) {
    // the new row into the cache (k_append_kv_incr, dev_residency.py:303-315)
    const size_t e0 = (size_t)len0 * A.nkv * HD + (size_t)g * HD;
#pragma unroll
    for (int i = 0; i < HD / 64; i++) {
      const int d = l + 64 * i;
      if (kF16) {
        ((uint16_t*)A.kc)[e0 + d] = ((const uint16_t*)sk)[d];
        ((uint16_t*)A.vc)[e0 + d] = lt_float_to_half_bits(sv[d]);
      } else {
        ((float*)A.kc)[e0 + d] = sk[d];
        ((float*)A.vc)[e0 + d] = sv[d];
      }
    }
  }

  // scores
  uint8_t* const kw = kbuf + w * 64 * kKRow;
  float mx = -1e30f, acc = 0.0f;
  for (int u0 = 0; u0 < nu; u0 += R) {
#pragma unroll
    for (int i = 0; i < R; i++) {
      const int u = u0 + i;
      if (u >= nu) break;
      const int t0 = (w + NW * (u / NL)) * 64, ln = u % NL;
      wave_fence();                                 // (the last line's reads, then this one's writes)
#pragma unroll
      for (int j = 0; j < 8; j++) *(u32x4*)(kw + (8 * j + (l >> 3)) * kKRow + (l & 7) * 16) = kr[i][j];
      load_k(krsrc, u + R, kr[i]);
      wave_fence();
      if (kStep && Lnew >= t0 && Lnew < t0 + 64) {  // the new row over its place
        if (l < 8)
          *(u32x4*)(kw + (Lnew - t0) * kKRow + l * 16) = *(const u32x4*)((const uint8_t*)sk + ln * 128 + l * 16);
        wave_fence();
      }
      if (NL == 1 || ln == 0) acc = 0.0f;
#pragma unroll
      for (int c = 0; c < 8; c++) {
        const u32x4 k = *(const u32x4*)(kw + l * kKRow + c * 16);
        const float* qc = sq + ln * (128 / kEb) + c * (16 / kEb);
        const uint32_t y[4] = {k.x, k.y, k.z, k.w};
#pragma unroll
        for (int e = 0; e < 4; e++) {
          if (kF16) {
            acc = fmaf(qc[2 * e], lt_h2f((uint16_t)(y[e] & 0xFFFFu)), acc);
            acc = fmaf(qc[2 * e + 1], lt_h2f((uint16_t)(y[e] >> 16)), acc);
          } else {
            acc = fmaf(qc[e], __uint_as_float(y[e]), acc);
          }
        }
      }
      if ((NL == 1 || ln == NL - 1) && t0 + l < n) {
        const float x = acc * A.scale;
        P[e_slot(t0 + l)] = x;
        mx = fmaxf(mx, x);
      }
    }
  }
  u32x4 vr[D];                                      // (under the softmax)
  if (w < NP) {
#pragma unroll
    for (int j = 0; j < D; j++)
      if (j < 2 || j * RB < nv) vr[j] = load_v(j * RB);
  }
  mx = wave_max(mx);
  if (l == 0) sm[w] = mx;
  __syncthreads();
  float m = -1e30f;
#pragma unroll
  for (int i = 0; i < NW; i++) m = fmaxf(m, sm[i]);
  // the exps; zeros up to whole groups of the O loop
  const int n_up = (nv + D * RB - 1) / (D * RB) * (D * RB);
  const int n_all = n_up > n ? n_up : n;
  if (n_all <= 64 * NW) {                           // one position a thread
    float e[1] = {P[e_slot(tid < n_all ? tid : 0)] - m};   // (the exps' LDS may end at n_all)
    lt_expf_n(e);
    if (tid < n_all) P[e_slot(tid)] = tid < n ? e[0] : 0.0f;
  } else {
    for (int t = tid; t < n_all; t += 128 * NW) {
      const int t1 = t + 64 * NW;
      float e[2];
      e[0] = P[e_slot(t)] - m;
      e[1] = P[e_slot(t1 < n_all ? t1 : t)] - m;
      lt_expf_n(e);
      P[e_slot(t)] = t < n ? e[0] : 0.0f;
      if (t1 < n_all) P[e_slot(t1)] = t1 < n ? e[1] : 0.0f;
    }
  }
  __syncthreads();
  if (w == NW - 1) {
    float z = 0.0f;
    for (int t = l; t < n; t += 64) z = z + P[e_slot(t)];
    z = wave_tree_dpp(z);
    if (l == 0) sm[NW] = z;
  }

  // O: the cached rows in ascending order; a step's new row, the last, from LDS
  f32x4 o[DT];
#pragma unroll
  for (int d = 0; d < DT; d++) o[d] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  if (w < NP) {
    uint8_t* const vw = vbuf + w * 2048;
    auto put_v = [&](int buf, u32x4 x) { *(u32x4*)(vw + buf * 1024 + l * 16) = x; };
    // block j: its lines written two blocks ahead, its operands read one block ahead
    constexpr int NS = RB / 4;                      // steps per block
    float va[2][NS][DT], ea[2][NS];
    auto read_block = [&](int buf, int p, float (&v)[NS][DT], float (&e)[NS]) {
#pragma unroll
      for (int i = 0; i < RB / 16; i++) {
        const f32x4 x = *(const f32x4*)(P + p + 16 * i + 4 * g4);
#pragma unroll
        for (int s = 0; s < 4; s++) {
          e[4 * i + s] = x[s];
          const uint8_t* y = vw + buf * 1024 + (16 * i + 4 * s + g4) * SB + n16 * kVB;
#pragma unroll
          for (int d = 0; d < DT; d++) v[4 * i + s][d] = kF16 ? lt_h2f(((const uint16_t*)y)[d]) : ((const float*)y)[d];
        }
      }
    };
    put_v(0, vr[0]);
    put_v(1, vr[1]);
    wave_fence();
    read_block(0, 0, va[0], ea[0]);
    for (int p = 0; p < nv; p += D * RB) {
#pragma unroll
      for (int j = 0; j < D; j++) {
        vr[j] = load_v(p + (j + D) * RB);
        wave_fence();
        read_block((j + 1) & 1, p + (j + 1) * RB, va[(j + 1) & 1], ea[(j + 1) & 1]);
        put_v(j & 1, vr[(j + 2) % D]);
#pragma unroll
        for (int i = 0; i < NS; i++)
#pragma unroll
          for (int d = 0; d < DT; d++)
            o[d] = mma(va[j & 1][i][d], ea[j & 1][i], o[d]);
        settle(o);
        if (p + (j + 1) * RB >= nv) break;          // (the rest of the group: zero rows)
      }
    }
  }
  __syncthreads();                                  // Z
  if (w < NP && n16 == 0) {
    const float z = sm[NW];
    const float en = kStep && valid ? P[e_slot(len0)] : 0.0f;
#pragma unroll
    for (int d = 0; d < DT; d++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int dim = db + DT * (4 * g4 + r) + d;
        float x = o[d][r];
        if (kStep) x = fmaf(en, sv[dim], x);
        so[dim] = valid ? x / z : 0.0f;
      }
  }
  __syncthreads();
  if (A.out && tid < HD) A.out[((size_t)b * A.nh + h) * HD + tid] = so[tid];
  if (A.oq && tid < HD) {
    const size_t blk = out_block(A, HD, b, h * (HD / 32) + (tid >> 5));
    quant_block_hw(so[tid], tid & 31, A.oq + blk * 32, A.od + blk);
  }
}

// Batched decode past one head per CU: a workgroup of 8 waves takes all heads of one KV group of
// one sequence, so its cache rows are read and converted once.  The heads are the columns of the
// matrix instructions (16, of which nh / nkv are used):
//   scores   tiles of 16 positions as in k_attn_mm, a wave every eighth tile, two tiles in flight;
//            a lane's four scores lie side by side by e_slot;
//   softmax  a wave per head: exps one, two or four at a time, Z by the 64-lane fold and tree;
//   O        as above with each head's exps in its own column, a wave per 16 dims.
// Bound by the serial chain over the positions and by one wave's exps; at most one workgroup runs
// per CU, so registers are not short.
template <bool kF16, int HD>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 4))) void k_attn_group(LtAttnHead A, int cap) {
  extern __shared__ __attribute__((aligned(16))) float lds[];
  constexpr int NW = 8;
  constexpr int kEb = kF16 ? 2 : 4;
  constexpr int NU = HD * kEb / 64;                 // 16-byte units per lane and K tile
  constexpr int NP = HD / 16;                       // waves that fold O, 16 dims each
  constexpr int SB = 16 * kEb;
  constexpr int RB = 1024 / SB;
  constexpr int D = 256 / RB;
  static_assert(NP <= NW, "k_attn_group: head size");
  const int rep = A.rep, ps = cap + 4;
  float* sm = lds;                                  // [NW][16] maxima, [16] Z
  uint8_t* vbuf = (uint8_t*)(sm + NW * 16 + 16);    // [NP][2][1024]
  float* P = (float*)(vbuf + NP * 2048);            // [rep][ps] exps by e_slot; then the outputs
  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63;
  const int n16 = l & 15, g4 = l >> 4;
  const int b = (int)blockIdx.y, g = (int)blockIdx.x;
  const int len0 = A.len[b];
  const uint32_t pitch = (uint32_t)A.nkv * HD * kEb;
  const size_t seq = (size_t)b * A.maxt * pitch;
  const uint32_t gb = (uint32_t)g * HD * kEb;
  auto rows_of = [&](void* c, int rows) {           // the sequence's first rows; later rows read zeros
    return __builtin_amdgcn_make_buffer_rsrc((uint8_t*)c + seq, 0, (int)((uint32_t)rows * pitch), 0x00020000);
  };

  // the queries first: loads return in order
  u32x4 qv[HD / 16];
  {
    const float* qs = A.q + (size_t)b * A.q_stride + (size_t)(g * rep + (n16 < rep ? n16 : 0)) * HD;
#pragma unroll
    for (int j = 0; j < HD / 16; j++) qv[j] = *(const u32x4_a4*)(qs + 16 * j + 4 * g4);
  }
  // K tile at position p: unit 4 j + g4 of the row that makes matrix row n16 position 4 (n16 & 3) +
  // n16 / 4, so that a lane's four scores lie side by side by e_slot
  const uint32_t kb0 = gb + (uint32_t)((n16 & 3) * 4 + (n16 >> 2)) * pitch + (uint32_t)g4 * 16u;
  auto load_unit = [&](__amdgpu_buffer_rsrc_t krsrc, int p, int j) {
    return __builtin_amdgcn_raw_buffer_load_b128(krsrc, (int)(kb0 + (uint32_t)p * pitch + 64u * j), 0, 0);
  };
  u32x4 kb[2][NU];
  constexpr int kEarly = 2;                         // tiles before the length (4 or 8: the same or slower)
  if (w < kEarly) {
    const __amdgpu_buffer_rsrc_t all = rows_of(A.kc, A.maxt);
#pragma unroll
    for (int j = 0; j < NU; j++) kb[0][j] = load_unit(all, w * 16, j);
  }
  const int n = len0 < 0 ? 0 : (len0 > A.maxt ? A.maxt : len0);
  const __amdgpu_buffer_rsrc_t krsrc = rows_of(A.kc, n), vrsrc = rows_of(A.vc, n);
#pragma unroll
  for (int i = 0; i < 2; i++) {
    const int p = (w + i * NW) * 16;
    if (p < n && (i == 1 || w >= kEarly)) {
#pragma unroll
      for (int j = 0; j < NU; j++) kb[i][j] = load_unit(krsrc, p, j);
    }
  }

  float qr[HD / 4];
#pragma unroll
  for (int j = 0; j < HD / 16; j++) {
    uint32_t r[4] = {qv[j].x, qv[j].y, qv[j].z, qv[j].w};
    transpose4(r);
#pragma unroll
    for (int e = 0; e < 4; e++) qr[4 * j + e] = __uint_as_float(r[e]);
  }
  // a tile's scores, its units replaced by those of the tile at `next` where there is one (a constant: a
  // branch around the loads would cut the chain into several blocks)
  auto s_tile = [&](u32x4 (&kt)[NU], int next, auto more) {
    f32x4 s[1] = {{0.0f, 0.0f, 0.0f, 0.0f}};
#pragma unroll
    for (int j = 0; j < NU; j++) {
      const u32x4 k = kt[j];
      if (kF16) {
        uint32_t r[4] = {__builtin_amdgcn_perm(k.z, k.x, 0x05040100u), __builtin_amdgcn_perm(k.z, k.x, 0x07060302u),
                         __builtin_amdgcn_perm(k.w, k.y, 0x05040100u), __builtin_amdgcn_perm(k.w, k.y, 0x07060302u)};
        if constexpr (decltype(more)::value) kt[j] = load_unit(krsrc, next, j);
        transpose4(r);
#pragma unroll
        for (int e = 0; e < 4; e++) {
          s[0] = mma(lt_h2f((uint16_t)(r[e] & 0xFFFFu)), qr[8 * j + 2 * e], s[0]);
          s[0] = mma(lt_h2f((uint16_t)(r[e] >> 16)), qr[8 * j + 2 * e + 1], s[0]);
        }
      } else {
        uint32_t r[4] = {k.x, k.y, k.z, k.w};
        if constexpr (decltype(more)::value) kt[j] = load_unit(krsrc, next, j);
        transpose4(r);
#pragma unroll
        for (int e = 0; e < 4; e++) s[0] = mma(__uint_as_float(r[e]), qr[4 * j + e], s[0]);
      }
    }
    settle(s);
    return s[0];
  };
  float mx = -1e30f;
  for (int p = w * 16; p < n; p += 32 * NW) {
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const int pi = p + 16 * NW * i, next = pi + 32 * NW;
      if (pi < n) {
        f32x4 s = next < n ? s_tile(kb[i], next, std::true_type{}) : s_tile(kb[i], next, std::false_type{});
#pragma unroll
        for (int r = 0; r < 4; r++) {
          s[r] = s[r] * A.scale;
          if (pi + 4 * r + g4 < n) mx = fmaxf(mx, s[r]);
        }
        if (n16 < rep) *(f32x4*)(P + n16 * ps + pi + 4 * g4) = s;
      }
    }
  }
  mx = max_over_groups(mx);
  if (l < 16) sm[w * 16 + l] = mx;
  // V block at row p: this wave's 16 dims
  const int vrow = l / (SB / 16);
  const uint32_t vb = gb + (uint32_t)(w < NP ? w : 0) * SB + (uint32_t)(l % (SB / 16)) * 16u;
  auto load_v = [&](int p) {
    return __builtin_amdgcn_raw_buffer_load_b128(vrsrc, (int)((uint32_t)(p + vrow) * pitch + vb), 0, 0);
  };
  u32x4 vr[D];
  if (w < NP) {
#pragma unroll
    for (int j = 0; j < D; j++)
      if (j < 2 || j * RB < n) vr[j] = load_v(j * RB);
  }
  __syncthreads();
  // lane l takes positions l, l + 64, ..., four at a time; zeros up to whole groups of the O loop
  const int n_up = (n + 255) & ~255;
  for (int h = w; h < rep; h += NW) {
    float m = -1e30f;
#pragma unroll
    for (int i = 0; i < NW; i++) m = fmaxf(m, sm[i * 16 + h]);
    float z = 0.0f;
    for (int t0 = 0; t0 < n_up; t0 += 256) {
      float* pe = P + h * ps + t0 + e_slot(l);
      auto part = [&](auto N) {                     // exps of the first N of the four
        float e[4] = {0.0f, 0.0f, 0.0f, 0.0f}, x[N];
#pragma unroll
        for (int u = 0; u < N; u++) x[u] = pe[64 * u] - m;
        lt_expf_n(x);
#pragma unroll
        for (int u = 0; u < N; u++) e[u] = t0 + 64 * u + l < n ? x[u] : 0.0f;
#pragma unroll
        for (int u = 0; u < 4; u++) {
          pe[64 * u] = e[u];
          if (u < N) z = z + e[u];
        }
      };
      if (n - t0 > 128) part(std::integral_constant<int, 4>{});
      else if (n - t0 > 64) part(std::integral_constant<int, 2>{});
      else part(std::integral_constant<int, 1>{});
    }
    z = wave_tree_dpp(z);
    if (l == 0) sm[NW * 16 + h] = z;
  }
  __syncthreads();
  f32x4 o[1] = {{0.0f, 0.0f, 0.0f, 0.0f}};
  if (w < NP) {
    uint8_t* const vw = vbuf + w * 2048;
    const float* pb = P + (n16 < rep ? n16 : 0) * ps + 4 * g4;
    auto put_v = [&](int buf, u32x4 x) { *(u32x4*)(vw + buf * 1024 + l * 16) = x; };
    constexpr int NS = RB / 4;
    float va[2][NS], ea[2][NS];
    auto read_block = [&](int buf, int p, float (&v)[NS], float (&e)[NS]) {
#pragma unroll
      for (int i = 0; i < RB / 16; i++) {
        const f32x4 x = *(const f32x4*)(pb + p + 16 * i);
#pragma unroll
        for (int s = 0; s < 4; s++) {
          e[4 * i + s] = x[s];
          const uint8_t* y = vw + buf * 1024 + (16 * i + 4 * s + g4) * SB + n16 * kEb;
          v[4 * i + s] = kF16 ? lt_h2f(*(const uint16_t*)y) : *(const float*)y;
        }
      }
    };
    put_v(0, vr[0]);
    put_v(1, vr[1]);
    wave_fence();
    read_block(0, 0, va[0], ea[0]);
    for (int p = 0; p < n; p += D * RB) {
#pragma unroll
      for (int j = 0; j < D; j++) {
        vr[j] = load_v(p + (j + D) * RB);
        wave_fence();
        read_block((j + 1) & 1, p + (j + 1) * RB, va[(j + 1) & 1], ea[(j + 1) & 1]);
        put_v(j & 1, vr[(j + 2) % D]);
#pragma unroll
        for (int i = 0; i < NS; i++) o[0] = mma(va[j & 1][i], ea[j & 1][i], o[0]);
        settle(o);
        if (p + (j + 1) * RB >= n) break;           // (the rest of the group: zero rows)
      }
    }
  }
  __syncthreads();                                  // the exps are free
  float* so = P;                                    // [rep][HD]
  if (w < NP && n16 < rep) {
    const float z = sm[NW * 16 + n16];
#pragma unroll
    for (int r = 0; r < 4; r++) so[n16 * HD + w * 16 + 4 * g4 + r] = o[0][r] / z;
  }
  __syncthreads();
  for (int i = tid; i < rep * HD; i += 512) {       // (whole half-waves: HD is a multiple of 32)
    if (A.out) A.out[((size_t)b * A.nh + (size_t)g * rep) * HD + i] = so[i];
    if (A.oq) {
      const size_t blk = out_block(A, HD, b, g * rep * (HD / 32) + (i >> 5));
      quant_block_hw(so[i], i & 31, A.oq + blk * 32, A.od + blk);
    }
  }
}

// LDS: vectors, a pair of V blocks per wave that folds O, K lines of 8 waves, the exps (read up to a
// block past the last group).
size_t head_lds(int hd, int maxt) {
  return (size_t)(4 * hd + 12 + hd / 16 * 512 + 8 * 64 * 36 + ((maxt + 255) & ~255) + 32) * sizeof(float);
}

int group_cap(int maxt) { return (maxt + 255) & ~255; }
size_t group_lds(int hd, int rep, int maxt) {
  const size_t exps = (size_t)rep * (group_cap(maxt) + 4) + 64, outs = (size_t)rep * hd;
  return (size_t)(8 * 16 + 16 + hd / 16 * 512 + (exps > outs ? exps : outs)) * sizeof(float);
}

}  // namespace

// One workgroup per CU is what both kernels are for: k_attn_head (85 KB of LDS at 1024 rows and heads of
// 64, 94 at 128, up to 256 registers a wave) takes the grids of at most one head per CU, k_attn_group
// those of more heads but at most one KV group per CU, up to its 16 matrix rows.  Past that the workgroups
// run one after the other and the smaller ones of lt_attn.hip are as fast or faster: 512 groups of 2 heads
// of 64, up to 500 rows of fp16, 18.4 us there, 19.6 here; 512 of 4 heads of 128 25.2 / 32.4.
//
// Per launch over 8 to 24 caches in turn, k_attn_w1 or k_attn_dec / here, in us; contexts of a batch
// spread over L/2 .. L.
//   step, rows          16          43          64          100         300         905
//   14 of 64, fp16      4.4 / 4.8   4.7 / 4.9   4.9 / 4.9   5.9 / 5.4   10.2 / 6.8  23.8 / 12.6
//   14 of 64, fp32      5.2 / 4.7   5.2 / 4.8   6.0 / 4.9   7.0 / 5.3   12.8 / 7.9  30.4 / 14.0
//   32 of 128, fp16     9.8 / 5.8   10.7 / 6.2  12.3 / 6.1  15.0 / 7.1  29.1 / 10.5 71.2 / 20
//   32 of 128, fp32     8.3 / 5.8   10.2 / 6.1  11.0 / 6.3  15.6 / 7.4  31.0 / 11.4 80.1 / 21
//   batch, L            8           40          64          100         200         500
//   8 x 14 of 64, fp16  4.9 / 4.3   5.0 / 4.4   5.1 / 4.5   6.8 / 4.7   10.4 / 5.6  17.8 / 8.0
//   8 x 32 of 128, fp16 5.3 / 5.0   5.2 / 5.2   5.2 / 5.4   7.6 / 6.6   11.7 / 9.1  20.3 / 13.3
//   k_attn_group:
//   64 x 14 of 64, fp16 4.8 / 4.8   4.8 / 5.0   4.8 / 5.1   6.8 / 6.1   10.4 / 7.9  17.9 / 12.1
//   64 x 14 of 64, fp32 5.1 / 4.8   5.2 / 5.1   5.4 / 5.5   7.5 / 6.2   11.5 / 8.2  19.9 / 13.9
//   32 x 32 of 128 fp16 5.4 / 5.8   5.8 / 6.3   5.9 / 6.4   8.1 / 8.1   12.2 / 11.3 21.0 / 18.9
//   32 x 32 of 128 fp32 8.2 / 6.0   10.9 / 6.3  11.5 / 6.8  16.0 / 8.4  24.1 / 12.7 47.4 / 24.8
// The length is not known at the launch, so the fp16 rows of at most 64 that lose up to 0.5 us stay.
static bool fits_cus(const lt_ctx* ctx, int batch, int heads) {
  return (size_t)batch * heads <= (size_t)(ctx->num_cus > 0 ? ctx->num_cus : 256);
}

bool lt_attn_head_covers(const lt_ctx* ctx, int batch, int nh, int nkv, int hd, int maxt, bool step) {
  if (hd != 64 && hd != 128) return false;
  if (fits_cus(ctx, batch, nh)) return head_lds(hd, maxt) <= 160 * 1024;
  return !step && fits_cus(ctx, batch, nkv) && nh / nkv <= 16 && (size_t)maxt * nkv * hd * 4 < ((size_t)1 << 31) &&
         group_lds(hd, nh / nkv, maxt) <= 160 * 1024;
}

int lt_attn_head(lt_ctx* ctx, LtAttnHead A, int hd, bool f16, bool step) {
  A.rep = A.nh / A.nkv;
  if (!fits_cus(ctx, A.batch, A.nh)) {
    const size_t shm = group_lds(hd, A.rep, A.maxt);
    const dim3 grid((unsigned)A.nkv, (unsigned)A.batch);
#define LT_GROUP_CASE(F, H) \
  if (f16 == F && hd == H) k_attn_group<F, H><<<grid, 512, shm, ctx->stream>>>(A, group_cap(A.maxt));
    LT_GROUP_CASE(true, 64) LT_GROUP_CASE(false, 64) LT_GROUP_CASE(true, 128) LT_GROUP_CASE(false, 128)
#undef LT_GROUP_CASE
    return lt_check_launch("k_attn_group");
  }
  const size_t shm = head_lds(hd, A.maxt);
  // pair / nkv as pair * rnkv >> 22: exact for the at most 1024 pairs of a grid (nkv <= pairs)
  A.rnkv = (1u << 22) / (uint32_t)A.nkv + 1u;
  const dim3 grid(8, (unsigned)A.rep, (unsigned)((A.batch * A.nkv + 7) / 8));
#define LT_HEAD_CASE(F, H, S)                                                        \
  if (f16 == F && hd == H && step == S) k_attn_head<F, H, 8, S><<<grid, 512, shm, ctx->stream>>>(A);
  LT_HEAD_CASE(true, 64, true) LT_HEAD_CASE(false, 64, true) LT_HEAD_CASE(true, 128, true)
  LT_HEAD_CASE(false, 128, true) LT_HEAD_CASE(true, 64, false) LT_HEAD_CASE(false, 64, false)
  LT_HEAD_CASE(true, 128, false) LT_HEAD_CASE(false, 128, false)
#undef LT_HEAD_CASE
  return lt_check_launch("k_attn_head");
}

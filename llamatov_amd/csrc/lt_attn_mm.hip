// lt_attn_mm.hip -- causal prefill attention on the fp32 matrix cores, bit-identical to the
// per-row kernels of lt_attn.hip.
//
// v_mfma_f32_16x16x4_f32 adds its four products to the accumulator one after the other in
// ascending k, each with one rounding: the sequential fma chain of the reference's scores
// (over the dims) and of its outputs (over the positions), for 16 x 16 chains at once.
// Checked on the device against fmaf chains of 512 terms over normal, subnormal and
// wide-range operands, zeros, infinities and nans (lt_selftest_attn_numerics: all bits equal);
// the parity tests compare whole results.
//
// One workgroup takes 16 consecutive query rows of one head, aligned to a cache position that
// is a multiple of 16, and its NW waves share the work:
//   scores   tiles of 16 positions, a wave every NW-th tile: A = 16 cache rows, B = the 16
//            queries (in registers), four dims per instruction; times scale into LDS [row][pos].
//            A lane loads 16-byte units of its cache row, and a 4 x 4 transpose over the four
//            16-lane groups (v_permlane32_swap / v_permlane16_swap) gives each group the dims
//            it feeds, so K never passes through LDS;
//   softmax  a wave's rows one after the other: lane l holds positions l, l + 64, ... as the
//            reference's 64-lane fold does (max order-free, Z the strided fold and the tree);
//   O        each wave owns 16 DT dims: A = V (four positions), B = the exps from LDS, four
//            positions per instruction in ascending order.
// Positions past LDS capacity are taken in chunks: a first pass over all scores finds the
// rows' maxima, then each chunk's scores are formed again, exponentiated and folded, the
// fold's partial sums and the output chains carried over.
//
// Rows of one tile attend up to 15 positions more or less; a masked exp is 0 and
// fma(0, v, o) = o for every finite v and every o but -0, which becomes +0.  (A chain that
// starts at +0 reaches -0 only where its products all underflow: there a zero's sign may differ
// from the per-row kernels'.)  Where V is not finite in the rows that only part of
// the tile attends, those steps run one position at a time with a select instead.
//
// Bound: the vector units' issue.  An fp32 matrix instruction holds its SIMD for 32 cycles (1024
// fmas, twice the plain vector rate) and vector instructions do not run beside it (a conversion
// before every one: 52 cycles a pair), so the conversions of fp16 rows, the transposes and the
// binary64 exps add to the matrix time.  Measured against the per-row kernel (k_attn_w1): T =
// 2048, 32 heads of 128 over 8 KV heads, fp16, one split: 1772 -> 572 us (60 TF of the 157 TF
// fp32 matrix peak; the second pass is 48% of its score work, a third of scores and outputs
// together); T = 512: 97 -> 39.6 us; T = 509, 14 heads of 64: 41.7 -> 18.5 us.
#include "lt_q8_device.h"

namespace {

using namespace lt;

constexpr uint32_t kNoRow = 0x80000000u;   // out-of-range buffer offset: reads zeros

// Whether one of a dword's values (two fp16 or one fp32) is not finite.
__device__ __forceinline__ int not_finite_bits(uint32_t w, bool f16) {
  return f16 ? (int)((w & 0x7C00u) == 0x7C00u) | (int)((w & 0x7C000000u) == 0x7C000000u)
             : (int)((w & 0x7F800000u) == 0x7F800000u);
}

// kSplit: nsplit splits of the context per row (a multiple of 16 of them, so that the rows of
// a tile, whose lengths lie in (16 c, 16 c + 16], share ceil(L / nsplit)), merged in ascending
// order as k_attn_merge does; all positions in LDS (cap >= maxt).
template <bool kF16, int HD, int NW, bool kSplit>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(2, 3))) void k_attn_mm(LtAttnMm A) {
  extern __shared__ __attribute__((aligned(16))) float lds[];
  constexpr int kEb = kF16 ? 2 : 4;
  constexpr int NU = HD * kEb / 64;                 // 16-byte units per lane and K tile
  constexpr int NP = NW < HD / 16 ? NW : HD / 16;   // waves that fold O
  constexpr int DT = HD / 16 / NP;                  // adjacent dims per lane in O
  constexpr int kVB = DT * kEb;                     // V bytes per lane and position
  static_assert(kVB == 2 || kVB == 4 || kVB == 8, "k_attn_mm: V element");
  constexpr int SB = 16 * kVB;                      // a wave's bytes of one V row
  constexpr int RB = 1024 / SB;                     // V rows per block (one 16-byte load per lane)
  constexpr int D = 4;                              // V blocks in flight
  constexpr int QPW = 16 / NW;                      // rows per wave in the softmax
  const int ps = A.cap + 4;                         // row pitch of P
  float* P = lds;                                   // [16][ps] (+ 64: reads past the last row's end)
  float* sm = P + 16 * ps + 64;                     // [NW][16] maxima of the waves' tiles
  float* sz = sm + NW * 16;                         // [16] Z
  uint8_t* sv = (uint8_t*)(sz + 16);                // [NP][2][1024] V blocks
  float* ssm = (float*)(sv + NP * 2048);            // kSplit: [16][nsplit] m_s, then w_s
  float* ssz = ssm + 16 * A.nsplit;                 // kSplit: [16][nsplit] Z_s
  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63;
  const int n = l & 15, g4 = l >> 4;                // this lane's row (or dim, position) and group

  // longest tiles first; consecutive workgroups go round the KV groups, which keeps a group's
  // cache rows on one XCD when there are 8 groups
  const int ti = (int)blockIdx.x / A.nh, hi = (int)blockIdx.x - ti * A.nh;
  const int g = hi % A.nkv, h = g * (A.nh / A.nkv) + hi / A.nkv;
  const int tj = A.ntiles - 1 - ti;
  const int len0 = *A.len;
  // row 0's query index and cache position: for splits the position is a multiple of 16
  const int t0 = kSplit ? ((len0 >> 4) + tj) * 16 - len0 : tj * 16;
  const int pf = t0 + len0;
  if (kSplit && (t0 >= A.T || t0 + 15 < 0)) return;
  auto clampL = [&](int L) { return L < 0 ? 0 : (L > A.maxt ? A.maxt : L); };
  const int tlo = t0 < 0 ? 0 : t0, thi = t0 + 15 < A.T - 1 ? t0 + 15 : A.T - 1;
  const int Lmin = clampL(len0 + tlo + 1), Lmax = clampL(len0 + thi + 1);
  auto rowL = [&](int r) { return t0 + r >= 0 && t0 + r < A.T ? clampL(pf + r + 1) : 0; };
  const int Ln = rowL(n);

  const uint32_t pitch = (uint32_t)A.nkv * HD * kEb;
  const uint32_t gb = (uint32_t)g * HD * kEb;
  auto rows_of = [&](const void* c, int rows) {     // the cache's first rows; later rows read zeros
    return __builtin_amdgcn_make_buffer_rsrc((void*)c, 0, (int)((uint32_t)rows * pitch), 0x00020000);
  };

  // loads return in order: the queries first, as B operands (register i of group g4 is q[row n][4i + g4])
  u32x4 qv[HD / 16];
  {
    const int tq = t0 + n < 0 ? 0 : (t0 + n < A.T ? t0 + n : A.T - 1);
    const float* qs = A.q + (size_t)tq * A.q_stride + (size_t)h * HD;
#pragma unroll
    for (int j = 0; j < HD / 16; j++) qv[j] = *(const u32x4_a4*)(qs + 16 * j + 4 * g4);
  }
  // K tile at position p: unit 4j + g4 of row p + n.  Only the first waves' first tiles are requested before
  // the length is known, all else through a descriptor that ends at it
  auto k_off = [&](int p) { return (uint32_t)(p + n) * pitch + gb + (uint32_t)g4 * 16u; };
  auto load_unit = [&](__amdgpu_buffer_rsrc_t k, uint32_t off, int j) {
    return __builtin_amdgcn_raw_buffer_load_b128(k, (int)(off + 64u * j), 0, 0);
  };
  u32x4 kb[2][NU];                                  // the wave's next two tiles
  constexpr int kEarly = 2;
  if (w < kEarly) {
    const __amdgpu_buffer_rsrc_t all = rows_of(A.kc, A.maxt);
#pragma unroll
    for (int j = 0; j < NU; j++) kb[0][j] = load_unit(all, k_off(w * 16), j);
  }
  const __amdgpu_buffer_rsrc_t krsrc = rows_of(A.kc, Lmax), vrsrc = rows_of(A.vc, Lmax);
  auto load_two = [&](int p, bool first) {
#pragma unroll
    for (int i = 0; i < 2; i++)
      if (!first || i == 1 || w >= kEarly) {
#pragma unroll
        for (int j = 0; j < NU; j++) kb[i][j] = load_unit(krsrc, k_off(p + (w + i * NW) * 16), j);
      }
  };
  load_two(0, true);

  // O: a wave's V dims of RB rows arrive by one 16-byte load per lane and pass through 1 KB of
  // LDS (the wave's own, two blocks in turn) to the lanes: lane (n, g4) feeds dims db + DT n ..
  // of position 4 i + g4
  const int db = w * 16 * DT;
  const int vrow = l / (SB / 16);
  const uint32_t vb = gb + (uint32_t)db * kEb + (uint32_t)(l % (SB / 16)) * 16u;
  u32x4 vr[D];

  float qr[HD / 4];
#pragma unroll
  for (int j = 0; j < HD / 16; j++) {
    uint32_t r[4] = {qv[j].x, qv[j].y, qv[j].z, qv[j].w};
    transpose4(r);
#pragma unroll
    for (int e = 0; e < 4; e++) qr[4 * j + e] = __uint_as_float(r[e]);
  }
  // a tile's scores: register r of (row n, group g4) is position 4 g4 + r; each unit is
  // replaced by that of the tile two ahead as soon as it is taken
  auto s_tile = [&](u32x4 (&kt)[NU], uint32_t next) {
    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int j = 0; j < NU; j++) {
      u32x4 k = kt[j];
      asm volatile("" : "+v"(k.x), "+v"(k.y), "+v"(k.z), "+v"(k.w));
      if (kF16) {
        // dims 32j + 8 g4 + e as pairs (e, e + 4): after the transpose, pair s is dims
        // 32j + 8s + g4 and + 4
        uint32_t r[4] = {__builtin_amdgcn_perm(k.z, k.x, 0x05040100u),
                         __builtin_amdgcn_perm(k.z, k.x, 0x07060302u),
                         __builtin_amdgcn_perm(k.w, k.y, 0x05040100u),
                         __builtin_amdgcn_perm(k.w, k.y, 0x07060302u)};
        kt[j] = load_unit(krsrc, next, j);
        transpose4(r);
#pragma unroll
        for (int s = 0; s < 4; s++) {
          acc = mma(lt_h2f((uint16_t)(r[s] & 0xFFFFu)), qr[8 * j + 2 * s], acc);
          acc = mma(lt_h2f((uint16_t)(r[s] >> 16)), qr[8 * j + 2 * s + 1], acc);
        }
      } else {
        uint32_t r[4] = {k.x, k.y, k.z, k.w};
        kt[j] = load_unit(krsrc, next, j);
        transpose4(r);
#pragma unroll
        for (int s = 0; s < 4; s++) acc = mma(__uint_as_float(r[s]), qr[4 * j + s], acc);
      }
    }
    return acc;
  };
  // the scores of positions [c0, c1) into P (kept) or into the running maximum only
  float mx = -1e30f;
  auto score = [&](int c0, int c1, bool keep, bool max) {
    for (int p = c0 + w * 16; p < c1; p += 32 * NW) {
#pragma unroll
      for (int i = 0; i < 2; i++) {
        const int pi = p + 16 * NW * i;
        if (pi < c1) {
          f32x4 s = s_tile(kb[i], k_off(pi + 32 * NW));
#pragma unroll
          for (int r = 0; r < 4; r++) {
            s[r] = s[r] * A.scale;
            if (max && pi + 4 * g4 + r < Ln) mx = fmaxf(mx, s[r]);
          }
          if (keep) *(f32x4*)(P + n * ps + (pi - c0) + 4 * g4) = s;
        }
      }
    }
  };

  uint8_t* const svw = sv + (w < NP ? w : 0) * 2048;
  auto load_v = [&](int row, int rows) {            // rows [row, row + rows), zeros past them
    return __builtin_amdgcn_raw_buffer_load_b128(
        vrsrc, vrow < rows ? (int)((uint32_t)(row + vrow) * pitch + vb) : (int)kNoRow, 0, 0);
  };
  auto put_v = [&](int buf, u32x4 x) { *(u32x4*)(svw + buf * 1024 + l * 16) = x; };
  f32x4 o[DT];
#pragma unroll
  for (int d = 0; d < DT; d++) o[d] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  // step i of the block in buffer buf: positions 4 i .. 4 i + 3, group g4 holding 4 i + g4
  auto get_v = [&](int buf, int i, float (&a)[DT]) {
    const uint8_t* x = svw + buf * 1024 + (4 * i + g4) * SB + n * kVB;
    if (kF16) {
      if (DT == 1) {
        a[0] = lt_h2f(*(const uint16_t*)x);
      } else {
        const uint32_t y = *(const uint32_t*)x;
        a[0] = lt_h2f((uint16_t)(y & 0xFFFFu));
        a[DT - 1] = lt_h2f((uint16_t)(y >> 16));
      }
    } else {
#pragma unroll
      for (int d = 0; d < DT; d++) a[d] = ((const float*)x)[d];
    }
  };
  auto fold = [&](int buf, int i, float b) {        // b: the exps of row n
    float a[DT];
    get_v(buf, i, a);
#pragma unroll
    for (int d = 0; d < DT; d++) o[d] = mma(a[d], b, o[d]);
  };
  // the same step with each row taking only the positions (p + k) it attends
  auto fold_masked = [&](int buf, int i, float b, int p) {
    float a[DT];
    get_v(buf, i, a);
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const bool mine = g4 == k;
#pragma unroll
      for (int d = 0; d < DT; d++) {
        const f32x4 y = mma(mine ? a[d] : 0.0f, mine ? b : 0.0f, o[d]);
#pragma unroll
        for (int r = 0; r < 4; r++) o[d][r] = p + k < Ln ? y[r] : o[d][r];
      }
    }
  };
  auto not_finite = [&](const u32x4& x) {
    return (not_finite_bits(x.x, kF16) | not_finite_bits(x.y, kF16) | not_finite_bits(x.z, kF16) |
            not_finite_bits(x.w, kF16)) != 0;
  };

  if constexpr (!kSplit) {
    const bool multi = Lmax > A.cap;
    // the maxima: with the scores where they all fit, in a pass of their own else
    if (multi) {
      score(0, Lmax, false, true);
      load_two(0, false);
    } else {
      score(0, Lmax, true, true);
    }
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    if (l < 16) sm[w * 16 + l] = mx;
    float m[QPW], zs[QPW];
    int Lq[QPW];
    for (int c0 = 0; c0 < Lmax; c0 += A.cap) {
      const int c1 = c0 + A.cap < Lmax ? c0 + A.cap : Lmax;
      if (multi) score(c0, c1, true, false);
      if (w < NP) {
#pragma unroll
        for (int j = 0; j < D; j++) vr[j] = load_v(c0 + j * RB, RB);
      }
      __syncthreads();
      if (c0 == 0) {
#pragma unroll
        for (int u = 0; u < QPW; u++) {
          m[u] = -1e30f;
          for (int i = 0; i < NW; i++) m[u] = fmaxf(m[u], sm[i * 16 + w * QPW + u]);
          zs[u] = 0.0f;
          Lq[u] = rowL(w * QPW + u);
        }
      }
      for (int t = l; t < ((c1 - c0 + 63) & ~63); t += 64) {
        float* pe = P + w * QPW * ps + t;
        float e[QPW];
#pragma unroll
        for (int u = 0; u < QPW; u++) e[u] = pe[u * ps] - m[u];
        lt_expf_n(e);
#pragma unroll
        for (int u = 0; u < QPW; u++) {
          e[u] = c0 + t < Lq[u] ? e[u] : 0.0f;
          pe[u * ps] = e[u];
          zs[u] = zs[u] + e[u];
        }
      }
      __syncthreads();
      if (w < NP) {
        const float* pb = P + n * ps + g4;
        const int cf = c1 < Lmin ? c1 : Lmin;       // every row attends the positions before cf
        int p = c0;
        // block j of a group of D in buffer j % 2, written one block ahead of its folds; the fence
        // keeps a block's folds behind its writes and before the next writes of its buffer
        put_v(0, vr[0]);
        for (; p + D * RB <= cf; p += D * RB) {
#pragma unroll
          for (int j = 0; j < D; j++) {
            vr[j] = load_v(p + (j + D) * RB, RB);
            wave_fence();
            put_v((j + 1) & 1, vr[(j + 1) % D]);
            const float* pj = pb + (p - c0) + j * RB;
#pragma unroll
            for (int i = 0; i < RB / 4; i++) fold(j & 1, i, pj[4 * i]);
          }
          settle(o);
        }
        for (; p < c1; p += D * RB) {               // the rows' last positions
#pragma unroll
          for (int j = 0; j < D; j++) {
            vr[j] = load_v(p + (j + D) * RB, RB);
            wave_fence();
            put_v((j + 1) & 1, vr[(j + 1) % D]);
            if (p + j * RB >= c1) continue;
            const float* pj = pb + (p - c0) + j * RB;
            if (__any(not_finite(*(const u32x4*)(svw + (j & 1) * 1024 + l * 16)))) {
              for (int i = 0; i < RB / 4; i++) fold_masked(j & 1, i, pj[4 * i], p + j * RB + 4 * i);
            } else {
#pragma unroll
              for (int i = 0; i < RB / 4; i++) fold(j & 1, i, pj[4 * i]);
            }
            settle(o);
          }
        }
      }
      if (multi) {
        load_two(c1, false);
        __syncthreads();                            // the next chunk rewrites P
      }
    }
    if (Lmax == 0) {
#pragma unroll
      for (int u = 0; u < QPW; u++) zs[u] = 0.0f;
    }
#pragma unroll
    for (int u = 0; u < QPW; u++) {
      const float z = wave_tree_dpp(zs[u]);
      if (l == 0) sz[w * QPW + u] = z;
    }
  } else {
    const int S = A.nsplit;
    const int per = (Lmax + S - 1) / S;             // the same for every row of the tile
    score(0, Lmax, true, false);
    auto in_split = [&](int s, int L) {             // positions of split s below L
      const int q0 = s * per;
      return q0 >= L ? 0 : (L - q0 < per ? L - q0 : per);
    };
    // V in blocks of RB rows (a split's last block holds fewer): block i in buffer i % 2,
    // written while block i - 1 is folded, D in flight
    struct Cur { int s, j, n; };                    // a block: rows j .. of split s, which holds n
    auto next = [&](Cur c) {
      const bool more = c.j + RB < c.n;
      const int s = c.n == 0 || more ? c.s : c.s + 1;
      return Cur{s, more ? c.j + RB : 0, more ? c.n : (s < S ? in_split(s, Lmax) : 0)};
    };
    auto load_cur = [&](Cur c) { return load_v(c.s * per + c.j, c.n - c.j); };
    Cur cur = {0, 0, in_split(0, Lmax)}, cl = cur;
    if (w < NP) {
#pragma unroll
      for (int j = 0; j < D; j++) {
        vr[j] = load_cur(cl);
        cl = next(cl);
      }
    }
    __syncthreads();
    // The wave's rows: per split the maximum m_s, then the exps of all positions, then Z_s.  A
    // half-wave takes a split of at most 32 positions (the upper half of the 64-lane tree then
    // adds zeros), a wave a longer one.
    const int r0 = w * QPW;
    float* const sv_spare = P + 16 * ps;            // written by the lanes that hold no sum
    int Lq[QPW];
#pragma unroll
    for (int u = 0; u < QPW; u++) Lq[u] = rowL(r0 + u);
    if (per <= 32) {
      const int hl = l & 31;
      for (int s = l >> 5; s < S; s += 2) {         // S is even
#pragma unroll
        for (int u = 0; u < QPW; u++) {
          const float x = P[(r0 + u) * ps + s * per + (hl < per ? hl : 0)];
          ssm[(r0 + u) * S + s] = halfwave_max(hl < in_split(s, Lq[u]) ? x : -1e30f);
        }
      }
    } else {
      for (int s = 0; s < S; s++) {
#pragma unroll
        for (int u = 0; u < QPW; u++) {
          float ms = -1e30f;
          for (int t = l; t < in_split(s, Lq[u]); t += 64) ms = fmaxf(ms, P[(r0 + u) * ps + s * per + t]);
          ssm[(r0 + u) * S + s] = wave_max(ms);
        }
      }
    }
    wave_fence();
    {
      // t / per by a multiplication: exact for t below 2^16 (the error of rper is below 2^-32)
      const uint32_t rper = per > 1 ? (uint32_t)(((1ull << 32) + per - 1) / (uint32_t)per) : 0u;
      for (int t = l; t < ((Lmax + 63) & ~63); t += 64) {
        int s = per > 1 ? (int)__umulhi((uint32_t)t, rper) : t;
        s = s < S ? s : S - 1;
        float* pe = P + r0 * ps + t;
        float e[QPW];
#pragma unroll
        for (int u = 0; u < QPW; u++) e[u] = pe[u * ps] - ssm[(r0 + u) * S + s];
        lt_expf_n(e);
#pragma unroll
        for (int u = 0; u < QPW; u++) pe[u * ps] = t < Lq[u] ? e[u] : 0.0f;
      }
    }
    wave_fence();
    if (per <= 32) {
      const int hl = l & 31;
      for (int s = l >> 5; s < S; s += 2) {
#pragma unroll
        for (int u = 0; u < QPW; u++) {
          const float x = P[(r0 + u) * ps + s * per + (hl < per ? hl : 0)];
          const float z = halfwave_tree_dpp(hl < in_split(s, Lq[u]) ? x : 0.0f);
          (hl == 0 ? ssz + (r0 + u) * S + s : sv_spare)[0] = z;
        }
      }
    } else {
      for (int s = 0; s < S; s++) {
#pragma unroll
        for (int u = 0; u < QPW; u++) {
          float z = 0.0f;
          for (int t = l; t < in_split(s, Lq[u]); t += 64) z = z + P[(r0 + u) * ps + s * per + t];
          z = wave_tree_dpp(z);
          (l == 0 ? ssz + (r0 + u) * S + s : sv_spare)[0] = z;
        }
      }
    }
    // w_s = exp(m_s - M) in place, Z = sum fma(w_s, Z_s) in ascending split order
    wave_fence();
#pragma unroll
    for (int u = 0; u < QPW; u++) {
      float* sr = ssm + (r0 + u) * S;
      float M = -1e30f;
      for (int s = l; s < S; s += 64) M = fmaxf(M, sr[s]);
      M = wave_max(M);
      for (int s = l; s < S; s += 64) sr[s] = lt_expf_sel(sr[s] - M);
    }
    wave_fence();
    if (l < QPW) {
      float Z = 0.0f;
      for (int s = 0; s < S; s++) Z = fmaf(ssm[(r0 + l) * S + s], ssz[(r0 + l) * S + s], Z);
      sz[r0 + l] = Z;
    }
    __syncthreads();
    if (w < NP) {
      f32x4 a[DT];
#pragma unroll
      for (int d = 0; d < DT; d++) a[d] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
      put_v(0, vr[0]);
      while (cur.n > 0) {
#pragma unroll
        for (int j = 0; j < D; j++) {
          vr[j] = load_cur(cl);
          cl = next(cl);
          wave_fence();
          put_v((j + 1) & 1, vr[(j + 1) % D]);
          if (cur.n > 0) {
            const int p = cur.s * per + cur.j, left = cur.n - cur.j;
            const float* pb = P + n * ps + p + g4;
            if (p + RB > Lmin && __any(not_finite(*(const u32x4*)(svw + (j & 1) * 1024 + l * 16)))) {
              for (int i = 0; i < RB / 4; i++)
                fold_masked(j & 1, i, 4 * i + g4 < left ? pb[4 * i] : 0.0f, p + 4 * i);
            } else {
#pragma unroll
              for (int i = 0; i < RB / 4; i += 2) {   // (pairs of steps: a short block skips the rest)
                if (4 * i >= left) break;
                const float b0 = pb[4 * i], b1 = pb[4 * i + 4];
                fold(j & 1, i, 4 * i + g4 < left ? b0 : 0.0f);
                fold(j & 1, i + 1, 4 * i + 4 + g4 < left ? b1 : 0.0f);
              }
            }
            settle(o);
            if (cur.j + RB >= cur.n) {                // the split's last block
              const float ws = ssm[n * S + cur.s];
#pragma unroll
              for (int d = 0; d < DT; d++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                  a[d][r] = fmaf(ws, o[d][r], a[d][r]);
                  o[d][r] = 0.0f;
                }
            }
            cur = next(cur);
          }
        }
      }
#pragma unroll
      for (int d = 0; d < DT; d++) o[d] = a[d];
    }
  }
  __syncthreads();
  // lane (row n, group g4): dims db + DT (4 g4 + r) + d
  if (w < NP && t0 + n >= 0 && t0 + n < A.T) {
    const float z = sz[n];
    float* dst = A.out + ((size_t)(t0 + n) * A.nh + h) * HD + db + DT * 4 * g4;
#pragma unroll
    for (int r = 0; r < 4; r++)
#pragma unroll
      for (int d = 0; d < DT; d++) dst[DT * r + d] = o[d][r] / z;
  }
}

constexpr int kLds = 160 * 1024;

size_t mm_lds(int cap, int nsplit) {
  return (size_t)(16 * (cap + 4) + 64 + 8 * 16 + 16 + 8 * 512 + (nsplit > 1 ? 32 * nsplit : 0)) * sizeof(float);
}

}  // namespace

// Splits cost a merge of the chains per split and tile whatever the length, so short prompts
// stay on the per-row kernel (16 splits, 32 heads of 128, maxt 1024, per-row / here: T = 100
// 19.0 / 22.3 us, 200 28.7 / 42.3, 512 106 / 95, and at maxt 512 87 / 71).  So do the shortest contexts, a
// tile or a few of which leave most waves idle, where the caller knows them (us over caches of 1024 rows):
//   T at 0 cached       16          32          48          64          100         135
//   14 of 64, fp16      3.9 / 5.4   4.0 / 5.5   4.6 / 5.9   4.7 / 6.0   6.9 / 7.2   9.8 / 8.8
//   14 of 64, fp32      4.0 / 5.5   4.1 / 5.7   4.9 / 6.0   5.0 / 6.3   8.2 / 7.2   13.3 / 8.9
//   32 of 128, fp16     5.9 / 7.3   6.0 / 7.3   8.0 / 8.0   8.2 / 8.2   13.0 / 10.1 24.2 / 12.9
//   32 of 128, fp32     5.3 / 7.5   5.8 / 7.7   8.0 / 8.2   8.8 / 8.8   14.2 / 10.4 25.3 / 13.6
// (16 at 100 cached: 6.0 / 7.7, 6.8 / 7.7, 12.1 / 10.3, 13.1 / 10.9; at 500: 17.2 / 16.3, 19.1 / 16.1,
// 40.5 / 23.1, 44.9 / 23.2).
bool lt_attn_mm_covers(int hd, bool f16, int T, int maxt, int end, int nsplit) {
  if (hd != 64 && hd != 128) return false;
  if (nsplit == 1) return end > (hd == 128 ? 32 : f16 ? 112 : 64);
  return (nsplit % 16 == 0 && T >= 384 && mm_lds((maxt + 63) & ~63, nsplit) <= (size_t)kLds);
}

int lt_attn_mm_prefill(lt_ctx* ctx, LtAttnMm A, int hd, bool f16) {
  const int all = (A.maxt + 63) & ~63;
  A.ntiles = A.nsplit > 1 ? (A.T + 30) / 16 : (A.T + 15) / 16;
  // Positions in LDS and waves per workgroup: 512 positions and 4 waves keep three workgroups
  // on a CU, which hide each other's loads and softmax (T = 2048 at 32 heads of 128, one split:
  // 572 us against 709 at 1024 positions and 8 waves; T = 512: 39.6 against 55.8).  A grid of
  // at most one workgroup per CU has nothing to hide behind and splits each tile over 8 waves,
  // with fewer second score passes (T = 37 at 900 cached, fp32: 36 against 54 us); so do splits
  // whose context passes 512 positions, all of which LDS holds (T = 512, 16 splits, maxt 1024:
  // 95 against 115; 512: 94 against 71).
  const int cus = ctx->num_cus > 0 ? ctx->num_cus : 256;
  const bool few = A.ntiles * A.nh <= cus;
  A.cap = A.nsplit > 1 ? all : few ? (all < 1024 ? all : 1024) : (all < 512 ? all : 512);
  const int nw = (A.nsplit > 1 ? A.cap > 512 : few) ? 8 : 4;
  const size_t shm = mm_lds(A.cap, A.nsplit);
  const dim3 grid((unsigned)A.ntiles * (unsigned)A.nh);
#define LT_MM_CASE(F, H, W)                                                          \
  if (f16 == F && hd == H && nw == W) {                                              \
    if (A.nsplit > 1)                                                                \
      k_attn_mm<F, H, W, true><<<grid, 64 * W, shm, ctx->stream>>>(A);               \
    else                                                                             \
      k_attn_mm<F, H, W, false><<<grid, 64 * W, shm, ctx->stream>>>(A);              \
  }
  LT_MM_CASE(true, 64, 4) LT_MM_CASE(true, 128, 4) LT_MM_CASE(false, 64, 4) LT_MM_CASE(false, 128, 4)
  LT_MM_CASE(true, 64, 8) LT_MM_CASE(true, 128, 8) LT_MM_CASE(false, 64, 8) LT_MM_CASE(false, 128, 8)
#undef LT_MM_CASE
  return lt_check_launch("k_attn_mm");
}

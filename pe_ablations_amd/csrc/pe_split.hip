// The fp32 compute type on the bf16 matrix cores (gfx950).  The fp32 matrix instruction does 64 FLOP a
// cycle and SIMD, the bf16 one 1024, so an fp32 product is formed from bf16 ones: every operand is the
// exact sum of three bf16 planes h + m + l (split_bf3), and of the nine plane products the six down to
// h l' + m m' + l h' are kept, six bf16 instructions for sixteen times the rate.  What is left out
// (m l' + l m' + l l') is below 2^-24 of the product, with the sign of rounding errors: less than the
// rounding of one fp32 product.  The products themselves are exact and the sums are fp32, as on the fp32
// unit.  Infinite operands give infinities and NaN where the fp32 unit gives them (split_big); a dS that
// overflows gives NaN in dq and dk.
//
// Operand rows hold their planes one after another (row_store8, DT_SPLIT), so a tile is three bf16 tiles
// of the 16-bit kernels' kind and everything about fragments, swizzles and the transpose load is theirs.
#include "pe_common.h"
#include "pe_internal.h"

namespace pe {

// c0 += the leading product h h', c1 += the five correction products, smallest first (c0 and c1 apart
// keep the corrections from being rounded at the size of the sum)
__device__ __forceinline__ void mma6(const u32x4 (&a)[3], const u32x4 (&b)[3], f32x16& c0, f32x16& c1) {
  using M = MT<0>;
  c1 = M::mma(a[2], b[0], c1);
  c1 = M::mma(a[0], b[2], c1);
  c1 = M::mma(a[1], b[1], c1);
  c1 = M::mma(a[1], b[0], c1);
  c1 = M::mma(a[0], b[1], c1);
  c0 = M::mma(a[0], b[0], c0);
}

// 8 consecutive C values (base j0) as the three operand fragments of the next product
__device__ __forceinline__ void split_frag(const f32x16& c, int j0, u32x4 (&f)[3]) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    uint32_t h, m, l;
    split_bf3(c[j0 + 2 * e], c[j0 + 2 * e + 1], h, m, l);
    f[0][e] = h; f[1][e] = m; f[2][e] = l;
  }
}

// Forward.  A workgroup of four waves owns 128 queries, each wave 32 of them with their q~ planes in
// registers (192 of 512 at QK width 256, one wave per SIMD), and streams 32-key tiles of the k~ and v
// planes through two double-buffered LDS rings (2 x 48 and 2 x 24 KiB at QK 256 / V 128).  Every fragment
// read (three planes) feeds six products, so the LDS is half used while the matrix cores run.  One wave per
// SIMD has no other wave to hide its vector work behind, so the steps are staggered: the scores of tile
// kb + 1 are formed while the exponentials and the split of P of tile kb run between their products
// (k~ therefore runs one tile ahead of v).  Only the row max of a tile stands alone.  With two waves per
// SIMD (narrow operands, OCC 2) the other wave fills those gaps and the steps follow each other.
template <int DQK, int DV, int OCC>
__global__ __launch_bounds__(256, OCC) void fwd_split_kernel(CoreArgs a, int o_vec) {
  constexpr int NW = 4, BM = 128, BN = 32;
  constexpr int NCK = DQK / 8, NCV = DV / 8, NQF = DQK / 16, NOT = DV / 32;
  constexpr int SK_PL = BN * NCK * 16, SV_PL = BN * NCV * 16, KT = 3 * SK_PL, VT = 3 * SV_PL;
  constexpr int SO_STRIDE = DV * 4 + 16;
  constexpr int SMEM = 2 * (KT + VT) > BM * SO_STRIDE ? 2 * (KT + VT) : BM * SO_STRIDE;
  __shared__ __attribute__((aligned(1024))) char smem[SMEM];  // k~ slots 0, 1, then v slots 0, 1

  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, g = lane >> 5, l32 = lane & 31;
  const int nqb = (a.Sq + BM - 1) / BM;
  int qb, bh;
  map_block(blockIdx.x, nqb, a.B * a.Hq, a.causal != 0, qb, bh);
  const int b = bh / a.Hq, h = bh % a.Hq, hk = h / (a.Hq / a.Hkv);
  const int q0 = qb * BM, qw = q0 + w * 32, myq = qw + l32;
  const int off = a.causal_off;

  u32x4 qf[NQF][3];
  {
    const uint16_t* qrow = (const uint16_t*)a.q + ((int64_t)(b * a.Hq + h) * a.Sq + (myq < a.Sq ? myq : a.Sq - 1)) * 3 * DQK;
#pragma unroll
    for (int kk = 0; kk < NQF; ++kk)
#pragma unroll
      for (int p = 0; p < 3; ++p) qf[kk][p] = *(const u32x4*)(qrow + p * DQK + kk * 16 + g * 8);
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): seen by the compiler, as in the 16-bit forward
  }

  int kend = a.Sk;
  if (a.causal) kend = min(a.Sk, q0 + BM + off);
  const int nkb = kend > 0 ? (kend + BN - 1) / BN : 0;
  const int64_t krs = 3 * DQK * 2, vrs = 3 * DV * 2;
  const char* kbase = (const char*)a.k + (int64_t)(b * a.Hkv + hk) * a.Sk * krs;
  const char* vbase = (const char*)a.v + (int64_t)(b * a.Hkv + hk) * a.Sk * vrs;

  const RowFrags<NCK, 0> rk(perm_row<0>(l32), g);
  const ColFrags<NCV, 1> cv(lane);
  // O^T: the leading products and, where the registers hold them apart (they spill at these two widths),
  // the corrections, added at the end
  constexpr bool OC = !(DQK == 256 && DV == 128) && !(DQK == 128 && OCC == 2);
  f32x16 o[NOT], oc_[OC ? NOT : 1];
  f32x16* const oc = OC ? oc_ : o;
#pragma unroll
  for (int t = 0; t < NOT; ++t)
#pragma unroll
    for (int j = 0; j < 16; ++j) { o[t][j] = 0.f; oc[t][j] = 0.f; }
  float m = -1e30f, l = 0.f;
  const float sl2 = a.scale * LOG2E;

  const DmaPlan<BN, NCK, NW, 0> plan_k(w, lane, (uint32_t)krs);
  const DmaPlan<BN, NCV, NW, 1> plan_v(w, lane, (uint32_t)vrs);
  const uint32_t smem_l = lds_addr(smem);
  auto issue_k = [&](int kb) {
    const int k0 = kb * BN, slot = (kb & 1) * KT;
    const char* src = kbase + (int64_t)k0 * krs;
    if (a.Sk - k0 >= BN) {
#pragma unroll
      for (int p = 0; p < 3; ++p) plan_k.full(src + p * DQK * 2, smem_l + (uint32_t)(slot + p * SK_PL), w, (uint32_t)krs);
    } else {
      int ln = lane;
      asm volatile("" : "+v"(ln));
#pragma unroll
      for (int p = 0; p < 3; ++p) dma_tile<BN, NCK, NW, 0>(smem + slot + p * SK_PL, src + p * DQK * 2, krs, a.Sk - k0, w, ln);
    }
  };
  auto issue_v = [&](int kb) {
    const int k0 = kb * BN, slot = 2 * KT + (kb & 1) * VT;
    const char* src = vbase + (int64_t)k0 * vrs;
    if (a.Sk - k0 >= BN) {
#pragma unroll
      for (int p = 0; p < 3; ++p) plan_v.full(src + p * DV * 2, smem_l + (uint32_t)(slot + p * SV_PL), w, (uint32_t)vrs);
    } else {
      int ln = lane;
      asm volatile("" : "+v"(ln));
#pragma unroll
      for (int p = 0; p < 3; ++p) dma_tile<BN, NCV, NW, 1>(smem + slot + p * SV_PL, src + p * DV * 2, vrs, a.Sk - k0, w, ln);
    }
  };
  // tiles this wave has a visible key in (the rest lie above its diagonal)
  int nvis = nkb;
  if (a.causal) nvis = max(0, min(nkb, (qw + 31 + off) / BN + 1));
  if (qw + 31 + off < 0 && a.causal) nvis = 0;
  nvis = __builtin_amdgcn_readfirstlane(nvis);

  constexpr bool STAG = OCC == 1;
  f32x16 s;                // scores of the tile in hand
  u32x4 pf[2][3];          // its P as operand planes
  float rs = 0.f;
  // the scores of tile kn into s; with PREV the elements of sp (the previous tile's scaled scores)
  // become probabilities and operand planes between the products
  auto scores = [&](int kn, f32x16& sp, auto prev_tag) {
    constexpr bool PREV = decltype(prev_tag)::value;
    constexpr int EPS = 16 / NQF > 0 ? 16 / NQF : 1;  // elements of P per contraction step
    int slot = (kn & 1) * KT;
    asm volatile("" : "+s"(slot));
    const char* sK = smem + slot;
    f32x16 c0, c1;
#pragma unroll
    for (int j = 0; j < 16; ++j) { c0[j] = 0.f; c1[j] = 0.f; }
    u32x4 kq[2][3];
#pragma unroll
    for (int p = 0; p < 3; ++p) kq[0][p] = rk.read(sK + p * SK_PL, 0, 0);
#pragma unroll
    for (int kk = 0; kk < NQF; ++kk) {
      __builtin_amdgcn_sched_barrier(0);
      if (kk + 1 < NQF) {  // fragments one contraction step (192 cycles) ahead of their products
#pragma unroll
        for (int p = 0; p < 3; ++p) kq[(kk + 1) & 1][p] = rk.read(sK + p * SK_PL, 0, kk + 1);
      }
      mma6(kq[kk & 1], qf[kk], c0, c1);
      if constexpr (PREV) {
#pragma unroll
        for (int e = 0; e < EPS; ++e) {
          const int j = kk * EPS + e;
          const float p = fast_exp2(sp[j] - m);
          sp[j] = p;
          rs += p;
          if (j & 1) {
            uint32_t h, mm, ll;
            split_bf3(sp[j - 1], p, h, mm, ll);
            pf[j / 8][0][(j % 8) / 2] = h;
            pf[j / 8][1][(j % 8) / 2] = mm;
            pf[j / 8][2][(j % 8) / 2] = ll;
          }
        }
        // one product, then the vector work that runs beside it
#pragma unroll
        for (int i = 0; i < 6; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x402, 3 * EPS, 0);
        }
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    s = c0 + c1;
  };

  if (nkb > 0) {
    issue_k(0);
    dma_wait();
    __syncthreads();
    issue_v(0);
    if (nkb > 1) issue_k(1);
    if (nvis > 0) scores(0, s, std::false_type{});
  }
  for (int kb = 0; kb < nkb; ++kb) {
    const int k0 = kb * BN;
    f32x16 sp;
    if (kb < nvis) {  // scaled scores and row max of tile kb
      const bool edge = (a.causal && k0 + BN - 1 > qw + off) || (k0 + BN > a.Sk);
      float mx = m;
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        float x = s[j] * sl2;
        if (edge) {
          const int key = k0 + c_logical<0>(j, g);
          if (key >= a.Sk || (a.causal && key > myq + off)) x = -INFINITY;
        }
        sp[j] = x;
        mx = fmaxf(mx, x);
      }
      mx = fmaxf(mx, xor32(mx));
      if (__any(mx > m)) {
        const float alpha = fast_exp2(m - mx);
        m = mx;
        l *= alpha;
#pragma unroll
        for (int t = 0; t < NOT; ++t)
#pragma unroll
          for (int j = 0; j < 16; ++j) {
            o[t][j] *= alpha;
            if (OC) oc[t][j] *= alpha;
          }
      }
    }
    dma_wait();
    __syncthreads();  // k~ tile kb + 1 and v tile kb are in; k~ tile kb and v tile kb - 1 are done with
    if (kb + 2 < nkb) issue_k(kb + 2);
    if (kb + 1 < nkb) issue_v(kb + 1);
    if (kb >= nvis) continue;
    rs = 0.f;
    if (STAG && kb + 1 < nvis) {
      scores(kb + 1, sp, std::true_type{});
    } else {
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        const float p = fast_exp2(sp[j] - m);
        sp[j] = p;
        rs += p;
      }
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) split_frag(sp, ks * 8, pf[ks]);
    }
    l += rs;
    int vslot = 2 * KT + (kb & 1) * VT;
    asm volatile("" : "+s"(vslot));
    const char* sV = smem + vslot;
    {
      constexpr int NF = NOT * 2;  // O^T += v^T P^T: key step i / NOT of column tile i % NOT
      u32x4 vq[2][3];
#pragma unroll
      for (int p = 0; p < 3; ++p) vq[0][p] = cv.read(sV + p * SV_PL, 0, 0);
#pragma unroll
      for (int i = 0; i < NF; ++i) {
        __builtin_amdgcn_sched_barrier(0);
        if (i + 1 < NF) {
#pragma unroll
          for (int p = 0; p < 3; ++p)
            vq[(i + 1) & 1][p] = cv.read(sV + p * SV_PL, ((i + 1) / NOT) * 16, ((i + 1) % NOT) * 32);
        }
        __builtin_amdgcn_sched_barrier(0);
        mma6(vq[i & 1], pf[i / NOT], o[i % NOT], oc[i % NOT]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if (!STAG && kb + 1 < nvis) scores(kb + 1, sp, std::false_type{});
  }

  if constexpr (OC) {
#pragma unroll
    for (int t = 0; t < NOT; ++t) o[t] += oc[t];
  }
  const float lt = l + xor32(l);
  const float inv = lt > 0.f ? 1.f / lt : 0.f;
  __syncthreads();
#pragma unroll
  for (int t = 0; t < NOT; ++t)
#pragma unroll
    for (int j = 0; j < 16; ++j)
      *(float*)(smem + (w * 32 + l32) * SO_STRIDE + (t * 32 + c_row(j, g)) * 4) = o[t][j] * inv;
  if (g == 0 && myq < a.Sq)
    a.lse[(int64_t)(b * a.Hq + h) * a.Sq + myq] = lt > 0.f ? (m + log2f(lt)) * LN2 : -INFINITY;
  __syncthreads();
  float* obase = (float*)a.o + b * a.o_sb + h * a.o_sh;
  if (o_vec) {
    constexpr int CPR = DV / 4;
    for (int q = tid; q < BM * CPR; q += 256) {
      const int row = q / CPR, c = q % CPR;
      if (q0 + row < a.Sq)
        *(u32x4*)(obase + (int64_t)(q0 + row) * a.o_ss + c * 4) = *(const u32x4*)(smem + row * SO_STRIDE + c * 16);
    }
  } else {
    const int dvr = a.dv_real;
    for (int q = tid; q < BM * dvr; q += 256) {
      const int row = q / dvr, c = q % dvr;
      if (q0 + row < a.Sq) obase[(int64_t)(q0 + row) * a.o_ss + c] = *(const float*)(smem + row * SO_STRIDE + c * 4);
    }
  }
}

// The backward, the closed form of pe_bwd.hip's head with every product formed
// from planes.  P is recomputed in natural units, exp(fma(s, scale, -lse)), as the fp32 unit's kernels do.
// One launch holds both halves: query blocks (dq~) first, then key blocks (dk~, dv), whose work differs
// by a factor of up to Sq / 128 under the causal mask; the two share no data, and together they fill the
// chip where either alone leaves it half empty (4 x 8 -> 4 heads, 1024 rows: 256 query blocks, 128 key
// blocks).  Key blocks are further shared out over `qsplit` workgroups, each taking a range of the block's
// (query head, query tile) list and leaving fp32 partials for split_sum_kernel.  Both walk 32-row tiles
// with the operands of their own 32 rows per wave in registers (one wave per SIMD, 512 registers) and run
// the exponentials and the split of P beside the products of dP.  At QK width 256 the registers do not hold
// it all (158 spilled at V width 128): 8 heads of 128, 4096 rows, forward and backward, still take 2.79 ms
// against 7.24 on the fp32 unit.
constexpr int SPLIT_NW = 4;

// acc += sum over the two 16-deep steps of a tile, corrections and leading products in accumulators of the
// tile's own, added by the vector unit.  The matrix core does not round a product that is added to a larger
// accumulator to nearest but to one side: corrections first and leading products on top of them left a bias
// in dk~ that the phase bias's gradient, a sum over all keys, shows (2.4e-6 of its size against 4e-7 to
// 8e-7 on the fp32 unit; 4e-7 to 7e-7 this way), and chained on the running sum they took dV's error at
// 2048 rows 3 % past the fp32 unit's.
template <typename F>
__device__ __forceinline__ void tile_products(f32x16& acc, const u32x4 (&af)[2][3], F&& bfrag) {
  using M = MT<0>;
  f32x16 c = {};
  u32x4 b0[3], b1[3];
  bfrag(0, b0);
  bfrag(1, b1);
  c = M::mma(af[0][2], b0[0], c);
  c = M::mma(af[0][0], b0[2], c);
  c = M::mma(af[0][1], b0[1], c);
  c = M::mma(af[0][1], b0[0], c);
  c = M::mma(af[0][0], b0[1], c);
  c = M::mma(af[1][2], b1[0], c);
  c = M::mma(af[1][0], b1[2], c);
  c = M::mma(af[1][1], b1[1], c);
  c = M::mma(af[1][1], b1[0], c);
  c = M::mma(af[1][0], b1[1], c);
  f32x16 d = {};
  d = M::mma(af[0][0], b0[0], d);
  d = M::mma(af[1][0], b1[0], d);
#pragma unroll
  for (int j = 0; j < 16; ++j) acc[j] += c[j] + d[j];
}

template <int DQK, int DV>
__device__ __forceinline__ void dkdv_split_body(const CoreArgs& a, int bid, char* smem) {
  constexpr int BQ = 32, BNK = SPLIT_NW * 32;
  constexpr int NCQ = DQK / 8, NCO = DV / 8, NKF = DQK / 16, NVF = DV / 16, NDK = DQK / 32, NDV = DV / 32;
  constexpr int SQ_PL = BQ * NCQ * 16, SO_PL = BQ * NCO * 16, STAGE = 3 * (SQ_PL + SO_PL) + 2 * BQ * 4;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, g = lane >> 5, l32 = lane & 31;
  const int nkb = (a.Sk + BNK - 1) / BNK, nblk = nkb * a.nbh;
  const int jq = bid / nblk;
  int kb, bh;
  map_block(bid - jq * nblk, nkb, a.nbh, false, kb, bh);
  const int b = bh / a.Hkv, hk = bh % a.Hkv, grp = a.Hq / a.Hkv;
  const int k0 = kb * BNK, kw0 = k0 + w * 32, myk = kw0 + l32;
  const int off = a.causal_off;
  const int64_t qrs = 3 * DQK * 2, ors = 3 * DV * 2;

  u32x4 kf[NKF][3], vf[NVF][3];
  {
    const int64_t kr = (int64_t)(b * a.Hkv + hk) * a.Sk + (myk < a.Sk ? myk : a.Sk - 1);
    const uint16_t* krow = (const uint16_t*)a.k + kr * 3 * DQK;
    const uint16_t* vrow = (const uint16_t*)a.v + kr * 3 * DV;
#pragma unroll
    for (int kk = 0; kk < NKF; ++kk)
#pragma unroll
      for (int p = 0; p < 3; ++p) kf[kk][p] = *(const u32x4*)(krow + p * DQK + kk * 16 + g * 8);
#pragma unroll
    for (int kk = 0; kk < NVF; ++kk)
#pragma unroll
      for (int p = 0; p < 3; ++p) vf[kk][p] = *(const u32x4*)(vrow + p * DV + kk * 16 + g * 8);
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): seen by the compiler
  }
  f32x16 dk[NDK], dv[NDV];
#pragma unroll
  for (int t = 0; t < NDK; ++t)
#pragma unroll
    for (int j = 0; j < 16; ++j) dk[t][j] = 0.f;
#pragma unroll
  for (int t = 0; t < NDV; ++t)
#pragma unroll
    for (int j = 0; j < 16; ++j) dv[t][j] = 0.f;

  const int nqt = (a.Sq + BQ - 1) / BQ;
  int qb0 = 0;
  if (a.causal) qb0 = max(0, k0 - off) / BQ;
  if (qb0 > nqt) qb0 = nqt;
  const int nper = nqt - qb0, ntot = nper * grp;
  const int it0 = (int)((int64_t)ntot * jq / a.qsplit), it1 = (int)((int64_t)ntot * (jq + 1) / a.qsplit);

  const DmaPlan<BQ, NCQ, SPLIT_NW, 1> plan_q(w, lane, (uint32_t)qrs);
  const DmaPlan<BQ, NCO, SPLIT_NW, 1> plan_o(w, lane, (uint32_t)ors);
  const uint32_t smem_l = lds_addr(smem);
  auto issue = [&](int it) {
    const int h = hk * grp + it / nper, q0 = (qb0 + it % nper) * BQ, slot = (it & 1) * STAGE;
    const int64_t r0 = (int64_t)(b * a.Hq + h) * a.Sq + q0;
    const char* qsrc = (const char*)a.q + r0 * qrs;
    const char* osrc = (const char*)a.dO + r0 * ors;
    const uint32_t sl = smem_l + (uint32_t)slot;
    if (a.Sq - q0 >= BQ) {
#pragma unroll
      for (int p = 0; p < 3; ++p) {
        plan_q.full(qsrc + p * DQK * 2, sl + p * SQ_PL, w, (uint32_t)qrs);
        plan_o.full(osrc + p * DV * 2, sl + 3 * SQ_PL + p * SO_PL, w, (uint32_t)ors);
      }
    } else {
      int ln = lane;
      asm volatile("" : "+v"(ln));
#pragma unroll
      for (int p = 0; p < 3; ++p) {
        dma_tile<BQ, NCQ, SPLIT_NW, 1>(smem + slot + p * SQ_PL, qsrc + p * DQK * 2, qrs, a.Sq - q0, w, ln);
        dma_tile<BQ, NCO, SPLIT_NW, 1>(smem + slot + 3 * SQ_PL + p * SO_PL, osrc + p * DV * 2, ors, a.Sq - q0, w, ln);
      }
    }
    // the rows' lse (natural units, +inf on padding rows: P = 0) and Di
    const int64_t p0 = (int64_t)(b * a.Hq + h) * a.sq_pad + q0;
    if (w == 0 && lane < 16) dma16((lane < 8 ? a.L2 : a.Di) + p0 + (lane & 7) * 4, sl + 3 * (SQ_PL + SO_PL));
  };
  const RowFrags<NCQ, 1> rq(perm_row<0>(l32), g);
  const RowFrags<NCO, 1> ro(perm_row<0>(l32), g);
  const ColFrags<NCQ, 1> cq(lane);
  const ColFrags<NCO, 1> co(lane);

  if (it0 < it1) issue(it0);
  for (int it = it0; it < it1; ++it) {
    const int q0 = (qb0 + it % nper) * BQ;
    int slot = (it & 1) * STAGE;
    asm volatile("" : "+s"(slot));
    const char* sQ = smem + slot;
    const char* sO = sQ + 3 * SQ_PL;
    const float* sL = (const float*)(sO + 3 * SO_PL);
    const float* sD = sL + BQ;
    dma_wait();
    __syncthreads();  // tile `it` is in, and every wave has left the slot of tile it - 1
    if (it + 1 < it1) issue(it + 1);
    if (a.causal && kw0 > q0 + BQ - 1 + off) continue;  // every key of this wave is after every query

    f32x16 s, dp;
    {
      f32x16 c0 = {}, c1 = {};
      u32x4 fr[2][3];
#pragma unroll
      for (int p = 0; p < 3; ++p) fr[0][p] = rq.read(sQ + p * SQ_PL, 0, 0);
#pragma unroll
      for (int kk = 0; kk < NKF; ++kk) {
        __builtin_amdgcn_sched_barrier(0);
        if (kk + 1 < NKF) {
#pragma unroll
          for (int p = 0; p < 3; ++p) fr[(kk + 1) & 1][p] = rq.read(sQ + p * SQ_PL, 0, kk + 1);
        }
        mma6(fr[kk & 1], kf[kk], c0, c1);
      }
      __builtin_amdgcn_sched_barrier(0);
      s = c0 + c1;
    }
    u32x4 pf[2][3], df[2][3];
    // dP, and beside its products P and its planes; EDGE: some key of the wave lies after some query
    auto dp_and_p = [&](auto edge_tag) {
      constexpr bool EDGE = decltype(edge_tag)::value;
      constexpr int EPS = 16 / NVF;
      const int kd = myk - off - q0 - g * 8;
      f32x16 c0 = {}, c1 = {};
      u32x4 fr[2][3];
#pragma unroll
      for (int p = 0; p < 3; ++p) fr[0][p] = ro.read(sO + p * SO_PL, 0, 0);
      f32x4 lg[4];
#pragma unroll
      for (int G = 0; G < 4; ++G) lg[G] = *(const f32x4*)(sL + (G >> 1) * 16 + g * 8 + (G & 1) * 4);
#pragma unroll
      for (int kk = 0; kk < NVF; ++kk) {
        __builtin_amdgcn_sched_barrier(0);
        if (kk + 1 < NVF) {
#pragma unroll
          for (int p = 0; p < 3; ++p) fr[(kk + 1) & 1][p] = ro.read(sO + p * SO_PL, 0, kk + 1);
        }
        mma6(fr[kk & 1], vf[kk], c0, c1);
#pragma unroll
        for (int e = 0; e < EPS; ++e) {
          const int j = kk * EPS + e;
          float x = __builtin_fmaf(s[j], a.scale, -lg[j / 4][j % 4]) * LOG2E;
          if (EDGE) x = kd > ((j >> 3) << 4) + (j & 7) ? -INFINITY : x;
          s[j] = fast_exp2(x);
          if (j & 1) {
            uint32_t h, mm, ll;
            split_bf3(s[j - 1], s[j], h, mm, ll);
            pf[j / 8][0][(j % 8) / 2] = h;
            pf[j / 8][1][(j % 8) / 2] = mm;
            pf[j / 8][2][(j % 8) / 2] = ll;
          }
        }
#pragma unroll
        for (int i = 0; i < 6; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x402, 2 * EPS, 0);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      dp = c0 + c1;
    };
    if (__builtin_amdgcn_readfirstlane(a.causal && kw0 + 31 > q0 + off)) dp_and_p(std::true_type{});
    else dp_and_p(std::false_type{});
    {
      f32x4 dg[4];
#pragma unroll
      for (int G = 0; G < 4; ++G) dg[G] = *(const f32x4*)(sD + (G >> 1) * 16 + g * 8 + (G & 1) * 4);
#pragma unroll
      for (int j = 0; j < 16; ++j) dp[j] = s[j] * (dp[j] - dg[j / 4][j % 4]);
    }
    // dV, with the split of dS free to run beside it
#pragma unroll
    for (int t = 0; t < NDV; ++t)
      tile_products(dv[t], pf, [&](int ks, u32x4 (&f)[3]) {
#pragma unroll
        for (int p = 0; p < 3; ++p) f[p] = co.read(sO + p * SO_PL, ks * 16, t * 32);
      });
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) split_frag(dp, ks * 8, df[ks]);
#pragma unroll
    for (int t = 0; t < NDK; ++t)
      tile_products(dk[t], df, [&](int ks, u32x4 (&f)[3]) {
#pragma unroll
        for (int p = 0; p < 3; ++p) f[p] = cq.read(sQ + p * SQ_PL, ks * 16, t * 32);
      });
  }

  const int64_t units = (int64_t)a.B * a.Hkv;
  float* dkb = a.dk_t + ((int64_t)jq * units + bh) * a.Sk * DQK;
#pragma unroll
  for (int t = 0; t < NDK; ++t)
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const int key = kw0 + c_row(j, g);
      if (key < a.Sk) dkb[(int64_t)key * DQK + t * 32 + l32] = dk[t][j] * a.scale;
    }
  if (a.qsplit > 1) {
    float* dvp = a.dv_part + ((int64_t)jq * units + bh) * a.Sk * DV;
#pragma unroll
    for (int t = 0; t < NDV; ++t)
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        const int key = kw0 + c_row(j, g);
        if (key < a.Sk) dvp[(int64_t)key * DV + t * 32 + l32] = dv[t][j];
      }
  } else {
#pragma unroll
    for (int t = 0; t < NDV; ++t)
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        const int key = kw0 + c_row(j, g), col = t * 32 + l32;
        if (key < a.Sk && col < a.dv_real)
          store_from_float(a.dv, b * a.dv_sb + hk * a.dv_sh + (int64_t)key * a.dv_ss + col, a.dv_dtype, dv[t][j]);
      }
  }
}

template <int DQK, int DV>
__device__ __forceinline__ void dq_split_body(const CoreArgs& a, int bid, char* smem) {
  constexpr int BM = SPLIT_NW * 32, BN = 32;
  constexpr int NCK = DQK / 8, NCV = DV / 8, NQF = DQK / 16, NVF = DV / 16, NDQ = DQK / 32;
  constexpr int SK_PL = BN * NCK * 16, SV_PL = BN * NCV * 16, STAGE = 3 * (SK_PL + SV_PL);
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, g = lane >> 5, l32 = lane & 31;
  const int nqb = (a.Sq + BM - 1) / BM;
  int qb, bh;
  map_block(bid, nqb, a.B * a.Hq, a.causal != 0, qb, bh);
  const int b = bh / a.Hq, h = bh % a.Hq, hk = h / (a.Hq / a.Hkv);
  const int q0 = qb * BM, qw = q0 + w * 32, myq = qw + l32;
  const int off = a.causal_off;
  const int64_t krs = 3 * DQK * 2, vrs = 3 * DV * 2;
  const int64_t rowq = (int64_t)(b * a.Hq + h) * a.Sq + (myq < a.Sq ? myq : a.Sq - 1);

  u32x4 qf[NQF][3], of[NVF][3];
  {
    const uint16_t* qrow = (const uint16_t*)a.q + rowq * 3 * DQK;
    const uint16_t* orow = (const uint16_t*)a.dO + rowq * 3 * DV;
#pragma unroll
    for (int kk = 0; kk < NQF; ++kk)
#pragma unroll
      for (int p = 0; p < 3; ++p) qf[kk][p] = *(const u32x4*)(qrow + p * DQK + kk * 16 + g * 8);
#pragma unroll
    for (int kk = 0; kk < NVF; ++kk)
#pragma unroll
      for (int p = 0; p < 3; ++p) of[kk][p] = *(const u32x4*)(orow + p * DV + kk * 16 + g * 8);
  }
  const int64_t prow = (int64_t)(b * a.Hq + h) * a.sq_pad + myq;  // sq_pad is a multiple of 128
  const float lse = a.L2[prow], Dq = a.Di[prow];
  __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): seen by the compiler
  f32x16 dq[NDQ];
#pragma unroll
  for (int t = 0; t < NDQ; ++t)
#pragma unroll
    for (int j = 0; j < 16; ++j) dq[t][j] = 0.f;

  int kend = a.Sk;
  if (a.causal) kend = min(a.Sk, q0 + BM + off);
  const int nkb = kend > 0 ? (kend + BN - 1) / BN : 0;
  const char* kbase = (const char*)a.k + (int64_t)(b * a.Hkv + hk) * a.Sk * krs;
  const char* vbase = (const char*)a.v + (int64_t)(b * a.Hkv + hk) * a.Sk * vrs;
  const DmaPlan<BN, NCK, SPLIT_NW, 1> plan_k(w, lane, (uint32_t)krs);
  const DmaPlan<BN, NCV, SPLIT_NW, 0> plan_v(w, lane, (uint32_t)vrs);
  const uint32_t smem_l = lds_addr(smem);
  auto issue = [&](int kb) {
    const int k0 = kb * BN, slot = (kb & 1) * STAGE;
    const char* ksrc = kbase + (int64_t)k0 * krs;
    const char* vsrc = vbase + (int64_t)k0 * vrs;
    const uint32_t sl = smem_l + (uint32_t)slot;
    if (a.Sk - k0 >= BN) {
#pragma unroll
      for (int p = 0; p < 3; ++p) {
        plan_k.full(ksrc + p * DQK * 2, sl + p * SK_PL, w, (uint32_t)krs);
        plan_v.full(vsrc + p * DV * 2, sl + 3 * SK_PL + p * SV_PL, w, (uint32_t)vrs);
      }
    } else {
      int ln = lane;
      asm volatile("" : "+v"(ln));
#pragma unroll
      for (int p = 0; p < 3; ++p) {
        dma_tile<BN, NCK, SPLIT_NW, 1>(smem + slot + p * SK_PL, ksrc + p * DQK * 2, krs, a.Sk - k0, w, ln);
        dma_tile<BN, NCV, SPLIT_NW, 0>(smem + slot + 3 * SK_PL + p * SV_PL, vsrc + p * DV * 2, vrs, a.Sk - k0, w, ln);
      }
    }
  };
  const RowFrags<NCK, 1> rk(perm_row<0>(l32), g);
  const RowFrags<NCV, 0> rv(perm_row<0>(l32), g);
  const ColFrags<NCK, 1> ck(lane);

  if (nkb > 0) issue(0);
  for (int kb = 0; kb < nkb; ++kb) {
    const int k0 = kb * BN;
    int slot = (kb & 1) * STAGE;
    asm volatile("" : "+s"(slot));
    const char* sK = smem + slot;
    const char* sV = sK + 3 * SK_PL;
    dma_wait();
    __syncthreads();
    if (kb + 1 < nkb) issue(kb + 1);
    if (a.causal && k0 > qw + 31 + off) continue;
    const bool edge = (a.causal && k0 + BN - 1 > qw + off) || (k0 + BN > a.Sk);

    f32x16 s, dp;
    {
      f32x16 c0 = {}, c1 = {};
      u32x4 fr[2][3];
#pragma unroll
      for (int p = 0; p < 3; ++p) fr[0][p] = rk.read(sK + p * SK_PL, 0, 0);
#pragma unroll
      for (int kk = 0; kk < NQF; ++kk) {
        __builtin_amdgcn_sched_barrier(0);
        if (kk + 1 < NQF) {
#pragma unroll
          for (int p = 0; p < 3; ++p) fr[(kk + 1) & 1][p] = rk.read(sK + p * SK_PL, 0, kk + 1);
        }
        mma6(fr[kk & 1], qf[kk], c0, c1);
      }
      __builtin_amdgcn_sched_barrier(0);
      s = c0 + c1;
    }
    auto dp_and_p = [&](auto edge_tag) {
      constexpr bool EDGE = decltype(edge_tag)::value;
      constexpr int EPS = 16 / NVF;
      f32x16 c0 = {}, c1 = {};
      u32x4 fr[2][3];
#pragma unroll
      for (int p = 0; p < 3; ++p) fr[0][p] = rv.read(sV + p * SV_PL, 0, 0);
#pragma unroll
      for (int kk = 0; kk < NVF; ++kk) {
        __builtin_amdgcn_sched_barrier(0);
        if (kk + 1 < NVF) {
#pragma unroll
          for (int p = 0; p < 3; ++p) fr[(kk + 1) & 1][p] = rv.read(sV + p * SV_PL, 0, kk + 1);
        }
        mma6(fr[kk & 1], of[kk], c0, c1);
#pragma unroll
        for (int e = 0; e < EPS; ++e) {
          const int j = kk * EPS + e;
          float x = __builtin_fmaf(s[j], a.scale, -lse) * LOG2E;
          if (EDGE) {
            const int key = k0 + c_logical<0>(j, g);
            if (key >= a.Sk || (a.causal && key > myq + off)) x = -INFINITY;
          }
          s[j] = fast_exp2(x);
        }
#pragma unroll
        for (int i = 0; i < 6; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x402, EPS, 0);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      dp = c0 + c1;
    };
    if (__builtin_amdgcn_readfirstlane(edge)) dp_and_p(std::true_type{});
    else dp_and_p(std::false_type{});
#pragma unroll
    for (int j = 0; j < 16; ++j) dp[j] = s[j] * (dp[j] - Dq);
    u32x4 df[2][3];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) split_frag(dp, ks * 8, df[ks]);
#pragma unroll
    for (int t = 0; t < NDQ; ++t)
      tile_products(dq[t], df, [&](int ks, u32x4 (&f)[3]) {
#pragma unroll
        for (int p = 0; p < 3; ++p) f[p] = ck.read(sK + p * SK_PL, ks * 16, t * 32);
      });
  }

  float* dqb = a.dq_t + (int64_t)(b * a.Hq + h) * a.Sq * DQK;
#pragma unroll
  for (int t = 0; t < NDQ; ++t)
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const int q = qw + c_row(j, g);
      if (q < a.Sq) dqb[(int64_t)q * DQK + t * 32 + l32] = dq[t][j] * a.scale;
    }
}

template <int DQK, int DV>
__global__ __launch_bounds__(SPLIT_NW * 64, 1) void bwd_split_kernel(CoreArgs a, int ndq) {
  constexpr int TILE = 3 * 32 * (DQK + DV) * 2;
  __shared__ __attribute__((aligned(1024))) char smem[2 * (TILE + 2 * 32 * 4)];
  if ((int)blockIdx.x < ndq) dq_split_body<DQK, DV>(a, blockIdx.x, smem);
  else dkdv_split_body<DQK, DV>(a, blockIdx.x - ndq, smem);
}

// The qsplit partials of dk~ (left in slice 0 for the inverse transform) and dV (to its view) added in
// slice order, four columns a thread.
template <int DQK, int DV> __global__ __launch_bounds__(256) void split_sum_kernel(CoreArgs a) {
  constexpr int CPR = (DQK + DV) / 4;
  const int64_t gid = (int64_t)blockIdx.x * 256 + threadIdx.x, row = gid / CPR;
  const int c = (int)(gid % CPR) * 4;
  const int64_t rows = (int64_t)a.B * a.Hkv * a.Sk;
  if (row >= rows) return;
  if (c < DQK) {
    float* d0 = a.dk_t + row * DQK + c;
    f32x4 x = *(const f32x4*)d0;
    for (int j = 1; j < a.qsplit; ++j) x += *(const f32x4*)(d0 + j * rows * DQK);
    *(f32x4*)d0 = x;
  } else {
    const int cv = c - DQK;
    const float* d0 = a.dv_part + row * DV + cv;
    f32x4 x = *(const f32x4*)d0;
    for (int j = 1; j < a.qsplit; ++j) x += *(const f32x4*)(d0 + j * rows * DV);
    const int key = (int)(row % a.Sk), bh = (int)(row / a.Sk);
    const int64_t o = (bh / a.Hkv) * a.dv_sb + (bh % a.Hkv) * a.dv_sh + (int64_t)key * a.dv_ss + cv;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (cv + e < a.dv_real) store_from_float(a.dv, o + e, a.dv_dtype, x[e]);
  }
}

// Measured against the fp32 unit's two kernels, forward and backward: 4 x 8 -> 4 heads of the split form, 1024
// rows, 882 -> 320 us; 2 x 8 heads of 64, 2048 rows, 1214 -> 588 us; 8 heads of 128, 4096 rows, 7.24 -> 2.79
// ms.  dq / dk / dv errors against float64 are 0.6 to 0.9 of the fp32 unit's.
template <int DQK, int DV>
static int run_bwd_split(const CoreArgs& a, hipStream_t s) {
  const int64_t ndq = (int64_t)((a.Sq + 127) / 128) * a.B * a.Hq;
  const int64_t ndk = (int64_t)((a.Sk + 127) / 128) * a.nbh * a.qsplit;
  if (ndq + ndk > 0x7fffffff) return -2;
  hipLaunchKernelGGL((bwd_split_kernel<DQK, DV>), dim3((unsigned)(ndq + ndk)), dim3(SPLIT_NW * 64), 0, s, a, (int)ndq);
  if (a.qsplit > 1) {
    const int64_t nthr = (int64_t)a.B * a.Hkv * a.Sk * ((DQK + DV) / 4);
    hipLaunchKernelGGL((split_sum_kernel<DQK, DV>), dim3((unsigned)((nthr + 255) / 256)), dim3(256), 0, s, a);
  }
  return hipGetLastError() == hipSuccess ? 0 : -7;
}

int launch_bwd_split(int dqk, int dv, const CoreArgs& a, hipStream_t s) {
  if (dqk == 64 && dv == 64) return run_bwd_split<64, 64>(a, s);
  if (dqk == 64 && dv == 128) return run_bwd_split<64, 128>(a, s);
  if (dqk == 128 && dv == 64) return run_bwd_split<128, 64>(a, s);
  if (dqk == 128 && dv == 128) return run_bwd_split<128, 128>(a, s);
  if (dqk == 256 && dv == 64) return run_bwd_split<256, 64>(a, s);
  if (dqk == 256 && dv == 128) return run_bwd_split<256, 128>(a, s);
  return -3;
}

// Measured against the fp32 matrix unit's kernel: 16 heads of 128, 16384 rows, 15.41 -> 9.32 ms (the six
// products alone, at the rate a large bf16 product reaches here, 8.2 ms); 8 heads of 64, 2 x 2048 rows, 305 ->
// 186 us; 4 -> 2 heads of the split form, 333 rows, 65 -> 51 us.  Error of the output against float64 at
// these shapes 8.0e-7 -> 6.8e-7, 3.5e-7 -> 2.7e-7 and 2.0e-7 -> 1.4e-7.
template <int DQK, int DV>
static int run_fwd_split(const CoreArgs& a, hipStream_t s) {
  // two workgroups a CU where the q~ planes leave room for them in the registers
  constexpr int OCC = DQK <= 128 && DV == 64 ? 2 : 1;
  const int grid = (a.Sq + 127) / 128 * a.B * a.Hq;
  const int o_vec = a.dv_real == DV && (uintptr_t)a.o % 16 == 0 && a.o_ss % 4 == 0 && a.o_sh % 4 == 0 && a.o_sb % 4 == 0;
  hipLaunchKernelGGL((fwd_split_kernel<DQK, DV, OCC>), dim3(grid), dim3(256), 0, s, a, o_vec);
  return hipGetLastError() == hipSuccess ? 0 : -7;
}

int launch_fwd_split(int dqk, int dv, const CoreArgs& a, hipStream_t s) {
  if (dqk == 64 && dv == 64) return run_fwd_split<64, 64>(a, s);
  if (dqk == 64 && dv == 128) return run_fwd_split<64, 128>(a, s);
  if (dqk == 128 && dv == 64) return run_fwd_split<128, 64>(a, s);
  if (dqk == 128 && dv == 128) return run_fwd_split<128, 128>(a, s);
  if (dqk == 256 && dv == 64) return run_fwd_split<256, 64>(a, s);
  if (dqk == 256 && dv == 128) return run_fwd_split<256, 128>(a, s);
  return -3;
}

}  // namespace pe

// Decode attention over long caches, split over the keys: four launches in place of the one
// block per (row, head) of k_attention_qkv. Same arithmetic (the q/k/v epilogue, RoPE, qrow, scores, softmax and p.V of
// exact_llm.py:164-176), same outputs and cache contents.
//
// The softmax needs the row's maximum before any exponent and the sum of exponents before any p (both integer
// roundings), so a row cannot be folded chunk by chunk; the launch boundaries are these synchronisations. A block of each
// launch takes 128 keys of one (row, KV head) for all the query heads of the group, so a group reads its keys and values
// once:
//   k_dec_scores  the query heads from the totals, the chunk's scores and their maximum; the chunk that holds the new
//                 position also writes its key and value
//   k_dec_exp     exponentials and their sum
//   k_dec_pv      p and p.V of the chunk, added to the totals
//   k_dec_out     the outputs and their bit lengths
// Together, in a graph: one row of 6002 positions, 28 heads over 4 KV heads, 182 -> 21.4 us (31 MB of keys and values: 6.2 us
// at the card's copy rate of 4.96 TB/s); 8 rows of 1240 to 1793 positions 112 us in two launches -> 31.8.
// The grids cover the cache, as a captured launch serves every position: blocks past a row's position leave at once, which at 8 rows
// of 8 KV heads costs 36 us in a cache of 8192 positions (4096 blocks a launch), so the caller's line counts them.
#include "exact_common.h"
#include "abi_util.h"

namespace exact {

#define DEC_CK 128        // keys a block: 16 a wave in k_dec_scores, 32 in k_dec_pv
#define DEC_A_THREADS 512
#define DEC_C_THREADS 256
#define DEC_SMAX 8192
#define DEC_NCH (DEC_SMAX / DEC_CK)   // chunks of the longest cache: one a lane

// grid (ceil(Smax / DEC_CK), KV, R). sc[(r H + h) Sp + key]: the scores of the keys 0 .. pos[r]. Blocks of chunks past the
// position leave at once. q.k on the matrix cores from int8 digits x = 256 hi + lo + 128 (every digit sum is below 2^22):
//   q.k = 65536 HH + 256 (HL + LH) + LL + 128 (sum q + sum k) - 16384 HD
// A wave takes 16 keys as the rows of v_mfma_i32_16x16x64_i8; columns 0 .. 7 are the heads' high digits and 8 .. 15 their
// low ones, so four products give a head all its digit sums, and four more against all-ones columns the keys' sums. Dot
// products of int16 pairs, widened to int64 each, kept the vector units busy instead: 8 rows of 1240 to 1793 positions, 28
// heads over 4 KV heads, 13.8 -> 11.2 us a launch; one row of 6002 8.9 -> 7.8, of 17 6.1 -> 5.0 (its chain of dependent
// steps: position, totals, RoPE, scores).
template <int HB, int HD>
__global__ __launch_bounds__(DEC_A_THREADS) void k_dec_scores(
    const int64_t* __restrict__ t, const int32_t* __restrict__ s, const int64_t* __restrict__ b,
    const int64_t* __restrict__ cos_t, const int64_t* __restrict__ sin_t, const int32_t* __restrict__ slot,
    const int32_t* __restrict__ pos, int16_t* __restrict__ kq, int32_t* __restrict__ sk, int64_t* __restrict__ v,
    int64_t* __restrict__ sc, int64_t* __restrict__ cm, int H, int KV, int Smax, int Sp, int INV) {
  constexpr int NT = DEC_A_THREADS, NW = NT / 64, KS = HD / 64;
  static_assert(HB <= 8 && DEC_CK == 16 * NW, "16 keys a wave, at most 8 heads");
  __shared__ int64_t y[HB + 2][HD];   // the group's query heads, the new key, the new value: shr(t, 28 - s) + b
  __shared__ __attribute__((aligned(16))) int8_t qd[2][HB][HD];   // the query heads' digits
  __shared__ int16_t qs[HB + 1][HD];  // quantised query heads and new key, for the new position's own scores
  __shared__ int shq[HB + 1], qsum[HB];
  __shared__ int64_t wm[NW + 1][8];   // the waves' maximum scores a head, then the new position's score
  const int c = blockIdx.x, kh = blockIdx.y, r = blockIdx.z, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int p = pos[r], sl = slot[r], k0 = c * DEC_CK;
  const int N = (H + 2 * KV) * HD, h0 = kh * HB;
  if (p < 0 || p >= Smax || k0 > p) return;   // uniform over the block
  const bool fresh = k0 + DEC_CK > p;         // this chunk holds the new position
  const int64_t cbase = ((int64_t)sl * KV + kh) * Smax;
  // loads that do not depend on the query first: lane holds dims 64 i + 16 (lane / 16) + [0, 16) of key lane % 16
  const int col = lane & 15, kw = k0 + 16 * wave, qt = lane >> 4;
  v4i kk[KS][2];
  {
    const int sj = kw + col < p ? kw + col : k0;   // past the cached keys: any key of the cache
    const v4i* kr = reinterpret_cast<const v4i*>(kq + (cbase + sj) * HD + 16 * qt);
#pragma unroll
    for (int i = 0; i < KS; ++i) {
      kk[i][0] = kr[8 * i];
      kk[i][1] = kr[8 * i + 1];
    }
  }
  int skv[4];   // the shifts of the keys of the lane's product rows
#pragma unroll
  for (int i = 0; i < 4; ++i) skv[i] = sk[cbase + (kw + 4 * qt + i < p ? kw + 4 * qt + i : k0)];
  int64_t cs[KS][2];   // the RoPE row
#pragma unroll
  for (int i = 0; i < KS; ++i) {
    cs[i][0] = cos_t[(int64_t)p * HD + lane + 64 * i];
    cs[i][1] = sin_t[(int64_t)p * HD + lane + 64 * i];
  }
  const int nh = fresh ? HB + 2 : HB, sh = 28 - s[r];
  for (int j = tid; j < nh * HD; j += NT) {
    const int w = j / HD, jj = j - w * HD;
    const int base = (w < HB ? h0 + w : (w == HB ? H + kh : H + KV + kh)) * HD + jj;
    const int64_t val = shr64(t[(int64_t)r * N + base], sh);
    y[w][jj] = b ? val + b[base] : val;
  }
  __syncthreads();
  const int nq = fresh ? HB + 1 : HB;
  for (int w = wave; w < nq; w += NW) {   // RoPE and qrow of a head, one wave each (k_qkv_rope_cache's steps)
    int64_t z[KS], m = 0;
#pragma unroll
    for (int i = 0; i < KS; ++i) {
      const int j = lane + 64 * i;
      const int64_t rot = j < HD / 2 ? -y[w][j + HD / 2] : y[w][j - HD / 2];
      z[i] = shr64(y[w][j] * cs[i][0] + rot * cs[i][1], EXACT_F);
      const int64_t a = abs64(z[i]);
      m = a > m ? a : m;
    }
    m = wave_max64(m);
    int q = bitlen64(m) - 15;
    if (q < 0) q = 0;
    int64_t sum = 0;
#pragma unroll
    for (int i = 0; i < KS; ++i) {
      const int64_t x = shr64(z[i], q);
      const int xc = (int)(x > 32767 ? 32767 : (x < -32767 ? -32767 : x));
      qs[w][lane + 64 * i] = (int16_t)xc;
      if (w < HB) {
        qd[0][w][lane + 64 * i] = (int8_t)(xc >> 8);
        qd[1][w][lane + 64 * i] = (int8_t)((xc & 255) - 128);
      }
      sum += xc;
    }
    sum = wave_sum64(sum);
    if (lane == 0) {
      shq[w] = q;
      if (w < HB) qsum[w] = (int)sum;
    }
  }
  __syncthreads();
  int64_t* scr = sc + ((int64_t)r * H + h0) * Sp;
  if (fresh) {   // the new position: into the cache, and its scores against the query heads
    for (int j = tid; j < HD; j += NT) {
      kq[(cbase + p) * HD + j] = qs[HB][j];
      v[(cbase + p) * HD + j] = y[HB + 1][j];
    }
    if (tid == 0) sk[cbase + p] = shq[HB];
    for (int w = wave; w < HB; w += NW) {
      int64_t ps = 0;
      for (int j = lane; j < HD; j += 64) ps += (int64_t)((int)qs[w][j] * (int)qs[HB][j]);
      const int64_t dot = wave_sum64(ps);
      if (lane == 0) {
        const int64_t val = shr64(dot * INV, 32 - shq[w] - shq[HB]);
        scr[(int64_t)w * Sp + p] = val;
        wm[NW][w] = val;
      }
    }
  }
  const int hb = (col & 7) < HB ? (col & 7) : HB - 1;
  const v4i ones = {0x01010101, 0x01010101, 0x01010101, 0x01010101};
  v4i ch = v4i{}, cl = v4i{}, sh1 = v4i{}, sl1 = v4i{};
#pragma unroll
  for (int i = 0; i < KS; ++i) {
    v4i khi, klo;
    split_digits(kk[i][0], kk[i][1], khi, klo);
    const v4i q = *reinterpret_cast<const v4i*>(&qd[col >> 3][hb][64 * i + 16 * qt]);
    ch = __builtin_amdgcn_mfma_i32_16x16x64_i8(khi, q, ch, 0, 0, 0);
    cl = __builtin_amdgcn_mfma_i32_16x16x64_i8(klo, q, cl, 0, 0, 0);
    sh1 = __builtin_amdgcn_mfma_i32_16x16x64_i8(khi, ones, sh1, 0, 0, 0);
    sl1 = __builtin_amdgcn_mfma_i32_16x16x64_i8(klo, ones, sl1, 0, 0, 0);
  }
  int64_t mx = INT64_MIN;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    // lane col < 8 holds HH and LH of its head, lane col + 8 HL and LL
    const int hl = dpp32<0x128>(ch[i]), ll = dpp32<0x128>(cl[i]);   // row rotated by 8
    const int ksum = 256 * sh1[i] + sl1[i] + 128 * HD;
    const int64_t dot = ((int64_t)ch[i] << 16) + ((int64_t)(hl + cl[i]) << 8) + ll + 128 * ((int64_t)qsum[hb] + ksum) - 16384 * HD;
    const int si = kw + 4 * qt + i;
    if (si < p) {
      const int64_t val = shr64(dot * INV, 32 - shq[hb] - skv[i]);
      if (col < HB) scr[(int64_t)col * Sp + si] = val;
      mx = val > mx ? val : mx;
    }
  }
  mx = max64(mx, (int64_t)__shfl_xor((long long)mx, 16));
  mx = max64(mx, (int64_t)__shfl_xor((long long)mx, 32));
  if (lane < HB) wm[wave][lane] = mx;
  __syncthreads();
  if (tid < HB) {
    int64_t m = fresh ? wm[NW][tid] : INT64_MIN;
#pragma unroll
    for (int w = 0; w < NW; ++w) m = max64(m, wm[w][tid]);
    cm[((int64_t)r * H + h0 + tid) * DEC_NCH + c] = m;
  }
}

// grid (chunks, KV, R), a wave a head: the row's maximum from the chunks', then e = exp LUT(max - score) of this chunk's
// keys (between two int32 table entries) and their sum. The first chunk's block clears the head's p.V totals.
template <int HB>
__global__ __launch_bounds__(64 * HB) void k_dec_exp(const int64_t* __restrict__ sc, const int64_t* __restrict__ cm,
                                                     const int32_t* __restrict__ pos, const int32_t* __restrict__ expt,
                                                     int32_t* __restrict__ el, int64_t* __restrict__ cs, int64_t* __restrict__ acc,
                                                     int H, int hd, int Smax, int Sp) {
  constexpr int EPT = DEC_CK / 64;
  const int c = blockIdx.x, r = blockIdx.z, lane = threadIdx.x & 63, k0 = c * DEC_CK, p = pos[r];
  const int64_t row = (int64_t)r * H + blockIdx.y * HB + (threadIdx.x >> 6);
  if (p < 0 || p >= Smax || k0 > p) return;
  int64_t mx = lane <= p / DEC_CK ? cm[row * DEC_NCH + lane] : INT64_MIN, x[EPT];
#pragma unroll
  for (int j = 0; j < EPT; ++j) x[j] = sc[row * Sp + k0 + lane + 64 * j];   // score rows are padded to whole chunks
  if (c == 0)
    for (int d = lane; d < hd; d += 64) acc[row * hd + d] = 0;
  mx = wave_max64(mx);
  int64_t es = 0;
#pragma unroll
  for (int j = 0; j < EPT; ++j) {
    const int i = k0 + lane + 64 * j;
    const int e = i <= p ? (int)lut_exp(expt, mx - x[j]) : 0;
    el[row * Sp + i] = e;
    es += e;
  }
  es = wave_sum64(es);
  if (lane == 0) cs[row * DEC_NCH + c] = es;
}

// grid (chunks, KV, R): p of the chunk's keys for all the group's heads (into LDS, 0 past the position), and their p.V over
// the chunk, added to the heads' totals (64-bit atomics, exact in any order). Every lane holds two dimensions, so a wave's
// value load is whole rows and a p is one LDS broadcast; all the chunk's value loads are in flight while p is made.
// Bound by the value rows: 8 rows of 1240 to 1793 positions (49 MB) 14.6 us = 3.4 TB/s, one row of 6002 (24.6 MB) 9.0 us.
// Blocks of 8 or 16 dimensions over all keys, which need no totals, had the p of every key loaded into each lane (19 us for
// the row of 6002, on 64 CUs).
template <int HB, int HD>
__global__ __launch_bounds__(DEC_C_THREADS) void k_dec_pv(const int32_t* __restrict__ el, const int64_t* __restrict__ cs,
                                                          const int64_t* __restrict__ v, const int32_t* __restrict__ slot,
                                                          const int32_t* __restrict__ pos, int64_t* __restrict__ acc, int H,
                                                          int KV, int Smax, int Sp) {
  constexpr int NT = DEC_C_THREADS, NW = NT / 64, LPK = HD / 2, KPI = 64 / LPK;   // lanes a key, keys a load
  constexpr int KPW = DEC_CK / NW, NL = KPW / KPI, HPW = (HB + NW - 1) / NW, EPT = DEC_CK / 64;
  __shared__ __attribute__((aligned(16))) int32_t pq[HB][DEC_CK];
  __shared__ int64_t part[NW * KPI][HB][HD], hes[HB];
  const int c = blockIdx.x, kh = blockIdx.y, r = blockIdx.z, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int p = pos[r], k0 = c * DEC_CK;
  if (p < 0 || p >= Smax || k0 > p) return;
  const int64_t row0 = (int64_t)r * H + kh * HB;
  // the exponentials and the chunks' sums first: loads complete in order
  int64_t cv[HPW];
  int ev[HPW][EPT];
#pragma unroll
  for (int i = 0; i < HPW; ++i) {
    const int64_t row = row0 + (wave + i * NW < HB ? wave + i * NW : HB - 1);
    cv[i] = lane <= p / DEC_CK ? cs[row * DEC_NCH + lane] : 0;
#pragma unroll
    for (int j = 0; j < EPT; ++j) ev[i][j] = el[row * Sp + k0 + lane + 64 * j];
  }
  // the lane's keys: a run of NL, so that a head's p of four of them is one LDS read
  const int kb = wave * KPW + (lane / LPK) * NL;
  const int64_t* vb = v + ((int64_t)slot[r] * KV + kh) * Smax * HD + 2 * (lane % LPK);
  v4i vv[NL];
#pragma unroll
  for (int i = 0; i < NL; ++i) {   // keys past the last load the last (their p is 0)
    const int si = k0 + kb + i <= p ? k0 + kb + i : p;
    vv[i] = *reinterpret_cast<const v4i*>(vb + (int64_t)si * HD);
  }
  __builtin_amdgcn_sched_barrier(0);
  int big = 0;
#pragma unroll
  for (int i = 0; i < HPW; ++i) {
    const int hb = wave + i * NW;
    if (hb < HB) {
      const int64_t es = wave_sum64(cv[i]);
      const double res = 1.0 / (double)es;   // one reciprocal; each quotient estimate is corrected exactly
#pragma unroll
      for (int j = 0; j < EPT; ++j) {
        const int64_t q = floordiv_rcp((int64_t)((uint64_t)(int64_t)ev[i][j] << 20), es, res);
        big |= q < 0 || q > 0x7fffffff;   // an exp table with negative entries
        pq[hb][lane + 64 * j] = (int32_t)q;
      }
      if (lane == 0) hes[hb] = es;
    }
  }
  big = __syncthreads_or(big);
  int64_t a0[HB], a1[HB];
#pragma unroll
  for (int hb = 0; hb < HB; ++hb) a0[hb] = a1[hb] = 0;
#pragma unroll
  for (int i = 0; i < NL; ++i) big |= (vv[i][1] ^ (vv[i][0] >> 31)) | (vv[i][3] ^ (vv[i][2] >> 31));
  if (!__any(big)) {   // p in [0, 2^31), v in int32 (all but extreme values): one 32 x 32 + 64 multiply-add each
#pragma unroll
    for (int hb = 0; hb < HB; ++hb) {
#pragma unroll
      for (int i = 0; i < NL; i += 4) {
        const v4i q = *reinterpret_cast<const v4i*>(&pq[hb][kb + i]);
#pragma unroll
        for (int f = 0; f < 4; ++f) {
          a0[hb] += (int64_t)q[f] * vv[i + f][0];
          a1[hb] += (int64_t)q[f] * vv[i + f][2];
        }
      }
    }
  } else {   // any p and v: 64-bit products, from memory
#pragma unroll 1
    for (int i = 0; i < NL; ++i) {
      const int si = k0 + kb + i;
      if (si > p) break;
      const uint64_t lo = vb[(int64_t)si * HD], hi = vb[(int64_t)si * HD + 1];
#pragma unroll
      for (int hb = 0; hb < HB; ++hb) {
        const uint64_t q = floordiv_rcp((int64_t)((uint64_t)(int64_t)el[(row0 + hb) * Sp + si] << 20), hes[hb], 1.0 / (double)hes[hb]);
        a0[hb] = (int64_t)((uint64_t)a0[hb] + q * lo);
        a1[hb] = (int64_t)((uint64_t)a1[hb] + q * hi);
      }
    }
  }
#pragma unroll
  for (int hb = 0; hb < HB; ++hb) {
    int64_t* d = &part[wave * KPI + lane / LPK][hb][2 * (lane % LPK)];
    d[0] = a0[hb];
    d[1] = a1[hb];
  }
  __syncthreads();
  for (int i = tid; i < HB * HD; i += NT) {
    uint64_t tot = 0;
#pragma unroll
    for (int w = 0; w < NW * KPI; ++w) tot += (uint64_t)(&part[w][0][0])[i];
    atomicAdd(reinterpret_cast<unsigned long long*>(acc + row0 * HD + i), (unsigned long long)tot);
  }
}

// grid (H, R), block HD: out = shr(p.V, 20) and the bit lengths of its slices
template <int HD>
__global__ __launch_bounds__(HD) void k_dec_out(const int64_t* __restrict__ acc, const int32_t* __restrict__ pos,
                                                int64_t* __restrict__ out, int32_t* __restrict__ obits, int obn, int H, int Smax) {
  __shared__ int bl[HD / 16];
  const int64_t row = (int64_t)blockIdx.y * H + blockIdx.x;
  const int d = threadIdx.x, p = pos[blockIdx.y];
  const int64_t o = p < 0 || p >= Smax ? 0 : shr64(acc[row * HD + d], 20);
  out[row * HD + d] = o;
  if (!obits) return;
  int m = bitlen64(abs64(o));   // maxima of 16 lanes: lane ^ 1, lane ^ 2, the mirrored lanes of the half row and the row
  m = max(m, dpp32<0xB1>(m));
  m = max(m, dpp32<0x4E>(m));
  m = max(m, dpp32<0x141>(m));
  m = max(m, dpp32<0x140>(m));
  if ((d & 15) == 0) bl[d >> 4] = m;
  __syncthreads();
  if (d < obn) {
    const int n = HD / 16 / obn;
    int x = 0;
    for (int i = 0; i < n; ++i) x = max(x, bl[d * n + i]);
    obits[row * obn + d] = x;
  }
}

// score rows in the workspace are padded to whole chunks
static int dec_sp(int Smax) { return (Smax + DEC_CK - 1) / DEC_CK * DEC_CK; }

template <int HB, int HD>
static void dec_go(const int64_t* t, const int32_t* s, const int64_t* b, const int64_t* cos_t, const int64_t* sin_t,
                   const int32_t* slot, const int32_t* pos, int16_t* kq, int32_t* sk, int64_t* v, const int32_t* exp_t,
                   int64_t* out, int32_t* obits, int obn, int8_t* work, int R, int H, int KV, int Smax, int INV, hipStream_t st) {
  const int Sp = dec_sp(Smax);
  const int64_t rows = (int64_t)R * H;
  int64_t* sc = reinterpret_cast<int64_t*>(work);
  int64_t* acc = sc + rows * Sp;
  int64_t* cm = acc + rows * HD;
  int64_t* cs = cm + rows * DEC_NCH;
  int32_t* el = reinterpret_cast<int32_t*>(cs + rows * DEC_NCH);
  const dim3 grid(Sp / DEC_CK, KV, R);
  hipLaunchKernelGGL((k_dec_scores<HB, HD>), grid, dim3(DEC_A_THREADS), 0, st, t, s, b, cos_t, sin_t, slot, pos, kq, sk, v, sc,
                     cm, H, KV, Smax, Sp, INV);
  hipLaunchKernelGGL((k_dec_exp<HB>), grid, dim3(64 * HB), 0, st, sc, cm, pos, exp_t, el, cs, acc, H, HD, Smax, Sp);
  hipLaunchKernelGGL((k_dec_pv<HB, HD>), grid, dim3(DEC_C_THREADS), 0, st, el, cs, v, slot, pos, acc, H, KV, Smax, Sp);
  hipLaunchKernelGGL((k_dec_out<HD>), dim3(H, R), dim3(HD), 0, st, acc, pos, out, obits, obn, H, Smax);
}

}  // namespace exact

using namespace exact;

static bool dec_takes(int R, int H, int KV, int hd, int Smax) {
  if (R <= 0 || H <= 0 || KV <= 0 || H % KV || Smax <= 0 || Smax > DEC_SMAX || (hd != 64 && hd != 128)) return false;
  const int grp = H / KV;
  return (grp == 1 || grp == 2 || grp == 4 || grp == 5 || grp == 7 || grp == 8) && R <= 65535 && H <= 65535;
}

extern "C" int64_t exact_attention_decode_workspace(int32_t R, int32_t H, int32_t KV, int32_t hd, int32_t Smax) {
  if (!dec_takes(R, H, KV, hd, Smax)) return 0;
  // scores, p.V totals, the chunks' maxima and sums, exponentials
  return (int64_t)R * H * (dec_sp(Smax) * 12LL + hd * 8 + DEC_NCH * 16);
}

extern "C" int exact_attention_decode(const int64_t* t, const int32_t* s, const int64_t* b, const int64_t* cos_t,
                                      const int64_t* sin_t, const int32_t* slot, const int32_t* pos, int16_t* kq, int32_t* sk,
                                      int64_t* v, const int32_t* exp_t, int64_t* out, int32_t* obits, int32_t obn, void* work,
                                      int64_t work_bytes, int32_t R, int32_t H, int32_t KV, int32_t hd, int32_t Smax,
                                      int32_t INV, void* stream) {
  if (!t || !s || !cos_t || !sin_t || !slot || !pos || !kq || !sk || !v || !exp_t || !out || !work) return EXACT_E_ARG;
  if (R <= 0 || H <= 0 || KV <= 0 || H % KV || hd <= 0 || Smax <= 0) return EXACT_E_ARG;
  if (obn != 1 && obn != 2 && obn != 4) return EXACT_E_ARG;
  if (!dec_takes(R, H, KV, hd, Smax)) return EXACT_E_UNSUPPORTED;
  if ((reinterpret_cast<uintptr_t>(work) & 255) || work_bytes < exact_attention_decode_workspace(R, H, KV, hd, Smax))
    return EXACT_E_ARG;
  if ((reinterpret_cast<uintptr_t>(kq) & 15) || (reinterpret_cast<uintptr_t>(v) & 15)) return EXACT_E_UNSUPPORTED;
  const hipStream_t st = as_stream(stream);
#define DEC_ARGS t, s, b, cos_t, sin_t, slot, pos, kq, sk, v, exp_t, out, obits, obn, static_cast<int8_t*>(work), R, H, KV, Smax, INV, st
#define DEC_HB(HB) \
  case HB: \
    if (hd == 64) dec_go<HB, 64>(DEC_ARGS); \
    else dec_go<HB, 128>(DEC_ARGS); \
    break
  switch (H / KV) {
    DEC_HB(1);
    DEC_HB(2);
    DEC_HB(4);
    DEC_HB(5);
    DEC_HB(7);
    DEC_HB(8);
  }
#undef DEC_HB
#undef DEC_ARGS
  return launch_status("attention_decode");
}

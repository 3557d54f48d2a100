// Attention of a short prompt's rows (up to 128 positions, hd 64 or 128; exact_llm.py:170-176), results as exact_attention.
//
// exact_attention takes a 512-thread block per (row, head): of 41 rows' keys at most 41 threads have one, five block barriers
// order its steps, and 41 rows of 28 heads are 1148 such blocks. Here a wave takes a (row, head): 8 lanes a key make the scores
// (16-byte loads, whole rows of 256 bytes), after which lane l holds key l of each 64; maximum, exponentials and division are
// wave reductions, and p.V gives each lane two dimensions, so that a value load is whole rows too. No barrier, 4 waves a block.
// us a layer of 28 heads over 4 of 128, in a graph, this kernel / exact_attention / the matrix-core kernels: 8 rows 6.2 / 10.1 /
// -, 41 rows 10.1 / 14.7 / 23.7, 64 rows 12.2 / 21.7 / 24.1, 95 rows 20.4 / 32.1 / 23.8. Bound by the chain of a wave's loads and
// reductions; a wave that walks four chunks (4 rows at 254 positions) takes 34 against 15.5, so it ends at two.
#include "exact_common.h"
#include "abi_util.h"

namespace exact {

#define ROWS_WAVES 4
#define ROWS_VL 8   // value loads in flight

template <int HD, int NK>   // NK: 64-key chunks
__global__ __launch_bounds__(ROWS_WAVES * 64) void k_attention_rows(
    const int16_t* __restrict__ qq, const int32_t* __restrict__ sq, const int16_t* __restrict__ kq,
    const int32_t* __restrict__ sk, const int64_t* __restrict__ v, const int32_t* __restrict__ slot,
    const int32_t* __restrict__ pos, const int32_t* __restrict__ expt, int64_t* __restrict__ out, int32_t* __restrict__ obits,
    int R, int H, int KV, int Smax, int INV) {
  constexpr int EL = HD / 8, LPK = HD / 2, KPI = 64 / LPK;   // a lane's elements of a key; lanes of a value row, rows a load
  __shared__ __attribute__((aligned(16))) int64_t ps[ROWS_WAVES][NK * 64];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int w = blockIdx.x * ROWS_WAVES + wave, HB = H / KV;
  if (w >= R * H) return;
  // the heads of a KV head and the rows next to each other share a block's cache lines
  const int kh = w / (R * HB), r = (w - kh * R * HB) / HB, h = kh * HB + (w - kh * R * HB) % HB;
  const int S = min(min(pos[r] + 1, Smax), NK * 64);
  const int64_t cbase = ((int64_t)slot[r] * KV + kh) * Smax;
  const int sqv = sq[r * H + h], g = lane >> 3, l8 = lane & 7;
  v4i qv[EL / 8];
  const int16_t* qp = qq + ((int64_t)r * H + h) * HD + l8 * EL;
#pragma unroll
  for (int e = 0; e < EL / 8; ++e) qv[e] = reinterpret_cast<const v4i*>(qp)[e];
  int64_t x[NK], mx = INT64_MIN;
#pragma unroll
  for (int c = 0; c < NK; ++c) {
    x[c] = INT64_MIN;
    if (64 * c >= S) continue;   // uniform over the wave
    const int key = 64 * c + lane;
    const int skv = sk[cbase + (key < S ? key : S - 1)];
    v4i kv[8][EL / 8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {   // key 8 g + i of the chunk; keys past the last read the last
      const int ki = 64 * c + 8 * g + i < S ? 64 * c + 8 * g + i : S - 1;
      const v4i* kp = reinterpret_cast<const v4i*>(kq + (cbase + ki) * HD + l8 * EL);
#pragma unroll
      for (int e = 0; e < EL / 8; ++e) kv[i][e] = kp[e];
    }
    int64_t dot = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      int64_t a = 0;
#pragma unroll
      for (int e = 0; e < EL / 8; ++e)
#pragma unroll
        for (int f = 0; f < 4; ++f) {   // a pair of int16 products is exact in int32 (< 2^31)
          const int kk = kv[i][e][f], q2 = qv[e][f];
          a += (int64_t)((int32_t)(int16_t)kk * (int32_t)(int16_t)q2 + (kk >> 16) * (q2 >> 16));
        }
      a += dpp64<0xB1>(a);
      a += dpp64<0x4E>(a);
      a += dpp64<0x141>(a);
      dot = l8 == i ? a : dot;
    }
    if (key < S) x[c] = shr64(dot * INV, 32 - sqv - skv);
    mx = max64(mx, x[c]);
  }
  // the first values, in flight while p is made
  const int sub = lane / LPK, NS = (S + KPI - 1) / KPI;   // value loads of the row
  const int64_t* vb = v + cbase * HD + 2 * (lane % LPK);
  auto vload = [&](int i) {
    const int si = KPI * i + sub < S ? KPI * i + sub : (S > 0 ? S - 1 : 0);
    return *reinterpret_cast<const v4i*>(vb + (int64_t)si * HD);
  };
  v4i vv[ROWS_VL];
#pragma unroll
  for (int i = 0; i < ROWS_VL; ++i) vv[i] = vload(i);
  mx = wave_max64(mx);
  int64_t es = 0, e[NK];
#pragma unroll
  for (int c = 0; c < NK; ++c) {
    e[c] = 64 * c + lane < S ? lut_exp(expt, mx - x[c]) : 0;
    es += e[c];
  }
  es = wave_sum64(es);
  const double rb = 1.0 / (double)es;
  int big = 0;
#pragma unroll
  for (int c = 0; c < NK; ++c) {
    const int64_t p = 64 * c + lane < S ? floordiv_rcp(shl64(e[c], 20), es, rb) : 0;
    big |= p < 0 || p > 0x7fffffff;   // an exp table with negative entries
    ps[wave][64 * c + lane] = p;
  }
  big = __any(big);
  __builtin_amdgcn_wave_barrier();   // a wave's own LDS operations complete in order
  const int64_t* pw = ps[wave];
  uint64_t a0 = 0, a1 = 0;
  for (int i0 = 0; i0 < NS; i0 += ROWS_VL) {
    int wide = big;
#pragma unroll
    for (int i = 0; i < ROWS_VL; ++i) wide |= (vv[i][1] ^ (vv[i][0] >> 31)) | (vv[i][3] ^ (vv[i][2] >> 31));
    wide = __any(wide);
#pragma unroll
    for (int i = 0; i < ROWS_VL; ++i) {
      const int si = KPI * (i0 + i) + sub;   // p is 0 past the last key (the last of NK * 64 slots at most)
      const int64_t p = si < NK * 64 ? pw[si] : 0;
      if (!wide) {   // p and v in 32 bits: one multiply-add each
        a0 += (uint64_t)((int64_t)(int32_t)p * vv[i][0]);
        a1 += (uint64_t)((int64_t)(int32_t)p * vv[i][2]);
      } else {
        a0 += (uint64_t)p * (((uint64_t)(uint32_t)vv[i][1] << 32) | (uint32_t)vv[i][0]);
        a1 += (uint64_t)p * (((uint64_t)(uint32_t)vv[i][3] << 32) | (uint32_t)vv[i][2]);
      }
    }
    if (i0 + ROWS_VL < NS)
#pragma unroll
      for (int i = 0; i < ROWS_VL; ++i) vv[i] = vload(i0 + ROWS_VL + i);
  }
  if constexpr (KPI == 2) {
    a0 += (uint64_t)__shfl_xor((long long)a0, 32, 64);
    a1 += (uint64_t)__shfl_xor((long long)a1, 32, 64);
  }
  const int64_t o0 = shr64((int64_t)a0, 20), o1 = shr64((int64_t)a1, 20);
  if (sub == 0)
    *reinterpret_cast<longlong2*>(out + ((int64_t)r * H + h) * HD + 2 * (lane % LPK)) = make_longlong2(o0, o1);
  if (obits) {
    const int b0 = bitlen64(abs64(o0)), b1 = bitlen64(abs64(o1));
    const int m = wave_max_i32(b0 > b1 ? b0 : b1);
    if (lane == 0) obits[r * H + h] = m;
  }
}

}  // namespace exact

using namespace exact;

extern "C" int exact_attention_rows(const int16_t* qq, const int32_t* sq, const int16_t* kq, const int32_t* sk, const int64_t* v,
                                    const int32_t* slot, const int32_t* pos, const int32_t* exp_t, int64_t* out, int32_t* obits,
                                    int32_t R, int32_t H, int32_t KV, int32_t hd, int32_t Smax, int32_t nkeys, int32_t INV,
                                    void* stream) {
  if (!qq || !sq || !kq || !sk || !v || !slot || !pos || !exp_t || !out) return EXACT_E_ARG;
  if (R <= 0 || H <= 0 || KV <= 0 || H % KV || hd <= 0 || Smax <= 0 || nkeys <= 0) return EXACT_E_ARG;
  if ((hd != 64 && hd != 128) || nkeys > 128 || Smax > 8192 || (int64_t)R * H > INT32_MAX / 2) return EXACT_E_UNSUPPORTED;
  if (((uintptr_t)qq | (uintptr_t)kq | (uintptr_t)v | (uintptr_t)out) & 15) return EXACT_E_UNSUPPORTED;
  const dim3 grid((uint32_t)cdiv((int64_t)R * H, ROWS_WAVES)), block(ROWS_WAVES * 64);
#define ROWS_GO(HD, NK)                                                                                                  \
  hipLaunchKernelGGL((k_attention_rows<HD, NK>), grid, block, 0, as_stream(stream), qq, sq, kq, sk, v, slot, pos, exp_t, out, \
                     obits, R, H, KV, Smax, INV)
  const int nk = (nkeys + 63) / 64;
  if (hd == 64) {
    if (nk <= 1) ROWS_GO(64, 1);
    else ROWS_GO(64, 2);
  } else {
    if (nk <= 1) ROWS_GO(128, 1);
    else ROWS_GO(128, 2);
  }
#undef ROWS_GO
  return launch_status("attention_rows");
}

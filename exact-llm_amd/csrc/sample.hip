// Integer sampler on the device (sample_int, exact_llm.py:256-259):
//   a = shr(lg * tnum, 16); p = isoftmax_row(a) (Q20); cum = cumsum(p);
//   target = (u20 * cum[-1]) >> 20 with u20 = splitmix64(seed, step) >> 44;
//   token = searchsorted(cum, target, 'right') = #{i : cum[i] <= target}
// One workgroup of SAMPLE_THREADS per row. Wave w owns the contiguous span [w*span, (w+1)*span) of the
// row and walks it 64 lanes at a time (coalesced loads); the running prefix inside a wave comes from a
// lane scan, the prefix before a wave from a scan over the waves' span sums. Since p >= 0, cum is
// non-decreasing, so the token is the number of prefix sums <= target.
//
// Rows of a vocabulary are split: one workgroup walking 152064 logits four times (each walk waits for the one before)
// keeps R of 256 CUs busy (8 rows: 311 us; 20.6 split, of which the four dependent launches alone take about 15, the time
// of one short row). exact_sample_split runs the four walks as four launches of one block per
// (row, chunk of SAMPLE_CHUNK logits); a launch starts from the chunk results of the one before (row maximum, softmax
// denominator, sums of p), which every block reduces again for itself.
#include "exact_common.h"
#include "abi_util.h"

namespace exact {

#define SAMPLE_THREADS 1024

__device__ __forceinline__ int64_t wave_incl_scan64(int64_t v, int lane) {
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int64_t w = __shfl_up(v, o, 64);
    if (lane >= o) v = (int64_t)((uint64_t)v + (uint64_t)w);
  }
  return v;
}

__global__ __launch_bounds__(SAMPLE_THREADS) void k_sample(const int64_t* __restrict__ lg, int V, uint64_t seed,
                                                          const int32_t* __restrict__ step, int64_t tnum,
                                                          const int32_t* __restrict__ T, int32_t* __restrict__ ids,
                                                          int64_t* __restrict__ p_out) {
  __shared__ int64_t red_a[16], red_b[16], red_c[16];
  __shared__ int64_t wsum[SAMPLE_THREADS / 64];
  __shared__ int64_t wcnt[SAMPLE_THREADS / 64];
  const int r = blockIdx.x, tid = threadIdx.x, lane = tid & 63, w = tid >> 6, nw = blockDim.x >> 6;
  const int64_t* row = lg + (int64_t)r * V;
  const int span = ((V + nw - 1) / nw + 63) / 64 * 64;
  const int b0 = w * span, b1 = b0 + span < V ? b0 + span : V;
  // pass 1: row max of a
  int64_t mx = INT64_MIN;
  for (int i = b0 + lane; i < b1; i += 64) {
    const int64_t a = shr64(row[i] * tnum, EXACT_F);
    mx = a > mx ? a : mx;
  }
  mx = block_max64(mx, red_a);
  // pass 2: the softmax denominator
  int64_t es = 0;
  for (int i = b0 + lane; i < b1; i += 64) es += lut_exp(T, mx - shr64(row[i] * tnum, EXACT_F));
  es = block_sum64(es, red_b);
  // pass 3: each wave's sum of p
  int64_t ps = 0;
  for (int i = b0 + lane; i < b1; i += 64) ps += floordiv_pos(shl64(lut_exp(T, mx - shr64(row[i] * tnum, EXACT_F)), 20), es);
  ps = wave_sum64(ps);
  if (lane == 0) wsum[w] = ps;
  __syncthreads();
  int64_t pre = 0, total = 0;
  for (int j = 0; j < nw; ++j) {
    if (j < w) pre += wsum[j];
    total += wsum[j];
  }
  const int64_t u = (int64_t)(splitmix64(seed, (uint64_t)(int64_t)step[r]) >> 44);
  const int64_t target = (u * total) >> 20;
  // pass 4: count the prefix sums <= target, 64 at a time
  int64_t cnt = 0, carry = pre;
  for (int base = b0; base < b1; base += 64) {
    const int i = base + lane;
    int64_t p = 0;
    if (i < b1) p = floordiv_pos(shl64(lut_exp(T, mx - shr64(row[i] * tnum, EXACT_F)), 20), es);
    if (p_out && i < b1) p_out[(int64_t)r * V + i] = p;
    const int64_t c = carry + wave_incl_scan64(p, lane);
    if (i < b1 && c <= target) ++cnt;
    carry = __shfl(c, 63, 64);
  }
  cnt = wave_sum64(cnt);
  if (lane == 0) wcnt[w] = cnt;
  __syncthreads();
  if (tid == 0) {
    int64_t tok = 0;
    for (int j = 0; j < nw; ++j) tok += wcnt[j];
    ids[r] = (int32_t)tok;
  }
}

// ---- split over chunks: block b is chunk b % nch of row b / nch. A wave owns SAMPLE_PT * 64 consecutive logits, 64 a
// step, so loads coalesce and the count of prefix sums needs a lane scan a step and no exchange but the waves' sums.
#define SAMPLE_PT 4
#define SAMPLE_NT 256
#define SAMPLE_CHUNK (SAMPLE_PT * SAMPLE_NT)

struct SampleWork {   // int64 arrays of one call
  int64_t *mx, *es, *ps;   // [R * nch]: chunk maximum of a, sum of exponentials, sum of p
  uint64_t* u;             // [R]: the row's 20 random bits
  int64_t* neg;            // [R]: a negative exponential (of an exp table with negative entries): cum may decrease
  int32_t* e;              // [R * V]: exponentials (between two int32 table entries)
};
__host__ __forceinline__ SampleWork sample_work(int64_t* w, int64_t n, int64_t R) {
  return {w, w + n, w + 2 * n, (uint64_t*)(w + 3 * n), w + 3 * n + R, (int32_t*)(w + 3 * n + 2 * R)};
}

// floor(e * 2^20 / es), rb ~ 2^20 / es: for 0 <= e <= es the quotient is at most 2^20 and the float64 estimate within one
// of it; anything else (an exp table with negative entries, or one that leaves a row no exponential) takes the general
// division, which gives 0 for es <= 0
__device__ __forceinline__ int64_t sample_p(int32_t e, int64_t es, double rb) {
  if (e < 0 || e > es || es <= 0) return floordiv_pos(shl64(e, 20), es);
  uint32_t q = (uint32_t)((double)e * rb);
  const int64_t d = ((int64_t)e << 20) - (int64_t)q * es;
  return (int64_t)q + (d >= es) - (d < 0);
}

struct SampleBlock {
  int64_t r, base, i0;   // row, its first chunk, this lane's first logit
  int ch;
  bool ok[SAMPLE_PT];
  __device__ __forceinline__ SampleBlock(int V, int nch) {
    r = blockIdx.x / nch;
    ch = (int)(blockIdx.x - r * nch);
    base = r * nch;
    i0 = (int64_t)ch * SAMPLE_CHUNK + (threadIdx.x >> 6) * (SAMPLE_PT * 64) + (threadIdx.x & 63);
#pragma unroll
    for (int k = 0; k < SAMPLE_PT; ++k) ok[k] = i0 + 64 * k < V;
  }
  __device__ __forceinline__ void load(const int64_t* lg, int V, int64_t tnum, int64_t (&a)[SAMPLE_PT]) const {
    const int64_t* row = lg + r * V + i0;
#pragma unroll
    for (int k = 0; k < SAMPLE_PT; ++k) a[k] = ok[k] ? shr64(row[64 * k] * tnum, EXACT_F) : INT64_MIN;
  }
};

__device__ __forceinline__ int64_t chunk_max(const int64_t* v, int nch, int64_t* red) {
  int64_t m = INT64_MIN;
  for (int i = threadIdx.x; i < nch; i += SAMPLE_NT) m = max64(m, v[i]);
  return block_max64_1(m, red);
}
__device__ __forceinline__ int64_t chunk_sum(const int64_t* v, int nch, int64_t* red) {
  uint64_t s = 0;
  for (int i = threadIdx.x; i < nch; i += SAMPLE_NT) s += (uint64_t)v[i];
  return block_sum64_1((int64_t)s, red);
}

__global__ __launch_bounds__(SAMPLE_NT) void k_sample_max(const int64_t* __restrict__ lg, int V, int nch, uint64_t seed,
                                                          const int32_t* step, int64_t tnum, SampleWork wk, int32_t* ids) {
  __shared__ int64_t red[16];
  const SampleBlock B(V, nch);
  int64_t a[SAMPLE_PT], m = INT64_MIN;
  B.load(lg, V, tnum, a);
#pragma unroll
  for (int k = 0; k < SAMPLE_PT; ++k) m = max64(m, a[k]);
  m = block_max64_1(m, red);
  if (threadIdx.x == 0) {
    wk.mx[blockIdx.x] = m;
    if (B.ch == 0) {   // step read before ids is written: they may be one array
      wk.u[B.r] = splitmix64(seed, (uint64_t)(int64_t)step[B.r]) >> 44;
      wk.neg[B.r] = 0;
      ids[B.r] = V;
    }
  }
}

__global__ __launch_bounds__(SAMPLE_NT) void k_sample_exp(const int64_t* __restrict__ lg, int V, int nch, int64_t tnum,
                                                          const int32_t* __restrict__ T, SampleWork wk) {
  __shared__ int64_t red[2][16];
  const SampleBlock B(V, nch);
  int64_t a[SAMPLE_PT], es = 0;
  B.load(lg, V, tnum, a);
  const int64_t mx = chunk_max(wk.mx + B.base, nch, red[0]);
#pragma unroll
  for (int k = 0; k < SAMPLE_PT; ++k)
    if (B.ok[k]) {
      const int64_t e = lut_exp(T, mx - a[k]);
      wk.e[B.r * V + B.i0 + 64 * k] = (int32_t)e;
      if (e < 0) wk.neg[B.r] = 1;
      es += e;
    }
  es = block_sum64_1(es, red[1]);
  if (threadIdx.x == 0) wk.es[blockIdx.x] = es;
}

__device__ __forceinline__ void load_p(const SampleBlock& B, int V, const SampleWork& wk, int64_t es, int64_t (&p)[SAMPLE_PT]) {
  const double rb = 1048576.0 / (double)es;
  int32_t e[SAMPLE_PT];
#pragma unroll
  for (int k = 0; k < SAMPLE_PT; ++k) e[k] = B.ok[k] ? wk.e[B.r * V + B.i0 + 64 * k] : 0;
#pragma unroll
  for (int k = 0; k < SAMPLE_PT; ++k) p[k] = B.ok[k] ? sample_p(e[k], es, rb) : 0;
}

__global__ __launch_bounds__(SAMPLE_NT) void k_sample_psum(int V, int nch, SampleWork wk) {
  __shared__ int64_t red[2][16];
  const SampleBlock B(V, nch);
  int64_t p[SAMPLE_PT], sum = 0;
  load_p(B, V, wk, chunk_sum(wk.es + B.base, nch, red[0]), p);
#pragma unroll
  for (int k = 0; k < SAMPLE_PT; ++k) sum += p[k];
  sum = block_sum64_1(sum, red[1]);
  if (threadIdx.x == 0) wk.ps[blockIdx.x] = sum;
}

// The token is the number of prefix sums <= target. ids holds V: where no p is negative, the one chunk in which the sums
// pass the target writes it (no chunk if all sums are 0), and the other blocks end early; 64-bit counts of every wave
// added to ids instead, 4768 atomics to one line, took 24 us at 8 rows of 152064. With a negative p every chunk counts.
__global__ __launch_bounds__(SAMPLE_NT) void k_sample_pick(int V, int nch, SampleWork wk, int32_t* __restrict__ ids,
                                                           int64_t* __restrict__ p_out) {
  __shared__ int64_t red[4][16];
  const SampleBlock B(V, nch);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int64_t total = chunk_sum(wk.ps + B.base, nch, red[0]);
  int64_t carry = chunk_sum(wk.ps + B.base, B.ch, red[1]);
  const int64_t target = ((int64_t)wk.u[B.r] * total) >> 20;
  const bool neg = wk.neg[B.r] != 0, here = carry <= target && target < carry + wk.ps[blockIdx.x];
  if (!here && !neg && !p_out) return;
  int64_t p[SAMPLE_PT], sum = 0;
  load_p(B, V, wk, chunk_sum(wk.es + B.base, nch, red[2]), p);
#pragma unroll
  for (int k = 0; k < SAMPLE_PT; ++k) sum += p[k];
  sum = wave_sum64(sum);
  if (lane == 0) red[3][w] = sum;
  __syncthreads();
  for (int j = 0; j < w; ++j) carry += red[3][j];
  int over = 0;   // prefix sums above the target
#pragma unroll
  for (int k = 0; k < SAMPLE_PT; ++k) {
    if (p_out && B.ok[k]) p_out[B.r * V + B.i0 + 64 * k] = p[k];
    const int64_t c = carry + wave_incl_scan64(p[k], lane);
    over += __popcll(__ballot(B.ok[k] && c > target));
    carry = readlane64(c, 63);
  }
  if (!here && !neg) return;
  if (neg) {
    if (lane == 0 && over) atomicAdd(&ids[B.r], -over);
  } else {
    __shared__ int32_t wover[16];
    if (lane == 0) wover[w] = over;
    __syncthreads();
    if (threadIdx.x == 0) {
      for (int j = 1; j < SAMPLE_NT / 64; ++j) over += wover[j];
      const int64_t end = ((int64_t)B.ch + 1) * SAMPLE_CHUNK;
      ids[B.r] = (int32_t)((end < V ? end : V) - over);
    }
  }
}

}  // namespace exact

using namespace exact;

extern "C" int exact_sample(const int64_t* lg, int32_t R, int32_t V, uint64_t seed, const int32_t* step, int64_t tnum,
                            const int32_t* exp_t, int32_t* ids, int64_t* p_out, void* stream) {
  if (!lg || !step || !exp_t || !ids || R <= 0 || V <= 0 || tnum <= 0) return EXACT_E_ARG;
  hipLaunchKernelGGL(k_sample, dim3(R), dim3(SAMPLE_THREADS), 0, as_stream(stream), lg, V, seed, step, tnum, exp_t, ids,
                     p_out);
  return launch_status("sample");
}

extern "C" int64_t exact_sample_workspace(int32_t R, int32_t V) {
  if (R <= 0 || V <= 0) return 0;
  return ((3 * cdiv(V, SAMPLE_CHUNK) + 2) * 8 + (int64_t)V * 4) * R;
}

extern "C" int exact_sample_split(const int64_t* lg, int32_t R, int32_t V, uint64_t seed, const int32_t* step, int64_t tnum,
                                  const int32_t* exp_t, int32_t* ids, int64_t* p_out, void* work, int64_t work_bytes,
                                  void* stream) {
  if (!lg || !step || !exp_t || !ids || !work || R <= 0 || V <= 0 || tnum <= 0) return EXACT_E_ARG;
  if ((uintptr_t)work % 8 || work_bytes < exact_sample_workspace(R, V)) return EXACT_E_ARG;
  const int64_t nch = cdiv(V, SAMPLE_CHUNK);
  if (nch * R > INT32_MAX) return EXACT_E_UNSUPPORTED;
  const SampleWork wk = sample_work((int64_t*)work, nch * R, R);
  const dim3 g((uint32_t)(nch * R)), b(SAMPLE_NT);
  hipStream_t st = as_stream(stream);
  hipLaunchKernelGGL(k_sample_max, g, b, 0, st, lg, V, (int)nch, seed, step, tnum, wk, ids);
  hipLaunchKernelGGL(k_sample_exp, g, b, 0, st, lg, V, (int)nch, tnum, exp_t, wk);
  hipLaunchKernelGGL(k_sample_psum, g, b, 0, st, V, (int)nch, wk);
  hipLaunchKernelGGL(k_sample_pick, g, b, 0, st, V, (int)nch, wk, ids, p_out);
  return launch_status("sample_split");
}

// softmax (norms.rs:44-56) over rows: max, e = expf(x - max), the sum of e as
// the reference's left-to-right fold, e * (1/sum).
//
// Long rows (a vocabulary) are cut into chunks of about 1024 values, a
// workgroup each, in five launches (seven from a million values on):
//   1. each chunk's maximum
//   2. each chunk's sum of exponentials, in any order
//   3. each chunk's part of the ordered sum as a map: while the running sum
//      stays inside one binade, a run of additions is a pair of integer
//      increments (exact_sum.h), and the sums of launch 2 predict the binade
//      at a chunk's start. Steps that may leave it (predicted within
//      pred_margin units of a binade boundary) are listed as plain additions
//      between two such runs.
//   4. one workgroup per row walks the chunks' records from the first chunk's
//      exact sum, checking that each run starts and ends in the binade its
//      map assumed; a chunk that fails is summed by the whole workgroup from
//      the exact value before it
//   5. the probabilities
// A chunk's record lives in the first words of the chunk in `out` until
// launch 5 overwrites it (each workgroup there reads its own record only), so
// the path needs no scratch and its launches keep nothing between calls; the
// exponentials are recomputed from `in` where they are needed, so in and out
// must not overlap. Bound by the latency of the five launches and the walk:
// one row of 151936 values 26-27 us, of 32000 21 us, against 3845 and 744 us on
// the one-workgroup kernel (an ordered pass of 256 lanes per binade); walking
// the 149 records one by one took 36 of then 48 us.
#include <climits>

#include "common.h"
#include "exact_sum.h"
#include "kernels.h"

namespace prana {

namespace {

// ---------------------------------------------------------------- short rows
// norms.rs:44-56, one workgroup per row; the sum is the sequential fold,
// evaluated exactly by the workgroup.
__global__ __launch_bounds__(256) void softmax_kernel(const float* __restrict__ in, int n, float* __restrict__ out) {
  __shared__ float s_red[4];
  const float* row = in + (size_t)blockIdx.x * n;
  float* dst = out + (size_t)blockIdx.x * n;
  float mx = -INFINITY;
  for (int i = threadIdx.x; i < n; i += 256) mx = fmaxf(mx, row[i]);
  mx = wave_max_f32(mx);
  if ((threadIdx.x & 63) == 0) s_red[threadIdx.x >> 6] = mx;
  __syncthreads();
  mx = fmaxf(fmaxf(s_red[0], s_red[1]), fmaxf(s_red[2], s_red[3]));
  for (int i = threadIdx.x; i < n; i += 256) dst[i] = dev_expf(row[i] - mx);
  __syncthreads();
  const float sum = exact::block_seq_sum_nonneg<256, false>(dst, n);  // norms.rs:53 order
  const float inv = sum > 0.0f ? 1.0f / sum : 0.0f;
  for (int i = threadIdx.x; i < n; i += 256) dst[i] = dst[i] * inv;
}


// ---------------------------------------------------------------- long rows
constexpr int kSmNT = 256;
constexpr int kSmCT = 4;                 // consecutive values per lane
constexpr int kSmChunk = kSmNT * kSmCT;  // values of a chunk at most
constexpr int kSmPlain = 256;            // plain additions a record may hold
constexpr int kSmSlots = 16;             // chunks whose plain terms are fetched ahead, per 64 records
// A chunk's record: launch 1 writes its maximum, launch 2 its sum and the
// row's maximum, launch 3 the maps (e0 o0 e1 o1), the plain additions and the
// binades of the two runs (chunk 0: its exact sum, in kRecMap), launch 4 the
// factor 1/sum.
enum {
  kRecMax = 0, kRecSum = 1, kRecMap = 2, kRecPlain = 6, kRecB0 = 7, kRecB1 = 8, kRecInv = 9, kRecRowMax = 10, kRecPre = 11
};
constexpr int kComplex = 1 << 30;        // kRecPlain: no map, sum the chunk from the value before it

// Chunk c of the row is [begin(c), begin(c + 1)): 512 values at least.
struct SmRow {
  const float* in;
  float* out;
  int n, chunks;
  __device__ int begin(int c) const { return static_cast<int>(static_cast<long long>(c) * n / chunks); }
  __device__ float* rec(int c) const { return out + begin(c); }
};

__device__ __forceinline__ SmRow sm_row(const float* in, float* out, int n, int chunks) {
  const size_t r = blockIdx.y;
  return SmRow{in + r * n, out + r * n, n, chunks};
}

// The maximum over the workgroup (every lane).
__device__ __forceinline__ float sm_block_max(float mx, float* s_red) {
  mx = wave_max_f32(mx);
  if ((threadIdx.x & 63) == 0) s_red[threadIdx.x >> 6] = mx;
  __syncthreads();
  return fmaxf(fmaxf(s_red[0], s_red[1]), fmaxf(s_red[2], s_red[3]));
}

__global__ __launch_bounds__(kSmNT) void softmax_max_kernel(const float* in, float* out, int n, int chunks) {
  __shared__ float s_red[kSmNT / 64];
  const SmRow R = sm_row(in, out, n, chunks);
  const int c = blockIdx.x, b = R.begin(c), e = R.begin(c + 1);
  float mx = -INFINITY;
#pragma unroll
  for (int u = 0; u < kSmCT; u++) mx = fmaxf(mx, R.in[min(b + static_cast<int>(threadIdx.x) + kSmNT * u, e - 1)]);
  mx = sm_block_max(mx, s_red);
  if (threadIdx.x == 0) R.rec(c)[kRecMax] = mx;
}

// Rows of more than kSmMany chunks (about a million values): the row's maximum and the sums before each
// chunk are formed by one workgroup per row, where otherwise every chunk's
// workgroup reads the other chunks' records (work that grows with the square of
// their number).
constexpr int kSmScanNT = 1024;

__global__ __launch_bounds__(kSmScanNT) void softmax_row_max_kernel(const float* in, float* out, int n, int chunks) {
  __shared__ float s_red[kSmScanNT / 64];
  const SmRow R = sm_row(in, out, n, chunks);
  float mx = -INFINITY;
  for (int c = threadIdx.x; c < chunks; c += kSmScanNT) mx = fmaxf(mx, R.rec(c)[kRecMax]);
  mx = wave_max_f32(mx);
  if ((threadIdx.x & 63) == 0) s_red[threadIdx.x >> 6] = mx;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < kSmScanNT / 64; w++) mx = fmaxf(mx, s_red[w]);
    R.out[kRecRowMax] = mx;
  }
}

// kRecPre of every chunk: the sums before it, in any order.
__global__ __launch_bounds__(kSmScanNT) void softmax_prefix_kernel(const float* in, float* out, int n, int chunks) {
  __shared__ float s_wave[2][kSmScanNT / 64];
  const SmRow R = sm_row(in, out, n, chunks);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  float carry = 0.0f, next = tid < chunks ? R.rec(tid)[kRecSum] : 0.0f;
  for (int c0 = 0, b = 0; c0 < chunks; c0 += kSmScanNT, b ^= 1) {
    const int c = c0 + tid;
    const float inc = exact::scan_add_f32(next);
    next = c + kSmScanNT < chunks ? R.rec(c + kSmScanNT)[kRecSum] : 0.0f;
    if (lane == 63) s_wave[b][wave] = inc;
    __syncthreads();  // (the buffer of the pass before last is free again)
    const float before = __int_as_float(exact::wave_shr1(__float_as_int(inc)));  // the lane before's, 0 in lane 0
    float pre = carry;
    for (int w = 0; w < kSmScanNT / 64; w++) {
      if (w == wave && c < chunks) R.rec(c)[kRecPre] = pre + before;
      pre += s_wave[b][w];
    }
    carry = pre;
  }
}

template <bool MANY>  // the row's maximum is in the first record
__global__ __launch_bounds__(kSmNT) void softmax_sum_kernel(const float* in, float* out, int n, int chunks) {
  __shared__ float s_red[kSmNT / 64], s_sum[kSmNT / 64];
  const SmRow R = sm_row(in, out, n, chunks);
  const int c = blockIdx.x, b = R.begin(c), e = R.begin(c + 1), tid = threadIdx.x;
  float x[kSmCT], mx = -INFINITY;
#pragma unroll
  for (int u = 0; u < kSmCT; u++) x[u] = R.in[min(b + tid + kSmNT * u, e - 1)];
  if constexpr (MANY) {
    mx = R.out[kRecRowMax];
  } else {
    for (int d = tid; d < chunks; d += kSmNT) mx = fmaxf(mx, R.rec(d)[kRecMax]);
    mx = sm_block_max(mx, s_red);
  }
  float s = 0.0f;
#pragma unroll
  for (int u = 0; u < kSmCT; u++) {
    const float v = dev_expf(x[u] - mx);
    s += b + tid + kSmNT * u < e ? v : 0.0f;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
  if ((tid & 63) == 0) s_sum[tid >> 6] = s;
  __syncthreads();
  if (tid == 0) {
    R.rec(c)[kRecSum] = (s_sum[0] + s_sum[1]) + (s_sum[2] + s_sum[3]);
    if (!MANY || c > 0) R.rec(c)[kRecRowMax] = mx;
  }
}

// A lane's kSmCT consecutive exponentials of the chunk [b, b + len), zeros past it.
__device__ __forceinline__ void sm_terms(const SmRow& R, int b, int len, float mx, float (&v)[kSmCT]) {
  const int j0 = threadIdx.x * kSmCT;
#pragma unroll
  for (int i = 0; i < kSmCT; i++) v[i] = R.in[b + min(j0 + i, len - 1)];
#pragma unroll
  for (int i = 0; i < kSmCT; i++) {
    const float e = dev_expf(v[i] - mx);
    v[i] = j0 + i < len ? e : 0.0f;
  }
}

// The ordered sum of v (kSmCT consecutive terms per lane, zeros past the
// chunk) continued from the exact value s > 0: one workgroup scan per binade.
__device__ float sm_continue(float s, const float (&v)[kSmCT], int* s_wave, int* s_first, float* s_val, int* s_k) {
  const int j0 = threadIdx.x * kSmCT;
  int k = 0;
  while (k < kSmChunk) {
    int e;
    int32_t m;
    exact::decompose(s, &e, &m);
    exact::Pair pr[kSmCT], loc{0, 0};
#pragma unroll
    for (int i = 0; i < kSmCT; i++) {
      pr[i] = j0 + i >= k ? exact::term_pair_bits(__float_as_uint(v[i]), e) : exact::Pair{0, 0};
      loc = exact::compose(loc, pr[i]);
    }
    if (threadIdx.x == 0) *s_first = INT_MAX;
    exact::Pair total;
    const exact::Pair pre = exact::block_exclusive_scan<kSmNT>(loc, s_wave, &total);  // barrier
    int32_t mm = exact::apply(pre, m), mprev = 0;
    int first = INT_MAX;
    float fv = 0.0f;
#pragma unroll
    for (int i = 0; i < kSmCT; i++) {
      const int32_t m2 = exact::apply(pr[i], mm);
      if (first == INT_MAX && m2 >= (1 << 24)) {
        first = j0 + i;
        mprev = mm;
        fv = v[i];
      }
      mm = m2;
    }
    if (first != INT_MAX) atomicMin(s_first, first);
    __syncthreads();
    const int f = *s_first;
    if (f == INT_MAX ? threadIdx.x == 0 : first == f) {
      const float u = ldexpf(1.0f, e - 23);
      *s_val = f == INT_MAX ? static_cast<float>(exact::apply(total, m)) * u : static_cast<float>(mprev) * u + fv;
      *s_k = f == INT_MAX ? kSmChunk : f + 1;
    }
    __syncthreads();
    s = *s_val;
    k = *s_k;
    __syncthreads();  // before the next pass writes them
  }
  return s;
}

template <bool MANY>  // kRecPre holds the sums before the chunk
__global__ __launch_bounds__(kSmNT) void softmax_map_kernel(const float* in, float* out, int n, int chunks) {
  __shared__ float s_red[kSmNT / 64], s_pre[kSmNT / 64], s_term[exact::run_pad(kSmChunk)];
  __shared__ int s_wave[2 * (kSmNT / 64)], s_p0, s_p1, s_b1;
  const SmRow R = sm_row(in, out, n, chunks);
  const int c = blockIdx.x, b = R.begin(c), len = R.begin(c + 1) - b, tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6, j0 = tid * kSmCT;
  float v[kSmCT];
  sm_terms(R, b, len, R.rec(c)[kRecRowMax], v);
  if (c == 0) {  // the sum's start: exact from its first term
#pragma unroll
    for (int i = 0; i < kSmCT; i++) s_term[exact::run_pad(j0 + i)] = v[i];
    __syncthreads();
    const float s = exact::block_seq_sum_short<kSmNT>([](int i) { return s_term[exact::run_pad(i)]; }, len);
    if (tid == 0) R.out[kRecMap] = s;
    return;
  }
  // approximate sum before the chunk (any order), then before this lane
  float pre = 0.0f;
  if constexpr (MANY) {
    pre = tid == 0 ? R.rec(c)[kRecPre] : 0.0f;
  } else {
    for (int d = tid; d < c; d += kSmNT) pre += R.rec(d)[kRecSum];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) pre += __shfl_xor(pre, o, 64);
  }
  const float inc = exact::scan_add_f32((v[0] + v[1]) + (v[2] + v[3]));
  if (lane == 63) s_pre[wave] = inc;
  if (lane == 0) s_red[wave] = pre;
  if (tid == 0) s_p0 = INT_MAX, s_p1 = -1, s_b1 = exact::kPredAmb;
  __syncthreads();
  const float P0 = (s_red[0] + s_red[1]) + (s_red[2] + s_red[3]);
  float P = P0;
  for (int w = 0; w < wave; w++) P += s_pre[w];
  P += __int_as_float(exact::wave_shr1(__float_as_int(inc)));
  // steps that may leave the binade of the sum before them
  const int mr = exact::pred_margin(n), b0 = exact::binade_code(P0, mr);
  int ein = tid == 0 ? b0 : exact::binade_code(P, mr), ec[kSmCT];
  int lo = INT_MAX, hi = -1;
#pragma unroll
  for (int i = 0; i < kSmCT; i++) {
    P += v[i];
    ec[i] = exact::binade_code(P, mr);
    if (j0 + i < len && exact::seg_break(ec[i], ein)) {
      lo = min(lo, j0 + i);
      hi = j0 + i;
    }
    ein = ec[i];
  }
  if (lo != INT_MAX) {
    atomicMin(&s_p0, lo);
    atomicMax(&s_p1, hi);
  }
  __syncthreads();
  const int p0 = s_p0, p1 = s_p1;
#pragma unroll
  for (int i = 0; i < kSmCT; i++)
    if (j0 + i == p1) s_b1 = ec[i];
  __syncthreads();
  const int b1 = s_b1;
  exact::Pair a0{0, 0}, a1{0, 0};
#pragma unroll
  for (int i = 0; i < kSmCT; i++) {
    if (j0 + i < p0) a0 = exact::compose(a0, exact::term_pair_bits(__float_as_uint(v[i]), b0));
    if (p1 >= 0 && j0 + i > p1) a1 = exact::compose(a1, exact::term_pair_bits(__float_as_uint(v[i]), b1));
  }
  exact::Pair t0, t1;
  (void)exact::block_exclusive_scan<kSmNT>(a0, s_wave, &t0);
  __syncthreads();
  (void)exact::block_exclusive_scan<kSmNT>(a1, s_wave, &t1);
  if (tid == 0) {
    float* r = R.rec(c);
    const int cnt = p1 >= 0 ? p1 - p0 + 1 : 0;
    // (a run whose binade is not decided cannot be mapped)
    const bool ok = cnt <= kSmPlain && !(p0 > 0 && b0 == exact::kPredAmb) &&
                    !(p1 >= 0 && p1 + 1 < len && b1 == exact::kPredAmb);
    r[kRecMap] = __int_as_float(t0.e);
    r[kRecMap + 1] = __int_as_float(t0.o);
    r[kRecMap + 2] = __int_as_float(t1.e);
    r[kRecMap + 3] = __int_as_float(t1.o);
    r[kRecPlain] = __int_as_float(!ok ? kComplex : cnt ? p0 | cnt << 16 : 0);
    r[kRecB0] = __int_as_float(p0 > 0 ? b0 : exact::kPredAmb);  // kPredAmb: an empty run
    r[kRecB1] = __int_as_float(cnt && p1 + 1 < len ? b1 : exact::kPredAmb);
  }
}

// A run of additions inside binade E as its map; false when the value leaves
// or does not start in it.
__device__ __forceinline__ bool sm_apply(float& val, int E, int me, int mo) {
  if (E == exact::kPredAmb) return true;  // empty
  const float mf = ldexpf(val, 23 - E);
  const bool in = (mf < 16777216.0f) & ((E == -126) | (mf >= 8388608.0f));
  const int32_t m = exact::apply(exact::Pair{me, mo}, static_cast<int32_t>(fminf(mf, 16777216.0f)));
  if (!in || m >= (1 << 24)) return false;
  val = ldexpf(static_cast<float>(m), E - 23);
  return true;
}

// One workgroup per row. Every wave follows the same walk, 64 records at a
// time: lane l holds record c0 + l. Neighbouring records without plain
// additions and with one binade are composed by a wave scan and applied as
// one map (149 records of a 151936-value row: about twenty steps).
__global__ __launch_bounds__(kSmNT) void softmax_walk_kernel(const float* in, float* out, int n, int chunks) {
  __shared__ __align__(16) float s_plain[kSmSlots][kSmPlain];
  __shared__ int s_wave[2 * (kSmNT / 64)], s_first, s_k;
  __shared__ float s_val;
  const SmRow R = sm_row(in, out, n, chunks);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const float mx = R.out[kRecRowMax];
  float val = R.out[kRecMap];
  bool good = val <= 3.4028234663852886e38f;  // a NaN exponential (a NaN or +inf input) makes the sum NaN
  int rec[7];
  float sum = 0.0f;
  auto load = [&](int c0) {
    const float* r = R.rec(min(c0 + lane, chunks - 1));
    sum = r[kRecSum];
#pragma unroll
    for (int w = 0; w < 7; w++) rec[w] = __float_as_int(r[kRecMap + w]);
  };
  load(1);
  for (int c0 = 1; c0 < chunks && good; c0 += 64) {
    const int nc = min(64, chunks - c0);
    good = __builtin_amdgcn_ballot_w64(!(sum <= 3.4028234663852886e38f)) == 0;  // (lanes past nc repeat the last record)
    int cur[7];
#pragma unroll
    for (int w = 0; w < 7; w++) cur[w] = rec[w];
    const int plain = cur[kRecPlain - kRecMap], B0 = cur[kRecB0 - kRecMap];
    const uint64_t listed = __builtin_amdgcn_ballot_w64(lane < nc && plain > 0 && plain < kComplex);
    // runs of records that one map covers: those after `starts` up to the next start
    const int prevB = exact::wave_shr1(B0), prevPlain = exact::wave_shr1(plain);
    const bool start = lane == 0 || lane >= nc || plain != 0 || prevPlain != 0 || B0 != prevB;
    const exact::SegAcc run = exact::scan_seg(exact::SegAcc{exact::Pair{cur[0], cur[1]}, start ? 1 : 0});
    const uint64_t starts = __builtin_amdgcn_ballot_w64(start);
    if (c0 + 64 < chunks) load(c0 + 64);
    __syncthreads();  // the slots of the last 64 records are read
    {
      uint64_t m = listed;
      for (int s = 0; m && s < kSmSlots; s++, m &= m - 1) {
        if ((s & (kSmNT / 64 - 1)) != wave) continue;
        const int l = __builtin_ctzll(m), pl = __builtin_amdgcn_readlane(plain, l), cnt = pl >> 16;
        const int at = R.begin(c0 + l) + (pl & 0xffff);
        for (int u = lane; u < kSmPlain; u += 64) s_plain[s][u] = u < cnt ? dev_expf(R.in[at + u] - mx) : 0.0f;
      }
    }
    __syncthreads();
    int t = 0, single = 0;  // records before `single` are taken one by one
    while (t < nc && good) {
      auto get = [&](int w) { return __builtin_amdgcn_readlane(cur[w - kRecMap], t); };
      const int pl = get(kRecPlain);
      const float before = val;
      if (pl == 0 && t >= single) {  // t starts a run
        const uint64_t later = t < 63 ? starts >> (t + 1) << (t + 1) : 0;
        const int end = later ? __builtin_ctzll(later) : nc;
        if (sm_apply(val, get(kRecB0), __builtin_amdgcn_readlane(run.p.e, end - 1),
                     __builtin_amdgcn_readlane(run.p.o, end - 1))) {
          t = end;
          continue;
        }
        single = end;
      }
      bool ok = pl < kComplex && sm_apply(val, get(kRecB0), get(kRecMap), get(kRecMap + 1));
      if (ok && pl) {
        const int slot = __builtin_popcountll(listed & ((uint64_t{1} << t) - 1)), cnt = pl >> 16;
        if (slot < kSmSlots) {
          const float4* x = reinterpret_cast<const float4*>(s_plain[slot]);
          for (int u = 0; u < cnt; u += 16) {  // (zeros past cnt)
            const float4 y[4] = {x[u / 4], x[u / 4 + 1], x[u / 4 + 2], x[u / 4 + 3]};
#pragma unroll
            for (int k = 0; k < 4; k++) {
              val += y[k].x;
              val += y[k].y;
              val += y[k].z;
              val += y[k].w;
            }
          }
        } else {
          const int at = R.begin(c0 + t) + (pl & 0xffff);
          for (int u = 0; u < cnt; u++) val += dev_expf(R.in[at + u] - mx);
        }
        ok = sm_apply(val, get(kRecB1), get(kRecMap + 2), get(kRecMap + 3));
      }
      if (!ok) {  // (the same in every wave)
        const int b = R.begin(c0 + t), len = R.begin(c0 + t + 1) - b;
        float v[kSmCT];
        sm_terms(R, b, len, mx, v);
        val = sm_continue(before, v, s_wave, &s_first, &s_val, &s_k);
      }
      t++;
    }
  }
  const float inv = good && val > 0.0f ? 1.0f / val : 0.0f;
  for (int c = tid; c < chunks; c += kSmNT) R.rec(c)[kRecInv] = inv;
}

__global__ __launch_bounds__(kSmNT) void softmax_scale_kernel(const float* in, float* out, int n, int chunks) {
  const SmRow R = sm_row(in, out, n, chunks);
  const int c = blockIdx.x, b = R.begin(c), e = R.begin(c + 1), tid = threadIdx.x;
  float x[kSmCT];
#pragma unroll
  for (int u = 0; u < kSmCT; u++) x[u] = R.in[min(b + tid + kSmNT * u, e - 1)];
  const float mx = R.out[b + kRecRowMax], inv = R.out[b + kRecInv];
  __syncthreads();  // every lane has read the record
#pragma unroll
  for (int u = 0; u < kSmCT; u++) {
    const int i = b + tid + kSmNT * u;
    if (i < e) R.out[i] = dev_expf(x[u] - mx) * inv;
  }
}

// Chunks from which a row has launches of its own for its maximum and the sums
// before each chunk: 1 x 4M values 261 -> 199 us, 3 x 4M 491 -> 285, 1 x 17M 4.1 -> 2.5
// ms, 1 x 67M 76 -> 40 ms (3554 on the one-workgroup kernel); with fewer the two
// launches cost as much as they save (1 x 800000 56 against 59, 1 x 1000000 60
// against 62, 3 x 1000000 87 against 82).
constexpr int kSmMany = 1000;

// Rows of n values that the chunked launches take at most. They read the input
// five times and evaluate each exponential three times, so many rows, which
// fill the chip on one workgroup each, are the short kernel's: 64 rows of 8000
// 31 (chunked) against 36 us, 256 rows 43 against 36; 192 rows of 11000 0.94
// of its time, 256 1.14; 768 rows of 12000 0.96, 2048 1.15; 1 row of 7168 18
// against 24 us. From 13000 values on all rows are chunked: 1024 rows 0.95-0.98,
// 2048 1.05-1.14, 3000 0.89-0.96, and the short kernel folds a row whose
// predicted scan fails, or of more than 16416 values, in a pass per binade (1024
// rows of 16400 152 against 1130 us, of 32000 265 against 2434).
size_t long_rows(size_t n) {
  if (n < 7168) return 0;
  return n < 8000 ? 64 : n < 10000 ? 96 : n < 12000 ? 192 : n < 13000 ? 768 : 65535;
}

}  // namespace

int launch_softmax(const float* in, size_t rows, size_t n, float* out, hipStream_t s) {
  if (rows == 0 || n == 0) return kOk;
  const float *in1 = in + rows * n, *out1 = out + rows * n;
  const bool overlap = in < out1 && out < in1;
  if (rows > long_rows(n) || n > static_cast<size_t>(INT_MAX) / 2 || overlap) {
    hipLaunchKernelGGL(softmax_kernel, dim3(rows), dim3(256), 0, s, in, (int)n, out);
    PRANA_LAUNCH_CHECK();
    return kOk;
  }
  const size_t chunks = (n + kSmChunk - 1) / kSmChunk;
  const dim3 grid(chunks, rows), nt(kSmNT);
  const int ni = static_cast<int>(n), nc = static_cast<int>(chunks);
  hipLaunchKernelGGL(softmax_max_kernel, grid, nt, 0, s, in, out, ni, nc);
  if (nc > kSmMany) {
    hipLaunchKernelGGL(softmax_row_max_kernel, dim3(1, rows), dim3(kSmScanNT), 0, s, in, out, ni, nc);
    hipLaunchKernelGGL(softmax_sum_kernel<true>, grid, nt, 0, s, in, out, ni, nc);
    hipLaunchKernelGGL(softmax_prefix_kernel, dim3(1, rows), dim3(kSmScanNT), 0, s, in, out, ni, nc);
    hipLaunchKernelGGL(softmax_map_kernel<true>, grid, nt, 0, s, in, out, ni, nc);
  } else {
    hipLaunchKernelGGL(softmax_sum_kernel<false>, grid, nt, 0, s, in, out, ni, nc);
    hipLaunchKernelGGL(softmax_map_kernel<false>, grid, nt, 0, s, in, out, ni, nc);
  }
  hipLaunchKernelGGL(softmax_walk_kernel, dim3(1, rows), nt, 0, s, in, out, ni, nc);
  hipLaunchKernelGGL(softmax_scale_kernel, grid, nt, 0, s, in, out, ni, nc);
  PRANA_LAUNCH_CHECK();
  return kOk;
}

}  // namespace prana

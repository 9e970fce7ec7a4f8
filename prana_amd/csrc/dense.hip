// Dense f32 matrices: dot_f32_scalar (matmul.rs:377-391) for every (token,
// row). Four strided partial sums (class l adds x[4i+l]*w[4i+l] over i from
// 0.0, products and sums rounded separately), combined ((a0+a1)+a2)+a3, then
// the tail of cols % 4 elements. The four classes are independent chains, so
// the kernels keep them in separate lanes. Those for a few tokens and for
// batches stage x and w in LDS class by class: four consecutive terms of a
// chain are one 16-byte read. Chunks are zero-padded past cols/4: adding +0.0
// leaves a chain (started from +0.0) unchanged.
#include "common.h"
#include "kernels.h"

namespace prana {

namespace {

typedef float f4 __attribute__((ext_vector_type(4)));  // (arrays of these stay in registers)

__device__ __forceinline__ void store_dense(const GemvOut& o, size_t tok, size_t r, float acc) {
  float* dst = o.out + tok * o.ldo + r;
  if (o.residual)
    *dst = *dst + acc;
  else if (o.bias)
    *dst = acc + o.bias[r];
  else
    *dst = acc;
}

// Elements 4i..4i+3 of a row, zeros from quad nq on. VEC: rows are 16-byte
// aligned (cols % 4 == 0 and an aligned base).
template <bool VEC>
__device__ __forceinline__ f4 load_quad(const float* row, int i, int nq) {
  const int j = i < nq ? i : nq - 1;  // in bounds
  f4 v;
  if constexpr (VEC) {
    v = *reinterpret_cast<const f4*>(row + 4 * j);
  } else {
    v = f4{row[4 * j], row[4 * j + 1], row[4 * j + 2], row[4 * j + 3]};
  }
  return i < nq ? v : f4{0, 0, 0, 0};
}

// ---------------------------------------------------------------- narrow rows
// One lane per class and row, operands read from memory (a row is a cache line
// or a few): no staging to wait for. Bound by launch and load latency.
__global__ __launch_bounds__(256) void gemv_f32_narrow_kernel(const float* __restrict__ w, int rows, int cols,
                                                              const float* __restrict__ x, GemvOut o) {
  __shared__ float part[256];
  const int tok = blockIdx.y, l = threadIdx.x & 3;
  const size_t r = (size_t)blockIdx.x * 64 + (threadIdx.x >> 2);
  const float* xr = x + (size_t)tok * cols;
  const float* wr = w + r * cols;
  float acc = 0.0f;
  if (r < static_cast<size_t>(rows))
    for (int i = 0; i < cols / 4; i++) acc += xr[i * 4 + l] * wr[i * 4 + l];
  part[threadIdx.x] = acc;
  __syncthreads();
  if (l == 0 && r < static_cast<size_t>(rows)) {
    float sum = part[threadIdx.x] + part[threadIdx.x + 1] + part[threadIdx.x + 2] + part[threadIdx.x + 3];
    for (int i = cols / 4 * 4; i < cols; i++) sum += xr[i] * wr[i];
    store_dense(o, tok, r, sum);
  }
}

// Short rows give the staging kernels one part-filled chunk and nothing to read
// ahead, so little work is done sooner without it (staged against this
// kernel): 32000 x 24 at one token 7.4 against 3.5 us, at 8 8.7 against 6.6, 4096 x
// 17 at 20 4.8 against 3.6, 1000 x 40 at 300 10.4 against 6.8, and one token over
// many rows up to 200 columns (32000 x 192 8.7 against 6.2, 256 9.2 against 8.9).
// The line falls as rows leave the cache line (10000 x 24 at 40 6.2 against 9.4, x
// 55 at 8 5.3 against 7.1); rows below four columns are staged by nothing
// (32000 x 1 at 8 3.8 against 3.4, at 40 6.8 against 9.5).
bool narrow_takes(size_t rows, size_t cols, size_t n_tok) {
  if (n_tok == 1 && rows >= 16000 && cols <= (rows >= 24000 ? 200u : 140u)) return true;
  if (n_tok == 2 && rows >= 16000 && rows <= 40000 && cols <= 110) return true;
  const size_t most = cols < 4 ? (n_tok <= 16 ? 3600000 : 2000000)
                      : cols <= 17 ? 26000000
                      : cols <= 24 ? (n_tok <= 16 ? 15000000 : 9000000)
                      : n_tok <= 4 ? 6000000
                      : rows > 5000 ? 3200000
                      : rows < 1000 ? 4000000
                      : cols <= 56 ? 13500000 : 6000000;
  return cols < 96 && n_tok <= 65535 && rows * n_tok * (cols + 4) <= most;
}

// ---------------------------------------------------------------- a few tokens
// One workgroup per 16 rows; the chunk of 256 elements of every row is loaded
// by all lanes, coalesced, three chunks ahead. Lane (row, l) of wave w then folds
// class l of its row for tokens w, w+4, ...: at one token wave 0 folds while
// the others only load. Bound by the weight stream; a lane's chain is cols/4
// dependent additions (~4.5 us at 4096 columns) under it. 4096 x 4096: 18 us
// at one token, 25 at 8 (112 and 113 with a lane per class and row that read
// its operands from memory; 25 and 33 with one chunk in flight instead of
// three).
constexpr int kDvNT = 256;
constexpr int kDvRows = 16;
constexpr int kDvQ = 64;           // quads (groups of four elements) per chunk
constexpr int kDvS = kDvQ + 4;     // padded chain: neighbouring lanes' 16-byte reads fall on different banks
constexpr int kDvMaxTok = 16;
constexpr size_t kDvMaxJobs = 400;  // (tiles of 16 tokens x 64 rows)

template <int TPW, bool VEC>  // tokens per wave: up to 4 * TPW tokens
__global__ __launch_bounds__(kDvNT) void gemv_f32_kernel(const float* __restrict__ w, int rows, int cols,
                                                         const float* __restrict__ x, int n_tok, GemvOut o) {
  constexpr int XROWS = 4 * TPW;
  __shared__ __align__(16) float s_w[2][kDvRows * 4 * kDvS];
  __shared__ __align__(16) float s_x[2][XROWS * 4 * kDvS];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r0 = blockIdx.x * kDvRows, t0 = blockIdx.y * XROWS;
  const int nq = cols / 4, n_ch = (nq + kDvQ - 1) / kDvQ;
  struct Regs {
    f4 w[kDvRows / 4], x[TPW];
  };
  // (loads past the last chunk read the last quad: the loop stays straight)
  auto load = [&](Regs& g, int c) __attribute__((always_inline)) {  // wave v takes rows v, v+4, ..., tokens likewise
#pragma unroll
    for (int u = 0; u < kDvRows / 4; u++)
      g.w[u] = load_quad<VEC>(w + (size_t)min(r0 + 4 * u + wave, rows - 1) * cols, c * kDvQ + lane, nq);
#pragma unroll
    for (int u = 0; u < TPW; u++)
      g.x[u] = load_quad<VEC>(x + (size_t)min(t0 + 4 * u + wave, n_tok - 1) * cols, c * kDvQ + lane, nq);
  };
  auto store = [&](const Regs& g, int b) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < kDvRows / 4; u++)
#pragma unroll
      for (int l = 0; l < 4; l++) s_w[b][((4 * u + wave) * 4 + l) * kDvS + lane] = g.w[u][l];
#pragma unroll
    for (int u = 0; u < TPW; u++)
#pragma unroll
      for (int l = 0; l < 4; l++) s_x[b][((4 * u + wave) * 4 + l) * kDvS + lane] = g.x[u][l];
  };
  float acc[TPW];
#pragma unroll
  for (int t = 0; t < TPW; t++) acc[t] = 0.0f;
  auto fold = [&](int c) __attribute__((always_inline)) {
    if (t0 + wave >= n_tok) return;  // uniform per wave
    const f4* wp = reinterpret_cast<const f4*>(s_w[c & 1] + lane * kDvS);
    const f4* xp = reinterpret_cast<const f4*>(s_x[c & 1] + (wave * 4 + (lane & 3)) * kDvS);
    const int ng = min(kDvQ / 4, (nq - c * kDvQ + 3) / 4);
#pragma unroll 4
    for (int g = 0; g < ng; g++) {
      const f4 a = wp[g];
#pragma unroll
      for (int t = 0; t < TPW; t++) {
        const f4 b = xp[t * 4 * kDvS + g];  // token wave + 4t: 16 chains further on
#pragma unroll
        for (int j = 0; j < 4; j++) acc[t] += b[j] * a[j];
      }
    }
  };
  if (n_ch > 0) {
    Regs g0, g1, g2;
    load(g0, 0);
    load(g1, 1);
    load(g2, 2);
    store(g0, 0);
    __syncthreads();
    for (int c = 0;; c += 3) {  // chunk c + 1 sits in g1, c + 2 in g2
      load(g0, c + 3);
      fold(c);
      if (c + 1 >= n_ch) break;
      store(g1, (c + 1) & 1);
      __syncthreads();
      load(g1, c + 4);
      fold(c + 1);
      if (c + 2 >= n_ch) break;
      store(g2, c & 1);
      __syncthreads();
      load(g2, c + 5);
      fold(c + 2);
      if (c + 3 >= n_ch) break;
      store(g0, (c + 1) & 1);
      __syncthreads();
    }
  }
  const int r = r0 + lane / 4;
#pragma unroll
  for (int t = 0; t < TPW; t++) {
    const int tok = t0 + wave + 4 * t;
    const float a0 = __shfl(acc[t], lane & ~3, 64), a1 = __shfl(acc[t], (lane & ~3) + 1, 64),
                a2 = __shfl(acc[t], (lane & ~3) + 2, 64), a3 = __shfl(acc[t], (lane & ~3) + 3, 64);
    if ((lane & 3) == 0 && r < rows && tok < n_tok) {
      float sum = a0 + a1 + a2 + a3;
      for (int i = 4 * nq; i < cols; i++) sum += x[(size_t)tok * cols + i] * w[(size_t)r * cols + i];
      store_dense(o, tok, r, sum);
    }
  }
}

// ---------------------------------------------------------------- batches
// One workgroup per TT tokens x 64 rows; wave l owns class l, each lane TT/8
// tokens x 8 rows of it: TT/8 + 8 16-byte LDS reads feed TT*8 vector
// operations. Chunks of 64 elements, loaded two ahead. Bound by the vector
// ALU (two operations per product): 4096 x 4096 over 512 tokens runs at 47
// Tops/s of the 65-68 that many independent chains reach on this card. 2048 x
// 2048 over 301 tokens: 86 us, 706 with a lane per class and row reading both
// operands from memory. Reading LDS further ahead (a full unroll of the
// chunk, 220 registers) is faster with one workgroup per compute unit and
// slower with more (512 tokens: 640 against 339 us).
constexpr int kDmNT = 256;
constexpr int kDmRows = 64;
constexpr int kDmQ = 16;        // quads per chunk
constexpr int kDmS = kDmQ + 4;  // padded chain

template <int TT, bool VEC>
__global__ __launch_bounds__(kDmNT) void gemm_f32_kernel(const float* __restrict__ w, int rows, int cols,
                                                         const float* __restrict__ x, int n_tok, GemvOut o) {
  constexpr int TL = TT / 8, WLD = kDmRows * kDmQ / kDmNT, XLD = TT * kDmQ / kDmNT;
  constexpr int WF = 4 * kDmRows * kDmS, XF = 4 * TT * kDmS;
  static_assert(2 * (WF + XF) >= 4 * TT * (kDmRows + 1), "the classes' sums fit the staging buffers");
  __shared__ __align__(16) float smem[2 * (WF + XF)];
  const int tid = threadIdx.x, lane = tid & 63;
  const int l = __builtin_amdgcn_readfirstlane(tid >> 6);  // this wave's class
  const int r0 = blockIdx.x * kDmRows, t0 = blockIdx.y * TT;
  const int nq = cols / 4, n_ch = (nq + kDmQ - 1) / kDmQ;
  struct Regs {
    f4 w[WLD], x[XLD];
  };
  auto load = [&](Regs& g, int c) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < WLD; u++) {
      const int e = tid + kDmNT * u;
      g.w[u] = load_quad<VEC>(w + (size_t)min(r0 + e / kDmQ, rows - 1) * cols, c * kDmQ + e % kDmQ, nq);
    }
#pragma unroll
    for (int u = 0; u < XLD; u++) {
      const int e = tid + kDmNT * u;
      g.x[u] = load_quad<VEC>(x + (size_t)min(t0 + e / kDmQ, n_tok - 1) * cols, c * kDmQ + e % kDmQ, nq);
    }
  };
  auto store = [&](const Regs& g, int b) __attribute__((always_inline)) {
    float* sw = smem + b * (WF + XF);
    float* sx = sw + WF;
#pragma unroll
    for (int u = 0; u < WLD; u++) {
      const int e = tid + kDmNT * u;
#pragma unroll
      for (int k = 0; k < 4; k++) sw[(k * kDmRows + e / kDmQ) * kDmS + e % kDmQ] = g.w[u][k];
    }
#pragma unroll
    for (int u = 0; u < XLD; u++) {
      const int e = tid + kDmNT * u;
#pragma unroll
      for (int k = 0; k < 4; k++) sx[(k * TT + e / kDmQ) * kDmS + e % kDmQ] = g.x[u][k];
    }
  };
  const int rg = lane & 7, tg = lane >> 3;  // rows rg + 8j, tokens tg + 8i
  float acc[TL][8];
#pragma unroll
  for (int i = 0; i < TL; i++)
#pragma unroll
    for (int j = 0; j < 8; j++) acc[i][j] = 0.0f;
  auto compute = [&](int c) __attribute__((always_inline)) {
    const float* sw = smem + (c & 1) * (WF + XF) + (l * kDmRows + rg) * kDmS;
    const float* sx = smem + (c & 1) * (WF + XF) + WF + (l * TT + tg) * kDmS;
#pragma unroll 2
    for (int g = 0; g < kDmQ / 4; g++) {
      f4 b[TL];
#pragma unroll
      for (int i = 0; i < TL; i++) b[i] = *reinterpret_cast<const f4*>(sx + 8 * i * kDmS + 4 * g);
#pragma unroll
      for (int j = 0; j < 8; j++) {
        const f4 a = *reinterpret_cast<const f4*>(sw + 8 * j * kDmS + 4 * g);
#pragma unroll
        for (int k = 0; k < 4; k++)
#pragma unroll
          for (int i = 0; i < TL; i++) acc[i][j] += b[i][k] * a[k];
      }
    }
  };
  if (n_ch > 0) {
    Regs g0, g1;
    load(g0, 0);
    load(g1, 1);
    store(g0, 0);
    __syncthreads();
    for (int c = 0;; c += 2) {  // chunk c + 1 sits in g1
      load(g0, c + 2);
      compute(c);
      if (c + 1 >= n_ch) break;
      store(g1, 1);
      __syncthreads();
      load(g1, c + 3);
      compute(c + 1);
      if (c + 2 >= n_ch) break;
      store(g0, 0);
      __syncthreads();
    }
  }
  __syncthreads();
  // the four classes' sums meet in LDS: [class][token][row]
#pragma unroll
  for (int i = 0; i < TL; i++)
#pragma unroll
    for (int j = 0; j < 8; j++) smem[(l * TT + tg + 8 * i) * (kDmRows + 1) + rg + 8 * j] = acc[i][j];
  __syncthreads();
  for (int e = tid; e < TT * kDmRows; e += kDmNT) {
    const int t = e / kDmRows, r = e % kDmRows;
    if (t0 + t >= n_tok || r0 + r >= rows) continue;
    const float* p = smem + t * (kDmRows + 1) + r;
    constexpr int CS = TT * (kDmRows + 1);
    float sum = p[0] + p[CS] + p[2 * CS] + p[3 * CS];
    for (int i = 4 * nq; i < cols; i++) sum += x[(size_t)(t0 + t) * cols + i] * w[(size_t)(r0 + r) * cols + i];
    store_dense(o, t0 + t, r0 + r, sum);
  }
}

template <bool VEC>
int launch_dense(const float* w, int rows, int cols, const float* x, int n_tok, const GemvOut& o, hipStream_t s) {
  if (narrow_takes(rows, cols, n_tok)) {
    hipLaunchKernelGGL(gemv_f32_narrow_kernel, dim3((rows + 63) / 64, n_tok), dim3(256), 0, s, w, rows, cols, x, o);
    PRANA_LAUNCH_CHECK();
    return kOk;
  }
  const size_t rt = (rows + kDmRows - 1) / kDmRows;
  auto jobs = [&](size_t tt) { return rt * ((n_tok + tt - 1) / tt); };
  // Larger batches with few tiles run as groups of eight tokens (4096 x 4096
  // at 64 tokens 89 against 161 us on the batch kernel, 100 x 8000 at 64 tokens
  // 43 against 240; at 128 tokens the batch kernel's 151 us are less).
  if (n_tok <= kDvMaxTok || jobs(16) < kDvMaxJobs) {
    const unsigned rg = (rows + kDvRows - 1) / kDvRows;
    const dim3 nt(kDvNT);
    auto grid = [&](unsigned tt) { return dim3(rg, (n_tok + tt - 1) / tt); };
    if (n_tok <= 4)
      hipLaunchKernelGGL((gemv_f32_kernel<1, VEC>), grid(4), nt, 0, s, w, rows, cols, x, n_tok, o);
    else if (n_tok <= 8 || n_tok > kDvMaxTok)
      hipLaunchKernelGGL((gemv_f32_kernel<2, VEC>), grid(8), nt, 0, s, w, rows, cols, x, n_tok, o);
    else
      hipLaunchKernelGGL((gemv_f32_kernel<4, VEC>), grid(16), nt, 0, s, w, rows, cols, x, n_tok, o);
    PRANA_LAUNCH_CHECK();
    return kOk;
  }
  const dim3 nt(kDmNT);
  if (jobs(64) >= 512)
    hipLaunchKernelGGL((gemm_f32_kernel<64, VEC>), dim3(rt, (n_tok + 63) / 64), nt, 0, s, w, rows, cols, x, n_tok, o);
  else if (jobs(32) >= 512)
    hipLaunchKernelGGL((gemm_f32_kernel<32, VEC>), dim3(rt, (n_tok + 31) / 32), nt, 0, s, w, rows, cols, x, n_tok, o);
  else
    hipLaunchKernelGGL((gemm_f32_kernel<16, VEC>), dim3(rt, (n_tok + 15) / 16), nt, 0, s, w, rows, cols, x, n_tok, o);
  PRANA_LAUNCH_CHECK();
  return kOk;
}

}  // namespace

int launch_gemv_f32(const DevMat& m, const float* x, size_t n_tok, const GemvOut& o, hipStream_t s) {
  PRANA_CHECK(x != nullptr, "gemv f32: dense activations required");
  PRANA_CHECK(m.rows <= INT32_MAX - 64u && m.cols <= INT32_MAX - 64u && n_tok <= (1u << 20), "gemv f32: shape out of range");
  const float* w = reinterpret_cast<const float*>(m.qs);
  const bool vec = m.cols % 4 == 0 && reinterpret_cast<uintptr_t>(x) % 16 == 0 && reinterpret_cast<uintptr_t>(w) % 16 == 0;
  const int rows = static_cast<int>(m.rows), cols = static_cast<int>(m.cols), n = static_cast<int>(n_tok);
  return vec ? launch_dense<true>(w, rows, cols, x, n, o, s) : launch_dense<false>(w, rows, cols, x, n, o, s);
}

}  // namespace prana

// Prefill attention (attention.rs:236-284) over the f32 K/V of a prompt as
// two register-tiled products around a softmax, in the reference's exact
// evaluation order:
//   score_t = (fold_d q[d]*k_t[d] from -0.0) * (1/sqrt(hd))
//   e_t = expf(score_t - max), sum = fold_t e_t, p_t = e_t * (1/sum)
//   out[d] = fold_t p_t * v_t[d] from 0.0
// Products and sums round separately (no FMA), so both products run on the
// vector ALU at two operations per (row, key, dim), which is what bounds the
// kernel; the tiling exists to keep the operand reads below that.
//
// One 256-lane workgroup takes one head's block of BQ consecutive query rows
// through three phases:
//   1. scores. Tiles of 8192/BQ keys, 8 rows x 4 keys per lane (BQ = 16: 256
//      keys, 4 rows x 4 keys): twelve 16-byte LDS reads (q rows broadcast) per 4
//      dims feed 256 vector operations (16: eight and 128). K is staged 16 KB
//      at a time, one stage ahead. Scores go to the workgroup's slot of
//      global scratch (they stay in the caches).
//   2. softmax. All lanes turn a tile's scores into exponentials (back to the
//      slot, and to LDS); one wave then folds the previous tile's
//      exponentials with one lane per query row, so the left-to-right sums of
//      all BQ rows run side by side at one addition per term. Waves take the
//      tiles in turn.
//   3. P.V. Tiles of 32 keys of p (formed as e * inv on the way in) and V in
//      LDS; each lane owns RT rows x 4*DW dims and folds key after key.
// Workgroups take several blocks each, longest first and then in alternating
// order, so that all of them cover about the same number of keys; when the
// heads divide by 8, an XCD works on whole heads and shares their K and V in
// its L2.
//
// Measured (one MI355X, one call): 14 heads x 64 dims at 2048 positions 275
// us and at 3001 505 us, 32 heads x 128 at 2048 963 us; the kernels before
// took 550 (eight query rows per workgroup, one key row gathered per lane),
// 5590 and 1760. At 32 x 128 x 2048 the counters show 1.09 vector instructions
// per SIMD and four cycles (two waves can issue together; a probe of
// independent operations reaches 1.9), 15 % of them not products or sums of
// the two contractions (the causal diagonal, exponentials, addresses), and
// waves waiting for memory and barriers 31 % of their time.
#include <algorithm>

#include "common.h"
#include "kernels.h"

namespace prana {

namespace {

typedef float f4 __attribute__((ext_vector_type(4)));  // (arrays of these stay in registers)
typedef f4 f4_any __attribute__((aligned(4)));         // the same 16-byte load from any f32 address

constexpr int kPtNT = 256;
constexpr int kPtTK = 256;      // keys of the longest score tile
constexpr int kPtVK = 32;       // keys per P.V tile
constexpr int kPtCus = 256;      // compute units

template <int BQ, int HDP>
struct PtCfg {
  static constexpr int RL = BQ >= 32 ? 8 : 4;      // query rows per lane (scores), each with 4 keys
  static constexpr int TK = 1024 * RL / BQ;        // keys per score tile
  static constexpr int DC = 4096 / TK;             // dims per staged K chunk
  static constexpr int KL = TK / 4;                // lanes across a score tile's keys
  static constexpr int TE = 4096 / BQ;             // keys per softmax tile
  static constexpr int ES = TE + 4;                // padded row of exponentials
  static constexpr int ELD = 4;                    // float4 words per lane and softmax tile
  static constexpr int DW = BQ * HDP / (256 * 16) > 1 ? BQ * HDP / (256 * 16) : 1;  // float4 dims per lane (P.V)
  static constexpr int COLS = HDP / 4 / DW;        // lanes across the head's dims
  static constexpr int RT = BQ * COLS / kPtNT;     // query rows per lane (P.V)
  static constexpr int PS = BQ + 4;                // padded probability row of one key
  static constexpr int VLD = kPtVK * HDP / 4 / kPtNT;
  static constexpr int PLD = (BQ * kPtVK / 4 + kPtNT - 1) / kPtNT;
  static constexpr int K_FLOATS = 2 * TK * DC, KQ_FLOATS = K_FLOATS + BQ * (HDP + 4);
  static constexpr int E_FLOATS = 2 * BQ * ES;
  static constexpr int P_FLOATS = 2 * kPtVK * (HDP + PS);
  static constexpr int FLOATS = KQ_FLOATS > E_FLOATS ? (KQ_FLOATS > P_FLOATS ? KQ_FLOATS : P_FLOATS)
                                                     : (E_FLOATS > P_FLOATS ? E_FLOATS : P_FLOATS);
  static_assert(kPtNT % COLS == 0 && (RT == 1 || RT == 2 || RT == 4) && RT * (kPtNT / COLS) == BQ, "whole lane tiles");
  static_assert(BQ * TE / 4 == ELD * kPtNT && VLD >= 1 && PLD >= 1, "whole words per lane");
};

__host__ __device__ constexpr size_t pt_stride(size_t seq) { return (seq + kPtTK - 1) / kPtTK * kPtTK; }

// scratch: gridDim.x slots of BQ rows of sstride floats. nx: 8 when heads are
// dealt to the XCDs, else 1 (gridDim.x is a multiple of nx).
template <int BQ, int HDP, int WPC>
__global__ __launch_bounds__(kPtNT, WPC) void attn_prefill_tile(const float* __restrict__ q, const float* __restrict__ k,
                                                           const float* __restrict__ v, int seq, int n_heads,
                                                           int group, int hd, float* __restrict__ out,
                                                           float* __restrict__ scratch, int sstride,
                                                           int8_t* __restrict__ qd, float* __restrict__ qsa,
                                                           int* __restrict__ qsum, int nx) {
  using C = PtCfg<BQ, HDP>;
  __shared__ __align__(16) float smem[C::FLOATS];
  __shared__ float s_mx[BQ], s_sum[BQ], s_inv[BQ];
  __shared__ uint64_t s_tab[32];  // expf's table
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kv_dim = (n_heads / group) * hd;
  const int nqb = (seq + BQ - 1) / BQ;
  const int hpx = n_heads / nx;  // heads of this workgroup's share
  const int xw = blockIdx.x % nx, wl = blockIdx.x / nx, nwl = gridDim.x / nx;
  const int jobs = nqb * hpx;
  float* slot = scratch + (size_t)blockIdx.x * BQ * sstride;
  const float scale = 1.0f / sqrtf(static_cast<float>(hd));
  if (tid < 32) s_tab[tid] = kExp2Tab[tid];  // read after phase 1's barriers

  for (int round = 0;; round++) {
    // job order: the longest blocks first, heads fastest; odd rounds reversed
    const int job = round * nwl + ((round & 1) ? nwl - 1 - wl : wl);
    if (round * nwl >= jobs) break;  // uniform over the share
    if (job >= jobs) continue;
    const int h = xw * hpx + job % hpx;
    const int i0 = (nqb - 1 - job / hpx) * BQ;
    const int nk = min(i0 + BQ, seq);  // keys any row of the block attends
    const float* kh = k + (size_t)(h / group) * hd;
    const float* vh = v + (size_t)(h / group) * hd;

    // ---- 1. scores
    {
      const int n_kt = (nk + C::TK - 1) / C::TK;
      const int n_dc = (hd + C::DC - 1) / C::DC;
      const int n_st = n_kt * n_dc;
      constexpr int D4 = C::DC / 4;
      f4* kbuf = reinterpret_cast<f4*>(smem);  // [2][D4][TK], keys swizzled by the dim word's parity
      float* qbuf = smem + C::K_FLOATS;                // [BQ][qs]
      const int qs = hd + 4;
      for (int e = tid; e < BQ * (hd / 4); e += kPtNT) {
        const int r = e / (hd / 4), d = 4 * (e % (hd / 4));  // rows past seq repeat the last one (not used)
        *reinterpret_cast<f4*>(qbuf + r * qs + d) =
            *reinterpret_cast<const f4*>(q + ((size_t)min(i0 + r, seq - 1) * n_heads + h) * hd + d);
      }
      f4 kr[4];
      auto load = [&](int kt, int dc) {
#pragma unroll
        for (int u = 0; u < 4; u++) {
          const int idx = tid + kPtNT * u, key = idx / D4, d = dc * C::DC + 4 * (idx % D4);
          // keys past nk and dims past hd read valid words that no result uses
          kr[u] = *reinterpret_cast<const f4*>(kh + (size_t)min(kt * C::TK + key, nk - 1) * kv_dim +
                                                   min(d, hd - 4));
        }
      };
      auto store = [&](int buf) {
#pragma unroll
        for (int u = 0; u < 4; u++) {
          const int idx = tid + kPtNT * u, key = idx / D4, d4 = idx % D4;
          kbuf[(buf * D4 + d4) * C::TK + (key ^ ((d4 & 1) << 3))] = kr[u];
        }
      };
      const int kl = tid % C::KL, rg = tid / C::KL * C::RL;  // this lane's keys kl + KL*c and rows rg..
      float mx[C::RL], acc[C::RL][4];
#pragma unroll
      for (int r = 0; r < C::RL; r++) mx[r] = -INFINITY;
      load(0, 0);
      store(0);
      __syncthreads();
      int kt = 0, dc = 0;
      for (int st = 0; st < n_st; st++) {
        const int dc1 = dc + 1 < n_dc ? dc + 1 : 0, kt1 = dc + 1 < n_dc ? kt : kt + 1;
        if (st + 1 < n_st) load(kt1, dc1);
        if (dc == 0) {
#pragma unroll
          for (int r = 0; r < C::RL; r++)
#pragma unroll
            for (int c = 0; c < 4; c++) acc[r][c] = -0.0f;
        }
        const f4* kb = kbuf + (st & 1) * D4 * C::TK;
        const float* qb = qbuf + rg * qs + dc * C::DC;
        const int nd4 = min(C::DC, hd - dc * C::DC) / 4;  // uniform
        const int live = (nk - kt * C::TK + C::KL - 1) / C::KL;  // key groups of this tile with a key below nk
        if (live >= 4) {
          for (int d4 = 0; d4 < nd4; d4++) {
            const int sw = (d4 & 1) << 3;
            f4 kv[4];
#pragma unroll
            for (int c = 0; c < 4; c++) kv[c] = kb[d4 * C::TK + C::KL * c + (kl ^ sw)];
#pragma unroll
            for (int r = 0; r < C::RL; r++) {
              const f4 qv = *reinterpret_cast<const f4*>(qb + r * qs + 4 * d4);
#pragma unroll
              for (int j = 0; j < 4; j++)
#pragma unroll
                for (int c = 0; c < 4; c++) acc[r][c] += qv[j] * kv[c][j];
            }
          }
        } else {  // the window's last tile: one key group after the other
#pragma unroll
          for (int c = 0; c < 3; c++) {
            if (c >= live) continue;
            for (int d4 = 0; d4 < nd4; d4++) {
              const f4 kv = kb[d4 * C::TK + C::KL * c + (kl ^ ((d4 & 1) << 3))];
#pragma unroll
              for (int r = 0; r < C::RL; r++) {
                const f4 qv = *reinterpret_cast<const f4*>(qb + r * qs + 4 * d4);
#pragma unroll
                for (int j = 0; j < 4; j++) acc[r][c] += qv[j] * kv[j];
              }
            }
          }
        }
        if (dc + 1 == n_dc) {
          // row i attends keys 0..i; the slot's words past nk are scratch too
#pragma unroll
          for (int r = 0; r < C::RL; r++) {
            float* dst = slot + (size_t)(rg + r) * sstride + kt * C::TK + kl;
#pragma unroll
            for (int c = 0; c < 4; c++) {
              const float s = acc[r][c] * scale;
              dst[C::KL * c] = s;
              mx[r] = kt * C::TK + C::KL * c + kl <= i0 + rg + r ? fmaxf(mx[r], s) : mx[r];
            }
          }
        }
        if (st + 1 < n_st) store((st + 1) & 1);
        __syncthreads();
        kt = kt1;
        dc = dc1;
      }
#pragma unroll
      for (int r = 0; r < C::RL; r++) {
        float m = mx[r];
#pragma unroll
        for (int o = 1; o < C::KL; o <<= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
        if (kl == 0) s_mx[rg + r] = m;
      }
      if (tid < BQ) s_sum[tid] = -0.0f;
      __syncthreads();
    }

    // ---- 2. exponentials and their left-to-right sums (norms.rs:44-56)
    {
      const int n_et = (nk + C::TE - 1) / C::TE;
      float* ebuf = smem;  // [2][BQ][ES]
      const int row = tid / (kPtNT / BQ), part = tid % (kPtNT / BQ);
      float* srow = slot + (size_t)row * sstride;
      const float mx = s_mx[row];
      const int last = min(i0 + row, seq - 1);
      f4 x[C::ELD];
      auto load = [&](int c) {
#pragma unroll
        for (int u = 0; u < C::ELD; u++)
          x[u] = *reinterpret_cast<const f4*>(srow + c * C::TE + 4 * (part + (kPtNT / BQ) * u));
      };
      load(0);
      for (int c = 0; c < n_et; c++) {
#pragma unroll
        for (int u = 0; u < C::ELD; u++) {
          const int off = 4 * (part + (kPtNT / BQ) * u), t = c * C::TE + off;
          f4 e;
          e.x = dev_expf_tab(x[u].x - mx, s_tab);
          e.y = dev_expf_tab(x[u].y - mx, s_tab);
          e.z = dev_expf_tab(x[u].z - mx, s_tab);
          e.w = dev_expf_tab(x[u].w - mx, s_tab);
          e.x = t <= last ? e.x : 0.0f;
          e.y = t + 1 <= last ? e.y : 0.0f;
          e.z = t + 2 <= last ? e.z : 0.0f;
          e.w = t + 3 <= last ? e.w : 0.0f;
          *reinterpret_cast<f4*>(srow + t) = e;
          *reinterpret_cast<f4*>(ebuf + ((c & 1) * BQ + row) * C::ES + off) = e;
        }
        if (c + 1 < n_et) load(c + 1);
        __syncthreads();
        // tile c's fold runs beside tile c+1's exponentials; zeros past a
        // row's window leave its sum (of terms >= +0) unchanged
        if (wave == (c & 3) && lane < BQ) {
          const f4* er = reinterpret_cast<const f4*>(ebuf + ((c & 1) * BQ + lane) * C::ES);
          float s = s_sum[lane];
#pragma unroll 8
          for (int u = 0; u < C::TE / 4; u++) {
            const f4 e = er[u];
            s += e.x;
            s += e.y;
            s += e.z;
            s += e.w;
          }
          s_sum[lane] = s;
        }
      }
      __syncthreads();
      if (tid < BQ) s_inv[tid] = s_sum[tid] > 0.0f ? 1.0f / s_sum[tid] : 0.0f;
      __syncthreads();
    }

    // ---- 3. P.V
    {
      float* vbuf = smem;                           // [2][kPtVK][HDP]
      float* pbuf = smem + 2 * kPtVK * HDP;         // [2][kPtVK][PS]
      const int n_t = (nk + kPtVK - 1) / kPtVK;
      f4 vr[C::VLD], pr[C::PLD];
      auto load = [&](int c) {
#pragma unroll
        for (int u = 0; u < C::VLD; u++) {
          const int idx = tid + kPtNT * u, key = idx / (HDP / 4), d = 4 * (idx % (HDP / 4));
          const int t = min(c * kPtVK + key, nk - 1);
          vr[u] = d < hd ? static_cast<f4>(*reinterpret_cast<const f4_any*>(vh + (size_t)t * kv_dim + d)) : f4{0, 0, 0, 0};
        }
#pragma unroll
        for (int u = 0; u < C::PLD; u++) {
          const int idx = (tid + kPtNT * u) % (BQ * kPtVK / 4);  // (16 rows: half the lanes repeat the others' words)
          pr[u] = *reinterpret_cast<const f4*>(slot + (size_t)(idx / (kPtVK / 4)) * sstride + c * kPtVK +
                                                   4 * (idx % (kPtVK / 4)));
        }
      };
      auto store = [&](int buf) {
#pragma unroll
        for (int u = 0; u < C::VLD; u++)
          reinterpret_cast<f4*>(vbuf + buf * kPtVK * HDP)[tid + kPtNT * u] = vr[u];
#pragma unroll
        for (int u = 0; u < C::PLD; u++) {
          const int idx = (tid + kPtNT * u) % (BQ * kPtVK / 4), row = idx / (kPtVK / 4), key = 4 * (idx % (kPtVK / 4));
          const float inv = s_inv[row];
          float* p = pbuf + (buf * kPtVK + key) * C::PS + row;
          p[0] = pr[u].x * inv;
          p[C::PS] = pr[u].y * inv;
          p[2 * C::PS] = pr[u].z * inv;
          p[3 * C::PS] = pr[u].w * inv;
        }
      };
      const int col = tid % C::COLS, r0 = tid / C::COLS * C::RT;
      float acc[C::RT][4 * C::DW];
#pragma unroll
      for (int r = 0; r < C::RT; r++)
#pragma unroll
        for (int d = 0; d < 4 * C::DW; d++) acc[r][d] = 0.0f;
      // one key; ALL: every row of the block attends it
      auto step = [&](const float* vb, const float* pb, int t, auto all) {
        float p[C::RT];
        if constexpr (C::RT == 4) {
          const f4 p4 = *reinterpret_cast<const f4*>(pb + r0);
          p[0] = p4.x, p[1] = p4.y, p[2] = p4.z, p[3] = p4.w;
        } else if constexpr (C::RT == 1) {
          p[0] = pb[r0];
        } else {
          const float2 p2 = *reinterpret_cast<const float2*>(pb + r0);
          p[0] = p2.x, p[1] = p2.y;
        }
#pragma unroll
        for (int w = 0; w < C::DW; w++) {
          const f4 v4 = reinterpret_cast<const f4*>(vb)[w * C::COLS + col];
          const float vv[4] = {v4.x, v4.y, v4.z, v4.w};
#pragma unroll
          for (int r = 0; r < C::RT; r++) {
            const bool live = decltype(all)::value || t <= i0 + r0 + r;
#pragma unroll
            for (int d = 0; d < 4; d++) {
              const float n = acc[r][4 * w + d] + p[r] * vv[d];
              acc[r][4 * w + d] = live ? n : acc[r][4 * w + d];
            }
          }
        }
      };
      load(0);
      store(0);
      __syncthreads();
      for (int c = 0; c < n_t; c++) {
        if (c + 1 < n_t) load(c + 1);
        const float* vb = vbuf + (c & 1) * kPtVK * HDP;
        const float* pb = pbuf + (c & 1) * kPtVK * C::PS;
        const int t0 = c * kPtVK;
        if (t0 + kPtVK <= i0 + 1) {
#pragma unroll 8
          for (int u = 0; u < kPtVK; u++) step(vb + u * HDP, pb + u * C::PS, t0 + u, std::true_type{});
        } else {  // the diagonal: keys past a row's position are skipped (not added as zeros: V may hold inf or NaN)
          const int nu = min(kPtVK, nk - t0);
          for (int u = 0; u < nu; u++) step(vb + u * HDP, pb + u * C::PS, t0 + u, std::false_type{});
        }
        if (c + 1 < n_t) store((c + 1) & 1);
        __syncthreads();
      }
#pragma unroll
      for (int w = 0; w < C::DW; w++) {
        const int d = 4 * (w * C::COLS + col);
#pragma unroll
        for (int r = 0; r < C::RT; r++) {
          const int i = i0 + r0 + r;
          const bool live = i < seq && d < hd;
          const size_t gi = ((size_t)min(i, seq - 1) * n_heads + h) * hd + min(d, hd - 4);
          if (live) {
#pragma unroll
            for (int j = 0; j < 4; j++) out[gi + j] = acc[r][4 * w + j];
          }
          if (qd) {  // hd % 32 == 0: a 32-block is eight neighbouring lanes of one row, all live or none
            float qscale;
            int qv[4], qs;
            quantize_quad8(&acc[r][4 * w], qv, &qscale, &qs);
            if (live) {
#pragma unroll
              for (int j = 0; j < 4; j++) qd[gi + j] = static_cast<int8_t>(qv[j]);
              if ((col & 7) == 0) {
                qsa[gi >> 5] = qscale;
                qsum[gi >> 5] = qs;
              }
            }
          }
        }
      }
    }
  }
}

// Query rows per block: the larger a block, the fewer operand reads per
// product, but the placement of workgroups is not ours, so a launch of one
// round leaves compute units with unequal blocks. Blocks of 64 rows are
// taken once every slot gets two (2048 positions of 32 heads: 963 us), of 32
// rows from 2.5 per compute unit (1024 positions: 254 us against 437 with 64
// rows; 800: 204 against 252 with 16), else 16 (511: 96 us against 133 with
// 32).
int pt_block(size_t seq, size_t n_heads) {
  auto jobs = [&](size_t bq) { return (seq + bq - 1) / bq * n_heads; };
  return jobs(64) >= 4 * kPtCus ? 64 : jobs(32) >= kPtCus * 5 / 2 ? 32 : 16;
}

// Workgroups per compute unit (compiled for that many, and as many slots).
// Three from about four blocks per compute unit on, where LDS allows (14 heads
// x 64 at 3001 positions 505 us against 575 with two; 32 x 128 at 1024 254
// against 289); with fewer blocks the registers that two leave free are worth
// more (14 x 64 at 2048 275 against 299). 16-row blocks always take three (32 x
// 128 at 511 96 against 120; 8 x 256 at 1500 367 against 395, though only two
// fit).
int pt_wpc(int bq, size_t seq, size_t n_heads, size_t hd) {
  if (bq == 16) return 3;
  // (64-row blocks are taken from 1024 on)
  return hd <= (bq == 64 ? 64u : 128u) && (seq + bq - 1) / bq * n_heads >= 1000 ? 3 : 2;
}
size_t pt_slots(int bq, int wpc, size_t seq, size_t n_heads) {
  return std::min((seq + bq - 1) / bq * n_heads, size_t{kPtCus} * wpc);
}

// The launch a shape takes: query rows per block, padded head width,
// workgroups per compute unit.
struct PtPlan {
  int bq, hdp, wpc;
};
PtPlan pt_plan(size_t seq, size_t n_heads, size_t hd) {
  const int bq = pt_block(seq, n_heads), hdp = hd > 128 ? 256 : hd > 64 ? 128 : 64;
  if (bq == 16) return PtPlan{16, hdp, 3};
  if (hdp == 256) return PtPlan{32, hdp, 2};  // (wide heads have no 64-row instance)
  return PtPlan{bq, hdp, pt_wpc(bq, seq, n_heads, hd)};
}

template <int BQ, int HDP, int WPC>
int launch_tile(const float* q, const float* k, const float* v, size_t seq, size_t n_heads, size_t n_kv_heads,
                size_t hd, float* out, float* scratch, const ActQuant* aq, hipStream_t s) {
  const int nx = n_heads % 8 == 0 ? 8 : 1;
  const size_t grid = pt_slots(BQ, WPC, seq, n_heads);  // a multiple of nx
  hipLaunchKernelGGL((attn_prefill_tile<BQ, HDP, WPC>), dim3(grid), dim3(kPtNT), 0, s, q, k, v, (int)seq, (int)n_heads,
                     (int)(n_heads / n_kv_heads), (int)hd, out, scratch, (int)pt_stride(seq), aq ? aq->q : nullptr,
                     aq ? aq->sa : nullptr, aq ? aq->sums : nullptr, nx);
  PRANA_LAUNCH_CHECK();
  return kOk;
}

}  // namespace

size_t prefill_tile_scratch_floats(size_t seq, size_t n_heads, size_t hd) {
  const PtPlan p = pt_plan(seq, n_heads, hd);
  return pt_slots(p.bq, p.wpc, seq, n_heads) * p.bq * pt_stride(seq);
}

// Below these (query row, head) counts the one-launch kernel's workgroup per
// row and head is faster. Its time grows with rows x positions x head width,
// the tiled kernel's with positions and the padded width, so the line falls
// with more heads and with a fuller padded width: 1 head x 16 at 1500 positions
// 77 against 96 us, at 2600 166 against 157; 1 x 48 at 1000 72 against 87; 2 x
// 80 at 600 75 against 96; 4 x 128 at 250 56 against 55; 16 x 96 at 44 28
// against 28; 256-wide heads, 8 x 120 61 against 67, 8 x 300 211 against 111.
static size_t pt_min_rows(size_t n_heads, size_t hd) {
  static const unsigned rows[4][5] = {// heads 1, 2, 3-5, 6-15, 16 and more
                                      {2100, 1450, 1050, 750, 700},    // up to 32 dims
                                      {1400, 1220, 1080, 1040, 700},   // 64
                                      {1800, 1600, 1400, 1080, 840},   // 112
                                      {1250, 1200, 1180, 1080, 900}};  // 128
  if (hd > 128) return 1100;
  return rows[hd <= 32 ? 0 : hd <= 64 ? 1 : hd <= 112 ? 2 : 3]
             [n_heads < 3 ? n_heads - 1 : n_heads < 6 ? 2 : n_heads < 16 ? 3 : 4];
}
bool prefill_tile_takes(size_t seq, size_t n_heads, size_t hd) {
  return hd % 4 == 0 && hd <= 256 && seq >= 16 && n_heads > 0 && seq * n_heads >= pt_min_rows(n_heads, hd) &&
         seq <= static_cast<size_t>(INT32_MAX) / 2;
}
// (v may sit at any f32 address: 14 heads x 64 at 2048 positions take the one-launch
// kernel 4868 us)
bool prefill_tile_aligned(const float* q, const float* k) {
  return reinterpret_cast<uintptr_t>(q) % 16 == 0 && reinterpret_cast<uintptr_t>(k) % 16 == 0;
}

int launch_prefill_tile(const float* q, const float* k, const float* v, size_t seq, size_t n_heads,
                        size_t n_kv_heads, size_t hd, float* out, float* scratch, const ActQuant* aq,
                        bool* quantized, hipStream_t s) {
  PRANA_CHECK(prefill_tile_takes(seq, n_heads, hd) && prefill_tile_aligned(q, k) && scratch,
              "prefill attention: shape out of range");
  const ActQuant* fuse = aq && aq->q && hd % 32 == 0 ? aq : nullptr;
  if (quantized) *quantized = fuse != nullptr;
  const PtPlan p = pt_plan(seq, n_heads, hd);
  auto go = [&](auto hdp) {
    constexpr int HDP = decltype(hdp)::value;
    if constexpr (HDP <= 128) {
      if (p.bq == 64)
        return launch_tile<64, HDP, HDP == 64 ? 3 : 2>(q, k, v, seq, n_heads, n_kv_heads, hd, out, scratch, fuse, s);
      if (p.bq == 32 && p.wpc == 3)
        return launch_tile<32, HDP, 3>(q, k, v, seq, n_heads, n_kv_heads, hd, out, scratch, fuse, s);
    }
    if (p.bq == 32) return launch_tile<32, HDP, 2>(q, k, v, seq, n_heads, n_kv_heads, hd, out, scratch, fuse, s);
    return launch_tile<16, HDP, 3>(q, k, v, seq, n_heads, n_kv_heads, hd, out, scratch, fuse, s);
  };
  if (p.hdp == 256) return go(std::integral_constant<int, 256>());
  if (p.hdp == 128) return go(std::integral_constant<int, 128>());
  return go(std::integral_constant<int, 64>());
}

}  // namespace prana

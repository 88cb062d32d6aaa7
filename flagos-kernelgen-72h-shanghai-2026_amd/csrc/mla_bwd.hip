// mla_bwd.hip - gfx950 MLA backward (NoPE, shared K = V = C): dQ and dC as
// the reference's Task 03 operator computes them (C ABI: include/fagq_mla.h).
//
// Function (reference: src/task03_mla_bwd_nope_dkdv.py:401-425, :453-480):
//   rows i < E = min(16, S) of every (b, h): exact dq_i = sum_j dS_ij c_j with
//     P_ij = bf16(exp2((q_i . c_j * scale - lse_i) * log2 e)), j <= i,
//     dS_ij = bf16(P_ij (do_i . c_j - delta_i) scale), delta_i = out_i . do_i
//   rows i >= E: dq_i = scale * do_i
//   dc_j = sum_{i >= j} hs_i / (i + 1), hs_i = sum_h do[h, i]
//
// Kernels, in stream order.  The long form (see pick_form):
//   K1 mla_stream_do   - the one pass over dO (all the HBM traffic): per row
//                        and all H heads, dq = scale * do (rows >= E) and the
//                        head sum, stored as hs_i / (i + 1) in the workspace.
//                        A lane owns 8 consecutive dims (16-byte loads), a
//                        workgroup 2048 / D rows, so each head contributes a
//                        contiguous 4 KB (D = 512) segment per workgroup.
//                        With two head planes each half of the heads is a
//                        workgroup of its own, with its own plane of sums.
//   K2 mla_block_totals - per block of 16-64 rows: fp32 totals of hs / (i + 1);
//                        two planes are added here, the sum into the first.
//   K3 mla_exact_rows_suffix_scan - one launch of 1024-thread workgroups, two
//                        kinds:
//                        * exact rows, one per (b, h): q, do and c rows 0..E-1
//                          in LDS, the logits and dP by bf16 MFMAs with fp32
//                          accumulation (one wave), P and dS rounded to bf16
//                          where the reference rounds, dq rows 0..E-1 (which
//                          K1 does not write);
//                        * per block: carry = totals of all later blocks, then
//                          the reverse running sum over the block's rows,
//                          written as dc.
//                        The exact rows depend on nothing K1 or K2 writes;
//                        sharing the last launch with the few scan workgroups
//                        runs them in the part of the chip those leave idle.
// K2 and K3 issue each thread's loads as one batch: at these sizes they are
// latency-bound: every dependent round trip to memory adds its full latency.
// The short form, two launches: mla_short_do (the dO pass with the running sums
// of 8-row blocks, and the exact rows) and mla_short_scan.
//
// D above kSliceD (512) runs as column slices of at most kSliceD dims: K1, the
// block totals and K3 are per column, so each slice runs them on its columns
// (the tensors' row stride stays D, the workspace holds one slice), and the
// exact rows, whose dot products span all of D, run once over all columns in
// the first slice's K3, staging the rows in chunks of kSliceD dims.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>
#include <mutex>
#include <type_traits>

#include "fagq.h"
#include "fagq_diag.h"
#include "fagq_dispatch.hpp"
#include "fagq_mla.h"

namespace fagq {
namespace mla {
namespace {

constexpr int kThreads = 256;
constexpr int kE = FAGQ_MLA_EXACT_ROWS;
constexpr int kSliceD = FAGQ_MLA_SLICE_D;   // dims per column slice
constexpr int kPadElems = 8;             // LDS row padding (bf16 elements), exact rows
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

struct MArgs {
  const uint16_t* q;
  const uint16_t* c;
  const uint16_t* out;
  const uint16_t* dout;
  const float* lse;
  void* dq;
  void* dc;
  float* hs;          // workspace: [planes, B, S, D] head sums / (i + 1); in the short form
                      // their reverse running sums within blocks of kBlockRows rows
  float* tot;         // workspace: [B, nblk, D] block totals
  int64_t hs_plane;   // elements between the planes (B * S * D)
  int32_t planes;     // 1, or 2: the heads' halves, each with its plane
  int32_t brows;      // rows per scan block
  int32_t nblk;       // ceil(S / brows)
  int32_t H, S;
  int32_t D;          // dims of this column slice (the width K1, K2 and K3's scan handle)
  int32_t ld;         // elements between rows of q, c, out, dout, dq and dc (the full D);
                      // their pointers point at the slice's first column
  int32_t nexact;     // K3 workgroups (x < nexact) running exact rows: H in the first slice
  int32_t erows;      // min(16, S)
  float scale;
  int32_t dq_bf16;    // dq is bf16 (else fp32)
  int32_t dc_bf16;
};

__device__ __forceinline__ float bf16_to_f(uint32_t h) { return __uint_as_float(h << 16); }

// fp32 -> bf16 bits, round to nearest even (v_cvt_pk_bf16_f32).
__device__ __forceinline__ uint32_t f_to_bf16(float v) { return pack_bf16x2(v, 0.0f) & 0xffffu; }
__device__ __forceinline__ float round_bf16(float v) { return bf16_to_f(f_to_bf16(v)); }

// Stores 8 fp32 values at element offset e of an fp32 or bf16 tensor.
__device__ __forceinline__ void store8(const rsrc_t& rs, bool bf16, uint32_t e, const float (&v)[8]) {
  if (bf16) {
    const u32x4 w = {pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]), pack_bf16x2(v[4], v[5]),
                     pack_bf16x2(v[6], v[7])};
    __builtin_amdgcn_raw_buffer_store_b128(w, rs, e * 2u, 0, kNonTemporal);
  } else {
    const u32x4 a = {__float_as_uint(v[0]), __float_as_uint(v[1]), __float_as_uint(v[2]),
                     __float_as_uint(v[3])};
    const u32x4 b = {__float_as_uint(v[4]), __float_as_uint(v[5]), __float_as_uint(v[6]),
                     __float_as_uint(v[7])};
    __builtin_amdgcn_raw_buffer_store_b128(a, rs, e * 4u, 0, kNonTemporal);
    __builtin_amdgcn_raw_buffer_store_b128(b, rs, e * 4u + 16u, 0, kNonTemporal);
  }
}

// ------------------------------------------------------------------ the dO pass

// 8 fp32 values of a lane: one 16-byte bf16 or two 16-byte fp32 stores at
// element xa (HALVES: fp32, the second at xb).
template <bool HALVES>
__device__ __forceinline__ void store_lane(const rsrc_t& rs, bool bf16, uint32_t xa, uint32_t xb,
                                           const float (&v)[8]) {
  if constexpr (HALVES) {
    const u32x4 x = {__float_as_uint(v[0]), __float_as_uint(v[1]), __float_as_uint(v[2]),
                     __float_as_uint(v[3])};
    const u32x4 y = {__float_as_uint(v[4]), __float_as_uint(v[5]), __float_as_uint(v[6]),
                     __float_as_uint(v[7])};
    __builtin_amdgcn_raw_buffer_store_b128(x, rs, xa * 4u, 0, kNonTemporal);
    __builtin_amdgcn_raw_buffer_store_b128(y, rs, xb * 4u, 0, kNonTemporal);
  } else {
    store8(rs, bf16, xa, v);
  }
}

// A lane's 8 elements of one row over heads hbeg .. hend - 1 of batch b: dq =
// scale * dO (rows >= E) and their sum, acc.  The elements are 8 consecutive
// from ea (of head 0), or with HALVES 4 from ea and 4 from eb.  Heads in
// batches of U, software-pipelined: the loads of batch i + 1 are issued before
// batch i is consumed.  Heads past hend re-read head hend - 1 (in bounds) and
// are not used.
template <int U, bool HALVES>
__device__ __forceinline__ void stream_heads(const MArgs& g, int b, int row, uint32_t ea,
                                             uint32_t eb, int hbeg, int hend, float (&acc)[8]) {
  const uint32_t hsd = (uint32_t)g.H * (uint32_t)g.S * (uint32_t)g.ld;   // elements per batch
  // The slice's elements of batch b end at (H S - 1) ld + D (the descriptors'
  // size, so they stay inside the tensors whatever the slice's first column).
  const uint32_t span = hsd - (uint32_t)g.ld + (uint32_t)g.D;
  const rsrc_t rdo = make_rsrc(g.dout + (int64_t)b * hsd, span * 2u);
  const rsrc_t rdq = make_rsrc((const uint8_t*)g.dq + (int64_t)b * hsd * (g.dq_bf16 ? 2 : 4),
                               span * (g.dq_bf16 ? 2u : 4u));
  const uint32_t hstride = (uint32_t)g.S * (uint32_t)g.ld;
  const bool write_dq = row >= g.erows;
  const bool dq_bf16 = g.dq_bf16 != 0;
  auto load_batch = [&](int h0, u32x4 (&v)[U]) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int h = h0 + u < hend ? h0 + u : hend - 1;
      const uint32_t ho = (uint32_t)h * hstride;
      if constexpr (HALVES) {
        const u32x2 x = __builtin_amdgcn_raw_buffer_load_b64(rdo, (ea + ho) * 2u, 0, kNonTemporal);
        const u32x2 y = __builtin_amdgcn_raw_buffer_load_b64(rdo, (eb + ho) * 2u, 0, kNonTemporal);
        v[u] = u32x4{x[0], x[1], y[0], y[1]};
      } else {
        v[u] = __builtin_amdgcn_raw_buffer_load_b128(rdo, (ea + ho) * 2u, 0, kNonTemporal);
      }
    }
  };
  u32x4 cur[U], nxt[U];
  load_batch(hbeg, cur);
  for (int h0 = hbeg; h0 < hend; h0 += U) {
    if (h0 + U < hend) load_batch(h0 + U, nxt);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (h0 + u < hend) {
        float f[8];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          f[2 * k] = bf16_lo(cur[u][k]);
          f[2 * k + 1] = bf16_hi(cur[u][k]);
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) acc[k] += f[k];
        if (write_dq) {
          float d[8];
#pragma unroll
          for (int k = 0; k < 8; ++k) d[k] = f[k] * g.scale;
          const uint32_t ho = (uint32_t)(h0 + u) * hstride;
          store_lane<HALVES>(rdq, dq_bf16, ea + ho, eb + ho, d);
        }
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) cur[u] = nxt[u];
  }
}

// The heads of a plane: [h0, h1), never empty (two planes have 40 heads or more).
__device__ __forceinline__ void plane_heads(const MArgs& g, int plane, int& h0, int& h1) {
  const int hpp = (g.H + g.planes - 1) >> (g.planes - 1);
  h0 = plane * hpp;
  h1 = h0 + hpp < g.H ? h0 + hpp : g.H;
}

// K1.  grid (ceil(S / rows_per_wg), B, planes); rows_per_wg = 256 / (D / 8).  U
// heads' loads are in flight per lane: U = 2 with bf16 dq (50 VGPRs, 8 workgroups
// per CU) and U = 1 with fp32 dq, whose stores are twice the loads' bytes (2 B / 4
// B, 2 x 64 x 4096 x 512: 297 against 308 us for the pass; 2 x 64 x 1900 x 512
// 147.9 us per call against 157.2 with U = 8); U = 8 (110 VGPRs, 4 per CU) with
// bf16 dq for grids that fit 4 per CU (figures: pick_form).
template <int U, bool HALVES>
__global__ void __launch_bounds__(kThreads) mla_stream_do(const MArgs g) {
  const int lpr = g.D / 8;                        // lanes per row
  const int t = threadIdx.x;
  // When lpr does not divide kThreads, the last kThreads % lpr threads hold
  // no whole row of this workgroup (their t / lpr would be the next
  // workgroup's first row), and stop here.
  if (t / lpr >= kThreads / lpr) return;
  const int row = (int)blockIdx.x * (kThreads / lpr) + t / lpr;
  if (row >= g.S) return;
  const int b = (int)blockIdx.y;
  // HALVES: eb = ea + D / 2, so that each of the lane's two 16-byte fp32
  // stores lies in a contiguous half-row span of the row's lanes.  wa / wb:
  // the same elements in the workspace's head sums, rows of D.
  const uint32_t lo = (uint32_t)(t % lpr) * (HALVES ? 4u : 8u);
  const uint32_t ea = (uint32_t)row * (uint32_t)g.ld + lo;
  const uint32_t wa = (uint32_t)row * (uint32_t)g.D + lo;
  const uint32_t half = (uint32_t)g.D / 2u;
  float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  int h0, h1;
  plane_heads(g, (int)blockIdx.z, h0, h1);
  stream_heads<U, HALVES>(g, b, row, ea, ea + half, h0, h1, acc);
  const float n1 = (float)(row + 1);
  float o[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) o[k] = acc[k] / n1;
  const uint32_t sd = (uint32_t)g.S * (uint32_t)g.D;
  const rsrc_t rhs = make_rsrc(g.hs + (int64_t)blockIdx.z * g.hs_plane + (int64_t)b * sd, sd * 4u);
  store_lane<HALVES>(rhs, false, wa, wa + half, o);
}

// ------------------------------------------------------------------ K3: exact rows

constexpr int kWide = 1024;               // threads of K2 and K3 (16 waves)

// Exact rows 0..E-1 of (b, h) by NW waves (16 or 8), wave m owning query rows
// m, m + NW, .. for delta and dq; wave 0 computes all 16 x 16 logits and dP with
// MFMAs.  The rows' D = ld dims go through LDS in chunks of W = min(D,
// kSliceD): per chunk, every global load is issued before the first LDS store
// (wave m loads 16-byte piece `lane` of its q, do and out rows, thread t piece
// t % (W / 8) of c row t / (W / 8)); buffer descriptors over rows 0..E-1 return
// zeros for the rest.  The logits, dP and delta accumulate over the chunks; dS follows; then
// dq, chunk by chunk (c staged again when D > W).  Dynamic LDS: q, do and c
// rows 0..15 of one chunk (padded by 16 bytes), then dS [16][16] and delta [16].
template <int NW>
__device__ __forceinline__ void exact_rows(const MArgs& g, int b, int h) {
  constexpr int RPW = kE / NW;                    // query rows per wave
  static_assert(RPW * NW == kE, "the waves share the rows evenly");
  extern __shared__ __align__(16) uint8_t smem[];
  const int D = g.ld, E = g.erows;
  const int W = D < kSliceD ? D : kSliceD;
  const int ldl = W + kPadElems;                  // bf16 elements per LDS row
  uint16_t* qs = reinterpret_cast<uint16_t*>(smem);
  uint16_t* dos = qs + kE * ldl;
  uint16_t* cs = dos + kE * ldl;
  float* dS = reinterpret_cast<float*>(cs + kE * ldl);
  float* deltas = dS + kE * kE;                   // [kE], after dS
  const int t = threadIdx.x, lane = t & 63, m = t >> 6;
  const int bh = b * g.H + h;
  const int64_t qrow0 = (int64_t)bh * g.S * D;    // q, do, out rows of (b, h)
  const uint32_t rbytes = (uint32_t)(E * D * 2);
  const rsrc_t rq = make_rsrc(g.q + qrow0, rbytes);
  const rsrc_t rdo = make_rsrc(g.dout + qrow0, rbytes);
  const rsrc_t rout = make_rsrc(g.out + qrow0, rbytes);
  const rsrc_t rc = make_rsrc(g.c + (int64_t)b * g.S * D, rbytes);
  // c rows 0..15 of the W-wide chunk at dim c0: 16 W / 8 <= 1024 pieces, RPW or
  // fewer per thread.
  auto load_c = [&](int c0, int cpr, u32x4 (&cv)[RPW]) {
#pragma unroll
    for (int i = 0; i < RPW; ++i) {
      const int e = t + i * 64 * NW, cr = e / cpr;
      const uint32_t coff = cr < E ? (uint32_t)(cr * D + c0 + (e % cpr) * 8) * 2u : rbytes;
      cv[i] = __builtin_amdgcn_raw_buffer_load_b128(rc, coff, 0, 0);
    }
  };
  auto put_c = [&](int cpr, const u32x4 (&cv)[RPW]) {
#pragma unroll
    for (int i = 0; i < RPW; ++i) {
      const int e = t + i * 64 * NW;
      if (e < kE * cpr) *reinterpret_cast<u32x4*>(cs + (e / cpr) * ldl + (e % cpr) * 8) = cv[i];
    }
  };

  // Logits and dP of query row qm = lane % 16 with keys n = 4 (lane / 16) +
  // r (r < 4), by wave 0 alone: v_mfma_f32_16x16x32_bf16 with A = c rows
  // (key), B = q or dO rows (query), K = the chunk's dims in steps of 32.
  // Lane l supplies row l % 16 of both operands, 8 consecutive dims (the same
  // ones for both) per step, and receives D[4 (l / 16) + r][l % 16] (checked
  // on the GPU).  Rows past E were staged as zeros.
  const int qm = lane & 15, k0 = (lane >> 4) * 8;
  f32x4 lg = {0.0f, 0.0f, 0.0f, 0.0f}, dpv = lg;
  float delta[RPW];
#pragma unroll
  for (int i = 0; i < RPW; ++i) delta[i] = 0.0f;
  for (int c0 = 0; c0 < D; c0 += W) {
    const int w = D - c0 < W ? D - c0 : W;        // a multiple of 64
    const int cpr = w / 8;                        // 16-byte pieces per row (8..64)
    if (c0 > 0) __syncthreads();                  // the previous chunk's reads are done
    u32x4 a[RPW], d[RPW], o[RPW], cv[RPW];
#pragma unroll
    for (int i = 0; i < RPW; ++i) {
      const int row = m + i * NW;
      const uint32_t off = row < E && lane < cpr ? (uint32_t)(row * D + c0 + lane * 8) * 2u : rbytes;
      a[i] = __builtin_amdgcn_raw_buffer_load_b128(rq, off, 0, 0);
      d[i] = __builtin_amdgcn_raw_buffer_load_b128(rdo, off, 0, 0);
      o[i] = __builtin_amdgcn_raw_buffer_load_b128(rout, off, 0, 0);
    }
    load_c(c0, cpr, cv);
    put_c(cpr, cv);
#pragma unroll
    for (int i = 0; i < RPW; ++i) {
      if (lane < cpr) {
        *reinterpret_cast<u32x4*>(qs + (m + i * NW) * ldl + lane * 8) = a[i];
        *reinterpret_cast<u32x4*>(dos + (m + i * NW) * ldl + lane * 8) = d[i];
      }
      // delta_m = out_m . do_m, this lane's part.
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        delta[i] += bf16_lo(o[i][j]) * bf16_lo(d[i][j]);
        delta[i] += bf16_hi(o[i][j]) * bf16_hi(d[i][j]);
      }
    }
    __syncthreads();
    if (m == 0) {
      const uint16_t* cr = cs + qm * ldl + k0;
      const uint16_t* qr = qs + qm * ldl + k0;
      const uint16_t* dr = dos + qm * ldl + k0;
      auto ld8 = [](const uint16_t* p) { return *reinterpret_cast<const bf16x8*>(p); };
#pragma unroll 2
      for (int k = 0; k < w; k += 64) {           // w % 64 == 0: two steps per pass
        const bf16x8 c0v = ld8(cr + k), q0 = ld8(qr + k), d0 = ld8(dr + k);
        const bf16x8 c1v = ld8(cr + k + 32), q1 = ld8(qr + k + 32), d1 = ld8(dr + k + 32);
        lg = __builtin_amdgcn_mfma_f32_16x16x32_bf16(c0v, q0, lg, 0, 0, 0);
        dpv = __builtin_amdgcn_mfma_f32_16x16x32_bf16(c0v, d0, dpv, 0, 0, 0);
        lg = __builtin_amdgcn_mfma_f32_16x16x32_bf16(c1v, q1, lg, 0, 0, 0);
        dpv = __builtin_amdgcn_mfma_f32_16x16x32_bf16(c1v, d1, dpv, 0, 0, 0);
      }
    }
  }
#pragma unroll
  for (int i = 0; i < RPW; ++i) {
#pragma unroll
    for (int s = 32; s > 0; s >>= 1) delta[i] += __shfl_xor(delta[i], s, 64);
    if (lane == 0) deltas[m + i * NW] = delta[i];
  }
  __syncthreads();
  if (m == 0) {
    const float lse = qm < E ? g.lse[(int64_t)bh * g.S + qm] : 0.0f;
    const float dlt = deltas[qm];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int kn = 4 * (lane >> 4) + r;
      float sv = 0.0f;
      if (qm < E && kn <= qm) {
        const float p = round_bf16(exp2f((lg[r] * g.scale - lse) * 1.4426950408889634f));
        sv = round_bf16(p * (dpv[r] - dlt) * g.scale);
      }
      dS[qm * kE + kn] = sv;
    }
  }
  __syncthreads();

  // dq row m, chunk by chunk: lane owns dims c0 + 8 lane .. + 7.
  const rsrc_t rdq = make_rsrc((const uint8_t*)g.dq + qrow0 * (g.dq_bf16 ? 2 : 4),
                               (uint32_t)(E * D) * (g.dq_bf16 ? 2u : 4u));
  for (int c0 = 0; c0 < D; c0 += W) {
    const int w = D - c0 < W ? D - c0 : W;
    if (D > W) {                                  // c of this chunk (one chunk: still staged)
      __syncthreads();
      u32x4 cv[RPW];
      load_c(c0, w / 8, cv);
      put_c(w / 8, cv);
      __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < RPW; ++i) {
      const int row = m + i * NW;
      if (row >= E || lane * 8 >= w) continue;
      const int k = lane * 8;
      float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
      for (int j = 0; j <= row; ++j) {
        const float sv = dS[row * kE + j];
        const u32x4 c = *reinterpret_cast<const u32x4*>(cs + j * ldl + k);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          acc[2 * e] = fmaf(sv, bf16_lo(c[e]), acc[2 * e]);
          acc[2 * e + 1] = fmaf(sv, bf16_hi(c[e]), acc[2 * e + 1]);
        }
      }
      store8(rdq, g.dq_bf16 != 0, (uint32_t)(row * D + c0 + k), acc);
    }
  }
}

// Dynamic LDS of K3: the exact rows' rows and dS.
size_t exact_lds_bytes(int64_t D) {
  const int64_t W = D < kSliceD ? D : kSliceD;
  return (size_t)3 * kE * (W + kPadElems) * 2 + (size_t)(kE * kE + kE) * 4;
}
constexpr size_t kBlockTotalLds = (size_t)kWide * 16;   // dynamic LDS of K2: the parts' join

// ------------------------------------------------------------------ K2: block totals

constexpr int kBatch = 16;                // loads issued before they are used

__device__ __forceinline__ void add4(float4& a, const float4& b) {
  a.x += b.x;
  a.y += b.y;
  a.z += b.z;
  a.w += b.w;
}

// Thread layout of K2's block totals and K3 over D columns: cpt = D / 4 column
// threads (16..128) per part, np = kWide / cpt parts (8..64); thread t owns
// columns 4 (t % cpt) .. + 3 of part t / cpt (threads of parts >= np idle).
struct Parts {
  int cpt, np, p, col;
  __device__ explicit Parts(int D) : cpt(D >> 2), np(kWide / (D >> 2)), p((int)threadIdx.x / (D >> 2)),
                                     col((int)threadIdx.x - p * (D >> 2)) {}
};

// Totals of block blk (g.brows rows) of batch b: part p of the block's threads
// sums rows r0 + p, r0 + p + np, ..., kBatch / PL of them loaded together; the
// parts' totals are joined in LDS, in part order.  PL 2: each row's two planes are
// added, and the sum written over the first, the only one that K3 reads.
template <int PL>
__device__ __forceinline__ void block_total(const MArgs& g, int b, int blk) {
  constexpr int R = kBatch / PL;
  extern __shared__ __align__(16) uint8_t smem[];
  float4* part = reinterpret_cast<float4*>(smem);
  const Parts P(g.D);
  const int r0 = blk * g.brows;
  const int r1 = r0 + g.brows < g.S ? r0 + g.brows : g.S;
  float* __restrict__ hs = g.hs + (int64_t)b * g.S * g.D + 4 * P.col;
  float4 a = make_float4(0.f, 0.f, 0.f, 0.f);
  if (P.p < P.np) {
    for (int r = r0 + P.p; r < r1; r += R * P.np) {
      float4 v[R][PL];
#pragma unroll
      for (int i = 0; i < R; ++i) {
        // Clamped to a row that no other thread writes (PL 2); r0 is one load for all.
        const int rr = r + i * P.np < r1 ? r + i * P.np : PL == 2 ? r : r0;
#pragma unroll
        for (int p = 0; p < PL; ++p)
          v[i][p] = *reinterpret_cast<const float4*>(hs + p * g.hs_plane + (int64_t)rr * g.D);
      }
#pragma unroll
      for (int i = 0; i < R; ++i) {
        if (r + i * P.np >= r1) continue;
        if constexpr (PL == 2) {
          add4(v[i][0], v[i][1]);
          *reinterpret_cast<float4*>(hs + (int64_t)(r + i * P.np) * g.D) = v[i][0];
        }
        add4(a, v[i][0]);
      }
    }
  }
  part[threadIdx.x] = a;
  __syncthreads();
  if (P.p == 0) {
    for (int q = 1; q < P.np; ++q) add4(a, part[q * P.cpt + P.col]);
    *reinterpret_cast<float4*>(g.tot + ((int64_t)b * g.nblk + blk) * g.D + 4 * P.col) = a;
  }
}

// grid (nblk, B)
template <int PL>
__global__ void __launch_bounds__(kWide) mla_block_totals(const MArgs g) {
  block_total<PL>(g, (int)blockIdx.y, (int)blockIdx.x);
}

// ------------------------------------------------------------------ K3

constexpr int kChunkRows = 8;             // >= ceil(64 / 8): rows per part of a block

// Block blk of batch b.  The block's rows are np chunks of cr = ceil(brows /
// np) rows (cr <= 8 since brows <= 64 and np >= 8); part p scans chunk p.
// Part p first sums (1) the totals of later blocks blk + 1 + p, blk + 1 + p +
// np, ... and (2) the rows of its chunk (kept in registers); after one
// barrier its carry is all parts' (1), in part order, plus the (2) of the
// chunks above it, then the reverse running sum over the chunk is written as
// dc.
__device__ __forceinline__ void suffix_scan(const MArgs& g, int b, int blk) {
  __shared__ float4 later[kWide], chunk[kWide];
  const Parts P(g.D);
  const int r0 = blk * g.brows;
  const int r1 = r0 + g.brows < g.S ? r0 + g.brows : g.S;
  const int cr = (g.brows + P.np - 1) / P.np;
  const int c0 = r0 + P.p * cr < r1 ? r0 + P.p * cr : r1;
  const int c1 = c0 + cr < r1 ? c0 + cr : r1;
  // The workspace and dc never overlap (checked at launch): restrict lets the
  // loads issue together ahead of the stores.
  const float* __restrict__ hs = g.hs + (int64_t)b * g.S * g.D + 4 * P.col;
  const float* __restrict__ tot = g.tot + (int64_t)b * g.nblk * g.D + 4 * P.col;
  float4 rows[kChunkRows];
  float4 lat = make_float4(0.f, 0.f, 0.f, 0.f), own = lat;
  if (P.p < P.np) {
#pragma unroll
    for (int k = 0; k < kChunkRows; ++k)        // rows c1 - 1 - k (clamped)
      rows[k] = *reinterpret_cast<const float4*>(hs + (int64_t)(c1 - 1 - k >= c0 ? c1 - 1 - k : r0) * g.D);
    for (int x = blk + 1 + P.p; x < g.nblk; x += kBatch * P.np) {
      float4 v[kBatch];
#pragma unroll
      for (int k = 0; k < kBatch; ++k) {
        const int xx = x + k * P.np;
        v[k] = *reinterpret_cast<const float4*>(tot + (int64_t)(xx < g.nblk ? xx : x) * g.D);
      }
#pragma unroll
      for (int k = 0; k < kBatch; ++k)
        if (x + k * P.np < g.nblk) add4(lat, v[k]);
    }
#pragma unroll
    for (int k = 0; k < kChunkRows; ++k)
      if (c1 - 1 - k >= c0) add4(own, rows[k]);
  }
  later[threadIdx.x] = lat;
  chunk[threadIdx.x] = own;
  __syncthreads();
  if (P.p >= P.np || c0 >= c1) return;
  float4 cy = make_float4(0.f, 0.f, 0.f, 0.f);
  for (int q = 0; q < P.np; ++q) add4(cy, later[q * P.cpt + P.col]);
  for (int q = P.np - 1; q > P.p; --q) add4(cy, chunk[q * P.cpt + P.col]);
  float* __restrict__ dcf = static_cast<float*>(g.dc) + (int64_t)b * g.S * g.ld + 4 * P.col;
  uint16_t* __restrict__ dch = static_cast<uint16_t*>(g.dc) + (int64_t)b * g.S * g.ld + 4 * P.col;
  const bool bf16 = g.dc_bf16 != 0;
#pragma unroll
  for (int k = 0; k < kChunkRows; ++k) {
    const int r = c1 - 1 - k;
    if (r >= c0) {
      add4(cy, rows[k]);
      if (bf16) {
        const uint2 wv = {pack_bf16x2(cy.x, cy.y), pack_bf16x2(cy.z, cy.w)};
        *reinterpret_cast<uint2*>(dch + (int64_t)r * g.ld) = wv;
      } else {
        *reinterpret_cast<float4*>(dcf + (int64_t)r * g.ld) = cy;
      }
    }
  }
}

// grid (nexact + nblk, B): x < nexact (H in the first column slice, else 0)
// are the exact rows of head x, the rest the scan of block x - nexact.
// Uniform per workgroup, so every barrier sees all its waves.
__global__ void __launch_bounds__(kWide) mla_exact_rows_suffix_scan(const MArgs g) {
  const int x = (int)blockIdx.x, b = (int)blockIdx.y;
  if (x < g.nexact)
    exact_rows<kWide / 64>(g, b, x);
  else
    suffix_scan(g, b, x - g.nexact);
}

// ------------------------------------------------------------------ short sequences

// The dO pass of a short sequence.  Whole rows give few workgroups there, so a
// workgroup takes 8 rows of a column tile of CW dims, and its 8 waves split them
// and the heads (1 to 8 head groups): the groups' sums are joined in LDS, and
// the block's reverse running sums (with the 1 / (i + 1)) go to the workspace,
// whose rows 0, 8, 16, .. then are the blocks' totals.  One launch replaces a
// pass that wrote up to 8 partial planes and a kernel for the totals, and the
// last one only adds the later blocks' totals.  With two planes each half of the
// heads is a workgroup of its own: few tiles of many heads leave CUs idle, and a
// wave's chain of heads is long.  The exact rows, which depend on nothing else,
// are the grid's first workgroups and run beside the dO pass.  Bound by the dO
// pass's bytes, and below about 20 us by the two launches' latency (figures:
// pick_form).
constexpr int kBlockRows = 8;
constexpr int kShortWaves = 8;

template <int CW, int U, bool HALVES>
__global__ void __launch_bounds__(64 * kShortWaves) mla_short_do(const MArgs g) {
  constexpr int LPR = CW / 8, WR = 64 / LPR;             // lanes per row, rows per wave
  constexpr int RW = kBlockRows / WR, HG = kShortWaves / RW;
  constexpr int C4 = CW / 4, T = 64 * kShortWaves;
  static_assert(RW * WR == kBlockRows && HG * RW == kShortWaves, "waves tile the block");
  extern __shared__ __align__(16) uint8_t smem[];        // HG x 8 x CW floats, or the exact rows'
  const int b = (int)blockIdx.y;
  if ((int)blockIdx.x < g.nexact) {                      // uniform over the workgroup
    exact_rows<kShortWaves>(g, b, (int)blockIdx.x);
    return;
  }
  float4* const part = reinterpret_cast<float4*>(smem);
  const int t = threadIdx.x, lane = t & 63;
  const int w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int rw = w % RW, hg = w / RW;
  const int y = (int)blockIdx.x - g.nexact;
  const int plane = y & (g.planes - 1), x = y >> (g.planes - 1);
  const int ncol = g.D / CW, ct = x % ncol, blk = x / ncol;   // CW divides D
  const int r0 = blk * kBlockRows;
  const int brow = rw * WR + lane / LPR, row = r0 + brow;     // the lane's row in the block, of S
  const int li = lane % LPR;
  int h0, h1;
  plane_heads(g, plane, h0, h1);
  const int hps = (h1 - h0 + HG - 1) / HG;
  const int hbeg = h0 + hg * hps < h1 ? h0 + hg * hps : h1;
  const int hend = hbeg + hps < h1 ? hbeg + hps : h1;
  float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  if (row < g.S && hbeg < hend) {
    const uint32_t ea = (uint32_t)row * (uint32_t)g.ld + (uint32_t)(ct * CW + li * (HALVES ? 4 : 8));
    stream_heads<U, HALVES>(g, b, row, ea, ea + CW / 2, hbeg, hend, acc);
  }
  float4* const mine = part + (hg * kBlockRows + brow) * C4;
  mine[HALVES ? li : 2 * li] = make_float4(acc[0], acc[1], acc[2], acc[3]);
  mine[HALVES ? li + C4 / 2 : 2 * li + 1] = make_float4(acc[4], acc[5], acc[6], acc[7]);
  __syncthreads();
  // Heads' sums in group order, into group 0's place.
  for (int e = t; e < kBlockRows * C4; e += T) {
    float4 v = part[e];
#pragma unroll
    for (int q = 1; q < HG; ++q) add4(v, part[q * kBlockRows * C4 + e]);
    part[e] = v;
  }
  __syncthreads();
  if (t < C4) {
    float4 v[kBlockRows];
#pragma unroll
    for (int k = 0; k < kBlockRows; ++k) v[k] = part[k * C4 + t];
    float* const hs = g.hs + plane * g.hs_plane + ((int64_t)b * g.S + r0) * g.D + ct * CW + 4 * t;
    float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int k = kBlockRows - 1; k >= 0; --k) {          // rows past S hold zeros
      const float n1 = (float)(r0 + k + 1);
      add4(s, make_float4(v[k].x / n1, v[k].y / n1, v[k].z / n1, v[k].w / n1));
      if (r0 + k < g.S) *reinterpret_cast<float4*>(hs + (int64_t)k * g.D) = s;
    }
  }
}

// dc of a short sequence.  grid (nblk, B), g.brows rows each (a multiple of
// kBlockRows): a row's dc is its running sum within its block of 8 rows plus
// the totals of the later blocks.  Part p (see Parts) owns cr consecutive rows,
// cr a power of two up to CR, so all in one block; it sums the totals of every
// np-th block past the workgroup's rows, and after one barrier adds all parts'
// sums, in part order, and the totals of the workgroup's own later blocks.  PL 2:
// every row and total is the sum of its two planes; both are loaded together, for
// which the registers suffice where brows is 16 (CR 2, one later block).  Its sums
// are kept in 64 bits until they are written: the planes' own roundings are two where
// one plane has one (relative error of dc at 1 x 128 x 100 x 512: 5.2e-8; 7.0e-8 with sums in
// 32 bits, 6.4e-8 with one plane).
struct Sum64 {
  double x, y, z, w;
};
__device__ __forceinline__ void add4(Sum64& a, const Sum64& b) {
  a.x += b.x;
  a.y += b.y;
  a.z += b.z;
  a.w += b.w;
}
template <int PL, int CR>
__global__ void __launch_bounds__(kWide) mla_short_scan(const MArgs g) {
  constexpr int NEAR = CR == 2 ? 1 : kBlockRows - 1;     // later blocks in the workgroup's rows
  constexpr int LB = kBlockRows / PL;                    // far totals loaded together
  using Sum = std::conditional_t<PL == 2, Sum64, float4>;
  __shared__ Sum later[kWide];
  const int b = (int)blockIdx.y;
  const Parts P(g.D);
  const int r0 = (int)blockIdx.x * g.brows;
  const int r1 = r0 + g.brows < g.S ? r0 + g.brows : g.S;
  int cr = 1;
  while (cr * P.np < g.brows) cr *= 2;                   // <= 8: brows <= 64, np >= 8
  const int c0 = r0 + P.p * cr < r1 ? r0 + P.p * cr : r1;
  const int c1 = c0 + cr < r1 ? c0 + cr : r1;
  const int nb = (g.S + kBlockRows - 1) / kBlockRows;    // blocks of 8 rows of the sequence
  const int next = (r0 + g.brows) / kBlockRows;          // the first past the workgroup's rows
  const float* __restrict__ hs = g.hs + (int64_t)b * g.S * g.D + 4 * P.col;
  auto load = [&](int row, float4 (&v)[PL]) {
#pragma unroll
    for (int p = 0; p < PL; ++p)
      v[p] = *reinterpret_cast<const float4*>(hs + p * g.hs_plane + (int64_t)row * g.D);
  };
  auto add = [](Sum& a, const float4 (&v)[PL]) {
    if constexpr (PL == 2)
      add4(a, Sum64{(double)v[0].x + v[1].x, (double)v[0].y + v[1].y, (double)v[0].z + v[1].z,
                    (double)v[0].w + v[1].w});
    else
      add4(a, v[0]);
  };
  float4 rows[CR][PL], near[NEAR][PL];
  Sum lat = {0, 0, 0, 0};
  const int own = c0 / kBlockRows;                       // the block of the part's rows
  const int nnear = (next < nb ? next : nb) - own - 1;   // later blocks of this workgroup
  if (P.p < P.np && c0 < c1) {
#pragma unroll
    for (int k = 0; k < CR; ++k)
      if (k < cr) load(c0 + k < c1 ? c0 + k : c0, rows[k]);
#pragma unroll
    for (int k = 0; k < NEAR; ++k)
      if (k < nnear) load((own + 1 + k) * kBlockRows, near[k]);
  }
  if (P.p < P.np) {
    for (int x = next + P.p; x < nb; x += LB * P.np) {
      float4 v[LB][PL];
#pragma unroll
      for (int k = 0; k < LB; ++k) {
        const int xx = x + k * P.np;
        load((xx < nb ? xx : x) * kBlockRows, v[k]);
      }
#pragma unroll
      for (int k = 0; k < LB; ++k)
        if (x + k * P.np < nb) add(lat, v[k]);
    }
  }
  later[threadIdx.x] = lat;
  __syncthreads();
  if (P.p >= P.np || c0 >= c1) return;
  Sum cy = {0, 0, 0, 0};
  for (int q = 0; q < P.np; ++q) add4(cy, later[q * P.cpt + P.col]);
#pragma unroll
  for (int k = NEAR - 1; k >= 0; --k)
    if (k < nnear) add(cy, near[k]);
  float* __restrict__ dcf = static_cast<float*>(g.dc) + (int64_t)b * g.S * g.ld + 4 * P.col;
  uint16_t* __restrict__ dch = static_cast<uint16_t*>(g.dc) + (int64_t)b * g.S * g.ld + 4 * P.col;
  const bool bf16 = g.dc_bf16 != 0;
#pragma unroll
  for (int k = 0; k < CR; ++k) {
    const int r = c0 + k;
    if (k < cr && r < c1) {
      Sum sum = cy;
      add(sum, rows[k]);
      const float4 o = make_float4((float)sum.x, (float)sum.y, (float)sum.z, (float)sum.w);
      if (bf16) {
        const uint2 wv = {pack_bf16x2(o.x, o.y), pack_bf16x2(o.z, o.w)};
        *reinterpret_cast<uint2*>(dch + (int64_t)r * g.ld) = wv;
      } else {
        *reinterpret_cast<float4*>(dcf + (int64_t)r * g.ld) = o;
      }
    }
  }
}

bool aligned(const void* p, uintptr_t a) { return (reinterpret_cast<uintptr_t>(p) & (a - 1)) == 0; }

bool overlap(const void* a, int64_t na, const void* b, int64_t nb) {
  const uintptr_t x = reinterpret_cast<uintptr_t>(a), y = reinterpret_cast<uintptr_t>(b);
  return na > 0 && nb > 0 && x < y + (uintptr_t)nb && y < x + (uintptr_t)na;
}

constexpr int kMinK1Groups = 1024;        // K1 workgroups wanted (4 per CU)

// K1's workgroups for a column slice of D dims.
int64_t k1_groups(int64_t B, int64_t S, int64_t D) {
  const int64_t rows_per_wg = kThreads / (D / 8);
  return ((S + rows_per_wg - 1) / rows_per_wg) * B;
}

// Planes of head sums a slice of D dims may need, whatever its heads and types
// (pick_form halves the heads below kMinK1Groups only).
int64_t workspace_planes(int64_t B, int64_t S, int64_t D) {
  return D >= 64 && k1_groups(B, S, D) < kMinK1Groups ? 2 : 1;
}

// Rows per scan block: S / 64 rounded up to a multiple of 16, within [16, 64],
// so short sequences still spread over many blocks and each thread's carry and
// in-block loops stay short.
int64_t block_rows(int64_t S) {
  int64_t r = ((S + 63) / 64 + 15) / 16 * 16;
  return r < 16 ? 16 : r > 64 ? 64 : r;
}

// How one column slice of ds dims runs.
struct Form {
  int cw;                 // short form: dims of a column tile; 0: the long form
  int unroll;             // heads in flight per lane
  int planes;             // 1, or 2 head halves, each with its plane of head sums
  const void* kernel;     // the dO pass
};
template <int CW, int U>
Form short_form(bool halves, int planes) {
  return {CW, U, planes, halves ? reinterpret_cast<const void*>(&mla_short_do<CW, U, true>)
                                : reinterpret_cast<const void*>(&mla_short_do<CW, U, false>)};
}
Form long_form(bool halves, bool fits, int planes) {
  if (halves) return {0, 1, planes, reinterpret_cast<const void*>(&mla_stream_do<1, true>)};
  if (fits) return {0, 8, planes, reinterpret_cast<const void*>(&mla_stream_do<8, false>)};
  return {0, 2, planes, reinterpret_cast<const void*>(&mla_stream_do<2, false>)};
}

// The form of a slice, `nexact` exact-row workgroups per batch beside it.  The lines
// were drawn on 2520 shapes (B 1 .. 8, H 8 .. 128, S 8 .. 8192, D 64 .. 512, both types of
// dq), each timed in every form.  us per call in a replayed graph; B x H x S x D.
Form pick_form(int64_t B, int64_t H, int64_t S, int64_t ds, int64_t nexact, bool halves) {
  const int64_t groups = k1_groups(B, S, ds);
  const int64_t blocks = B * ((S + kBlockRows - 1) / kBlockRows);
  auto tiles = [&](int64_t cw) { return blocks * (ds / cw); };

  // The long form where K1's grid is large: 4 workgroups per CU, or 2 with fp32 dq,
  // whose stores set the pass's rate (fp32, 2 x 64 x 1900 x 512: 147.9 against 154.1 in
  // the short form; 2 x 64 x 1024 x 512: 84.6 against 85.0).  Also where only 64-dim
  // tiles fit and few heads leave their 8 head groups one or two heads each (bf16, 1
  // x 8 x 3000 x 448: 22.4 against 30.9; 1 x 8 x 1500 x 448: 18.2 against 17.8).
  // U = 8 fills the chip once with 4 workgroups per CU: at 1000 to 1028 of them 26.4
  // against 28.6 with U = 2 (1 x 8 x 4000 x 448), 109.5 against 113.9 (2 x 64 x 2048 x
  // 512), 207.8 against 220.6 (4 x 128 x 1025 x 512); from 1050 on 117.1 with U = 2
  // against 118.4 (2 x 64 x 2100 x 512), 121.8 against 127.3 (2200).  Multiples of 128
  // dims meet it at 1024 workgroups only: below, the short form takes them.
  const bool narrow_few = ds % 128 != 0 && H < 16 && tiles(64) > 1500;
  if (groups >= (halves ? kMinK1Groups / 2 : kMinK1Groups) || narrow_few)
    return long_form(halves, groups <= kMinK1Groups, 1);

  // Many heads make a short-form workgroup's chain long and its last round costly:
  // there the heads are halved over workgroups, each half with its plane of sums.
  const bool fits = tiles(128) + B * nexact <= 320;   // 128-dim tiles and exact rows: one round
  if (H >= 40) {
    // Two planes need scan blocks of 16 rows (mla_short_scan); behind hundreds of exact
    // rows a call of a few rows gains nothing (bf16 8 x 128 x 11 x 512 21.9, not halved 19.5).
    const bool pairs = S <= 1024 && (S >= 32 || B * H <= 512);
    if (ds % 128 != 0) {
      // fp32 1 x 128 x 265 x 192 16.3 against 21.6, 2 x 128 x 197 x 192 24.7 / 33.8, 1 x 64 x 313
      // x 192 13.3 / 14.6; past the line 1 x 64 x 281 x 448 (252 tiles) 18.9 / 18.0; 4 x 128 x 103 x
      // 320, 39.1 / 31.8, is the one shape measured more than 8 % slower.
      if (pairs && ((tiles(64) <= 128 && (S >= 32 || B == 1)) || (H >= 112 && tiles(64) <= 400)))
        return short_form<64, 4>(halves, 2);
    } else {
      // Halved 128-dim tiles of at most one per CU: fp32 1 x 128 x 100 x 512 18.3 against
      // 24.9, 1 x 128 x 185 23.3 / 28.9, 1 x 64 x 200 16.1 / 17.3, 1 x 64 x 246 (124 tiles) 18.0 /
      // 17.6; past the line 1 x 64 x 300 (152) 21.0 / 17.7.  Fewer yet: 64-dim tiles, fp32 1 x
      // 128 x 34 14.0 / 20.5, bf16 1 x 128 x 64 12.5 / 19.1.  Where the tiles and the exact rows do
      // not fit one round, halved tiles even the rounds (not halved: 64-dim tiles, which do
      // so too): fp32 1 x 128 x 420 x 512 41.9 / 48.8, 3 x 128 x 102 44.1 / 57.4, 2 x 64 x 300 31.2 /
      // 36.1, bf16 2 x 64 x 300 24.9 / 26.1.  8 heads in flight where a wave has 16 heads.
      if (pairs && tiles(64) <= 96) return short_form<64, 4>(halves, 2);
      if (pairs && (tiles(128) <= 128 || (tiles(128) < 320 && !fits)))
        return H >= 112 && B <= 2 ? short_form<128, 8>(halves, 2) : short_form<128, 4>(halves, 2);
      if (ds % 256 == 0 && tiles(256) >= 320) {
        // The long form halved, smaller workgroups than tiles that fill a second or
        // third round badly: fp32 1 x 128 x 1300 x 512 101.6 against 126.0, 1 x 64 x 1500
        // 64.0 / 71.3, past the line 1 x 64 x 1657 (416 tiles) 78.6 / 76.7; bf16 1 x 128 x 2400
        // 123.6 / 140.8, 1 x 64 x 2700 80.0 / 82.4, 2 x 128 x 1100 121.3 / 128.1, but 1 x 64 x 1800
        // (450 tiles) 60.2 / 54.7, 1 x 64 x 3400 (850) 96.7 / 93.5, 2 x 64 x 1500 (752) 84.3 / 79.4.
        if (halves ? B <= 2 && H >= 48 && tiles(256) <= 384
                   : tiles(256) >= 520 && (B == 1 ? H >= 64 && tiles(256) < 760
                                                  : B == 2 && H >= 96 && tiles(256) < 640))
          return long_form(halves, false, 2);
        // Three batches' exact rows and wide tiles: fp32 4 x 64 x 420 x 512 70.4 against
        // 85.9, bf16 4 x 128 x 420 92.3 / 106.4, 3 x 64 x 687 62.3 / 66.2, 4 x 64 x 850 93.7 / 103.2.
        if (B >= 3 && H >= 64) return short_form<128, 8>(halves, pairs ? 2 : 1);
      } else if (B >= 3 && pairs && tiles(128) >= 320) {
        // bf16 4 x 128 x 199 x 512 52.7 against 64.1 not halved, 8 x 64 x 132 37.8 / 41.2, fp32 4 x
        // 64 x 223 42.4 / 50.8; with two batches 2 x 128 x 457 60.0 / 57.7.
        return short_form<128, 8>(halves, 2);
      }
    }
  }
  // The widest tile with at least 320 workgroups, whose longer contiguous pieces of a
  // row memory serves faster; else 128 dims with all of a wave's 8 or more heads in
  // flight where they fit one round with the exact rows, else 64 dims.  320 is a measured
  // line, H = 64, D = 512, bf16 (B x S: the tile of this rule, the others in the order 512
  // / 256 / 128 / 64): 1 x 300, fp32: 128: 17.9, others 43.4 / 29.5 / - / 25.1; 2 x 1024: 256: 60.0, 68.5 /
  // - / 62.4 / 69.9; 2 x 1900: 512: 102.2, - / 116.6 / 111.5 / 121.9.  Before the short form (partial
  // planes, block totals, scan with the exact rows): 25.6, 62.1 and 109.3.
  if (ds % 512 == 0 && tiles(512) >= 320) return short_form<512, 4>(halves, 1);
  if (ds % 256 == 0 && tiles(256) >= 320) return short_form<256, 4>(halves, 1);
  if (ds % 128 == 0 && tiles(128) >= 320) return short_form<128, 4>(halves, 1);
  if (ds % 128 == 0 && fits) return short_form<128, 8>(halves, 1);
  return short_form<64, 4>(halves, 1);
}

// Dims of column slice `i` of D (slices of kSliceD, the last one shorter).
int64_t slice_dims(int64_t D, int64_t i) {
  const int64_t rest = D - i * kSliceD;
  return rest < kSliceD ? rest : kSliceD;
}

// The workspace holds one column slice at a time: the most any of D's slices
// (kSliceD wide, the last one D % kSliceD when that is not 0) needs.
int64_t workspace_bytes(int64_t B, int64_t S, int64_t D) {
  if (B < 0 || S < 0 || D < 0 || B > (1 << 20) || S > (1ll << 31) || D > (1ll << 31)) return -1;
  const int64_t nblk = (S + block_rows(S) - 1) / block_rows(S);
  auto slice_bytes = [&](int64_t w) {
    return (workspace_planes(B, S, w) * B * S + B * nblk) * w * 4;
  };
  const int64_t a = slice_bytes(D < kSliceD ? D : kSliceD);
  const int64_t b = D > kSliceD && D % kSliceD ? slice_bytes(D % kSliceD) : 0;
  return a > b ? a : b;
}

}  // namespace
}  // namespace mla
}  // namespace fagq

using namespace fagq;
using namespace fagq::mla;

extern "C" {

FAGQ_API int64_t fagq_mla_bwd_workspace_bytes(int64_t B, int64_t S, int64_t D) {
  return workspace_bytes(B, S, D);
}

}  // extern "C"

namespace fagq {
namespace mla {
namespace {

int check_sizes(int64_t B, int64_t H, int64_t S, int64_t D) {
  if (B < 0 || H < 1 || S < 1 || D < 64 || D % 64 != 0) return FAGQ_E_SHAPE;
  if (B > 65535 || H > 65535 || H * S * D * 4 >= (1ll << 32)) return FAGQ_E_TOO_LARGE;
  return FAGQ_OK;
}

// Argument checks shared by both entry points (everything but the workspace);
// *need receives the workspace bytes the call uses.
int check_args(const void* q, const void* c_kv, const void* out, const void* dout,
               const float* lse, void* dq, void* dc_kv, int64_t B, int64_t H, int64_t S,
               int64_t D, float sm_scale, int dq_dtype, int dc_dtype, int64_t* need) {
  if (!q || !c_kv || !out || !dout || !lse || !dq || !dc_kv) return FAGQ_E_NULL;
  if ((dq_dtype != FAGQ_MLA_F32 && dq_dtype != FAGQ_MLA_BF16) ||
      (dc_dtype != FAGQ_MLA_F32 && dc_dtype != FAGQ_MLA_BF16))
    return FAGQ_E_FORMAT;
  if (!(sm_scale == sm_scale)) return FAGQ_E_SHAPE;
  const int sizes = check_sizes(B, H, S, D);
  if (sizes != FAGQ_OK) return sizes;
  *need = workspace_bytes(B, S, D);
  if (*need < 0) return FAGQ_E_TOO_LARGE;
  if (!aligned(q, 16) || !aligned(c_kv, 16) || !aligned(out, 16) || !aligned(dout, 16) ||
      !aligned(lse, 4) || !aligned(dq, 16) || !aligned(dc_kv, 16))
    return FAGQ_E_ALIGN;
  return FAGQ_OK;
}

// Overlap checks with the workspace, the device check and the launches.
int launch(const void* q, const void* c_kv, const void* out, const void* dout, const float* lse,
           void* dq, void* dc_kv, void* workspace, int64_t need, int64_t B, int64_t H, int64_t S,
           int64_t D, float sm_scale, int dq_dtype, int dc_dtype, void* stream) {
  const int64_t nq = B * H * S * D * 2, nc = B * S * D * 2, nl = B * H * S * 4;
  const int64_t ndq = B * H * S * D * (dq_dtype == FAGQ_MLA_BF16 ? 2 : 4);
  const int64_t ndc = B * S * D * (dc_dtype == FAGQ_MLA_BF16 ? 2 : 4);
  const void* ins[5] = {q, c_kv, out, dout, lse};
  const int64_t nin[5] = {nq, nc, nq, nq, nl};
  void* outs[3] = {dq, dc_kv, workspace};
  const int64_t nout[3] = {ndq, ndc, need};
  for (int i = 0; i < 3; ++i) {
    for (int j = 0; j < 5; ++j)
      if (overlap(outs[i], nout[i], ins[j], nin[j])) return FAGQ_E_ALIAS;
    for (int j = i + 1; j < 3; ++j)
      if (overlap(outs[i], nout[i], outs[j], nout[j])) return FAGQ_E_ALIAS;
  }
  const int dcheck = device_check();
  if (dcheck != FAGQ_OK) return dcheck;

  // One pass per column slice; every slice's kernels run in stream order, so
  // each reuses the workspace after the previous slice's K3 has read it.
  const int64_t nslice = (D + kSliceD - 1) / kSliceD;
  const int64_t qb = dq_dtype == FAGQ_MLA_BF16 ? 2 : 4, cb = dc_dtype == FAGQ_MLA_BF16 ? 2 : 4;
  hipStream_t st = static_cast<hipStream_t>(stream);
  for (int64_t sl = 0; sl < nslice; ++sl) {
    const int64_t col = sl * kSliceD, ds = slice_dims(D, sl);
    MArgs g;
    g.q = static_cast<const uint16_t*>(q);         // the exact rows (first slice) read all of D
    g.c = static_cast<const uint16_t*>(c_kv);
    g.out = static_cast<const uint16_t*>(out);
    g.dout = static_cast<const uint16_t*>(dout) + col;
    g.lse = lse;
    g.dq = static_cast<uint8_t*>(dq) + col * qb;   // K1's rows; the exact rows run with col = 0
    g.dc = static_cast<uint8_t*>(dc_kv) + col * cb;
    g.nexact = sl == 0 ? (int32_t)H : 0;
    const Form f = pick_form(B, H, S, ds, g.nexact, dq_dtype == FAGQ_MLA_F32);
    g.planes = f.planes;
    g.hs_plane = B * S * ds;
    g.hs = static_cast<float*>(workspace);
    g.brows = (int32_t)block_rows(S);
    g.nblk = (int32_t)((S + g.brows - 1) / g.brows);
    g.tot = g.hs + g.planes * g.hs_plane;
    g.H = (int32_t)H;
    g.S = (int32_t)S;
    g.D = (int32_t)ds;
    g.ld = (int32_t)D;
    g.erows = (int32_t)(S < kE ? S : kE);
    g.scale = sm_scale;
    g.dq_bf16 = dq_dtype == FAGQ_MLA_BF16;
    g.dc_bf16 = dc_dtype == FAGQ_MLA_BF16;
    void* args[] = {&g};
    if (f.cw != 0) {
      const int64_t blocks = (S + kBlockRows - 1) / kBlockRows * (ds / f.cw) * f.planes;
      const size_t join = (size_t)kShortWaves * 64 * 8 * 4;   // 8 floats of each lane
      const size_t exact = g.nexact ? exact_lds_bytes(D) : 0;
      // nexact + blocks < 2^17 + 2^27: H S D 4 < 2^32 and D >= 64.
      int ls = launch_kernel(f.kernel, dim3((unsigned)(g.nexact + blocks), (unsigned)B),
                             dim3(64 * kShortWaves), args, join > exact ? join : exact, st);
      if (ls != FAGQ_OK) return ls;
      const void* scan = f.planes == 2 ? reinterpret_cast<const void*>(&mla_short_scan<2, 2>)
                                       : reinterpret_cast<const void*>(&mla_short_scan<1, kBlockRows>);
      ls = launch_kernel(scan, dim3((unsigned)g.nblk, (unsigned)B), dim3(kWide), args, 0, st);
      if (ls != FAGQ_OK) return ls;
      continue;
    }
    const int rows_per_wg = kThreads / (int)(ds / 8);
    const dim3 k1_grid((unsigned)((S + rows_per_wg - 1) / rows_per_wg), (unsigned)B,
                       (unsigned)f.planes);
    int ls = launch_kernel(f.kernel, k1_grid, dim3(kThreads), args, 0, st);
    if (ls != FAGQ_OK) return ls;
    // nblk < 2^20 and nexact + nblk < 2^17 + 2^20: nblk <= S / 16 + 1 and
    // H S D 4 < 2^32 with D >= 64.
    const void* totals = f.planes == 2 ? reinterpret_cast<const void*>(&mla_block_totals<2>)
                                       : reinterpret_cast<const void*>(&mla_block_totals<1>);
    ls = launch_kernel(totals, dim3((unsigned)g.nblk, (unsigned)B), dim3(kWide), args,
                       kBlockTotalLds, st);
    if (ls != FAGQ_OK) return ls;
    ls = launch_kernel(reinterpret_cast<const void*>(&mla_exact_rows_suffix_scan),
                       dim3((unsigned)(g.nexact + g.nblk), (unsigned)B), dim3(kWide), args,
                       g.nexact ? exact_lds_bytes(D) : 0, st);
    if (ls != FAGQ_OK) return ls;
  }
  return FAGQ_OK;
}

// The workspace of fagq_mla_bwd_launch_noalloc: one array per GPU the library
// runs on, held until the process ends.  Host code never passes `scratch`
// itself to a kernel (in host code the name is a stand-in, not the device
// address): the device address is looked up once per device, with that
// device current, and used instead.
static __device__ __align__(256) uint8_t scratch[FAGQ_MLA_SCRATCH_BYTES];

constexpr int kMaxScratchDevices = 64;
std::atomic<void*> g_scratch_addr[kMaxScratchDevices];
std::mutex g_scratch_mu;

// Device address of the current device's `scratch`; FAGQ_OK or an error.
int scratch_address(void** out) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return -(int)e;
  if (dev < 0 || dev >= kMaxScratchDevices) return FAGQ_E_DEVICE;
  void* p = g_scratch_addr[dev].load(std::memory_order_acquire);
  if (!p) {
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    p = g_scratch_addr[dev].load(std::memory_order_relaxed);
    if (!p) {
      e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
      if (e != hipSuccess) return -(int)e;
      if (!p) return FAGQ_E_DEVICE;
      g_scratch_addr[dev].store(p, std::memory_order_release);
    }
  }
  *out = p;
  return FAGQ_OK;
}

}  // namespace
}  // namespace mla
}  // namespace fagq

extern "C" {

FAGQ_API int fagq_mla_bwd_launch(const void* q, const void* c_kv, const void* out, const void* dout,
                                 const float* lse, void* dq, void* dc_kv, void* workspace,
                                 int64_t ws_bytes, int64_t B, int64_t H, int64_t S, int64_t D,
                                 float sm_scale, int dq_dtype, int dc_dtype, void* stream) {
  int64_t need = 0;
  const int v = check_args(q, c_kv, out, dout, lse, dq, dc_kv, B, H, S, D, sm_scale, dq_dtype,
                           dc_dtype, &need);
  if (v != FAGQ_OK) return v;
  if (!workspace) return FAGQ_E_NULL;
  if (ws_bytes < need) return FAGQ_E_SHAPE;
  if (!aligned(workspace, 16)) return FAGQ_E_ALIGN;
  if (B == 0) return FAGQ_OK;
  return launch(q, c_kv, out, dout, lse, dq, dc_kv, workspace, need, B, H, S, D, sm_scale,
                dq_dtype, dc_dtype, stream);
}

FAGQ_API int fagq_mla_bwd_query_route(int64_t B, int64_t H, int64_t S, int64_t D, int dq_dtype,
                                      int64_t slice, fagq_mla_route* route) {
  if (!route) return FAGQ_E_NULL;
  if (dq_dtype != FAGQ_MLA_F32 && dq_dtype != FAGQ_MLA_BF16) return FAGQ_E_FORMAT;
  const int sizes = check_sizes(B, H, S, D);
  if (sizes != FAGQ_OK) return sizes;
  if (slice < 0 || slice >= (D + kSliceD - 1) / kSliceD) return FAGQ_E_SHAPE;
  const int64_t ds = slice_dims(D, slice);
  const Form f = pick_form(B, H, S, ds, slice == 0 ? H : 0, dq_dtype == FAGQ_MLA_F32);
  route->dims = (int32_t)ds;
  route->tile_dims = f.cw;
  route->heads_in_flight = f.unroll;
  route->head_planes = f.planes;
  return FAGQ_OK;
}

FAGQ_API int fagq_mla_bwd_launch_noalloc(const void* q, const void* c_kv, const void* out,
                                         const void* dout, const float* lse, void* dq,
                                         void* dc_kv, int64_t B, int64_t H, int64_t S, int64_t D,
                                         float sm_scale, int dq_dtype, int dc_dtype, void* stream) {
  int64_t need = 0;
  const int v = check_args(q, c_kv, out, dout, lse, dq, dc_kv, B, H, S, D, sm_scale, dq_dtype,
                           dc_dtype, &need);
  if (v != FAGQ_OK) return v;
  if (need > FAGQ_MLA_SCRATCH_BYTES) return FAGQ_E_TOO_LARGE;
  if (B == 0) return FAGQ_OK;
  const int dcheck = device_check();
  if (dcheck != FAGQ_OK) return dcheck;
  void* ws = nullptr;
  const int sa = scratch_address(&ws);
  if (sa != FAGQ_OK) return sa;
  return launch(q, c_kv, out, dout, lse, dq, dc_kv, ws, need, B, H, S, D, sm_scale, dq_dtype,
                dc_dtype, stream);
}

}  // extern "C"

// MI355X (gfx950) kernels of the Davidson sigma step and the C-ABI around them.
//
// One H.C is a list of GEMM pairs (the flattened two-operator TensorMultiply
// of operatorfunctions.C:485-537), grouped by the V block they update:
//   W = alpha_a op(A) C        (first GEMM, operatorfunctions.C:512-516)
//   V += alpha W op(B)^T       (second GEMM, operatorfunctions.C:530)
// By the size of the V block and of a pair's depths:
//   up to 32: k_small (small_f64.h), a wavefront per work unit, W in registers;
//   up to 96, FP64: k_panel (panel_f64.h), 16 rows per wavefront, C in LDS;
//   33 to 64, split precision: k_sigma_bf, a workgroup per V tile that forms W
//   in LDS chunks from pre-split BF16 slices (v_mfma_f32_16x16x32_bf16) and
//   contracts each with B' at once;
//   larger: k_gemm (gemm_f64.h) and k_gemm_bf (gemm_bf.h), the two products as
//   LDS tiles of their own, W in scratch.
// k_sigma (k_sigma_bf's FP64 counterpart) and k_wave (one 16-row tile per
// wavefront) run where a tile-table rule names them.  Long pair lists are cut
// into work units whose partial tiles k_reduce adds in a fixed order, so V is
// reduced without atomics and bitwise reproducibly.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <array>
#include <atomic>
#include <functional>
#include <map>
#include <memory>
#include <mutex>
#include <thread>
#include <tuple>
#include <type_traits>
#include <unordered_map>
#include <cstdio>
#include <cstring>
#include <string>
#include <vector>

#include "../../include/block_sigma.h"

namespace {

thread_local std::string g_err;
int fail(int code, const std::string& msg) {
  g_err = msg;
  // a HIP error reported here is not the next launch's
  if (code != BSG_ERR_ARG) (void)hipGetLastError();
  return code;
}
#define HIPCHK(x)                                                                             \
  do {                                                                                        \
    hipError_t e_ = (x);                                                                      \
    if (e_ != hipSuccess) return fail(BSG_ERR_HIP, std::string(#x) + ": " + hipGetErrorString(e_)); \
  } while (0)

constexpr int TK = 16;  // K depth of one LDS slice

typedef double dbl4 __attribute__((ext_vector_type(4)));

struct TileRef {
  int32_t item, tm, tn, pad;
};

// Several right-hand sides (roots) in one launch: root r reads c + r
// wstride, accumulates into v + r wstride, keeps its partial tiles at part +
// r pstride, its BF16 C slices at cslices + r cstride and its W scratch at
// tstride times r.
struct RootSet {
  int32_t n;
  int32_t pad;
  int64_t wstride, pstride, cstride, tstride;
};
// Workgroup L of a launch over rs.n roots -> (tile t, root): the roots of one
// tile are dispatched next to each other, eight workgroups apart, so tile t
// runs on XCD t mod 8 (workgroup L runs on XCD L mod 8) for every root, and
// the roots share the tile's operator blocks in that XCD's L2.  The launch
// has roundup(ntiles, 8) rs.n workgroups.
__device__ inline int root_of(int L, int nroot, int& t) {
  const int g = L / (8 * nroot), rem = L - g * 8 * nroot;
  t = g * 8 + (rem & 7);
  return rem >> 3;
}



// A work unit: pairs [first, first+count) of one V block.  p_off < 0: the
// unit owns the whole pair list and accumulates into V; otherwise it writes
// its partial tile to P[p_off...] for k_reduce.
struct Seg {
  int32_t vb, first, count, pad;
  int64_t p_off;
};
// Ordered reduction of the partial tiles of one V block slice:
// V[v_off + e] += sum_s P[p_off + s*mn + e] for e in [e0, e0+len), len <= 64.
// Bound by the chain of loads (a V block has up to some hundred partial
// tiles): each wavefront takes every fourth tile with eight loads under way.
// On the D2h superblock at M = 1000 60 us with one thread per element, 27 us
// so (2.4 TB/s).
struct RedItem {
  int64_t v_off, p_off;
  int32_t nseg, mn, e0, len;
};

__global__ __launch_bounds__(256) void k_reduce(const RedItem* __restrict__ items, const double* __restrict__ part,
                                                double* __restrict__ v, RootSet rs) {
  __shared__ double sum[4][64];
  const RedItem it = items[blockIdx.x];
  part += blockIdx.y * rs.pstride;
  v += blockIdx.y * rs.wstride;
  const int e = threadIdx.x & 63, w = threadIdx.x >> 6;
  const bool in = e < it.len;
  const double* p = part + it.p_off + it.e0 + (in ? e : 0);
  double s = 0.0;
  int q = w;
  for (; q + 28 < it.nseg; q += 32) {
    double x[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = p[(int64_t)(q + 4 * i) * it.mn];
#pragma unroll
    for (int i = 0; i < 8; ++i) s += x[i];
  }
  {
    double x[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = q + 4 * i < it.nseg ? p[(int64_t)(q + 4 * i) * it.mn] : 0.0;
#pragma unroll
    for (int i = 0; i < 8; ++i) s += x[i];
  }
  sum[w][e] = s;
  __syncthreads();
  if (w == 0 && in) v[it.v_off + it.e0 + e] += (sum[0][e] + sum[1][e]) + (sum[2][e] + sum[3][e]);
}

// ---------------------------------------------------------------- FP64 grouped kernel
// Runs by tile-table rule.  A workgroup of 4 wavefronts owns a V
// panel tile: rows [row0, row0 + TM) and one column group of width JC (the
// whole block when n <= JC), with the waves arranged WR x WC (WR WC = 4),
// each wave owning NR 16-row blocks and PB = 2 16-wide column blocks (wc,
// wc + WC).  Per tile geometry (WR, NR) is chosen by the host per V block:
// TM = 16 NR WR <= 64, JC = 32 WC.  Two waves per SIMD (register budget 256).  Each W block is formed once per tile and
// padding is 16-granular.
//   GEMM 1: W chunk (TM x JC of W) = alpha_a op(A) C: op(A) staged through LDS
//           in 32-deep K chunks (double-buffered, shared by the waves of a
//           wave row), C column blocks straight into MFMA B operands; the
//           next chunk's loads are issued before the current chunk's MFMAs.
//   GEMM 2: V += alpha W B': the W chunk in LDS is the MFMA A operand, B'
//           column blocks go straight into B operands, 32 K deep per batch.
// Operand loads are raw buffer loads: masked lanes use an out-of-range offset
// and read zero, so no select follows a load.
constexpr int PB = 2;      // column blocks per wave
constexpr int PKC = 32;    // K depth of one staged op(A) chunk
constexpr int GTM = 64;    // largest tile height
constexpr int GP = GTM + 1;        // LDS pitch of k-major rows (doubles)
constexpr int GWS = 16 * PB * 4 * 33;  // W chunk doubles: max over geometries of JC (TM + 1)
constexpr uint32_t OOB = 0x80000000u;

__device__ inline __amdgpu_buffer_rsrc_t block_rsrc(const double* p, int64_t n) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)p, (short)0, (int)(n * 8), 0x00020000);
}
__device__ inline double bload(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0));
}
// voff: per-lane byte offset (OOB for a masked lane); soff: uniform byte offset
__device__ inline double bload2(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
  return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, 0));
}

// ---- split precision: three BF16 slices on the fly ----------------------
// An FP64 operand x is rounded to FP32 (error <= 2^-24 |x|) and split into
// BF16 slices h + m + l that represent that FP32 value exactly (8 + 8 + 8
// significant bits); BF16 keeps FP32's exponent range, so no block scale is
// needed.  A product keeps the six slice products of order <= 2^-16 (i+j <=
// 2), summed smallest first in FP32 by v_mfma_f32_16x16x32_bf16 (exact BF16
// products) for one 32-deep K group, and each group's FP32 result is added
// into FP64 accumulators.
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
__device__ inline void split_f32(double x, __bf16& h, __bf16& m, __bf16& l) {
  const float f = (float)x;
  h = (__bf16)f;
  const float r = f - (float)h;
  m = (__bf16)r;
  l = (__bf16)(r - (float)m);
}
// acc[r][t] += A(row blocks of this wave, 4-deep K step at k) * b[t] for the
// first nv column blocks and the first nr row blocks; A k-major in LDS.
template <int NRM, int NB>
__device__ inline void mma_step(int nv, int nr, dbl4 (&acc)[NRM][NB], const double* Al, int P, int arow, int k, int li,
                                int lk, const double (&b)[NB]) {
  const double a0 = Al[(k + lk) * P + arow + li];
  double a1 = 0.0;
  if (NRM > 1 && nr > 1) a1 = Al[(k + lk) * P + arow + 16 + li];
#pragma unroll
  for (int t = 0; t < NB; ++t) {
    if (t < nv) {
      acc[0][t] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b[t], acc[0][t], 0, 0, 0);
      if constexpr (NRM > 1)
        if (nr > 1) acc[1][t] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b[t], acc[1][t], 0, 0, 0);
    }
  }
}
// S K steps (4 S deep) from k0; steps at or past kend skipped, column slots
// past nv skipped (uniform branches)
template <int NRM, int NB, int S = 4>
__device__ inline void mma_run(int nv, int nr, dbl4 (&acc)[NRM][NB], const double* Al, int P, int arow, int k0, int kend,
                               int li, int lk, const double (&b)[S][NB]) {
  if (nv <= 0) return;
#pragma unroll
  for (int s = 0; s < S; ++s)
    if (k0 + 4 * s < kend) mma_step<NRM, NB>(nv, nr, acc, Al, P, arow, k0 + 4 * s, li, lk, b[s]);
}

// Tile geometry code in TileRef::pad: bits 0-1 log2(WR), bit 2 (NR - 1);
// NRM: row blocks per wave the accumulators hold (NR <= NRM).
// NV: V column blocks per wave (the V tile is 16 NV WC wide); the W chunk of
// GEMM 1 is PB blocks per wave (16 PB WC wide), so a V tile wider than the W
// chunk forms every W column once and contracts it into NV / PB chunks' worth
// of V columns.
// NWV: wavefronts per workgroup; with 8 they form one wave row of 8 columns
// of waves (a 16 x 768 tile for NV = 6 with the registers of the 384-wide
// one), so V blocks up to 768 wide form each W column once per row panel.
template <int NRM, int NV, int PBW = PB, int NWV = 4>
__global__ __launch_bounds__(64 * NWV) __attribute__((amdgpu_waves_per_eu(NV == 4 ? 3 : 2))) void k_sigma(
    const bsg_vblock_t* __restrict__ vbs, const bsg_pair_t* __restrict__ prs, const Seg* __restrict__ segs,
    const TileRef* __restrict__ tiles, int ntiles, const double* __restrict__ arena, const double* __restrict__ c,
    double* __restrict__ v, double* __restrict__ part, RootSet rs) {
  static_assert(NV % PBW == 0, "V tile width is a whole number of W chunks");
  static_assert(NWV == 4 || (NWV == 8 && NRM == 1 && PBW == PB), "eight waves: one wave row, 16-row tiles");
  constexpr int NT = 64 * NWV;
  // GEMM 1 uses two op(A) chunk buffers, GEMM 2 the W chunk; they share the
  // LDS (barriers separate the phases).  Both k-major: X[k * P + row].
  // W chunk: JC (TM + 1) doubles, JC = 16 PBW WC
  constexpr int WSD = NWV == 8 ? 16 * PBW * 8 * 17 : (PBW == PB ? GWS : 16 * PBW * 4 * 17);
  constexpr int LDSD = 2 * PKC * GP > WSD ? 2 * PKC * GP : WSD;
  __shared__ double lds[LDSD];
  double* const As0 = lds;
  double* const As1 = lds + PKC * GP;
  double* const Ws = lds;
  int tid;
  const int root = root_of(blockIdx.x, rs.n, tid);
  if (tid >= ntiles) return;
  c += root * rs.wstride;
  v += root * rs.wstride;
  part += root * rs.pstride;
  const TileRef tr = tiles[tid];
  if (tr.item < 0) return;  // padding of the XCD-interleaved order
  const Seg sg = segs[tr.item];
  const bsg_vblock_t vb = vbs[sg.vb];
  const int lwr = tr.pad & 3, nr = min(((tr.pad >> 2) & 1) + 1, NRM);
  const int WR = NWV == 8 ? 1 : 1 << lwr, WC = NWV == 8 ? 8 : 4 >> lwr;
  const int TM = 16 * nr * WR, JC = 16 * PBW * WC, JV = 16 * NV * WC, P = TM + 1;
  const int row0 = tr.tm * TM, colg = tr.tn * JV;
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wr = w / WC, wc = w % WC;
  const int arow = wr * nr * 16;  // first panel row of this wave
  const int li = lane & 15, lk = lane >> 4;
  // row blocks of this wave inside the block (0, 1 or 2)
  int nrw = (vb.m - row0 - arow + 15) / 16;
  nrw = nrw < 0 ? 0 : (nrw > nr ? nr : nrw);
  int nvb = 0;  // V column blocks of this wave that exist
  for (int t = 0; t < NV; ++t)
    if (colg + (wc + WC * t) * 16 < vb.n) nvb = t + 1;
  if (nrw == 0) nvb = 0;
  dbl4 accV[NRM][NV];
#pragma unroll
  for (int r = 0; r < NRM; ++r)
#pragma unroll
    for (int t = 0; t < NV; ++t) accV[r][t] = dbl4{0.0, 0.0, 0.0, 0.0};
  int abuf = 0;
  for (int q = 0; q < sg.count; ++q) {
    const bsg_pair_t pr = prs[sg.first + q];
    const __amdgpu_buffer_rsrc_t rC = block_rsrc(c + pr.c_off, (int64_t)pr.k1 * pr.k2);
    if (pr.a_off < 0 && pr.b_off < 0) {
      // identity A and B': V += alpha C
#pragma unroll
      for (int r = 0; r < NRM; ++r)
#pragma unroll
        for (int t = 0; t < NV; ++t) {
          const int col = colg + (wc + WC * t) * 16 + li;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int row = row0 + arow + r * 16 + lk + 4 * i;
            const bool ok = r < nr && row < vb.m && col < vb.n;
            accV[r][t][i] += pr.alpha * bload(rC, ok ? (uint32_t)(row * pr.k2 + col) * 8u : OOB);
          }
        }
      continue;
    }
    for (int j0 = 0; j0 < pr.k2; j0 += JC) {
      // identity B': only the W chunks of this tile's V columns
      if (pr.b_off < 0 && (j0 < colg || j0 >= colg + JV)) continue;
      const int jw = min(JC, pr.k2 - j0);        // W columns in this chunk
      int nwb = 0;                               // W column blocks of this wave in the chunk
      for (int t = 0; t < PBW; ++t)
        if ((wc + WC * t) * 16 < jw) nwb = t + 1;
      if (nrw == 0) nwb = 0;
      if (pr.a_off < 0) {
        // identity A: W = alpha C (panel rows of C)
        for (int e = threadIdx.x; e < TM * JC; e += NT) {
          const int j = e % JC, i = e / JC;
          const int gi = row0 + i;
          const bool ok = gi < vb.m && j < jw;
          Ws[j * P + i] = pr.alpha * bload(rC, ok ? (uint32_t)(gi * pr.k2 + j0 + j) * 8u : OOB);
        }
      } else {
        const __amdgpu_buffer_rsrc_t rA = block_rsrc(arena + pr.a_off, (int64_t)vb.m * pr.k1);
        dbl4 accW[NRM][PBW];
#pragma unroll
        for (int r = 0; r < NRM; ++r)
#pragma unroll
          for (int t = 0; t < PBW; ++t) accW[r][t] = dbl4{0.0, 0.0, 0.0, 0.0};
        // Pipeline over 32-deep chunks, each consumed in two 16-deep halves:
        // the op(A) elements of a chunk and the C operands of its first half
        // are loaded during the previous chunk's second half, the C operands
        // of the second half during the first half.  Per-lane offsets are
        // loop-invariant; the K position goes in the uniform offset.  Loads
        // past the end of a block read zero (buffer range check); op(A)
        // elements loaded past k1 inside the block only meet zero C rows.
        // wide tiles are always one 16-row block per wave in one wave row
        constexpr int AE = (NV > PB ? 16 : GTM) * PKC / NT;
        uint32_t aoff[AE];
#pragma unroll
        for (int u = 0; u < AE; ++u) {
          const int e = threadIdx.x + u * NT;
          const int i = pr.a_trans ? e % TM : e / PKC, p = pr.a_trans ? e / TM : e % PKC;
          const int gi = row0 + i;
          aoff[u] = e < TM * PKC ? (uint32_t)(pr.a_trans ? p * vb.m + gi : gi * pr.k1 + p) * 8u : OOB;
        }
        const uint32_t astep = (uint32_t)(pr.a_trans ? vb.m : 1) * 8u;  // bytes per K index
        uint32_t coff[PBW];
#pragma unroll
        for (int t = 0; t < PBW; ++t) {
          const int col = j0 + (wc + WC * t) * 16 + li;
          coff[t] = (t < nwb && col < pr.k2) ? (uint32_t)(lk * pr.k2 + col) * 8u : OOB;
        }
        const uint32_t crow = (uint32_t)pr.k2 * 8u;  // bytes per C row
        // C operands in batches of S1 K steps (8 deep for the 256-wide W
        // chunks: register budget); each batch is loaded while the previous
        // one runs, and the last batch of a chunk overlaps the next chunk's
        // op(A) and first C loads
        constexpr int S1 = PBW > PB ? 2 : 4;
        double an[AE], bn[S1][PBW];
        auto load_a = [&](int k0) {
#pragma unroll
          for (int u = 0; u < AE; ++u)
            if (u * NT < TM * PKC) an[u] = bload2(rA, aoff[u], (uint32_t)k0 * astep);
        };
        auto load_c = [&](int k0, int kh) {  // C rows k0 + kh .. k0 + kh + 4 S1 - 1
#pragma unroll
          for (int s4 = 0; s4 < S1; ++s4)
#pragma unroll
            for (int t = 0; t < PBW; ++t) bn[s4][t] = bload2(rC, coff[t], (uint32_t)(k0 + kh + 4 * s4) * crow);
        };
        load_a(0);
        load_c(0, 0);
        for (int k0 = 0; k0 < pr.k1; k0 += PKC) {
          const int kc = min(PKC, pr.k1 - k0);
          double* Ab = abuf ? As1 : As0;
          abuf ^= 1;
#pragma unroll
          for (int u = 0; u < AE; ++u) {
            const int e = threadIdx.x + u * NT;
            if (u * NT < TM * PKC && e < TM * PKC) {
              const int i = pr.a_trans ? e % TM : e / PKC, p = pr.a_trans ? e / TM : e % PKC;
              Ab[p * P + i] = pr.alpha_a * an[u];
            }
          }
          double bc[S1][PBW];
#pragma unroll
          for (int s4 = 0; s4 < S1; ++s4)
#pragma unroll
            for (int t = 0; t < PBW; ++t) bc[s4][t] = bn[s4][t];
          __syncthreads();
          if constexpr (S1 == 4) {
            // two 16-deep halves
            if (kc > 16) load_c(k0, 16);
            mma_run<NRM, PBW>(nwb, nrw, accW, Ab, P, arow, 0, kc, li, lk, bc);
            if (kc > 16) {
#pragma unroll
              for (int s4 = 0; s4 < 4; ++s4)
#pragma unroll
                for (int t = 0; t < PBW; ++t) bc[s4][t] = bn[s4][t];
            }
            if (k0 + PKC < pr.k1) {
              load_a(k0 + PKC);
              load_c(k0 + PKC, 0);
            }
            if (kc > 16) mma_run<NRM, PBW>(nwb, nrw, accW, Ab, P, arow, 16, kc, li, lk, bc);
          } else {
            for (int kh = 0; kh < kc; kh += 4 * S1) {
              const bool more = kh + 4 * S1 < kc;
              if (more) {
                load_c(k0, kh + 4 * S1);
              } else if (k0 + PKC < pr.k1) {
                load_a(k0 + PKC);
                load_c(k0 + PKC, 0);
              }
              mma_run<NRM, PBW, S1>(nwb, nrw, accW, Ab, P, arow, kh, kc, li, lk, bc);
              if (more) {
#pragma unroll
                for (int s4 = 0; s4 < S1; ++s4)
#pragma unroll
                  for (int t = 0; t < PBW; ++t) bc[s4][t] = bn[s4][t];
              }
            }
          }
        }
        __syncthreads();  // op(A) buffers done before W (same LDS) is written
        if (pr.b_off < 0) {
          // identity B': the W blocks of this wave are V blocks t + ch PBW
          // of the tile, ch = the chunk's position in the tile
          const int ch = (j0 - colg) / JC;
#pragma unroll
          for (int cc = 0; cc < NV / PBW; ++cc)
            if (cc == ch)
#pragma unroll
              for (int r = 0; r < NRM; ++r)
#pragma unroll
                for (int t = 0; t < PBW; ++t)
#pragma unroll
                  for (int i = 0; i < 4; ++i) accV[r][cc * PBW + t][i] += pr.alpha * accW[r][t][i];
          continue;
        }
#pragma unroll
        for (int r = 0; r < NRM; ++r)
#pragma unroll
          for (int t = 0; t < PBW; ++t) {
            const int cb = wc + WC * t;
            if (r < nr)
#pragma unroll
              for (int i = 0; i < 4; ++i) Ws[(cb * 16 + li) * P + arow + r * 16 + lk + 4 * i] = pr.alpha * accW[r][t][i];
          }
      }
      __syncthreads();
      // GEMM 2: V[tile] += W chunk * B'[j0:j0+jw, tile columns]; W columns
      // past jw up to the next multiple of 4 are zero.  B' operands of the
      // next batch (16 deep, 8 for the widest tiles: register budget) are
      // loaded while the current one runs.
      {
        constexpr int S2 = NV >= 6 || PBW > PB ? 2 : 4;
        const __amdgpu_buffer_rsrc_t rB = block_rsrc(arena + pr.b_off, (int64_t)vb.n * pr.k2);
        // B'(k, col) at k * ks + col * cs inside the block
        const int ks = pr.b_trans ? 1 : vb.n, cs = pr.b_trans ? pr.k2 : 1;
        // per-lane offsets loop-invariant, K position in the uniform offset;
        // rows past k2 read zero or meet zero W columns
        uint32_t boff[NV];
#pragma unroll
        for (int t = 0; t < NV; ++t) {
          const int col = colg + (wc + WC * t) * 16 + li;
          boff[t] = (t < nvb && col < vb.n) ? (uint32_t)(lk * ks + col * cs) * 8u : OOB;
        }
        const uint32_t bstep = (uint32_t)ks * 8u;
        double bn[S2][NV];
        auto load_b = [&](int kg) {
#pragma unroll
          for (int s4 = 0; s4 < S2; ++s4)
#pragma unroll
            for (int t = 0; t < NV; ++t) bn[s4][t] = bload2(rB, boff[t], (uint32_t)(j0 + kg + 4 * s4) * bstep);
        };
        load_b(0);
        for (int kg = 0; kg < jw; kg += 4 * S2) {
          double bb[S2][NV];
#pragma unroll
          for (int s4 = 0; s4 < S2; ++s4)
#pragma unroll
            for (int t = 0; t < NV; ++t) bb[s4][t] = bn[s4][t];
          if (kg + 4 * S2 < jw) load_b(kg + 4 * S2);
          mma_run<NRM, NV, S2>(nvb, nrw, accV, Ws, P, arow, kg, jw, li, lk, bb);
        }
      }
      __syncthreads();
    }
  }
  const bool direct = sg.p_off < 0;
  double* out = direct ? v + vb.v_off : part + sg.p_off;
#pragma unroll
  for (int r = 0; r < NRM; ++r)
#pragma unroll
    for (int t = 0; t < NV; ++t) {
      const int col = colg + (wc + WC * t) * 16 + li;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = row0 + arow + r * 16 + lk + 4 * i;
        if (r < nr && row < vb.m && col < vb.n) {
          if (direct)
            out[(size_t)row * vb.n + col] += accV[r][t][i];
          else
            out[(size_t)row * vb.n + col] = accV[r][t][i];
        }
      }
    }
}

// ---------------------------------------------------------------- split-precision grouped kernel
// The grouped kernel's tiles and work units with every operand already in
// three BF16 slices (x = h + m + l, the exact FP32 rounding of x):
//   op(A) blocks, row-major with K contiguous   (built once per arena)
//   B' blocks, [V column][K] with K contiguous  (built once per arena)
//   C blocks transposed, [k2][k1]               (built per application)
// each slice padded to a multiple of 8 along K and zero there.  A lane's 8
// K slots are then one 16-byte load per slice (K = 8 lk .. 8 lk + 7 for lane
// (li, lk), the same bijection for both MFMA operands).  GEMM 1 runs in the
// transposed orientation W^T = C^T op(A)^T so that a lane's result registers
// hold 4 consecutive W columns of one W row: they are scaled, split and
// written to LDS as one 8-byte store per slice, the layout GEMM 2 reads as
// its A operand.  Identity-B' pairs keep the direct orientation, whose result
// layout is the V accumulators'.  Each 32-deep K group is 6 slice products
// (i + j <= 2, smallest first) in FP32, added into FP64 accumulators.
typedef int i32x4 __attribute__((ext_vector_type(4)));
struct PairS {
  int64_t a, b, c;  // BF16 element offsets of the op(A), B' and C^T slice 0 (-1: identity)
};
struct SliceItem {
  // element (r, k) of the sliced matrix is src[trans ? k rows + r : r cols + k]
  // for k < cols, zero for cols <= k < pitch; slice s at dst + s rows pitch
  int64_t src, dst;
  int32_t rows, cols, pitch, trans;
};
struct Frag {
  bf16x8 h, m, l;
};
__device__ inline bf16x8 bload8(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
  return __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0));
}
__device__ inline __amdgpu_buffer_rsrc_t slice_rsrc(const __bf16* p, int64_t elems) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)p, (short)0, (int)(elems * 2), 0x00020000);
}
__device__ inline void mma6(dbl4& acc, const Frag& a, const Frag& b) {
  f32x4 x = {0.f, 0.f, 0.f, 0.f};
  x = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.l, b.h, x, 0, 0, 0);
  x = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.m, b.m, x, 0, 0, 0);
  x = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.h, b.l, x, 0, 0, 0);
  x = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.m, b.h, x, 0, 0, 0);
  x = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.h, b.m, x, 0, 0, 0);
  x = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.h, b.h, x, 0, 0, 0);
#pragma unroll
  for (int i = 0; i < 4; ++i) acc[i] += (double)x[i];
}

// A wavefront's share of the slicing: groups of 8 K (one 16-byte store per
// slice) [first, first + SLICE_GROUPS) of an item.
struct SliceChunk {
  int32_t item, first;
};
constexpr int SLICE_GROUPS = 256;
// lanes of an item's groups, padded to whole tiles
__host__ __device__ inline int slice_groups(const SliceItem& it) {
  return it.trans ? ((it.rows + 15) >> 4) * ((it.pitch + 31) >> 5) * 64 : it.rows * (it.pitch >> 3);
}
// Groups run along K where the source's K is contiguous; where its rows are, a
// wavefront takes tiles of 16 rows x 32 K, so that it reads 128 bytes and
// writes 64 bytes at a time.  (One
// workgroup per block and one element per thread left a superblock of few
// large blocks on a few CUs and stored 2 bytes at a time: 0.195 ms for the
// 24 blocks of a 315,905-element wavefunction.)
__global__ __launch_bounds__(256) void k_slices(const SliceChunk* __restrict__ chunks, int nchunks,
                                                const SliceItem* __restrict__ items, const double* __restrict__ src,
                                                __bf16* __restrict__ dst, int64_t src_stride, int64_t dst_stride) {
  const int ci = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (ci >= nchunks) return;
  const SliceChunk ch = chunks[ci];
  const SliceItem it = items[ch.item];
  src += blockIdx.y * src_stride + it.src;
  dst += blockIdx.y * dst_stride + it.dst;
  const int gk = it.pitch >> 3;
  const int64_t tot = (int64_t)it.rows * it.pitch;
  const int last = min(ch.first + SLICE_GROUPS, slice_groups(it)), lane = threadIdx.x & 63;
  const int tr = (it.rows + 15) >> 4;  // tiles along the rows
  for (int g0 = ch.first; g0 < last; g0 += 64) {
    int r, k0;
    if (it.trans) {
      const int t = g0 >> 6, tk = t / tr;
      r = 16 * (t - tk * tr) + (lane >> 2);
      k0 = 32 * tk + 8 * (lane & 3);
      if (r >= it.rows || k0 >= it.pitch) continue;
    } else {
      const int g = g0 + lane;
      r = g / gk;
      k0 = 8 * (g - r * gk);
      if (r >= it.rows) continue;
    }
    const double* q = src + (it.trans ? (int64_t)k0 * it.rows + r : (int64_t)r * it.cols + k0);
    const int64_t step = it.trans ? it.rows : 1;
    double x[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = k0 + e < it.cols ? q[e * step] : 0.0;
    bf16x8 h, m, l;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      __bf16 a, b, c;
      split_f32(x[e], a, b, c);
      h[e] = a;
      m[e] = b;
      l[e] = c;
    }
    __bf16* o = dst + (int64_t)r * it.pitch + k0;
    *(bf16x8*)o = h;
    *(bf16x8*)(o + tot) = m;
    *(bf16x8*)(o + 2 * tot) = l;
  }
}

constexpr int SAP = 40;                 // LDS pitch (BF16) of a staged op(A) row: 32 K + 8
constexpr int SAB = 3 * GTM * SAP;      // one staged op(A) chunk, 3 slices
constexpr int SWMAX = 3 * 64 * 72;      // W chunk slices: max over geometries of 3 TM (JC + 8)

// NRM, NV: as for the FP64 kernel (row blocks per wave the accumulators
// hold, V column blocks per wave).  NWV: wavefronts per workgroup; with 8
// they form one wave row of 8 columns of waves (16 x 512 for NV = 4, the
// registers of the 256-wide tile), so V blocks up to 512 wide form each W
// column once per row panel.
template <int NRM, int NV, int NWV = 4>
__global__ __launch_bounds__(64 * NWV) __attribute__((amdgpu_waves_per_eu(2))) void k_sigma_bf(
    const bsg_vblock_t* __restrict__ vbs, const bsg_pair_t* __restrict__ prs, const PairS* __restrict__ pss,
    const Seg* __restrict__ segs, const TileRef* __restrict__ tiles, int ntiles, const __bf16* __restrict__ slices,
    const __bf16* __restrict__ cslices, const double* __restrict__ c, double* __restrict__ v,
    double* __restrict__ part, RootSet rs) {
  // two op(A) chunk buffers for GEMM 1, the W chunk for GEMM 2 (aliased,
  // barriers separate the phases)
  constexpr int LDSE = 2 * SAB > SWMAX ? 2 * SAB : SWMAX;
  __shared__ __attribute__((aligned(16))) __bf16 lds[LDSE];
  int tid;
  const int root = root_of(blockIdx.x, rs.n, tid);
  if (tid >= ntiles) return;
  c += root * rs.wstride;
  v += root * rs.wstride;
  part += root * rs.pstride;
  cslices += root * rs.cstride;
  const TileRef tr = tiles[tid];
  if (tr.item < 0) return;
  const Seg sg = segs[tr.item];
  const bsg_vblock_t vb = vbs[sg.vb];
  static_assert(NV % PB == 0, "V tile width is a whole number of W chunks");
  static_assert(NWV == 4 || (NWV == 8 && NRM == 1), "eight waves: one wave row, 16-row tiles");
  constexpr int NT = 64 * NWV;
  const int lwr = tr.pad & 3, nr = min(((tr.pad >> 2) & 1) + 1, NRM);
  const int WR = NWV == 8 ? 1 : 1 << lwr, WC = NWV == 8 ? 8 : 4 >> lwr;
  const int TM = 16 * nr * WR, JC = 16 * PB * WC, JV = 16 * NV * WC, WP = JC + 8;
  const int row0 = tr.tm * TM, colg = tr.tn * JV;
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wr = w / WC, wc = w % WC;
  const int arow = wr * nr * 16;
  const int li = lane & 15, lk = lane >> 4;
  int nrw = (vb.m - row0 - arow + 15) / 16;
  nrw = nrw < 0 ? 0 : (nrw > nr ? nr : nrw);
  int nvb = 0;
  for (int t = 0; t < NV; ++t)
    if (colg + (wc + WC * t) * 16 < vb.n) nvb = t + 1;
  if (nrw == 0) nvb = 0;
  dbl4 accV[NRM][NV];
#pragma unroll
  for (int r = 0; r < NRM; ++r)
#pragma unroll
    for (int t = 0; t < NV; ++t) accV[r][t] = dbl4{0.0, 0.0, 0.0, 0.0};
  // op(A) staging: piece u (8 BF16) of a chunk is slice u / (4 TM), row
  // (u / 4) % TM, K quarter u % 4; three pieces per thread at most (one on
  // the wide tiles, which are 16 rows)
  constexpr int SPT = ((NV > PB ? 16 : GTM) * 12 + NT - 1) / NT;
  int abuf = 0;
  for (int q = 0; q < sg.count; ++q) {
    const bsg_pair_t pr = prs[sg.first + q];
    const PairS ps = pss[sg.first + q];
    const int k1p = (pr.k1 + 7) & ~7, k2p = (pr.k2 + 7) & ~7;
    if (pr.a_off < 0 && pr.b_off < 0) {  // V += alpha C
      const __amdgpu_buffer_rsrc_t rC = block_rsrc(c + pr.c_off, (int64_t)pr.k1 * pr.k2);
#pragma unroll
      for (int r = 0; r < NRM; ++r)
#pragma unroll
        for (int t = 0; t < NV; ++t) {
          const int col = colg + (wc + WC * t) * 16 + li;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int row = row0 + arow + r * 16 + 4 * lk + i;
            const bool ok = r < nr && row < vb.m && col < vb.n;
            accV[r][t][i] += pr.alpha * bload(rC, ok ? (uint32_t)(row * pr.k2 + col) * 8u : OOB);
          }
        }
      continue;
    }
    for (int j0 = 0; j0 < pr.k2; j0 += JC) {
      // identity B': only the W chunks of this tile's V columns
      if (pr.b_off < 0 && (j0 < colg || j0 >= colg + JV)) continue;
      const int jw = min(JC, pr.k2 - j0);
      int nwb = 0;
      for (int t = 0; t < PB; ++t)
        if ((wc + WC * t) * 16 < jw) nwb = t + 1;
      if (nrw == 0) nwb = 0;
      if (pr.a_off < 0) {
        const __amdgpu_buffer_rsrc_t rC = block_rsrc(c + pr.c_off, (int64_t)pr.k1 * pr.k2);
        // W = alpha C (panel rows), split into the W slices
        for (int e = threadIdx.x; e < TM * JC; e += NT) {
          const int j = e % JC, i = e / JC;
          const int gi = row0 + i;
          const bool ok = gi < vb.m && j < jw;
          __bf16 h, m, l;
          split_f32(pr.alpha * bload(rC, ok ? (uint32_t)(gi * pr.k2 + j0 + j) * 8u : OOB), h, m, l);
          lds[i * WP + j] = h;
          lds[TM * WP + i * WP + j] = m;
          lds[2 * TM * WP + i * WP + j] = l;
        }
      } else {
        const __amdgpu_buffer_rsrc_t rA = slice_rsrc(slices + ps.a, 3 * (int64_t)vb.m * k1p);
        const __amdgpu_buffer_rsrc_t rC = slice_rsrc(cslices + ps.c, 3 * (int64_t)pr.k2 * k1p);
        const uint32_t aslice = (uint32_t)vb.m * k1p * 2u, cslice = (uint32_t)pr.k2 * k1p * 2u;  // bytes per slice
        dbl4 accW[NRM][PB];
#pragma unroll
        for (int r = 0; r < NRM; ++r)
#pragma unroll
          for (int t = 0; t < PB; ++t) accW[r][t] = dbl4{0.0, 0.0, 0.0, 0.0};
        uint32_t aoff[SPT];
        int alds[SPT], aq[SPT];
#pragma unroll
        for (int x = 0; x < SPT; ++x) {
          const int u = threadIdx.x + NT * x;
          const int s = u / (4 * TM), i = (u >> 2) % TM, kq = u & 3;
          const bool ok = u < 12 * TM && row0 + i < vb.m;
          aoff[x] = ok ? (uint32_t)s * aslice + (uint32_t)((row0 + i) * k1p + 8 * kq) * 2u : OOB;
          alds[x] = u < 12 * TM ? (s * GTM + i) * SAP + 8 * kq : -1;
          aq[x] = 8 * kq;
        }
        uint32_t coff[PB];
#pragma unroll
        for (int t = 0; t < PB; ++t) {
          const int j = j0 + (wc + WC * t) * 16 + li;
          coff[t] = (t < nwb && j < pr.k2) ? (uint32_t)(j * k1p + 8 * lk) * 2u : OOB;
        }
        i32x4 an[SPT];
        Frag cn[PB];
        auto load_a = [&](int k0) {
#pragma unroll
          for (int x = 0; x < SPT; ++x)
            an[x] = __builtin_amdgcn_raw_buffer_load_b128(rA, k0 + aq[x] < k1p ? aoff[x] : OOB, (uint32_t)k0 * 2u, 0);
        };
        auto load_c = [&](int k0) {
          const bool in = k0 + 8 * lk < k1p;
#pragma unroll
          for (int t = 0; t < PB; ++t) {
            const uint32_t o = in ? coff[t] : OOB;
            cn[t].h = bload8(rC, o, (uint32_t)k0 * 2u);
            cn[t].m = bload8(rC, o, cslice + (uint32_t)k0 * 2u);
            cn[t].l = bload8(rC, o, 2u * cslice + (uint32_t)k0 * 2u);
          }
        };
        load_a(0);
        load_c(0);
        for (int k0 = 0; k0 < pr.k1; k0 += PKC) {
          __bf16* Ab = lds + abuf * SAB;
          abuf ^= 1;
#pragma unroll
          for (int x = 0; x < SPT; ++x)
            if (alds[x] >= 0) *(i32x4*)(Ab + alds[x]) = an[x];
          Frag cc[PB];
#pragma unroll
          for (int t = 0; t < PB; ++t) cc[t] = cn[t];
          __syncthreads();
          if (k0 + PKC < pr.k1) {
            load_a(k0 + PKC);
            load_c(k0 + PKC);
          }
          Frag af[NRM];
#pragma unroll
          for (int r = 0; r < NRM; ++r) {
            if (r >= nr) {
              af[r] = af[0];
              continue;
            }
            const int o = (arow + r * 16 + li) * SAP + 8 * lk;
            af[r].h = *(const bf16x8*)(Ab + o);
            af[r].m = *(const bf16x8*)(Ab + GTM * SAP + o);
            af[r].l = *(const bf16x8*)(Ab + 2 * GTM * SAP + o);
          }
#pragma unroll
          for (int t = 0; t < PB; ++t)
            if (t < nwb)
#pragma unroll
              for (int r = 0; r < NRM; ++r)
                if (r < nrw) {
                  if (pr.b_off < 0)
                    mma6(accW[r][t], af[r], cc[t]);  // W block: (row 4 lk + i, col li)
                  else
                    mma6(accW[r][t], cc[t], af[r]);  // W^T block: (W col 4 lk + i, W row li)
                }
        }
        __syncthreads();  // op(A) buffers done before the W slices (same LDS) are written
        const double aw = pr.alpha * pr.alpha_a;
        if (pr.b_off < 0) {
          // identity B': the W blocks of this wave are V blocks t + ch PB
          const int ch = (j0 - colg) / JC;
#pragma unroll
          for (int cc = 0; cc < NV / PB; ++cc)
            if (cc == ch)
#pragma unroll
              for (int r = 0; r < NRM; ++r)
#pragma unroll
                for (int t = 0; t < PB; ++t)
#pragma unroll
                  for (int i = 0; i < 4; ++i) accV[r][cc * PB + t][i] += aw * accW[r][t][i];
          continue;
        }
        // lane holds W(arow + 16 r + li, 16 cb + 4 lk + i), i < 4
#pragma unroll
        for (int r = 0; r < NRM; ++r)
          if (r < nr)
#pragma unroll
            for (int t = 0; t < PB; ++t) {
              const int cb = wc + WC * t;
              __bf16 hs[4], ms[4], ls[4];
#pragma unroll
              for (int i = 0; i < 4; ++i) split_f32(aw * accW[r][t][i], hs[i], ms[i], ls[i]);
              const int o = (arow + r * 16 + li) * WP + cb * 16 + 4 * lk;
              typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
              *(bf16x4*)(lds + o) = bf16x4{hs[0], hs[1], hs[2], hs[3]};
              *(bf16x4*)(lds + TM * WP + o) = bf16x4{ms[0], ms[1], ms[2], ms[3]};
              *(bf16x4*)(lds + 2 * TM * WP + o) = bf16x4{ls[0], ls[1], ls[2], ls[3]};
            }
      }
      __syncthreads();
      // GEMM 2: V[tile] += W chunk B'[j0 + .., tile columns], 32 deep per group
      {
        const __amdgpu_buffer_rsrc_t rB = slice_rsrc(slices + ps.b, 3 * (int64_t)vb.n * k2p);
        const uint32_t bslice = (uint32_t)vb.n * k2p * 2u;
        uint32_t boff[NV];
#pragma unroll
        for (int t = 0; t < NV; ++t) {
          const int col = colg + (wc + WC * t) * 16 + li;
          boff[t] = (t < nvb && col < vb.n) ? (uint32_t)(col * k2p + 8 * lk) * 2u : OOB;
        }
        Frag bn[NV];
        auto load_b = [&](int kg) {
          const bool in = j0 + kg + 8 * lk < k2p;
          const uint32_t so = (uint32_t)(j0 + kg) * 2u;
#pragma unroll
          for (int t = 0; t < NV; ++t) {
            const uint32_t o = in ? boff[t] : OOB;
            bn[t].h = bload8(rB, o, so);
            bn[t].m = bload8(rB, o, bslice + so);
            bn[t].l = bload8(rB, o, 2u * bslice + so);
          }
        };
        load_b(0);
        for (int kg = 0; kg < jw; kg += 32) {
          Frag bc[NV];
#pragma unroll
          for (int t = 0; t < NV; ++t) bc[t] = bn[t];
          if (kg + 32 < jw) load_b(kg + 32);
          Frag af[NRM];
#pragma unroll
          for (int r = 0; r < NRM; ++r) {
            if (r >= nr) {
              af[r] = af[0];
              continue;
            }
            const int o = (arow + r * 16 + li) * WP + kg + 8 * lk;
            af[r].h = *(const bf16x8*)(lds + o);
            af[r].m = *(const bf16x8*)(lds + TM * WP + o);
            af[r].l = *(const bf16x8*)(lds + 2 * TM * WP + o);
          }
#pragma unroll
          for (int r = 0; r < NRM; ++r)
            if (r < nrw)
#pragma unroll
              for (int t = 0; t < NV; ++t)
                if (t < nvb) mma6(accV[r][t], af[r], bc[t]);
        }
      }
      __syncthreads();
    }
  }
  const bool direct = sg.p_off < 0;
  double* out = direct ? v + vb.v_off : part + sg.p_off;
#pragma unroll
  for (int r = 0; r < NRM; ++r)
#pragma unroll
    for (int t = 0; t < NV; ++t) {
      const int col = colg + (wc + WC * t) * 16 + li;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = row0 + arow + r * 16 + 4 * lk + i;
        if (r < nr && row < vb.m && col < vb.n) {
          if (direct)
            out[(size_t)row * vb.n + col] += accV[r][t][i];
          else
            out[(size_t)row * vb.n + col] = accV[r][t][i];
        }
      }
    }
}

// ---------------------------------------------------------------- FP64 per-wave tiles
// Medium V blocks are latency-bound in the grouped kernel too: a pair's
// MFMAs are few next to its operand round trips, and a 4-wave tile runs one
// chain of round trips for 4 waves.  Here, as in the small-block kernel, each
// wavefront owns one tile of a V block (16 rows x 16 NB columns) for one work
// unit and walks the unit's pairs alone -- no LDS, no barriers, four
// unrelated tiles per workgroup -- so a CU keeps four times as many operand
// streams in flight.  A pair's op(A) row panel (16 rows x k1, k1 <= 4 KA)
// sits in registers; W^T = C^T op(A)^T is formed 16 W columns at a time and
// its result registers are at once GEMM 2's A operand against the matching
// 16 rows of B'.  On the 32-wide tiles (NB = 2) the C operands of the next
// 16 W columns are requested before the MFMAs of the current ones (two
// register sets, used in turn); the 64-wide tiles (NB = 4, which form each
// W column once for twice the V columns) spend that room on B' and keep one
// set.  The B' operands of a column group are requested before its GEMM 1
// MFMAs, and the next pair's descriptor before this pair's operands.
// Identity-B' pairs use the direct orientation W = op(A) C, whose result
// layout is the V accumulators'; identity-A pairs load W = alpha C straight
// into GEMM 2's operand layout.  Operands past a block's rows, columns or
// contraction depth read as zero (buffer range checks and masked lanes), and
// every C column past k2 is masked, so B' rows past k2 only meet zero W.
// 4-deep K steps of op(A) held in registers: k1 <= 64 on the 32-wide tiles,
// k1 <= 80 on the 64-wide ones (their single C register set leaves room)
constexpr int wave_ka(int nb) { return nb == 4 ? 20 : 16; }
template <int NB>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_wave(
    const bsg_vblock_t* __restrict__ vbs, const bsg_pair_t* __restrict__ prs, const Seg* __restrict__ segs,
    const TileRef* __restrict__ tiles, int ntiles, const double* __restrict__ arena, const double* __restrict__ c,
    double* __restrict__ v, double* __restrict__ part, RootSet rs) {
  constexpr int KA = wave_ka(NB);
  int g;
  const int root = root_of(blockIdx.x, rs.n, g);
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tid = g * 4 + w;
  if (tid >= ntiles) return;
  const TileRef tr = tiles[tid];
  if (tr.item < 0) return;  // padding: no tile for this wave (waves never synchronise here)
  c += root * rs.wstride;
  v += root * rs.wstride;
  part += root * rs.pstride;
  const Seg sg = segs[tr.item];
  const bsg_vblock_t vb = vbs[sg.vb];
  const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
  const int row0 = tr.tm * 16, col0 = tr.tn * 16 * NB;
  const bool rowok = row0 + li < vb.m;  // op(A) / W row li of the tile inside the block
  dbl4 accV[NB];  // register i of lane (li, lk): V(row0 + lk + 4 i, col0 + 16 t + li)
#pragma unroll
  for (int t = 0; t < NB; ++t) accV[t] = dbl4{0.0, 0.0, 0.0, 0.0};
  bsg_pair_t nxt = prs[sg.first];
  for (int q = 0; q < sg.count; ++q) {
    const bsg_pair_t pr = nxt;
    if (q + 1 < sg.count) nxt = prs[sg.first + q + 1];
    const __amdgpu_buffer_rsrc_t rC = block_rsrc(c + pr.c_off, (int64_t)pr.k1 * pr.k2);
    const uint32_t crow = (uint32_t)pr.k2 * 8u;
    if (pr.a_off < 0 && pr.b_off < 0) {  // identity A and B': V += alpha C
#pragma unroll
      for (int t = 0; t < NB; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int row = row0 + lk + 4 * i, col = col0 + t * 16 + li;
          const bool ok = row < vb.m && col < vb.n;
          accV[t][i] += pr.alpha * bload(rC, ok ? (uint32_t)(row * pr.k2 + col) * 8u : OOB);
        }
      continue;
    }
    const int nk1 = (pr.k1 + 3) / 4;
    double a[KA];  // a[s] = op(A)(row0 + li, 4 s + lk)
    if (pr.a_off >= 0) {
      const __amdgpu_buffer_rsrc_t rA = block_rsrc(arena + pr.a_off, (int64_t)vb.m * pr.k1);
      const int ar = pr.a_trans ? 1 : pr.k1, ak = pr.a_trans ? vb.m : 1;
      const uint32_t off = rowok ? (uint32_t)((row0 + li) * ar + lk * ak) * 8u : OOB;
#pragma unroll
      for (int s = 0; s < KA; ++s) a[s] = bload2(rA, s < nk1 ? off : OOB, (uint32_t)(s * ak) * 32u);
    }
    const double aw = pr.alpha_a * pr.alpha;
    if (pr.b_off < 0) {
      // identity B' (k2 = n): V(:, block t) += alpha alpha_a op(A) C(:, block t)
#pragma unroll
      for (int t = 0; t < NB; ++t) {
        const int col = col0 + t * 16 + li;
        if (col0 + t * 16 >= vb.n) break;
        const uint32_t coff = col < pr.k2 ? (uint32_t)(lk * pr.k2 + col) * 8u : OOB;
        double ct[KA];
#pragma unroll
        for (int s = 0; s < KA; ++s) ct[s] = bload2(rC, s < nk1 ? coff : OOB, (uint32_t)(4 * s) * crow);
        dbl4 accW = dbl4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int s4 = 0; s4 < KA; s4 += 4)
          if (s4 < nk1)
#pragma unroll
            for (int s = s4; s < s4 + 4; ++s) accW = __builtin_amdgcn_mfma_f64_16x16x4f64(a[s], ct[s], accW, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; ++i) accV[t][i] += aw * accW[i];
      }
      continue;
    }
    // B'(k, col) at k ks + col cs inside the block; per-lane offsets of the
    // tile's columns, the K position in the uniform offset
    const __amdgpu_buffer_rsrc_t rB = block_rsrc(arena + pr.b_off, (int64_t)vb.n * pr.k2);
    const int ks = pr.b_trans ? 1 : vb.n, cs = pr.b_trans ? pr.k2 : 1;
    uint32_t boff[NB];
#pragma unroll
    for (int t = 0; t < NB; ++t) {
      const int col = col0 + t * 16 + li;
      boff[t] = col < vb.n ? (uint32_t)(lk * ks + col * cs) * 8u : OOB;
    }
    const int njb = (pr.k2 + 15) / 16;
    if (pr.a_off < 0) {
      // identity A (k1 = m): W(row0 + li, 16 jb + 4 i + lk) = alpha C(...)
      for (int jb = 0; jb < njb; ++jb) {
        double wa[4], b[4][NB];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int k = jb * 16 + 4 * i + lk;
          wa[i] = pr.alpha * bload(rC, rowok && k < pr.k2 ? (uint32_t)((row0 + li) * pr.k2 + k) * 8u : OOB);
#pragma unroll
          for (int t = 0; t < NB; ++t) b[i][t] = bload2(rB, boff[t], (uint32_t)((jb * 16 + 4 * i) * ks) * 8u);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int t = 0; t < NB; ++t) accV[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(wa[i], b[i][t], accV[t], 0, 0, 0);
      }
      continue;
    }
    // W^T 16 columns at a time: ct[s] = C(4 s + lk, 16 jb + li) (columns past
    // k2 masked), b[i][t] = B'(16 jb + 4 i + lk, col0 + 16 t + li); the B'
    // operands of a column group are requested before its GEMM 1 MFMAs
    auto load_jb = [&](int jb, double (&ct)[KA]) {
      const int col = jb * 16 + li;
      const uint32_t coff = col < pr.k2 ? (uint32_t)(lk * pr.k2 + col) * 8u : OOB;
#pragma unroll
      for (int s = 0; s < KA; ++s) ct[s] = bload2(rC, s < nk1 ? coff : OOB, (uint32_t)(4 * s) * crow);
    };
    auto run_jb = [&](int jb, const double (&ct)[KA]) {
      double b[4][NB];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int t = 0; t < NB; ++t) b[i][t] = bload2(rB, boff[t], (uint32_t)((jb * 16 + 4 * i) * ks) * 8u);
      // register i of lane (li, lk): W(row0 + li, 16 jb + lk + 4 i)
      dbl4 accT = dbl4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int s4 = 0; s4 < KA; s4 += 4)
        if (s4 < nk1)
#pragma unroll
          for (int s = s4; s < s4 + 4; ++s) accT = __builtin_amdgcn_mfma_f64_16x16x4f64(ct[s], a[s], accT, 0, 0, 0);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const double wv = aw * accT[i];
#pragma unroll
        for (int t = 0; t < NB; ++t) accV[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(wv, b[i][t], accV[t], 0, 0, 0);
      }
    };
    if constexpr (NB <= 2) {
      double ct0[KA], ct1[KA];
      load_jb(0, ct0);
      for (int jb = 0; jb < njb; jb += 2) {
        if (jb + 1 < njb) load_jb(jb + 1, ct1);
        run_jb(jb, ct0);
        if (jb + 1 >= njb) break;
        if (jb + 2 < njb) load_jb(jb + 2, ct0);
        run_jb(jb + 1, ct1);
      }
    } else {  // one register set: the wider tile's B' operands take the room
      for (int jb = 0; jb < njb; ++jb) {
        double ct[KA];
        load_jb(jb, ct);
        run_jb(jb, ct);
      }
    }
  }
  const bool direct = sg.p_off < 0;
  double* out = direct ? v + vb.v_off : part + sg.p_off;
#pragma unroll
  for (int t = 0; t < NB; ++t) {
    const int col = col0 + t * 16 + li;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = row0 + lk + 4 * i;
      if (row < vb.m && col < vb.n) {
        if (direct)
          out[(size_t)row * vb.n + col] += accV[t][i];
        else
          out[(size_t)row * vb.n + col] = accV[t][i];
      }
    }
  }
}



#include "gemm_f64.h"
#include "panel_f64.h"
#include "small_f64.h"
#include "gemm_bf.h"

// Tile geometry of the grouped kernels for an m x n V block: waves WR x WC
// (WR WC = 4), NR 16-row blocks per wave (TM = 16 NR WR <= 64 rows), a W
// chunk of JC = 16 PB WC columns and a V tile of JV = 16 NV WC columns.
// NV = PB is the basic tile; the wide tiles (WR = 1, NR = 1, NV = 4 or 6)
// cover up to 256 or 384 V columns, so every W column of a pair is formed
// once per row panel instead of once per column group.  cls: the FP64
// kernel instantiation (0: <2, 2>, 1: <1, 4>, 2: <1, 6>, 3: <1, 6> of eight
// waves; split precision: 2: <1, 4> of eight waves).  Chosen to minimise
// the MFMA issue time of the block's tiles (per-wave MFMAs per pair, summed
// over tiles), which counts row padding, idle column slots and GEMM 1
// repeated per column group.
constexpr int NCLS = 4;
struct Geom {
  int lwr, nr, nv, tm, jc, jv, code, cls;
  int wc = 4, nw = 4;  // wave columns, waves per workgroup
};
// MFMAs of all waves of all tiles of a V block, in units of a 4-wave tile's
inline long geom_cost(const Geom& g, long m, long n, long k) {
  auto cdiv = [](long a, long b) { return (a + b - 1) / b; };
  const int wc = g.wc;
  const long panels = cdiv(m, g.tm), groups = cdiv(n, g.jv);
  const long wblk = cdiv(cdiv(k, 16), wc);  // W column blocks per wave (all chunks)
  const long vblk = std::max<long>(1, std::min<long>(g.nv, cdiv(std::min<long>(n, g.jv), 16 * wc)));
  return panels * groups * g.nr * (wblk + vblk) * cdiv(k, 4) * g.nw / 4;
}
inline Geom make_geom(int lwr, int nr, int nv) {
  Geom g;
  g.lwr = lwr;
  g.nr = nr;
  g.nv = nv;
  g.tm = 16 * nr * (1 << lwr);
  g.jc = 16 * PB * (4 >> lwr);
  g.jv = 16 * nv * (4 >> lwr);
  g.code = lwr | ((nr - 1) << 2);
  g.cls = nv / 2 - 1;
  g.wc = 4 >> lwr;
  return g;
}
// the 8-wave tiles: 16 rows, 8 wave columns of nv V column blocks (768 wide
// for the FP64 kernel's nv = 6, tile class 3; 512 for the split kernel's
// nv = 4, split tile class 2)
inline Geom make_geom_w8(int nv) {
  Geom g = make_geom(0, 1, nv);
  g.wc = 8;
  g.nw = 8;
  g.jc = 16 * PB * 8;
  g.jv = 16 * nv * 8;
  g.code = nv == 6 ? 8 : 16;
  g.cls = nv == 6 ? 3 : 2;
  return g;
}
// Measured tile choices (bsg_set_tile_table): for V blocks with m in
// [m_lo, m_hi] and n in [n_lo, n_hi], the index of the geometry to use in
// pick_geom's candidate list (FP64 and split-precision lists; -1: the
// model's choice).  Set before plans are created; read when they are.
struct TileRule {
  int32_t m_lo, m_hi, n_lo, n_hi, fp64, split;
};
struct RuleSet {
  std::vector<TileRule> rules;
  unsigned version = 0;  // pick_geom's cache key
};
std::shared_ptr<const RuleSet> g_tile_rules = std::make_shared<RuleSet>();
std::vector<Geom> geom_candidates(int max_nv) {
  std::vector<Geom> cand;
  for (int lwr = 0; lwr <= 2; ++lwr)
    for (int nr = 1; nr <= 2; ++nr) cand.push_back(make_geom(lwr, nr, PB));
  for (int nv = 4; nv <= max_nv; nv += 2) cand.push_back(make_geom(0, 1, nv));
  cand.push_back(make_geom_w8(max_nv >= 6 ? 6 : 4));
  return cand;
}
Geom pick_geom_uncached(const RuleSet& rs, int m, int n, int max_nv);
// pick_geom per V block shape, remembered per thread (plans repeat shapes)
inline Geom pick_geom(const RuleSet& rs, int m, int n, int max_nv) {
  thread_local std::unordered_map<uint64_t, Geom> cache;
  thread_local unsigned version = ~0u;
  if (version != rs.version) {
    cache.clear();
    version = rs.version;
  }
  const uint64_t key = ((uint64_t)(uint32_t)m << 33) | ((uint64_t)(uint32_t)n << 1) | (max_nv >= 6 ? 1u : 0u);
  auto f = cache.find(key);
  if (f != cache.end()) return f->second;
  const Geom g = pick_geom_uncached(rs, m, n, max_nv);
  cache.emplace(key, g);
  return g;
}
Geom pick_geom_uncached(const RuleSet& rs, int m, int n, int max_nv) {
  // typical contraction depth: the block's own dimensions
  const long k = std::max(m, n);
  // the two candidate lists, built once (pick_geom runs per V block)
  static const std::vector<Geom> cand_fp64 = geom_candidates(6), cand_split = geom_candidates(4);
  const std::vector<Geom>& cand = max_nv >= 6 ? cand_fp64 : cand_split;
  for (const TileRule& r : rs.rules)
    if (m >= r.m_lo && m <= r.m_hi && n >= r.n_lo && n <= r.n_hi) {
      const int idx = max_nv >= 6 ? r.fp64 : r.split;
      if (idx >= 0 && idx < (int)cand.size() && cand[idx].tm <= GTM) return cand[idx];
      break;
    }
  Geom best = cand[0];
  long bc = -1;
  for (const Geom& g : cand) {
    if (g.tm > GTM) continue;
    const long cst = geom_cost(g, m, n, k);
    if (bc < 0 || cst < bc || (cst == bc && g.tm > best.tm)) {
      bc = cst;
      best = g;
    }
  }
  return best;
}
// MFMA instructions of one pair in the small-block kernel plus an allowance
// for its loads (segment cost; the wave works alone)
template <class Pair>  // bsg_pair_t, PanelPair
inline long small_cost(int m, int n, const Pair& pr) {
  const long nrb = (m + 15) / 16, nnb = (n + 15) / 16, o = (std::max(pr.k1, pr.k2) + 7) / 8;
  return 2 * o * ((o + 1) / 2 * nrb + nrb * nnb) + 4;
}
// Per-wave tiles: 16 x 32 for V blocks up to 32 columns, 16 x 64 above
// (wave_nb).  In the FP64 column of the tile table the candidate index after
// the geometries selects them for a V block's pairs within their contraction
// depth (k1 <= 4 wave_ka, or identity A); the block's other pairs run on the
// geometry the model picks.  Without a rule, blocks stay on the grouped
// kernel.
inline int wave_nb(int n) { return n <= 32 ? 2 : 4; }
inline int wave_candidate() {
  static const int n = (int)geom_candidates(6).size();
  return n;
}
// candidate the tile table names for an m x n V block (-1: none)
inline int table_rule(const RuleSet& rs, int m, int n, bool split) {
  for (const TileRule& r : rs.rules)
    if (m >= r.m_lo && m <= r.m_hi && n >= r.n_lo && n <= r.n_hi) return split ? r.split : r.fp64;
  return -1;
}
// split-precision V blocks up to this on both sides stay on the grouped kernel
constexpr int SPLIT_GROUPED = 64;
// MFMA instructions of one pair in a per-wave tile plus a latency allowance
// (segment cost)
inline long wave_cost(int n, const bsg_pair_t& pr) {
  auto cdiv = [](long a, long b) { return (a + b - 1) / b; };
  const long nnb = std::min<long>(wave_nb(n), cdiv(n, 16)), njb = cdiv(pr.k2, 16), nk1 = cdiv(pr.k1, 4);
  if (pr.a_off < 0) return (pr.b_off < 0 ? 0 : njb * 4 * nnb) + 24;
  return (pr.b_off < 0 ? nnb * nk1 : njb * (nk1 + 4 * nnb)) + 24;
}
typedef GemmTile<2, 2, 2, 2, 4> GemmT;
typedef SplitTile<2, 4, 4, 2, 2> SplitBig;
typedef SplitTile<2, 2, 2, 2, 3> SplitSmall;
// 128 x 128 split tiles unless they pad an m x n product to much more than
// 64 x 64 ones would
inline int split_shape(int m, int n) {
  auto area = [&](int64_t t) { return ((m + t - 1) / t) * ((n + t - 1) / t) * t * t; };
  return 2 * area(128) <= 3 * area(64);
}
// ... in superblocks that fill the chip with such tiles.  The smaller shape
// alone and both take, by W tiles of 128: 4,900 0.71 and 0.74 ms (24 orbitals,
// C1, peak dimension 150), 11,000 1.04 to 1.20 and 1.05 to 1.20 (195 to 220),
// 10,900 of 20 orbitals 1.28 and 1.40, 13,300 1.80 and 1.69 (250), 17,800 2.28
// and 2.04 (280), 21,600 2.89 and 2.67 (313), 55,000 2.71 and 2.62 (36 orbitals,
// D2h, 79), 193,000 15.2 and 15.3 (190)
constexpr int64_t SPLIT_WIDE = 1 << 14;
// MFMA instructions per wavefront of one pair in a panel plus a latency
// allowance
inline long panel_cost(int n, int k1, int k2, bool a, bool b) {
  const long nb = (n + 15) / 16;
  if (!a && !b) return 8;
  if (!a || !b) return ((b ? k2 : k1) + 3) / 4 * nb + 24;
  return (k2 + 15) / 16 * (2L * ((k1 + 7) / 8) + 4 * nb) + 8;
}
inline long panel_cost(int n, const bsg_pair_t& pr) { return panel_cost(n, pr.k1, pr.k2, pr.a_off >= 0, pr.b_off >= 0); }
inline long panel_cost(int n, const PanelPair& pr) { return panel_cost(n, pr.k1, pr.k2, pr.a >= 0, pr.b >= 0); }
// The same of one pair in a V tile of the large blocks' products (16-deep
// chunks) plus its share of a chunk's overhead
inline long gemm_cost(const bsg_pair_t& pr) {
  if (pr.a_off < 0 && pr.b_off < 0) return 0;
  return ((pr.b_off < 0 ? pr.k1 : pr.k2) + GKC - 1) / GKC * 16 + 4;
}
// W scratch of the large blocks' rounds, in doubles: one round up to
// W_ONE_ROUND, else an even number of rounds of at most W_HALF each (W_HALF / 2
// and one unit's W where that is more: blocks of some 20,000 rows); roots
// share a launch while W_ROOTS holds all of them
constexpr int64_t W_ONE_ROUND = 1 << 23, W_HALF = 1 << 26, W_ROOTS = 1 << 29;
// MFMA instructions per wavefront of one pair in a tile (segment cost)
inline long pair_cost(const Geom& g, int n, const bsg_pair_t& pr) {
  auto cdiv = [](long a, long b) { return (a + b - 1) / b; };
  const int wc = g.wc;
  const long kw = pr.b_off < 0 ? std::min<long>(pr.k2, g.jv) : pr.k2;  // W columns formed per tile
  const long nch = cdiv(kw, g.jc);
  const long g1 = pr.a_off < 0 ? 0 : g.nr * cdiv(cdiv(kw, 16), wc) * cdiv(pr.k1, 4);
  const long g2 =
      pr.b_off < 0 ? 0 : g.nr * std::min<long>(g.nv, cdiv(cdiv(std::min<long>(n, g.jv), 16), wc)) * cdiv(pr.k2, 4);
  return g1 + g2 + 16 * nch;
}

// (cost, index) pairs, given by ascending index, to descending cost: counted
// into place where the costs are few (a rotation's tens of thousands of
// one-pair units; comparing them took a third of its plan's time)
inline void costliest_first(std::vector<std::pair<long, int>>& v) {
  constexpr long MOST = 1 << 16;
  long top = 0;
  for (const auto& x : v) top = std::max(top, x.first);
  if (v.size() < 512 || top >= MOST) {
    std::sort(v.begin(), v.end(), [](const std::pair<long, int>& a, const std::pair<long, int>& b) {
      return a.first != b.first ? a.first > b.first : a.second < b.second;
    });
    return;
  }
  std::vector<int32_t> at(top + 2, 0);
  for (const auto& x : v) ++at[top - x.first + 1];
  for (long k = 1; k <= top + 1; ++k) at[k] += at[k - 1];
  std::vector<std::pair<long, int>> to(v.size());
  for (const auto& x : v) to[at[top - x.first]++] = x;
  v.swap(to);
}

// Launch order of grouped tiles, panels and product tiles.  Workgroup i runs on XCD
// i mod 8, each XCD with its own L2: the tiles of one work unit share their
// C and B' blocks, so a unit's tiles go to one XCD, units are spread over
// the XCDs by cost (costliest first, to the least loaded XCD), each XCD's
// queue runs costliest units first, and the queues are interleaved
// (padding tiles with item -1 keep the positions aligned).
constexpr int NXCD = 8;
// a work unit's tiles: segment seg, ntm x ntn tiles of geometry code
struct GUnit {
  long cost = 0;
  int seg = 0, ntm = 0, ntn = 0, code = 0;
  long ntiles() const { return (long)ntm * ntn; }
};
inline std::vector<TileRef> xcd_order(std::vector<GUnit>& units) {
  // (work, index) pairs sorted by work descending, index ascending on ties
  std::vector<std::pair<long, int>> ord(units.size());
  for (size_t i = 0; i < ord.size(); ++i) ord[i] = {units[i].cost * units[i].ntiles(), (int)i};
  costliest_first(ord);
  std::vector<std::vector<TileRef>> q(NXCD);
  for (auto& v : q) v.reserve(units.size() / NXCD + 16);
  long load[NXCD] = {};
  for (const auto& o : ord) {
    int x = 0;
    for (int y = 1; y < NXCD; ++y)
      if (load[y] < load[x]) x = y;
    const GUnit& g = units[o.second];
    load[x] += o.first;
    for (int tm = 0; tm < g.ntm; ++tm)
      for (int tn = 0; tn < g.ntn; ++tn) q[x].push_back({g.seg, tm, tn, g.code});
  }
  size_t len = 0;
  for (auto& v : q) len = std::max(len, v.size());
  std::vector<TileRef> out;
  out.reserve(len * NXCD);
  for (size_t i = 0; i < len; ++i)
    for (int x = 0; x < NXCD; ++x) out.push_back(i < q[x].size() ? q[x][i] : TileRef{-1, 0, 0, 0});
  return out;
}

// ---------------------------------------------------------------- vector kernels
#include "vectors.h"

// one workgroup per chunk of at most COPY_CHUNK doubles
constexpr int64_t COPY_CHUNK = 16384;
__global__ __launch_bounds__(256) void k_copy_chunks(const bsg_copy_seg_t* __restrict__ chunks) {
  const bsg_copy_seg_t c = chunks[blockIdx.x];
  for (int64_t i = threadIdx.x; i < c.n; i += 256) c.dst[i] = c.src[i];
}

// Composite-operator build: groups of scaled block copies.  Group g owns the
// destination rectangle dst[r ld + c] (r < rows, c < cols) and the run of
// sources [first, first + count); its elements are numbered from
// estart[g] in one flat index space, 256 per workgroup, so small rectangles
// share workgroups.  Each element sums its sources in list order,
// (alpha a) beta per source, and adds the sum to the destination (zero
// beforehand): bitwise the host build's accumulation.
//
// Rectangles are some 10 x 10, so this is bound by the chain of loads that
// leads to an element's sources and by the cache lines that such rows touch.
// A wavefront looks for its first element's group together, 64 candidates a
// round, and its lanes take their groups from the 64 from there on.  17
// million elements of 152,000 rectangles: 506 us with a binary search for
// every element, 315 us so; a table of each workgroup's first group instead of
// the search takes 278 us, but the host longer to make than that saves.
__global__ __launch_bounds__(256) void k_build(const bsg_build_group_t* __restrict__ groups,
                                               const int64_t* __restrict__ estart, int ngroups,
                                               const bsg_build_src_t* __restrict__ srcs, int64_t nelem) {
  // no fused multiply-adds: the host build rounds every product and sum
#pragma clang fp contract(off)
  const int lane = threadIdx.x & 63;
  const int64_t e0 = (int64_t)blockIdx.x * 256 + (threadIdx.x & ~63), e = e0 + lane;
  if (e0 >= nelem) return;
  // last group whose start is <= e0: it is in [lo, lo + n)
  int lo = 0, n = ngroups;
  while (n > 1) {
    const int step = (n + 63) >> 6;
    const uint64_t le = __ballot((int64_t)lane * step < n && estart[lo + lane * step] <= e0);
    const int hit = 63 - __clzll(le);  // lane 0's holds
    lo += hit * step;
    n = min(step, n - hit * step);
  }
  // this lane's element: groups are not empty, so at most 63 further on
  const int64_t st = lane < ngroups - lo ? estart[lo + lane] : nelem;
  const uint64_t in = __ballot(st <= e0 + 63);
  int g0 = 0;
  int64_t x = e - __shfl(st, 0);
  for (int j = 1; j < 64 && ((in >> j) & 1); ++j) {
    const int64_t y = e - __shfl(st, j);
    if (y >= 0) {
      g0 = j;
      x = y;
    }
  }
  if (e >= nelem) return;
  const bsg_build_group_t g = groups[lo + g0];
  int r, c;
  if (x <= 0xffffffffLL) {
    r = (int)((uint32_t)x / (uint32_t)g.cols);
    c = (int)((uint32_t)x - (uint32_t)r * (uint32_t)g.cols);
  } else {
    r = (int)(x / g.cols);
    c = (int)(x % g.cols);
  }
  double* out = g.dst + (int64_t)r * g.ld + c;
  const double old = *out;
  double s = 0.0;
  for (int j = 0; j < g.count; ++j) {
    const bsg_build_src_t sj = srcs[g.first + j];
    const double a = sj.trans ? sj.src[(int64_t)c * sj.ld + r] : sj.src[(int64_t)r * sj.ld + c];
    s += (sj.alpha * a) * sj.beta;
  }
  *out = old + s;
}

// diag(H) by V block: item i covers elements [e0, e0 + 256) of the block of
// its term group; every thread sums the group's terms in list order for its
// element (alpha_t A_ii B_jj, identity partners read as 1).
struct DiagGroup {
  int32_t first, count;
};
struct DiagItem {
  int32_t group, e0;
};
__global__ __launch_bounds__(256) void k_diag(const bsg_diag_t* __restrict__ terms, const DiagGroup* __restrict__ groups,
                                              const DiagItem* __restrict__ items, const double* __restrict__ arena,
                                              double* __restrict__ diag) {
  const DiagItem it = items[blockIdx.x];
  const DiagGroup g = groups[it.group];
  const bsg_diag_t t0 = terms[g.first];
  const int64_t e = (int64_t)it.e0 + threadIdx.x;
  if (e >= (int64_t)t0.m * t0.n) return;
  const int i = (int)(e / t0.n), j = (int)(e % t0.n);
  double s = 0.0;
  for (int q = 0; q < g.count; ++q) {
    const bsg_diag_t t = terms[g.first + q];
    const double a = t.a_off < 0 ? 1.0 : arena[t.a_off + (int64_t)i * (t.m + 1)];
    const double b = t.b_off < 0 ? 1.0 : arena[t.b_off + (int64_t)j * (t.n + 1)];
    s += t.alpha * a * b;
  }
  diag[t0.v_off + e] += s;
}

// workgroups of a reduction over n elements, two per thread at least
int reduce_grid(int64_t n) { return (int)std::max<int64_t>(1, std::min<int64_t>(RMAXB, (n + 2 * RB - 1) / (2 * RB))); }
int grid_for(int64_t n) { return (int)std::max<int64_t>(1, std::min<int64_t>(2048, (n + 255) / 256)); }

}  // namespace

// ---------------------------------------------------------------- static scratch
// Partial tiles of bsg_sigma_apply_noalloc: a file-scope device array, one
// copy per GPU the library runs on, held until the process ends.  Host code
// never passes the array's name to a kernel (on the host it is a stand-in,
// not a device address): the address comes from hipGetSymbolAddress, once
// per device with that device current, and is kept per device.
__device__ __align__(256) double scratch[BSG_NOALLOC_SCRATCH_DOUBLES];
namespace {
constexpr int MAX_DEVICES = 64;
std::mutex g_scratch_mu;
double* g_scratch_ptr[MAX_DEVICES] = {};
// this device's scratch address (device current); nullptr with g_err set on failure
double* scratch_address(int device) {
  if (device < 0 || device >= MAX_DEVICES) {
    g_err = "static scratch: device index out of range";
    return nullptr;
  }
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (!g_scratch_ptr[device]) {
    void* ptr = nullptr;
    hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr) {
      g_err = std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e);
      return nullptr;
    }
    g_scratch_ptr[device] = static_cast<double*>(ptr);
  }
  return g_scratch_ptr[device];
}
}  // namespace

// ---------------------------------------------------------------- context and plan
// W scratch of the large blocks' products.  A context's applications run one
// after the other (its single stream; bsg_context::apply keeps the launches of
// calls from several threads apart), so its plans share one buffer: plans
// and their captured graphs keep the buffer they were made with, the context
// keeps the latest one up to W_ROOTS doubles for the next superblock's plan
// (until bsg_free), and the last holder frees it.  Sizes are whole powers of
// two up to there, so that a sweep's growing superblocks replace it a few times
// only: memory is cleared when it is given back, and freeing the 4 GB of four
// roots with every plan took 40 to 300 ms.
struct WScratch {
  double* ptr = nullptr;
  int64_t doubles = 0;
  ~WScratch() { (void)hipFree(ptr); }  // waits for the device
};

constexpr int COEF_SLOTS = 4;

struct bsg_context {
  int device = 0;
  std::mutex apply;                    // held while an application is enqueued or captured
  std::mutex wmu;                      // of wscratch
  std::shared_ptr<WScratch> wscratch;
  hipStream_t stream = nullptr;
  // second stream (default priority) for the kernels that run beside those on
  // `stream` (enqueue_chunk); fork/join events tie it to that
  hipStream_t side = nullptr;
  hipEvent_t fork = nullptr, join = nullptr;
  double* red = nullptr;  // two sets of two partial lists (RMAXB each)
  double* gpart = nullptr;  // Gram partials (GBLK GMAX^2) + coefficient slots (GRAM_MAX^2 each)
  bsg_copy_seg_t* copy_list = nullptr;  // chunk list of bsg_copy_segments (grown on demand)
  size_t copy_cap = 0;
  // page-locked staging of bsg_lincomb's coefficients, used in turn (GRAM_MAX^2
  // each), their last copies to the device, and results (GRAM_MAX^2)
  double* coef_pin = nullptr;
  hipEvent_t coef_done[COEF_SLOTS] = {};
  int coef_next = 0;
  double* res_pin = nullptr;
  double* scratch = nullptr;  // this device's copy of the static scratch (bsg_sigma_apply_noalloc)
  // operator-slice buffer lent to one split-precision plan at a time (grown
  // on demand), so successive superblocks do not allocate and free it
  __bf16* abs_buf = nullptr;
  size_t abs_cap = 0;  // elements
  bool abs_leased = false;
};

// One round of the large blocks' products: the W tiles, then the V tiles
// that read them.  Rounds alternate between the context stream and the side
// stream, each with its own half of the W scratch, so that one round's last
// tiles run beside the next round's first.
struct GemmRound {
  TileRef *d_w[2] = {}, *d_v[2] = {};  // W tiles, V tiles by tile shape (FP64: the first only)
  int n_w[2] = {}, n_v[2] = {};
};

// Launch lists of one precision mode of a chunk
struct ModeLists {
  bool ready = false;
  void* d_blob = nullptr;        // one device allocation holding the arrays below
  Seg* d_seg = nullptr;
  TileRef* d_g[NCLS] = {};       // grouped-kernel tiles per kernel class (split: basic, 256 wide, 512 wide)
  int n_g[NCLS] = {};
  int32_t* d_s[3] = {};          // FP64 small-block units (up to 16, 24, 32 wide)
  int n_s[3] = {};
  TileRef* d_w[2] = {};          // FP64 per-wave tiles (16 x 32, 16 x 64), 4 per workgroup (item -1: none), a multiple of 32
  int n_w[2] = {};
  TileRef* d_p[3] = {};          // FP64 panels (KB = 3, 5, 6)
  int n_p[3] = {};
  PanelPair* d_pp = nullptr;     // pairs of the panels and small blocks
  GemmUnit* d_gu = nullptr;      // FP64 product tiles, by round
  GemmSeg* d_gs = nullptr;
  GemmAdd* d_ga = nullptr;
  std::vector<GemmRound> rounds;
  RedItem* d_red = nullptr;
  int n_red = 0;
  int64_t part_doubles = 0;
  // whether an application launches anything on the side stream
  bool side() const { return n_s[1] > 0 || n_s[2] > 0 || n_g[0] > 0 || n_p[0] > 0 || rounds.size() > 1; }
};

struct PlanChunk {
  bsg_vblock_t* d_vb = nullptr;  // (with the FP64 lists)
  bsg_pair_t* d_pr = nullptr;    // pairs in device order and (split) their slice offsets, where the
  PairS* d_ps = nullptr;         // grouped or per-wave kernels read them
  // host copies for the launch lists: V blocks, pairs in device order (V
  // block i's at h_base[i], its first h_fast[i] the small-block or per-wave
  // kernel's)
  std::unique_ptr<bsg_pair_t[]> h_perm;
  int64_t n_pairs = 0;
  double flops = 0.0;
  std::vector<bsg_vblock_t> h_vb;
  std::vector<int32_t> h_base, h_fast;
  std::vector<PairS> h_ps;
  ModeLists ml[2];  // FP64, split (made by the first bsg_plan_split_arena)
};

struct bsg_plan {
  bsg_context* ctx = nullptr;
  std::vector<PlanChunk> chunks;
  // by precision mode: partial tiles of V blocks in several units, of `batch`
  // roots, part_doubles (the largest chunk's) apart
  double* part[2] = {};
  int64_t part_doubles[2] = {};
  mutable std::atomic<int64_t> split_partials{-1};  // part_doubles[1] to come, once asked for (-1: not yet)
  std::shared_ptr<const RuleSet> rules;  // the tile table when the plan was created
  int32_t batch = 1;         // roots per launch (bsg_plan_set_batch)
  // by precision mode: W scratch of the large blocks' rounds, wroots roots
  // w_doubles apart
  std::shared_ptr<WScratch> wscratch[2];
  int64_t w_doubles[2] = {};
  int32_t wroots[2] = {1, 1};  // roots per launch of the rounds
  bool cs_ready = false;     // d_cs holds C slices for `batch` roots
  bool slices_built = false; // slice recipes and pair slice offsets (first bsg_plan_split_arena)
  bool abs_from_ctx = false; // d_abs is the context's lent buffer
  int64_t wave_size = 0;
  int64_t arena_extent = 0;  // doubles of operator arena the pairs reach
  double flops = 0.0, flops1 = 0.0, flops2 = 0.0;
  double flops_split = 0.0;  // of flops: the grouped kernels' pairs (BF16 slices in split mode)
  double flops_past = 0.0;   // of flops: pairs with a side or depth past the panels'
  // split precision: the arena bsg_plan_split_arena sliced, the slice
  // recipes of the operator blocks (once per arena) and of the C blocks
  // (every application) and their BF16 buffers
  const double* split_src = nullptr;
  std::vector<SliceItem> ab_items, c_items;
  int64_t ab_elems = 0, c_elems = 0;
  SliceItem *d_ab_items = nullptr, *d_c_items = nullptr;
  SliceChunk *d_ab_chunks = nullptr, *d_c_chunks = nullptr;
  void* d_slice_lists = nullptr;  // the allocation of these
  int n_ab_chunks = 0, n_c_chunks = 0;
  __bf16 *d_abs = nullptr, *d_cs = nullptr;
  // one captured application (bsg_plan_capture): its executable graph and
  // what it was captured for
  hipGraphExec_t graph = nullptr;
  const double *g_arena = nullptr, *g_c = nullptr;
  double* g_v = nullptr;
  int32_t g_nvec = 0, g_precision = -1;
};

extern "C" {

const char* bsg_last_error(void) { return g_err.c_str(); }

int bsg_init(bsg_context** ctx, int device) {
  if (!ctx) return fail(BSG_ERR_ARG, "bsg_init: null ctx");
  int ndev = 0;
  HIPCHK(hipGetDeviceCount(&ndev));
  if (device < 0 || device >= ndev) return fail(BSG_ERR_ARG, "bsg_init: no such device");
  HIPCHK(hipSetDevice(device));
  auto* c = new bsg_context();
  c->device = device;
  hipError_t e = hipStreamCreate(&c->stream);
  if (e != hipSuccess) {
    delete c;
    return fail(BSG_ERR_HIP, std::string("hipStreamCreate: ") + hipGetErrorString(e));
  }
  e = hipMalloc(&c->red, sizeof(double) * 4 * RMAXB);
  if (e != hipSuccess) {
    (void)hipStreamDestroy(c->stream);
    delete c;
    return fail(BSG_ERR_NOMEM, "bsg_init: reduction buffer");
  }
  if (hipMalloc(&c->gpart, sizeof(double) * ((size_t)GBLK * GMAX * GMAX + COEF_SLOTS * GRAM_MAX * GRAM_MAX)) != hipSuccess) {
    (void)hipFree(c->red);
    (void)hipStreamDestroy(c->stream);
    delete c;
    return fail(BSG_ERR_NOMEM, "bsg_init: Gram scratch");
  }
  c->scratch = scratch_address(device);
  if (!c->scratch) {
    const std::string m = g_err;
    (void)hipFree(c->gpart);
    (void)hipFree(c->red);
    (void)hipStreamDestroy(c->stream);
    delete c;
    return fail(BSG_ERR_HIP, "bsg_init: " + m);
  }
  if (hipStreamCreate(&c->side) != hipSuccess || hipEventCreateWithFlags(&c->fork, hipEventDisableTiming) != hipSuccess ||
      hipEventCreateWithFlags(&c->join, hipEventDisableTiming) != hipSuccess ||
      [&] {
        for (hipEvent_t& e : c->coef_done)
          if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) return true;
        return false;
      }() ||
      hipHostMalloc((void**)&c->coef_pin, sizeof(double) * COEF_SLOTS * GRAM_MAX * GRAM_MAX, hipHostMallocDefault) != hipSuccess ||
      hipHostMalloc((void**)&c->res_pin, sizeof(double) * GRAM_MAX * GRAM_MAX, hipHostMallocDefault) != hipSuccess) {
    if (c->side) (void)hipStreamDestroy(c->side);
    if (c->fork) (void)hipEventDestroy(c->fork);
    if (c->join) (void)hipEventDestroy(c->join);
    for (hipEvent_t e : c->coef_done)
      if (e) (void)hipEventDestroy(e);
    if (c->coef_pin) (void)hipHostFree(c->coef_pin);
    if (c->res_pin) (void)hipHostFree(c->res_pin);
    (void)hipFree(c->gpart);
    (void)hipFree(c->red);
    (void)hipStreamDestroy(c->stream);
    delete c;
    return fail(BSG_ERR_HIP, "bsg_init: side stream");
  }
  *ctx = c;
  return BSG_OK;
}

int bsg_free(bsg_context* ctx) {
  if (!ctx) return BSG_OK;
  HIPCHK(hipSetDevice(ctx->device));
  HIPCHK(hipStreamSynchronize(ctx->stream));
  ctx->wscratch.reset();
  HIPCHK(hipFree(ctx->red));
  if (ctx->copy_list) HIPCHK(hipFree(ctx->copy_list));
  HIPCHK(hipStreamSynchronize(ctx->side));
  HIPCHK(hipFree(ctx->gpart));
  if (ctx->abs_buf) HIPCHK(hipFree(ctx->abs_buf));
  HIPCHK(hipHostFree(ctx->coef_pin));
  HIPCHK(hipHostFree(ctx->res_pin));
  for (hipEvent_t e : ctx->coef_done) HIPCHK(hipEventDestroy(e));
  HIPCHK(hipEventDestroy(ctx->fork));
  HIPCHK(hipEventDestroy(ctx->join));
  HIPCHK(hipStreamDestroy(ctx->side));
  HIPCHK(hipStreamDestroy(ctx->stream));
  delete ctx;
  return BSG_OK;
}

int bsg_synchronize(bsg_context* ctx) {
  if (!ctx) return fail(BSG_ERR_ARG, "null ctx");
  HIPCHK(hipStreamSynchronize(ctx->stream));
  return BSG_OK;
}

int bsg_malloc(bsg_context* ctx, size_t bytes, void** dptr) {
  if (!ctx || !dptr) return fail(BSG_ERR_ARG, "bsg_malloc: null argument");
  HIPCHK(hipSetDevice(ctx->device));
  hipError_t e = hipMalloc(dptr, std::max<size_t>(bytes, 8));
  if (e != hipSuccess) return fail(BSG_ERR_NOMEM, std::string("hipMalloc: ") + hipGetErrorString(e));
  return BSG_OK;
}
int bsg_mfree(bsg_context* ctx, void* dptr) {
  if (!ctx) return fail(BSG_ERR_ARG, "null ctx");
  HIPCHK(hipStreamSynchronize(ctx->stream));
  HIPCHK(hipFree(dptr));
  return BSG_OK;
}
int bsg_memcpy_h2d(bsg_context* ctx, void* dst, const void* src, size_t bytes) {
  if (!ctx) return fail(BSG_ERR_ARG, "null ctx");
  if (bytes == 0) return BSG_OK;
  HIPCHK(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, ctx->stream));
  HIPCHK(hipStreamSynchronize(ctx->stream));
  return BSG_OK;
}
int bsg_host_alloc(bsg_context* ctx, size_t bytes, void** hptr) {
  if (!ctx || !hptr) return fail(BSG_ERR_ARG, "bsg_host_alloc: null argument");
  hipError_t e = hipHostMalloc(hptr, std::max<size_t>(bytes, 8), hipHostMallocDefault);
  if (e != hipSuccess) return fail(BSG_ERR_NOMEM, std::string("hipHostMalloc: ") + hipGetErrorString(e));
  return BSG_OK;
}
int bsg_host_free(bsg_context* ctx, void* hptr) {
  if (!ctx) return fail(BSG_ERR_ARG, "null ctx");
  HIPCHK(hipStreamSynchronize(ctx->stream));
  HIPCHK(hipHostFree(hptr));
  return BSG_OK;
}
int bsg_memcpy_h2d_async(bsg_context* ctx, void* dst, const void* src, size_t bytes) {
  if (!ctx) return fail(BSG_ERR_ARG, "null ctx");
  if (bytes == 0) return BSG_OK;
  HIPCHK(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, ctx->stream));
  return BSG_OK;
}
int bsg_memcpy_d2h(bsg_context* ctx, void* dst, const void* src, size_t bytes) {
  if (!ctx) return fail(BSG_ERR_ARG, "null ctx");
  if (bytes == 0) return BSG_OK;
  HIPCHK(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, ctx->stream));
  HIPCHK(hipStreamSynchronize(ctx->stream));
  return BSG_OK;
}
int bsg_memset_zero(bsg_context* ctx, void* dst, size_t bytes) {
  if (!ctx) return fail(BSG_ERR_ARG, "null ctx");
  if (bytes == 0) return BSG_OK;
  HIPCHK(hipMemsetAsync(dst, 0, bytes, ctx->stream));
  return BSG_OK;
}

}  // extern "C"

namespace {
// Contiguous ranges of a chunk's V blocks with about equal pair counts, one
// per host thread; work(t, first, last) runs on them.  The V blocks are
// independent: the lists made per range are concatenated in V block order,
// so a plan does not depend on the number of threads.
template <class F>
int over_vblocks(const bsg_vblock_t* vbs, int n_vb, int64_t n_pairs, F&& work) {
  int nth = (int)std::min<long>(std::max(1u, std::thread::hardware_concurrency()), 16);
  // starting a thread costs about as much as planning a few thousand pairs
  nth = (int)std::max<int64_t>(1, std::min<int64_t>({nth, n_pairs / 6000, n_vb}));
  std::vector<int> bounds(nth + 1, n_vb);
  bounds[0] = 0;
  int64_t acc = 0, tot = 0;
  for (int i = 0; i < n_vb; ++i) tot += std::max(0, vbs[i].count) + 1;
  int t = 1;
  for (int i = 0; i < n_vb && t < nth; ++i) {
    acc += std::max(0, vbs[i].count) + 1;
    if (acc * nth >= tot * t) bounds[t++] = i + 1;
  }
  std::vector<std::thread> th;
  for (int t = 1; t < nth; ++t) th.emplace_back([&, t] { work(t, bounds[t], bounds[t + 1]); });
  work(0, bounds[0], bounds[1]);
  for (auto& x : th) x.join();
  return nth;
}
constexpr int MAX_PLAN_THREADS = 16;

// the context's W scratch if it holds n doubles, else a new one (null: no memory)
std::shared_ptr<WScratch> w_scratch(bsg_context* ctx, int64_t n) {
  std::lock_guard<std::mutex> lk(ctx->wmu);
  if (ctx->wscratch && ctx->wscratch->doubles >= n) return ctx->wscratch;
  const bool keep = n <= W_ROOTS;
  if (keep) {
    int64_t p = 1;
    while (p < n) p <<= 1;
    n = p;
  }
  auto w = std::make_shared<WScratch>();
  if (hipMalloc(&w->ptr, sizeof(double) * n) != hipSuccess) return nullptr;
  w->doubles = n;
  if (keep) ctx->wscratch = w;
  return w;
}

int32_t rounds_roots(int64_t w_doubles, int32_t nroot) {
  return (int32_t)std::max<int64_t>(1, std::min<int64_t>(nroot, W_ROOTS / std::max<int64_t>(1, w_doubles)));
}

// f(0) .. f(n - 1) on up to nth host threads
template <class F>
void on_threads(int nth, int n, F&& f) {
  std::atomic<int> next{0};
  auto run = [&] {
    for (int i; (i = next++) < n;) f(i);
  };
  std::vector<std::thread> th;
  for (int t = 1; t < std::min(nth, n); ++t) th.emplace_back(run);
  run();
  for (auto& x : th) x.join();
}

// Device arrays of one upload (256-byte aligned parts of one host buffer, sent
// with one allocation and one copy, their pointers set then).  The buffer is
// written once, by the jobs, on several threads: zeroed, grown and copied list
// by list it was half of a plan's time.
struct Blob {
  std::vector<std::pair<void**, size_t>> parts;
  std::vector<std::function<void(char*)>> jobs;  // each writes its share, given the buffer
  size_t bytes = 0;
  // room for an array: its place in the buffer
  template <class P>
  size_t place(P** d, size_t n) {
    if (n == 0) return 0;
    const size_t off = (bytes + 255) & ~(size_t)255;
    bytes = off + n;
    parts.push_back({(void**)d, off});
    return off;
  }
  template <class T, class P>
  void add(P** d, std::vector<T> h) {
    if (h.empty()) return;
    const size_t off = place(d, sizeof(T) * h.size());
    jobs.push_back([off, v = std::make_shared<std::vector<T>>(std::move(h))](char* to) {
      std::memcpy(to + off, v->data(), sizeof(T) * v->size());
    });
  }
  // false: no memory (nothing is left allocated)
  bool send(void** blob, int nth) {
    if (bytes == 0) return true;
    std::unique_ptr<char[]> h(new char[bytes]);
    on_threads(nth, (int)jobs.size(), [&](int i) { jobs[i](h.get()); });
    char* d = nullptr;
    if (hipMalloc((void**)&d, bytes) != hipSuccess || hipMemcpy(d, h.get(), bytes, hipMemcpyHostToDevice) != hipSuccess) {
      (void)hipFree(d);
      return false;
    }
    *blob = d;
    for (auto& x : parts) *x.first = d + x.second;
    return true;
  }
};

// kernels a work unit runs on
enum UnitKind : char { UK_GROUPED = 0, UK_WAVE = 2, UK_GEMM = 3, UK_PANEL = 4 /* + class 0 .. 2 */, UK_SMALL = 7 /* + class 0 .. 2 */ };

// MFMAs per wavefront of a work unit before its pair list is split (small
// blocks: by width class; half as much or twice as much in the first two
// takes 217 and 233 us for 208 on the D2h superblock at M = 250)
// A superblock of little work is cut finer, down to SEG_COST_MIN: to the cost
// that makes UNITS_MIN units of its flops, were every MFMA full (several short
// runs in flight beat one long chain of pairs: a whole application of the
// 12-site Hubbard chain from host vectors 232 -> 116 us; 192 at least: 143 us,
// 24: 120 us; 512 units instead of 2048: 185 us for 161 on the D2h superblock
// at M = 250).  Costs count padded MFMAs and an allowance per pair, so narrow
// blocks make more units: 36 orbitals, D2h, 9,500 at peak dimension 40, 13,000
// at 24, 32,000 at 12; 24 orbitals, C1, 1,600 at 60, 5,000 at 30.
constexpr long SEG_COST_MIN = 48, UNITS_MIN = 2048;
constexpr long SEG_COST = 2048, SEG_COST_SMALL[3] = {256, 768, 1024};

inline bool small_block(const bsg_vblock_t& vb) { return std::max(vb.m, vb.n) <= 32; }
// whether the small-block kernel takes a pair of a small block
inline bool small_pair(const bsg_pair_t& pr) {
  return (pr.a_off >= 0 && pr.k1 <= 32 && pr.k2 <= 32) || (pr.a_off < 0 && pr.b_off < 0);
}

// W of a large block's pair (doubles; 0: it needs none); split precision: three
// slices of W, K padded to 8, of an identity A too
inline int pad8(int k) { return (k + 7) & ~7; }
inline int64_t w_size(const bsg_vblock_t& vb, const bsg_pair_t& pr, bool split) {
  if (pr.b_off < 0 || (pr.a_off < 0 && !split)) return 0;
  const int64_t n = split ? (3 * (int64_t)vb.m * pad8(pr.k2) + 3) / 4 : (int64_t)vb.m * pr.k2;
  return (n + 1) & ~(int64_t)1;
}
// A V unit of the large blocks: the W units (and, split, additions) of its
// pairs, its segments and additions; then, where they start in the lists and
// its W in its round's half of the scratch
struct LargeUnit {
  int64_t w = 0, w0 = 0;
  int64_t wide = 0;  // W tiles of the larger split shape
  long cost = 0;
  int part = 0, seg = 0;  // the segment: host thread's part, index there
  int nw = 0, nwseg = 0, nv = 0, nadd = 0, round = 0;
  int gu0 = 0, gs0 = 0, ga0 = 0, wadd0 = 0;
  void pair(const bsg_vblock_t& vb, const bsg_pair_t& pr, bool split) {
    if (split) wide += ((vb.m + SplitBig::T - 1) / SplitBig::T) * (int64_t)((pr.k2 + SplitBig::T - 1) / SplitBig::T);
    if (pr.a_off < 0 && pr.b_off < 0) {
      ++nadd;
      return;
    }
    ++nv;
    cost += gemm_cost(pr);
    if (const int64_t x = w_size(vb, pr, split)) {
      w += x;
      ++nw;
      nwseg += pr.a_off >= 0;
    }
  }
};

// What one host thread's V blocks contribute to a mode's launch lists, with
// indices of its own
struct ListPart {
  std::vector<GUnit> gunits[NCLS];                 // grouped tiles by kernel class
  std::vector<std::pair<long, int>> sunits[3];     // (cost, segment) of small-block units (up to 16, 24, 32)
  std::vector<LargeUnit> bunits;                   // large blocks' units
  std::vector<GUnit> wunits[2], punits[3];         // per-wave tiles (16 x 32, 16 x 64), panels (KB = 3, 5, 6)
  std::vector<int> gq;                             // pairs of the large blocks' units (indices into h_perm)
  std::vector<PanelPair> pp;
  std::vector<Seg> segs;
  std::vector<RedItem> reds;
  int64_t poff = 0;                                // partial tiles (doubles)
};
// How finely pair lists are cut into units: 0 as the kernels like it, 1 to
// CUT_WHOLE - 1 at 4^level times the costs, CUT_WHOLE not at all (one unit per
// kernel that a V block's pairs need at least)
constexpr int CUT_WHOLE = 5;

// Every V block's pairs (in device order: the h_fast first ones are the
// small-block or per-wave kernel's) cut into work units of about SEG_COST MFMAs
// per wave; blocks with several units get partial tiles and an ordered
// reduction.  Returns the number of parts used.
int cut_lists(const bsg_plan* p, const PlanChunk& pc, bool split, int level, std::vector<ListPart>& loc) {
  loc.clear();
  loc.resize(MAX_PLAN_THREADS);
  const long fill = std::max(SEG_COST_MIN, (long)(pc.flops / (2048.0 * UNITS_MIN)));
  const int nvb = (int)pc.h_vb.size();
  // panels up to 96, beside blocks past twice that up to 80: blocks of 81 to 96
  // as panels and as product tiles take, by the widest block, 2.85 and 3.99 ms
  // (90, 36 orbitals, D2h), 4.40 and 5.92 (101), 6.96 and 7.18 (119), the same
  // within 1% from 137 to 277 (both symmetries), and 4.13 and 3.99 ms at 309 (24
  // orbitals, C1), where the few wide panels end after everything else
  int widest = 0;
  for (const bsg_vblock_t& vb : pc.h_vb) widest = std::max(widest, std::max(vb.m, vb.n));
  const int panel_max = widest <= 2 * PANEL_MAX ? PANEL_MAX : 80;
  return over_vblocks(pc.h_vb.data(), nvb, pc.n_pairs, [&](int t, int i0, int i1) {
    ListPart& L = loc[t];
    std::vector<std::pair<int, int>> units;  // (first, count)
    std::vector<char> ukind;
    std::vector<int> pan[3], big, few[3];
    for (int i = i0; i < i1; ++i) {
      const bsg_vblock_t& vb = pc.h_vb[i];
      const bsg_pair_t* perm = pc.h_perm.get();
      const int base = pc.h_base[i], nfast = pc.h_fast[i], ntot = vb.count;
      const bool sm = small_block(vb);
      const int rule = table_rule(*p->rules, vb.m, vb.n, split);
      const bool wave_vb = !split && !sm && rule == wave_candidate();
      units.clear();
      ukind.clear();
      Geom g;
      auto cost_of = [&](int kind, const bsg_pair_t& pr) -> long {
        switch (kind) {
          case UK_SMALL:
          case UK_SMALL + 1:
          case UK_SMALL + 2: return small_cost(vb.m, vb.n, pr);
          case UK_WAVE: return wave_cost(vb.n, pr);
          case UK_GEMM: return gemm_cost(pr);
          case UK_PANEL:
          case UK_PANEL + 1:
          case UK_PANEL + 2: return panel_cost(vb.n, pr);
          default: return pair_cost(g, vb.n, pr);
        }
      };
      // at(q): the list's q-th pair; first: its index where the units point
      auto cut = [&](int first, int n, int kind, auto at) {
        const long lim = std::min(kind == UK_GEMM ? fill / 2 : fill, kind >= UK_SMALL ? SEG_COST_SMALL[kind - UK_SMALL] : SEG_COST)
                         << (2 * level);
        int start = 0;
        long cost = 0;
        for (int q = 0; q < n; ++q) {
          cost += cost_of(kind, at(q));
          if ((cost >= lim && level < CUT_WHOLE) || q + 1 == n) {
            units.push_back({first + start, q + 1 - start});
            ukind.push_back((char)kind);
            start = q + 1;
            cost = 0;
          }
        }
      };
      auto in_perm = [&](int first) { return [&, first](int q) -> const bsg_pair_t& { return perm[first + q]; }; };
      const int slow = split && !sm ? 0 : nfast;  // pairs the small-block or per-wave kernel takes
      // a list's pairs by C block (identity partners first, else as given) as
      // the kernels that keep C read them; pad: pairs left in the run on one C
      // block
      auto cut_by_c = [&](std::vector<int>& list, int kind) {
        if (list.size() > 1) std::stable_sort(list.begin(), list.end(), [&](int x, int y) {
          const bsg_pair_t &a = perm[x], &b = perm[y];
          if (a.c_off != b.c_off) return a.c_off < b.c_off;
          return (a.a_off < 0 || a.b_off < 0) && !(b.a_off < 0 || b.b_off < 0);
        });
        const int first = (int)L.pp.size();
        for (int q : list) {
          const bsg_pair_t& x = perm[q];
          L.pp.push_back(PanelPair{x.a_off, x.c_off, x.b_off, x.a_off < 0 ? x.alpha : x.alpha * x.alpha_a, x.k1, x.k2,
                                   (x.a_trans ? 1 : 0) | (x.b_trans ? 2 : 0), 1});
        }
        for (int q = (int)L.pp.size() - 2; q >= first; --q) {
          PanelPair &x = L.pp[q], &y = L.pp[q + 1];
          if (x.c == y.c && x.k1 == y.k1 && x.k2 == y.k2) x.pad = y.pad + 1;
        }
        cut(first, (int)list.size(), kind, [&](int q) -> const bsg_pair_t& { return perm[list[q]]; });
      };
      if (slow > 0 && wave_vb) cut(base, slow, UK_WAVE, in_perm(base));
      // in FP64 it also takes the pairs of an identity A and a B' it has room for
      auto few_pair = [&](int q) {
        return q < base + slow || (!split && sm && level < CUT_WHOLE && std::max(perm[q].k1, perm[q].k2) <= 32);
      };
      if (sm) {
        for (auto& x : few) x.clear();
        for (int q = base; q < base + ntot; ++q) {
          if (!few_pair(q)) continue;
          const int k = std::max(std::max(vb.m, vb.n), std::max(perm[q].k1, perm[q].k2));
          few[level == CUT_WHOLE ? 2 : (k <= 16 ? 0 : (k <= 24 ? 1 : 2))].push_back(q);
        }
        for (int k = 0; k < 3; ++k)
          if (!few[k].empty()) cut_by_c(few[k], UK_SMALL + k);
      }
      if (slow < ntot) {
        if (wave_vb || (!sm && rule >= 0) || (split && std::max(vb.m, vb.n) <= SPLIT_GROUPED)) {
          g = pick_geom(*p->rules, vb.m, vb.n, split ? 4 : 6);
          cut(base + slow, ntot - slow, UK_GROUPED, in_perm(base + slow));
        } else {
          const bool med = !split && std::max(vb.m, vb.n) <= panel_max;
          for (auto& x : pan) x.clear();
          big.clear();
          for (int q = base + slow; q < base + ntot; ++q) {
            if (few_pair(q)) continue;
            const int k = std::max(perm[q].k1, perm[q].k2);
            if (!med || k > panel_max)
              big.push_back(q);
            else
              pan[std::max(k, vb.n) <= 48 ? 0 : (std::max(k, vb.n) <= 80 ? 1 : 2)].push_back(q);
          }
          if (level == CUT_WHOLE) {  // the widest class, or product tiles, for all
            std::vector<int>& to = !big.empty() ? big : (pan[2].empty() ? pan[1] : pan[2]);
            for (auto& x : pan)
              if (&x != &to) {
                to.insert(to.end(), x.begin(), x.end());
                x.clear();
              }
            std::sort(to.begin(), to.end());
          }
          for (int k = 0; k < 3; ++k)
            if (!pan[k].empty()) cut_by_c(pan[k], UK_PANEL + k);
          if (!big.empty()) {
            const int first = (int)L.gq.size();
            L.gq.insert(L.gq.end(), big.begin(), big.end());
            cut(first, (int)big.size(), UK_GEMM, [&](int q) -> const bsg_pair_t& { return perm[big[q]]; });
          }
        }
      }
      const int64_t mn = (int64_t)vb.m * vb.n;
      const int nseg = (int)units.size();
      const int64_t p0 = L.poff;
      for (int u = 0; u < nseg; ++u) {
        Seg sg;
        sg.vb = i;
        sg.first = units[u].first;
        sg.count = units[u].second;
        sg.pad = 0;
        sg.p_off = nseg == 1 ? -1 : p0 + (int64_t)u * mn;
        const int si = (int)L.segs.size();
        L.segs.push_back(sg);
        const int kind = ukind[u];
        if (kind == UK_GEMM) {
          LargeUnit b;
          b.part = t;
          b.seg = si;
          for (int q = 0; q < sg.count; ++q) b.pair(vb, perm[L.gq[sg.first + q]], split);
          L.bunits.push_back(b);
          continue;
        }
        long ucost = 0;
        if (kind >= UK_PANEL && kind < UK_SMALL)
          for (int q = 0; q < sg.count; ++q) ucost += panel_cost(vb.n, L.pp[sg.first + q]);
        else if (kind >= UK_SMALL)
          for (int q = 0; q < sg.count; ++q) ucost += small_cost(vb.m, vb.n, L.pp[sg.first + q]);
        else
          for (int q = 0; q < sg.count; ++q) ucost += cost_of(kind, perm[sg.first + q]);
        if (kind >= UK_SMALL) {
          L.sunits[kind - UK_SMALL].push_back({ucost, si});
          continue;
        }
        GUnit gu;
        gu.cost = ucost;
        gu.seg = si;
        if (kind == UK_WAVE) {
          const int nb = wave_nb(vb.n);
          gu.ntm = (vb.m + 15) / 16;
          gu.ntn = (vb.n + 16 * nb - 1) / (16 * nb);
          L.wunits[nb == 4].push_back(gu);
        } else if (kind >= UK_PANEL && kind < UK_SMALL) {
          const int np = (vb.m + 15) / 16;
          gu.ntm = (np + 3) / 4;                    // workgroups
          gu.code = (np + gu.ntm - 1) / gu.ntm;     // panels of each
          gu.cost = ucost * np / gu.ntm;            // of its wavefronts that have a panel
          gu.ntn = 1;
          L.punits[kind - UK_PANEL].push_back(gu);
        } else {
          gu.ntm = (vb.m + g.tm - 1) / g.tm;
          gu.ntn = (vb.n + g.jv - 1) / g.jv;
          gu.code = g.code;
          L.gunits[g.cls].push_back(gu);
        }
      }
      if (nseg > 1) {
        for (int64_t e0 = 0; e0 < mn; e0 += 64) {
          RedItem r;
          r.v_off = vb.v_off;
          r.p_off = p0;
          r.nseg = nseg;
          r.mn = (int32_t)mn;
          r.e0 = (int32_t)e0;
          r.len = (int32_t)std::min<int64_t>(64, mn - e0);
          L.reds.push_back(r);
        }
        L.poff += nseg * mn;
      }
    }
  });
}

// Partial tiles (doubles) of a chunk's FP64 and split lists together, were the
// pair lists cut at fixed costs for the small-block kernel (V blocks and depths
// up to 32, one class), the grouped and the per-wave tiles alone.
// BSG_NOALLOC_SCRATCH_DOUBLES was set for lists cut so: what they keep within
// it, the finer lists of the kernels that came later keep within it too (cut_to_fit).
int64_t fixed_cut_partials(const bsg_plan* p, const PlanChunk& pc) {
  int64_t part[MAX_PLAN_THREADS] = {};
  auto cdiv = [](long a, long b) { return (a + b - 1) / b; };
  over_vblocks(pc.h_vb.data(), (int)pc.h_vb.size(), pc.n_pairs, [&](int t, int i0, int i1) {
    for (int i = i0; i < i1; ++i) {
      const bsg_vblock_t& vb = pc.h_vb[i];
      const bsg_pair_t* prs = pc.h_perm.get() + pc.h_base[i];
      const bool sm = small_block(vb), wave_vb = !sm && table_rule(*p->rules, vb.m, vb.n, false) == wave_candidate();
      const Geom gm = pick_geom(*p->rules, vb.m, vb.n, 6), gs = pick_geom(*p->rules, vb.m, vb.n, 4);
      auto small = [&](const bsg_pair_t& pr) {
        const long nrb = cdiv(vb.m, 16), nnb = cdiv(vb.n, 16), njb = cdiv(pr.k2, 16);
        return (pr.a_off < 0 ? 0 : (pr.b_off < 0 ? nnb : njb) * cdiv(pr.k1, 4) * nrb) +
               (pr.b_off < 0 ? 0 : njb * 4 * nrb * nnb) + 24;
      };
      // units of the first nf pairs (small-block or per-wave tiles) and of the rest
      auto units = [&](const Geom& g, int nf) {
        int64_t n = 0;
        long cost = 0;
        for (int q = 0; q < vb.count; ++q) {
          cost += q >= nf ? pair_cost(g, vb.n, prs[q]) : (sm ? small(prs[q]) : wave_cost(vb.n, prs[q]));
          if (cost < (q < nf && sm ? 1024 : 2048) && q + 1 != nf && q + 1 != vb.count) continue;
          ++n;
          cost = 0;
        }
        return n > 1 ? n : 0;
      };
      const int nf = pc.h_fast[i];
      int64_t n = units(gm, nf);
      if (wave_vb)
        n += units(gs, 0);
      else if (gm.code != gs.code || gm.nv != gs.nv)
        n += units(gs, nf);
      part[t] += n * vb.m * vb.n;
    }
  });
  int64_t sum = 0;
  for (int64_t x : part) sum += x;
  return sum;
}

// The cut of one mode's lists; coarser than the kernels like it where only that
// keeps the partial tiles within the static scratch and lists cut at fixed costs
// would have stayed within it (30 blocks of 32 x 32 with 1000 pairs of depth 1
// each: 10.3 million doubles, 2.6 million one level coarser; 4000 blocks of 60 x
// 64 with one pair in each of three panel classes: 30.7 million, none as whole
// lists).  Returns the doubles of the partial tiles; nth: parts used.
int64_t cut_to_fit(const bsg_plan* p, const PlanChunk& pc, bool split, std::vector<ListPart>& loc, int& nth) {
  int64_t need = 0;
  for (int level = 0; level <= CUT_WHOLE; ++level) {
    nth = cut_lists(p, pc, split, level, loc);
    need = 0;
    for (int t = 0; t < nth; ++t) need += loc[t].poff;
    if (need <= BSG_NOALLOC_SCRATCH_DOUBLES) break;
    if (level == 0 && fixed_cut_partials(p, pc) > BSG_NOALLOC_SCRATCH_DOUBLES) break;
  }
  return need;
}

// The large blocks' products: the V units' segments and the W tiles they read, in
// rounds of about equal W size.  Every unit's place in the lists and its share
// of W come first, then the rounds' tiles, units and segments are written on nth
// threads.
void plan_products(bsg_plan* p, const PlanChunk& pc, ModeLists& ml, Blob& blob, const std::vector<ListPart>& loc,
                   const std::vector<int64_t>& part_at, bool split, int nth) {
  const bsg_pair_t* perm = pc.h_perm.get();
  auto units = std::make_shared<std::vector<LargeUnit>>();
  for (const ListPart& L : loc) units->insert(units->end(), L.bunits.begin(), L.bunits.end());
  std::vector<LargeUnit>& un = *units;
  const int nu = (int)un.size();
  if (nu == 0) return;
  int64_t wtot = 0, wunit = 0, wide_tiles = 0;  // doubles of W: all units, the largest
  for (const LargeUnit& u : un) {
    wtot += u.w;
    wunit = std::max(wunit, u.w);
    wide_tiles += u.wide;
  }
  const bool wide = wide_tiles >= SPLIT_WIDE;
  // an even number of rounds once W is large enough to be worth two
  // (a round is closed by the unit that fills it, which may take it past the
  // target by almost that unit's W)
  const int64_t room = std::max(W_HALF / 2, W_HALF - wunit);
  int64_t nround = 1;
  if (wtot > W_ONE_ROUND) nround = 2 * ((wtot + room * 2 - 1) / (room * 2));
  // (no pair with a W: one round)
  const int64_t target = std::max<int64_t>(1, (wtot + nround - 1) / nround);
  std::vector<int> first(1, 0);  // the rounds' first units
  int64_t wused = 0, wneed[2] = {};
  int ngu = 0, ngs = 0, nga = 0, nwadd = 0;
  for (int i = 0; i < nu; ++i) {
    LargeUnit& u = un[i];
    const int r = u.round = (int)first.size() - 1;
    u.w0 = wused;
    u.gu0 = ngu;
    u.gs0 = ngs;
    u.ga0 = nga;
    u.wadd0 = nwadd;
    ngu += u.nw + 1;
    ngs += u.nwseg + u.nv;
    nga += u.nadd;
    nwadd += u.nw - u.nwseg;
    wused += u.w;
    wneed[r & 1] = std::max(wneed[r & 1], wused);
    if (wused >= target && i + 1 < nu) {
      first.push_back(i + 1);
      wused = 0;
    }
  }
  first.push_back(nu);
  const int nr = (int)first.size() - 1;
  p->w_doubles[split] = std::max(p->w_doubles[split], wneed[0] + wneed[1]);
  // the rounds' tiles: W (kind 0) and V (kind 1) tiles by shape
  std::vector<std::array<std::vector<TileRef>, 4>> rt(nr);
  on_threads(nth, 2 * nr, [&](int j) {
    const int r = j >> 1, kind = j & 1;
    std::vector<GUnit> to[2];
    auto put = [&](int m, int n, int gu, long cost) {
      const int shape = wide ? split_shape(m, n) : 0;
      const int edge = split ? (shape ? SplitBig::T : SplitSmall::T) : GemmT::TM;
      GUnit t;
      t.cost = cost;
      t.seg = gu;
      t.ntm = (m + edge - 1) / edge;
      t.ntn = (n + edge - 1) / edge;
      to[shape].push_back(t);
    };
    for (int i = first[r]; i < first[r + 1]; ++i) {
      const LargeUnit& u = un[i];
      const ListPart& L = loc[u.part];
      const Seg& sg = L.segs[u.seg];
      const bsg_vblock_t& vb = pc.h_vb[sg.vb];
      if (kind) {
        put(vb.m, vb.n, u.gu0 + u.nw, u.cost);
        continue;
      }
      int gu = u.gu0;
      for (int q = 0; q < sg.count; ++q) {
        const bsg_pair_t& pr = perm[L.gq[sg.first + q]];
        if (w_size(vb, pr, split) > 0)  // W, split: W^T
          put(split ? pr.k2 : vb.m, split ? vb.m : pr.k2, gu++, (pr.k1 + (split ? 31 : GKC - 1)) / (split ? 32 : GKC) + 4);
      }
    }
    for (int k = 0; k < 2; ++k) rt[r][2 * kind + k] = xcd_order(to[k]);
  });
  ml.rounds.resize(nr);
  for (int r = 0; r < nr; ++r)
    for (int k = 0; k < 2; ++k) {
      ml.rounds[r].n_w[k] = (int)rt[r][k].size();
      ml.rounds[r].n_v[k] = (int)rt[r][2 + k].size();
      blob.add(&ml.rounds[r].d_w[k], std::move(rt[r][k]));
      blob.add(&ml.rounds[r].d_v[k], std::move(rt[r][2 + k]));
    }
  // units, segments, additions (the W units' own follow the V units'); the
  // second half of the scratch follows the first
  static_assert((int)SP_W == (int)BS_W, "one constant for both precisions");
  const size_t gu_at = blob.place(&ml.d_gu, sizeof(GemmUnit) * ngu), gs_at = blob.place(&ml.d_gs, sizeof(GemmSeg) * ngs),
               ga_at = blob.place(&ml.d_ga, sizeof(GemmAdd) * (nga + nwadd));
  const int64_t second = wneed[0];
  auto write = [=, &pc, &loc, &part_at](char* to, int i) {
    const LargeUnit& u = (*units)[i];
    const ListPart& L = loc[u.part];
    const Seg& sg = L.segs[u.seg];
    const bsg_vblock_t& vb = pc.h_vb[sg.vb];
    const int half = u.round & 1;
    GemmUnit* gu = (GemmUnit*)(to + gu_at) + u.gu0;
    GemmSeg *ws = (GemmSeg*)(to + gs_at) + u.gs0, *vs = ws + u.nwseg;
    GemmAdd *ga = (GemmAdd*)(to + ga_at) + u.ga0, *wadd = (GemmAdd*)(to + ga_at) + nga + u.wadd0;
    int gs0 = u.gs0, wadd0 = nga + u.wadd0;
    int64_t at = (split ? 4 : 1) * (u.w0 + (half ? second : 0));  // split: BF16 elements
    for (int q = 0; q < sg.count; ++q) {
      const int j = L.gq[sg.first + q];
      const bsg_pair_t& pr = perm[j];
      if (pr.a_off < 0 && pr.b_off < 0) {
        *ga++ = GemmAdd{pr.c_off, pr.alpha};
        continue;
      }
      const int64_t w = (split ? 4 : 1) * w_size(vb, pr, split);
      if (w > 0) {
        GemmUnit x{};
        x.out = at;
        x.kind = GU_W;
        x.m = split ? pr.k2 : vb.m;
        x.n = split ? vb.m : pr.k2;
        x.alpha = 1.0;
        if (pr.a_off >= 0) {
          x.alpha = pr.alpha * pr.alpha_a;
          x.first = gs0++;
          x.count = 1;
          *ws++ = split ? GemmSeg{pc.h_ps[j].c, pc.h_ps[j].a, 1.0, pad8(pr.k1), BS_C << SEG_LSPACE}
                        : GemmSeg{pr.a_off, pr.c_off, 1.0, pr.k1, (SP_C << SEG_RSPACE) | (pr.a_trans ? SEG_LT : 0)};
        } else {
          x.add_first = wadd0++;
          x.add_count = 1;
          *wadd++ = GemmAdd{pr.c_off, pr.alpha};
        }
        *gu++ = x;
      }
      if (split) {
        // operands are slices with K padded to 8; op(A) C is formed as W^T, and
        // an identity A's W = alpha C is split like any other W
        const PairS& ps = pc.h_ps[j];
        *vs++ = w > 0 ? GemmSeg{at, ps.b, 1.0, pad8(pr.k2), BS_W << SEG_LSPACE}
                      : GemmSeg{ps.a, ps.c, pr.alpha * pr.alpha_a, pad8(pr.k1), BS_C << SEG_RSPACE};
      } else if (w > 0) {  // V += W B'
        *vs++ = GemmSeg{at, pr.b_off, 1.0, pr.k2, (SP_W << SEG_LSPACE) | (pr.b_trans ? SEG_RT : 0)};
      } else if (pr.a_off < 0) {  // V += alpha C B'
        *vs++ = GemmSeg{pr.c_off, pr.b_off, pr.alpha, pr.k2, (SP_C << SEG_LSPACE) | (pr.b_trans ? SEG_RT : 0)};
      } else {  // V += alpha op(A) C
        *vs++ = GemmSeg{pr.a_off, pr.c_off, pr.alpha * pr.alpha_a, pr.k1, (SP_C << SEG_RSPACE) | (pr.a_trans ? SEG_LT : 0)};
      }
      at += w;
    }
    GemmUnit x{};
    x.out = sg.p_off < 0 ? vb.v_off : part_at[u.part] + sg.p_off;
    x.kind = sg.p_off < 0 ? GU_V : GU_PART;
    x.m = vb.m;
    x.n = vb.n;
    x.alpha = 1.0;
    x.first = u.gs0 + u.nwseg;
    x.count = u.nv;
    x.add_first = u.ga0;
    x.add_count = u.nadd;
    *gu = x;
  };
  constexpr int STEP = 64;  // units a thread takes at a time
  for (int u0 = 0; u0 < nu; u0 += STEP)
    blob.jobs.push_back([=](char* to) {
      for (int i = u0; i < std::min(nu, u0 + STEP); ++i) write(to, i);
    });
}

// The launch lists of one precision mode
int plan_lists(bsg_plan* p, PlanChunk& pc, bool split) {
  ModeLists& ml = pc.ml[split];
  std::vector<ListPart> loc;
  int nth = 0;
  cut_to_fit(p, pc, split, loc, nth);
  // concatenate with the parts' indices shifted: units and their order here, the
  // rest straight into the upload
  std::vector<GUnit> gunits[NCLS], wunits[2], punits[3];
  std::vector<std::pair<long, int>> sunits[3];
  struct Base {
    size_t segs = 0, pp = 0, reds = 0;
  };
  std::vector<Base> at(nth + 1);
  std::vector<int64_t> part_at(nth + 1, 0);  // partial tiles
  for (int t = 0; t < nth; ++t) {
    const ListPart& L = loc[t];
    const Base& x = at[t];
    at[t + 1] = Base{x.segs + L.segs.size(), x.pp + L.pp.size(), x.reds + L.reds.size()};
    part_at[t + 1] = part_at[t] + L.poff;
    auto shift = [&](std::vector<GUnit>& to, const std::vector<GUnit>& from) {
      for (GUnit u : from) {
        u.seg += (int)x.segs;
        to.push_back(u);
      }
    };
    for (int k = 0; k < NCLS; ++k) shift(gunits[k], L.gunits[k]);
    for (int k = 0; k < 2; ++k) shift(wunits[k], L.wunits[k]);
    for (int k = 0; k < 3; ++k) {
      shift(punits[k], L.punits[k]);
      for (const auto& u : L.sunits[k]) sunits[k].push_back({u.first, u.second + (int)x.segs});
    }
  }
  const Base& all = at[nth];
  ml.part_doubles = part_at[nth];
  Blob blob;
  if (!split) blob.add(&pc.d_vb, pc.h_vb);
  const size_t seg_at = blob.place(&ml.d_seg, sizeof(Seg) * all.segs),
               red_at = blob.place(&ml.d_red, sizeof(RedItem) * all.reds),
               pp_at = blob.place(&ml.d_pp, sizeof(PanelPair) * all.pp);
  ml.n_red = (int)all.reds;
  for (int t = 0; t < nth; ++t)
    blob.jobs.push_back([&, t](char* to) {
      const ListPart& L = loc[t];
      Seg* seg = (Seg*)(to + seg_at) + at[t].segs;
      for (size_t u = 0; u < L.segs.size(); ++u) {
        seg[u] = L.segs[u];
        if (seg[u].p_off >= 0) seg[u].p_off += part_at[t];
      }
      for (int k = 0; k < 3; ++k) {
        for (const GUnit& u : L.punits[k]) seg[u.seg].first += (int)at[t].pp;
        for (const auto& u : L.sunits[k]) seg[u.second].first += (int)at[t].pp;
      }
      if (!L.pp.empty()) std::memcpy(to + pp_at + sizeof(PanelPair) * at[t].pp, L.pp.data(), sizeof(PanelPair) * L.pp.size());
      RedItem* red = (RedItem*)(to + red_at) + at[t].reds;
      for (RedItem r : L.reds) {
        r.p_off += part_at[t];
        *red++ = r;
      }
    });
  // small-block units, costliest first
  for (int k = 0; k < 3; ++k) {
    auto& su = sunits[k];
    costliest_first(su);
    std::vector<int32_t> sq;
    sq.reserve(su.size());
    for (const auto& x : su) sq.push_back(x.second);
    ml.n_s[k] = (int)sq.size();
    blob.add(&ml.d_s[k], std::move(sq));
  }
  for (int k = 0; k < NCLS; ++k) {
    std::vector<TileRef> t = xcd_order(gunits[k]);
    ml.n_g[k] = (int)t.size();
    blob.add(&ml.d_g[k], std::move(t));
  }
  for (int k = 0; k < 3; ++k) {
    std::vector<TileRef> t = xcd_order(punits[k]);
    ml.n_p[k] = (int)t.size();
    blob.add(&ml.d_p[k], std::move(t));
  }
  // per-wave tiles of each width: units (costliest first) go to the least
  // loaded of the 8 XCDs, a unit's tiles in consecutive wave slots of that
  // XCD's workgroups (they share the unit's C and B' blocks in its L2);
  // workgroup 8 j + x is XCD x's j-th
  for (int k = 0; k < 2; ++k) {
    std::vector<std::pair<long, int>> order;
    for (int u = 0; u < (int)wunits[k].size(); ++u)
      order.push_back({wunits[k][u].cost * wunits[k][u].ntm * wunits[k][u].ntn, u});
    costliest_first(order);
    std::vector<TileRef> q[8];
    long load[8] = {};
    for (const auto& o : order) {
      const int x = (int)(std::min_element(load, load + 8) - load);
      const GUnit& gu = wunits[k][o.second];
      for (int tm = 0; tm < gu.ntm; ++tm)
        for (int tn = 0; tn < gu.ntn; ++tn) q[x].push_back(TileRef{gu.seg, tm, tn, 0});
      load[x] += o.first;
    }
    size_t nwg = 0;
    for (auto& e : q) nwg = std::max(nwg, (e.size() + 3) / 4);
    std::vector<TileRef> wt(nwg * 32, TileRef{-1, 0, 0, 0});
    for (int x = 0; x < 8; ++x)
      for (size_t e = 0; e < q[x].size(); ++e) wt[((e / 4) * 8 + x) * 4 + e % 4] = q[x][e];
    ml.n_w[k] = (int)wt.size();
    blob.add(&ml.d_w[k], std::move(wt));
  }
  plan_products(p, pc, ml, blob, loc, part_at, split, nth);
  // the pairs as the grouped and per-wave kernels read them, once a list has such units
  auto send_pairs = [&](auto** d, const auto* h) {
    if (*d) return true;
    const size_t bytes = sizeof(*h) * pc.n_pairs;
    if (hipMalloc((void**)d, bytes) == hipSuccess && hipMemcpy(*d, h, bytes, hipMemcpyHostToDevice) == hipSuccess)
      return true;
    (void)hipFree(*d);
    *d = nullptr;
    return false;
  };
  bool grouped = false;
  for (int k = 0; k < NCLS; ++k) grouped |= ml.n_g[k] > 0;
  if (((grouped || ml.n_w[0] > 0 || ml.n_w[1] > 0) && !send_pairs(&pc.d_pr, pc.h_perm.get())) ||
      (split && grouped && !send_pairs(&pc.d_ps, pc.h_ps.data())) || !blob.send(&ml.d_blob, nth))
    return fail(BSG_ERR_NOMEM, "plan lists");
  ml.ready = true;
  return BSG_OK;
}
}  // namespace

extern "C" {

int bsg_plan_create(bsg_context* ctx, const bsg_chunk_t* chunks, int32_t n_chunks, int64_t wave_size,
                    bsg_plan** plan) {
  if (!ctx || !plan || (n_chunks > 0 && !chunks) || wave_size < 0) return fail(BSG_ERR_ARG, "bsg_plan_create: bad args");
  HIPCHK(hipSetDevice(ctx->device));
  auto* p = new bsg_plan();
  p->ctx = ctx;
  p->wave_size = wave_size;
  p->rules = g_tile_rules;
  auto cleanup = [&](int code, const std::string& m) {
    bsg_plan_destroy(p);
    return fail(code, m);
  };
  p->chunks.resize(std::max(0, n_chunks));
  for (int ci = 0; ci < n_chunks; ++ci) {
    const bsg_chunk_t& ch = chunks[ci];
    PlanChunk& pc = p->chunks[ci];
    int64_t np = 0;
    pc.h_vb.assign(ch.vblocks, ch.vblocks + ch.n_vblocks);
    pc.h_base.resize(ch.n_vblocks);
    pc.h_fast.resize(ch.n_vblocks);
    for (int i = 0; i < ch.n_vblocks; ++i) {
      const bsg_vblock_t& vb = ch.vblocks[i];
      if (vb.m <= 0 || vb.n <= 0 || vb.v_off < 0 || vb.v_off + (int64_t)vb.m * vb.n > wave_size || vb.first < 0 ||
          vb.count < 0 || vb.first + (int64_t)vb.count > ch.n_pairs)
        return cleanup(BSG_ERR_ARG, "bsg_plan_create: vblock out of range");
      pc.h_base[i] = (int32_t)np;
      np += vb.count;
    }
    if (np > 0x7fffffff) return cleanup(BSG_ERR_ARG, "bsg_plan_create: too many pairs");
    pc.n_pairs = np;
    pc.h_perm.reset(new bsg_pair_t[std::max<int64_t>(1, np)]);
    // the V blocks' pairs in device order: the small-block (per-wave)
    // kernel's ones, then the rest
    struct Local {
      int64_t arena_extent = 0;
      double flops = 0.0, flops1 = 0.0, flops2 = 0.0, flops_split = 0.0, flops_past = 0.0;
      bool bad = false;
      std::vector<bsg_pair_t> rest;
    };
    std::vector<Local> loc(MAX_PLAN_THREADS);
    const int nth = over_vblocks(ch.vblocks, ch.n_vblocks, np, [&](int t, int i0, int i1) {
      Local& L = loc[t];
      for (int i = i0; i < i1; ++i) {
        const bsg_vblock_t& vb = ch.vblocks[i];
        const bool sm = small_block(vb), wave_vb = !sm && table_rule(*p->rules, vb.m, vb.n, false) == wave_candidate();
        bsg_pair_t* to = pc.h_perm.get() + pc.h_base[i];
        L.rest.clear();
        int nf = 0;
        for (int q = 0; q < vb.count; ++q) {
          const bsg_pair_t& pr = ch.pairs[vb.first + q];
          if (pr.k1 <= 0 || pr.k2 <= 0 || pr.c_off < 0 || pr.c_off + (int64_t)pr.k1 * pr.k2 > wave_size ||
              (pr.a_off < 0 && pr.k1 != vb.m) || (pr.b_off < 0 && pr.k2 != vb.n)) {
            L.bad = true;
            return;
          }
          double f1 = 0.0, f2 = 0.0;
          if (pr.a_off >= 0) {
            L.arena_extent = std::max(L.arena_extent, pr.a_off + (int64_t)vb.m * pr.k1);
            f1 = 2.0 * vb.m * pr.k1 * pr.k2;
          }
          if (pr.b_off >= 0) {
            L.arena_extent = std::max(L.arena_extent, pr.b_off + (int64_t)vb.n * pr.k2);
            f2 = 2.0 * vb.m * pr.k2 * vb.n;
          }
          L.flops += f1 + f2;
          L.flops1 += f1;
          L.flops2 += f2;
          if (std::max(std::max(vb.m, vb.n), std::max(pr.k1, pr.k2)) > PANEL_MAX) L.flops_past += f1 + f2;
          const bool f = sm ? small_pair(pr) : wave_vb && (pr.a_off < 0 || pr.k1 <= 4 * wave_ka(wave_nb(vb.n)));
          if (!f || wave_vb) L.flops_split += f1 + f2;  // split mode: every pair of a per-wave block runs on BF16 slices
          if (f)
            to[nf++] = pr;
          else
            L.rest.push_back(pr);
        }
        std::copy(L.rest.begin(), L.rest.end(), to + nf);
        pc.h_fast[i] = nf;
      }
    });
    for (int t = 0; t < nth; ++t) {
      const Local& L = loc[t];
      if (L.bad) return cleanup(BSG_ERR_ARG, "bsg_plan_create: pair out of range");
      p->flops += L.flops;
      pc.flops += L.flops;
      p->flops1 += L.flops1;
      p->flops2 += L.flops2;
      p->flops_split += L.flops_split;
      p->flops_past += L.flops_past;
      p->arena_extent = std::max(p->arena_extent, L.arena_extent);
    }
    if (plan_lists(p, pc, false) != BSG_OK) return cleanup(BSG_ERR_NOMEM, "bsg_plan_create: plan arrays");
  }
  for (const PlanChunk& pc : p->chunks) p->part_doubles[0] = std::max(p->part_doubles[0], pc.ml[0].part_doubles);
  if (p->part_doubles[0] > 0 && hipMalloc(&p->part[0], sizeof(double) * p->part_doubles[0]) != hipSuccess)
    return cleanup(BSG_ERR_NOMEM, "bsg_plan_create: partial-tile scratch");
  if (p->w_doubles[0] > 0 && !(p->wscratch[0] = w_scratch(ctx, p->w_doubles[0])))
    return cleanup(BSG_ERR_NOMEM, "bsg_plan_create: W scratch");
  *plan = p;
  return BSG_OK;
}

int bsg_plan_destroy(bsg_plan* p) {
  if (!p) return BSG_OK;
  if (p->ctx) (void)hipStreamSynchronize(p->ctx->stream);
  for (auto& c : p->chunks) {
    (void)hipFree(c.d_pr);
    (void)hipFree(c.d_ps);
    for (auto& ml : c.ml) (void)hipFree(ml.d_blob);
  }
  for (double* x : p->part) (void)hipFree(x);
  (void)hipFree(p->d_slice_lists);
  if (p->abs_from_ctx)
    p->ctx->abs_leased = false;
  else
    (void)hipFree(p->d_abs);
  (void)hipFree(p->d_cs);
  if (p->graph) (void)hipGraphExecDestroy(p->graph);
  delete p;
  return BSG_OK;
}

int64_t bsg_plan_arena_extent(const bsg_plan* p) { return p ? p->arena_extent : 0; }
int64_t bsg_plan_partial_doubles(const bsg_plan* p) {
  if (!p) return 0;
  int64_t split = p->split_partials;
  if (split < 0) {  // the split lists' cut, whether or not they are made yet
    split = 0;
    std::vector<ListPart> loc;
    int nth = 0;
    for (const PlanChunk& pc : p->chunks)
      split = std::max(split, pc.ml[1].ready ? pc.ml[1].part_doubles : cut_to_fit(p, pc, true, loc, nth));
    p->split_partials = split;
  }
  return std::max(p->part_doubles[0], split);
}

}  // extern "C"

namespace {
// open-addressing tables (no allocation per entry), grown by doubling at
// half load so that their size follows the distinct blocks, not the pairs:
// keys of the operator blocks (offset, orientation, rows, cols) and of the
// C blocks (offset, rows, cols)
struct SliceTable {
  struct E {
    int64_t off, key, val;  // off < 0: empty
  };
  std::vector<E> e;
  size_t n = 0;
  explicit SliceTable(size_t hint) {  // hint: entries expected at most
    size_t cap = 4096;
    while (cap < hint) cap <<= 1;
    e.assign(cap, E{-1, 0, 0});
  }
  static size_t hash(int64_t off, int64_t key) {
    uint64_t h = (uint64_t)off * 0x9E3779B97F4A7C15ull ^ (uint64_t)key * 0xC2B2AE3D27D4EB4Full;
    h ^= h >> 31;
    h *= 0xBF58476D1CE4E5B9ull;
    return (size_t)(h ^ (h >> 29));
  }
  E& slot(int64_t off, int64_t key) {
    const size_t mask = e.size() - 1;
    for (size_t h = hash(off, key) & mask;; h = (h + 1) & mask)
      if (e[h].off < 0 || (e[h].off == off && e[h].key == key)) return e[h];
  }
  // the value of (off, key), made by make() on first sight
  template <class F>
  int64_t get(int64_t off, int64_t key, F&& make) {
    if (2 * (n + 1) > e.size()) {
      std::vector<E> old(2 * e.size(), E{-1, 0, 0});
      old.swap(e);
      for (const E& x : old)
        if (x.off >= 0) slot(x.off, x.key) = x;
    }
    E& x = slot(off, key);
    if (x.off < 0) {
      x = E{off, key, make()};
      ++n;
    }
    return x.val;
  }
};
// BF16 slice recipes of a plan, one per distinct (operator block,
// orientation) and per C block its grouped-kernel pairs read, and the pairs'
// slice offsets; made on the first split-precision set-up, so FP64-only
// plans (the rotations, FP64 solves) never pay for them.
int build_slices(bsg_plan* p) {
  // the operator table sized by its references (most operator blocks of a
  // superblock are referenced once) and its item list reserved likewise;
  // the C blocks are few (one per wavefunction block)
  size_t n_ab = 0;
  // f(pair index, V block) for every pair that reads slices: all but the
  // small-block kernel's
  auto sliced = [](const PlanChunk& pc, auto f) {
    for (size_t i = 0; i < pc.h_vb.size(); ++i)
      for (int64_t j = pc.h_base[i] + (small_block(pc.h_vb[i]) ? pc.h_fast[i] : 0); j < pc.h_base[i] + pc.h_vb[i].count; ++j)
        f(j, pc.h_vb[i]);
  };
  for (auto& pc : p->chunks)
    sliced(pc, [&](int64_t j, const bsg_vblock_t&) { n_ab += (pc.h_perm[j].a_off >= 0) + (pc.h_perm[j].b_off >= 0); });
  SliceTable abt(n_ab), ct(0);
  p->ab_items.reserve(n_ab);
  auto slice_of = [&](std::vector<SliceItem>& items, int64_t& elems, int64_t src, int rows, int cols, int trans) {
    SliceItem it;
    it.src = src;
    it.dst = elems;
    it.rows = rows;
    it.cols = cols;
    it.pitch = (cols + 7) & ~7;
    it.trans = trans;
    items.push_back(it);
    elems += 3 * (int64_t)rows * it.pitch;
    return it.dst;
  };
  auto ab_slice = [&](int64_t off, int trans, int rows, int cols) {
    const int64_t key = ((int64_t)rows << 33) | ((int64_t)cols << 1) | trans;
    return abt.get(off, key, [&] { return slice_of(p->ab_items, p->ab_elems, off, rows, cols, trans); });
  };
  auto c_slice = [&](int64_t off, int k1, int k2) {
    // C^T: (j, p) = C[p k2 + j]; pairs may read one offset as different shapes
    const int64_t key = ((int64_t)k1 << 32) | k2;
    return ct.get(off, key, [&] { return slice_of(p->c_items, p->c_elems, off, k2, k1, 1); });
  };
  for (auto& pc : p->chunks) {
    std::vector<PairS>& ps = pc.h_ps;
    ps.assign(pc.n_pairs, PairS{-1, -1, -1});
    sliced(pc, [&](int64_t j, const bsg_vblock_t& vb) {
      const bsg_pair_t& pr = pc.h_perm[j];
      if (pr.a_off >= 0) {
        ps[j].a = ab_slice(pr.a_off, pr.a_trans, vb.m, pr.k1);  // op(A)(i, p), K = p contiguous
        ps[j].c = c_slice(pr.c_off, pr.k1, pr.k2);
      }
      if (pr.b_off >= 0) ps[j].b = ab_slice(pr.b_off, pr.b_trans ? 0 : 1, vb.n, pr.k2);  // B'(k, col) as [col][k]
    });
  }
  Blob blob;
  std::vector<int32_t> first[2];  // the items' first chunks
  for (int c = 0; c < 2; ++c) {  // operators, wavefunction
    const std::vector<SliceItem>& items = c ? p->c_items : p->ab_items;
    std::vector<int32_t>& at = first[c];
    at.assign(items.size() + 1, 0);
    for (size_t i = 0; i < items.size(); ++i) at[i + 1] = at[i] + (slice_groups(items[i]) + SLICE_GROUPS - 1) / SLICE_GROUPS;
    const size_t item_at = blob.place(c ? &p->d_c_items : &p->d_ab_items, sizeof(SliceItem) * items.size()),
                 chunk_at = blob.place(c ? &p->d_c_chunks : &p->d_ab_chunks, sizeof(SliceChunk) * at.back());
    constexpr size_t STEP = 4096;  // items a thread takes at a time
    for (size_t i0 = 0; i0 < items.size(); i0 += STEP)
      blob.jobs.push_back([&items, &at, item_at, chunk_at, i0](char* to) {
        for (size_t i = i0; i < std::min(items.size(), i0 + STEP); ++i) {
          ((SliceItem*)(to + item_at))[i] = items[i];
          SliceChunk* ch = (SliceChunk*)(to + chunk_at) + at[i];
          for (int g = 0; g < at[i + 1] - at[i]; ++g) ch[g] = SliceChunk{(int32_t)i, g * SLICE_GROUPS};
        }
      });
    (c ? p->n_c_chunks : p->n_ab_chunks) = at.back();
  }
  if (!blob.send(&p->d_slice_lists, MAX_PLAN_THREADS)) return fail(BSG_ERR_NOMEM, "bsg_plan_split_arena: slice recipes");
  p->slices_built = true;
  return BSG_OK;
}
}  // namespace

extern "C" {

int bsg_plan_split_arena(bsg_context* ctx, bsg_plan* p, const double* arena, int64_t n) {
  if (!ctx || !p || !arena || n < 0) return fail(BSG_ERR_ARG, "bsg_plan_split_arena: bad args");
  if (p->ctx != ctx) return fail(BSG_ERR_ARG, "bsg_plan_split_arena: plan belongs to another context");
  if (n < p->arena_extent) return fail(BSG_ERR_ARG, "bsg_plan_split_arena: arena smaller than the plan's extent");
  HIPCHK(hipSetDevice(ctx->device));
  // FP64-only plans (the rotations, FP64 solves) never pay for the split
  // lists and slice recipes
  if (!p->slices_built) {
    const int rc = build_slices(p);
    if (rc != BSG_OK) return rc;
  }
  for (auto& pc : p->chunks) {
    if (pc.ml[1].ready) continue;
    const int rc = plan_lists(p, pc, true);
    if (rc != BSG_OK) return rc;
    p->part_doubles[1] = std::max(p->part_doubles[1], pc.ml[1].part_doubles);
  }
  if (!p->part[1] && p->part_doubles[1] > 0 &&
      hipMalloc(&p->part[1], sizeof(double) * p->part_doubles[1] * p->batch) != hipSuccess)
    return fail(BSG_ERR_NOMEM, "bsg_plan_split_arena: partial-tile scratch");
  if (!p->wscratch[1] && p->w_doubles[1] > 0) {
    p->wroots[1] = rounds_roots(p->w_doubles[1], p->batch);
    if (!(p->wscratch[1] = w_scratch(ctx, p->w_doubles[1] * p->wroots[1])))
      return fail(BSG_ERR_NOMEM, "bsg_plan_split_arena: W scratch");
  }
  // operator slices (the small-block kernel stays FP64), and room for the C
  // slices of one launch's roots
  if (!p->d_abs && p->ab_elems > 0) {
    if (!ctx->abs_leased) {
      if (ctx->abs_cap < (size_t)p->ab_elems) {
        (void)hipFree(ctx->abs_buf);
        ctx->abs_buf = nullptr;
        ctx->abs_cap = 0;
        const size_t cap = (size_t)p->ab_elems + (size_t)p->ab_elems / 4;
        if (hipMalloc((void**)&ctx->abs_buf, 2 * cap) != hipSuccess)
          return fail(BSG_ERR_NOMEM, "bsg_plan_split_arena: operator slices");
        ctx->abs_cap = cap;
      }
      p->d_abs = ctx->abs_buf;
      ctx->abs_leased = true;
      p->abs_from_ctx = true;
    } else {
      hipError_t e = hipMalloc((void**)&p->d_abs, 2 * p->ab_elems);
      if (e != hipSuccess) return fail(BSG_ERR_NOMEM, "bsg_plan_split_arena: operator slices");
    }
  }
  if (!p->cs_ready && p->c_elems > 0) {
    hipError_t e = hipMalloc((void**)&p->d_cs, 2 * p->c_elems * p->batch);
    if (e != hipSuccess) return fail(BSG_ERR_NOMEM, "bsg_plan_split_arena: wavefunction slices");
  }
  p->cs_ready = true;
  if (!p->ab_items.empty())
    hipLaunchKernelGGL(k_slices, dim3((p->n_ab_chunks + 3) / 4), dim3(256), 0, ctx->stream, p->d_ab_chunks,
                       p->n_ab_chunks, p->d_ab_items, arena, p->d_abs,
                       (int64_t)0, (int64_t)0);
  HIPCHK(hipGetLastError());
  p->split_src = arena;
  return BSG_OK;
}

int bsg_set_tile_table(const int32_t* rules, int32_t n) {
  if (n < 0 || (n > 0 && !rules)) return fail(BSG_ERR_ARG, "bsg_set_tile_table: bad args");
  std::vector<TileRule> t;
  const int nfp = (int)geom_candidates(6).size(), nsp = (int)geom_candidates(4).size();
  for (int32_t i = 0; i < n; ++i) {
    const int32_t* e = rules + 6 * i;
    TileRule r{e[0], e[1], e[2], e[3], e[4], e[5]};
    if (r.m_lo > r.m_hi || r.n_lo > r.n_hi || r.fp64 < -1 || r.fp64 > nfp || r.split < -1 || r.split >= nsp)
      return fail(BSG_ERR_ARG, "bsg_set_tile_table: bad rule");
    t.push_back(r);
  }
  auto rs = std::make_shared<RuleSet>();
  rs->rules = t;
  rs->version = g_tile_rules->version + 1;
  g_tile_rules = rs;
  return BSG_OK;
}
int bsg_tile_candidates(int32_t precision) {
  // FP64: the geometries, then the per-wave kernel
  return precision == BSG_SPLIT_BF16 ? (int)geom_candidates(4).size() : (int)geom_candidates(6).size() + 1;
}

int bsg_plan_set_batch(bsg_context* ctx, bsg_plan* p, int32_t nroot) {
  if (!ctx || !p || nroot < 1) return fail(BSG_ERR_ARG, "bsg_plan_set_batch: bad args");
  if (p->ctx != ctx) return fail(BSG_ERR_ARG, "bsg_plan_set_batch: plan belongs to another context");
  if (nroot == p->batch) return BSG_OK;
  HIPCHK(hipSetDevice(ctx->device));
  HIPCHK(hipStreamSynchronize(ctx->stream));  // no queued work reads the old buffers
  if (p->graph) {  // it reads the buffers replaced below
    HIPCHK(hipGraphExecDestroy(p->graph));
    p->graph = nullptr;
  }
  // the rounds of large blocks take as many roots per launch as W_ROOTS
  // doubles of scratch hold
  int32_t wroots[2];
  for (int k = 0; k < 2; ++k) wroots[k] = rounds_roots(p->w_doubles[k], nroot);
  // every new buffer before any old one goes: a failure leaves the plan as it was
  double* np[2] = {};
  std::shared_ptr<WScratch> nw[2];
  __bf16* nc = nullptr;
  const bool cs = p->cs_ready && p->c_elems > 0;
  auto more_w = [&](int k) { return p->wscratch[k] && wroots[k] != p->wroots[k]; };
  if ((p->part[0] && hipMalloc(&np[0], sizeof(double) * p->part_doubles[0] * nroot) != hipSuccess) ||
      (p->part[1] && hipMalloc(&np[1], sizeof(double) * p->part_doubles[1] * nroot) != hipSuccess) ||
      (more_w(0) && !(nw[0] = w_scratch(ctx, p->w_doubles[0] * wroots[0]))) ||
      (more_w(1) && !(nw[1] = w_scratch(ctx, p->w_doubles[1] * wroots[1]))) ||
      (cs && hipMalloc((void**)&nc, 2 * p->c_elems * nroot) != hipSuccess)) {
    for (double* x : np) (void)hipFree(x);
    return fail(BSG_ERR_NOMEM, "bsg_plan_set_batch: scratch of the roots");
  }
  for (int k = 0; k < 2; ++k)
    if (np[k]) {
      (void)hipFree(p->part[k]);
      p->part[k] = np[k];
    }
  for (int k = 0; k < 2; ++k)
    if (nw[k]) {
      p->wscratch[k] = nw[k];
      p->wroots[k] = wroots[k];
    }
  if (nc) {
    (void)hipFree(p->d_cs);
    p->d_cs = nc;
  }
  p->batch = nroot;
  return BSG_OK;
}

double bsg_plan_flops(const bsg_plan* p) { return p ? p->flops : 0.0; }
double bsg_plan_split_share(const bsg_plan* p) { return p && p->flops > 0.0 ? p->flops_split / p->flops : 0.0; }
double bsg_plan_split_gain_share(const bsg_plan* p) { return p && p->flops > 0.0 ? p->flops_past / p->flops : 0.0; }
int bsg_plan_phase_flops(const bsg_plan* p, double* f1, double* f2) {
  if (!p || !f1 || !f2) return fail(BSG_ERR_ARG, "bsg_plan_phase_flops: bad args");
  *f1 = p->flops1;
  *f2 = p->flops2;
  return BSG_OK;
}

}  // extern "C"

namespace {
// Launch one chunk for rs.n roots: the widest blocks' kernels on the context
// stream with the side-stream kernels beside them, then the ordered
// reduction.  ev (optional) receives 5 events: before the fused kernels,
// around the side stream's kernels, before and after the reduction.
// launches (optional) counts the kernel dispatches.
int enqueue_chunk(bsg_context* ctx, const bsg_plan* p, const PlanChunk& ch, const double* arena, const double* c,
                  double* v, hipEvent_t* ev, bool split, double* part, const RootSet& rs, long* launches = nullptr) {
  hipStream_t st = ctx->stream;
  const ModeLists& ml = ch.ml[split];
  auto grid = [&](int n) { return dim3((unsigned)(((n + 7) / 8) * 8 * rs.n)); };
  long nl = 0;
  if (ev) HIPCHK(hipEventRecord(ev[0], st));
  // the side stream runs the small-block kernel and the basic tiles beside
  // the wide tiles on the context stream; they write disjoint V blocks and
  // partial tiles, and the reduction waits for both
  const int nbasic = ml.n_g[0];
  const int *ns = ml.n_s;
  const bool side = ml.side();
  // round r of the large blocks, in launches of the roots its scratch holds
  auto round = [&](size_t r, hipStream_t q) {
    const GemmRound& g = ml.rounds[r];
    double* wbuf = p->wscratch[split] ? p->wscratch[split]->ptr : nullptr;
    for (int r0 = 0; r0 < rs.n; r0 += p->wroots[split]) {
      RootSet sub = rs;
      sub.n = std::min(p->wroots[split], rs.n - r0);
      const double* cr = c + r0 * rs.wstride;
      const __bf16* csr = p->d_cs + r0 * rs.cstride;
      double *vr = v + r0 * rs.wstride, *pr = part + r0 * rs.pstride;
      auto tiles = [&](TileRef* const(&t)[2], const int(&n)[2]) {
        for (int k = 1; k >= 0; --k) {
          if (n[k] == 0) continue;
          const dim3 blocks((unsigned)(((n[k] + 7) / 8) * 8 * sub.n));
          if (!split)
            hipLaunchKernelGGL((k_gemm<GemmT>), blocks, dim3(GemmT::NT), 0, q, ml.d_gu, ml.d_gs, ml.d_ga, t[k], n[k],
                               arena, cr, vr, wbuf, pr, sub);
          else if (k == 1)
            hipLaunchKernelGGL((k_gemm_bf<SplitBig>), blocks, dim3(SplitBig::NT), 0, q, ml.d_gu, ml.d_gs, ml.d_ga, t[k],
                               n[k], p->d_abs, csr, cr, vr, (__bf16*)wbuf, pr, sub);
          else
            hipLaunchKernelGGL((k_gemm_bf<SplitSmall>), blocks, dim3(SplitSmall::NT), 0, q, ml.d_gu, ml.d_gs, ml.d_ga,
                               t[k], n[k], p->d_abs, csr, cr, vr, (__bf16*)wbuf, pr, sub);
          ++nl;
        }
      };
      tiles(g.d_w, g.n_w);
      tiles(g.d_v, g.n_v);
    }
  };
  if (side) {
    HIPCHK(hipEventRecord(ctx->fork, st));
    HIPCHK(hipStreamWaitEvent(ctx->side, ctx->fork, 0));
    if (ev) HIPCHK(hipEventRecord(ev[1], ctx->side));
    for (size_t r = 1; r < ml.rounds.size(); r += 2) round(r, ctx->side);
    if (ml.n_p[0] > 0) {
      hipLaunchKernelGGL((k_panel<3>), grid(ml.n_p[0]), dim3(256), 0, ctx->side, ch.d_vb, ml.d_pp, ml.d_seg, ml.d_p[0],
                         ml.n_p[0], arena, c, v, part, rs);
      ++nl;
    }
    if (ns[2] > 0) {
      hipLaunchKernelGGL((k_small<4>), grid(ns[2]), dim3(64), 0, ctx->side, ch.d_vb, ml.d_pp, ml.d_seg, ml.d_s[2],
                         ns[2], arena, c, v, part, rs);
      ++nl;
    }
    if (ns[1] > 0) {
      hipLaunchKernelGGL((k_small<3>), grid(ns[1]), dim3(64), 0, ctx->side, ch.d_vb, ml.d_pp, ml.d_seg, ml.d_s[1],
                         ns[1], arena, c, v, part, rs);
      ++nl;
    }
    if (nbasic > 0) {
      if (split)
        hipLaunchKernelGGL((k_sigma_bf<2, 2>), grid(nbasic), dim3(256), 0, ctx->side, ch.d_vb, ch.d_pr, ch.d_ps,
                           ml.d_seg, ml.d_g[0], nbasic, p->d_abs, p->d_cs, c, v, part, rs);
      else
        hipLaunchKernelGGL((k_sigma<2, 2>), grid(nbasic), dim3(256), 0, ctx->side, ch.d_vb, ch.d_pr, ml.d_seg,
                           ml.d_g[0], nbasic, arena, c, v, part, rs);
      ++nl;
    }
    if (ev) HIPCHK(hipEventRecord(ev[2], ctx->side));
    HIPCHK(hipEventRecord(ctx->join, ctx->side));
  }
  if (ns[0] > 0) {
    hipLaunchKernelGGL((k_small<2>), grid(ns[0]), dim3(64), 0, st, ch.d_vb, ml.d_pp, ml.d_seg, ml.d_s[0], ns[0],
                       arena, c, v, part, rs);
    ++nl;
  }
  for (size_t r = 0; r < ml.rounds.size(); r += 2) round(r, st);
  if (split) {
    if (ml.n_g[2] > 0) {
      hipLaunchKernelGGL((k_sigma_bf<1, 4, 8>), grid(ml.n_g[2]), dim3(512), 0, st, ch.d_vb, ch.d_pr, ch.d_ps,
                         ml.d_seg, ml.d_g[2], ml.n_g[2], p->d_abs, p->d_cs, c, v, part, rs);
      ++nl;
    }
    if (ml.n_g[1] > 0) {
      hipLaunchKernelGGL((k_sigma_bf<1, 4>), grid(ml.n_g[1]), dim3(256), 0, st, ch.d_vb, ch.d_pr, ch.d_ps, ml.d_seg,
                         ml.d_g[1], ml.n_g[1], p->d_abs, p->d_cs, c, v, part, rs);
      ++nl;
    }
  } else {
    if (ml.n_p[2] > 0) {
      hipLaunchKernelGGL((k_panel<6>), grid(ml.n_p[2]), dim3(256), 0, st, ch.d_vb, ml.d_pp, ml.d_seg, ml.d_p[2],
                         ml.n_p[2], arena, c, v, part, rs);
      ++nl;
    }
    if (ml.n_p[1] > 0) {
      hipLaunchKernelGGL((k_panel<5>), grid(ml.n_p[1]), dim3(256), 0, st, ch.d_vb, ml.d_pp, ml.d_seg, ml.d_p[1],
                         ml.n_p[1], arena, c, v, part, rs);
      ++nl;
    }
    if (ml.n_w[1] > 0) {
      hipLaunchKernelGGL((k_wave<4>), grid(ml.n_w[1] / 4), dim3(256), 0, st, ch.d_vb, ch.d_pr, ml.d_seg, ml.d_w[1],
                         ml.n_w[1], arena, c, v, part, rs);
      ++nl;
    }
    if (ml.n_w[0] > 0) {
      hipLaunchKernelGGL((k_wave<2>), grid(ml.n_w[0] / 4), dim3(256), 0, st, ch.d_vb, ch.d_pr, ml.d_seg, ml.d_w[0],
                         ml.n_w[0], arena, c, v, part, rs);
      ++nl;
    }
    if (ml.n_g[3] > 0) {
      hipLaunchKernelGGL((k_sigma<1, 6, PB, 8>), grid(ml.n_g[3]), dim3(512), 0, st, ch.d_vb, ch.d_pr, ml.d_seg,
                         ml.d_g[3], ml.n_g[3], arena, c, v, part, rs);
      ++nl;
    }
    if (ml.n_g[2] > 0) {
      hipLaunchKernelGGL((k_sigma<1, 6>), grid(ml.n_g[2]), dim3(256), 0, st, ch.d_vb, ch.d_pr, ml.d_seg, ml.d_g[2],
                         ml.n_g[2], arena, c, v, part, rs);
      ++nl;
    }
    if (ml.n_g[1] > 0) {
      hipLaunchKernelGGL((k_sigma<1, 4>), grid(ml.n_g[1]), dim3(256), 0, st, ch.d_vb, ch.d_pr, ml.d_seg, ml.d_g[1],
                         ml.n_g[1], arena, c, v, part, rs);
      ++nl;
    }
  }
  if (side) HIPCHK(hipStreamWaitEvent(st, ctx->join, 0));
  if (ev) HIPCHK(hipEventRecord(ev[3], st));
  if (ml.n_red > 0) {
    hipLaunchKernelGGL(k_reduce, dim3(ml.n_red, rs.n), dim3(256), 0, st, ml.d_red, part, v, rs);
    ++nl;
  }
  if (ev) HIPCHK(hipEventRecord(ev[4], st));
  HIPCHK(hipGetLastError());
  if (launches) *launches += nl;
  return BSG_OK;
}

int check_precision(const bsg_plan* p, const double* arena, int32_t precision) {
  if (precision == BSG_FP64) return BSG_OK;
  if (precision != BSG_SPLIT_BF16) return fail(BSG_ERR_ARG, "unknown precision mode");
  if (p->split_src != arena || !p->slices_built || (p->part_doubles[1] > 0 && !p->part[1]) || (p->w_doubles[1] > 0 && !p->wscratch[1]) || (p->ab_elems > 0 && !p->d_abs) || (p->c_elems > 0 && !p->d_cs))
    return fail(BSG_ERR_ARG, "split precision needs bsg_plan_split_arena on this arena first");
  return BSG_OK;
}
// v += H c for nvec vectors, at most `group` roots per launch, with the
// partial tiles of split V blocks in part (roots part_doubles apart; written
// before they are read within each launch, so no clearing).  launches
// (optional) counts the kernel dispatches; ev (optional) receives 5 events
// per chunk launch.
int sigma_apply_with(bsg_context* ctx, bsg_plan* p, const double* arena, const double* c, double* v, int32_t nvec,
                     int32_t precision, double* part, int group, long* launches = nullptr, hipEvent_t* ev = nullptr) {
  int rc = check_precision(p, arena, precision);
  if (rc) return rc;
  const bool split = precision == BSG_SPLIT_BF16;
  group = std::max(1, std::min(group, p->batch));
  for (int iv = 0; iv < nvec; iv += group) {
    RootSet rs;
    rs.n = std::min(group, nvec - iv);
    rs.pad = 0;
    rs.wstride = p->wave_size;
    rs.pstride = p->part_doubles[split];
    rs.cstride = p->c_elems;
    rs.tstride = p->w_doubles[split];
    const double* cv = c + (size_t)iv * p->wave_size;
    double* vv = v + (size_t)iv * p->wave_size;
    if (split && !p->c_items.empty()) {
      hipLaunchKernelGGL(k_slices, dim3((p->n_c_chunks + 3) / 4, rs.n), dim3(256), 0, ctx->stream, p->d_c_chunks,
                         p->n_c_chunks, p->d_c_items, cv,
                         p->d_cs, rs.wstride, rs.cstride);
      if (launches) ++*launches;
    }
    for (auto& ch : p->chunks) {
      if ((rc = enqueue_chunk(ctx, p, ch, arena, cv, vv, ev, split, part, rs, launches))) return rc;
      if (ev) ev += 5;
    }
  }
  return BSG_OK;
}
}  // namespace

extern "C" {

int bsg_sigma_apply(bsg_context* ctx, bsg_plan* p, const double* arena, const double* c, double* v, int32_t nvec,
                    int32_t precision) {
  if (!ctx || !p || !arena || !c || !v || nvec <= 0) return fail(BSG_ERR_ARG, "bsg_sigma_apply: bad args");
  if (p->ctx != ctx) return fail(BSG_ERR_ARG, "bsg_sigma_apply: plan belongs to another context");
  std::lock_guard<std::mutex> lk(ctx->apply);
  return sigma_apply_with(ctx, p, arena, c, v, nvec, precision, p->part[precision == BSG_SPLIT_BF16], p->batch);
}

int bsg_plan_capture(bsg_context* ctx, bsg_plan* p, const double* arena, const double* c, double* v, int32_t nvec,
                     int32_t precision) {
  if (!ctx || !p || !arena || !c || !v || nvec <= 0) return fail(BSG_ERR_ARG, "bsg_plan_capture: bad args");
  if (p->ctx != ctx) return fail(BSG_ERR_ARG, "bsg_plan_capture: plan belongs to another context");
  std::lock_guard<std::mutex> lk(ctx->apply);
  int rc = check_precision(p, arena, precision);
  if (rc) return rc;
  HIPCHK(hipSetDevice(ctx->device));
  HIPCHK(hipStreamSynchronize(ctx->stream));
  if (p->graph) {
    HIPCHK(hipGraphExecDestroy(p->graph));
    p->graph = nullptr;
    p->g_nvec = 0;
  }
  // the launches of one application on the context stream (the side stream
  // joins through the fork/join events and is captured with it); no memset
  // or allocation is recorded
  HIPCHK(hipStreamBeginCapture(ctx->stream, hipStreamCaptureModeThreadLocal));
  rc = sigma_apply_with(ctx, p, arena, c, v, nvec, precision, p->part[precision == BSG_SPLIT_BF16], p->batch);
  hipGraph_t g = nullptr;
  const hipError_t e = hipStreamEndCapture(ctx->stream, &g);
  if (rc) {
    if (g) (void)hipGraphDestroy(g);
    return rc;
  }
  if (e != hipSuccess) return fail(BSG_ERR_HIP, std::string("hipStreamEndCapture: ") + hipGetErrorString(e));
  hipGraphExec_t x = nullptr;
  const hipError_t e2 = hipGraphInstantiate(&x, g, nullptr, nullptr, 0);
  (void)hipGraphDestroy(g);
  if (e2 != hipSuccess) return fail(BSG_ERR_HIP, std::string("hipGraphInstantiate: ") + hipGetErrorString(e2));
  p->graph = x;
  p->g_arena = arena;
  p->g_c = c;
  p->g_v = v;
  p->g_nvec = nvec;
  p->g_precision = precision;
  return BSG_OK;
}

int bsg_plan_replay(bsg_context* ctx, bsg_plan* p) {
  if (!ctx || !p || !p->graph) return fail(BSG_ERR_ARG, "bsg_plan_replay: no captured application");
  if (p->ctx != ctx) return fail(BSG_ERR_ARG, "bsg_plan_replay: plan belongs to another context");
  // the slices the split kernels read must still be those of the captured arena
  int rc = check_precision(p, p->g_arena, p->g_precision);
  if (rc) return rc;
  std::lock_guard<std::mutex> lk(ctx->apply);  // not between the launches of another thread's application
  HIPCHK(hipGraphLaunch(p->graph, ctx->stream));
  return BSG_OK;
}

int bsg_sigma_apply_noalloc(bsg_context* ctx, bsg_plan* p, const double* arena, const double* c, double* v,
                            int32_t nvec, int32_t precision) {
  if (!ctx || !p || !arena || !c || !v || nvec <= 0) return fail(BSG_ERR_ARG, "bsg_sigma_apply_noalloc: bad args");
  if (p->ctx != ctx) return fail(BSG_ERR_ARG, "bsg_sigma_apply_noalloc: plan belongs to another context");
  std::lock_guard<std::mutex> lk(ctx->apply);
  if (!ctx->scratch) return fail(BSG_ERR_ARG, "bsg_sigma_apply_noalloc: no scratch address for this device");
  const int64_t need = p->part_doubles[precision == BSG_SPLIT_BF16];
  if (need > BSG_NOALLOC_SCRATCH_DOUBLES)
    return fail(BSG_ERR_ARG, "bsg_sigma_apply_noalloc: the plan needs " + std::to_string(need) +
                                 " doubles of partial tiles, more than the " +
                                 std::to_string((long long)BSG_NOALLOC_SCRATCH_DOUBLES) + " of the static scratch");
  // as many roots per launch as the scratch holds partial tiles for
  const int group = need > 0 ? (int)std::min<int64_t>(p->batch, BSG_NOALLOC_SCRATCH_DOUBLES / need) : p->batch;
  return sigma_apply_with(ctx, p, arena, c, v, nvec, precision, ctx->scratch, group);
}

int bsg_sigma_profile(bsg_context* ctx, bsg_plan* p, const double* arena, const double* c, double* v, int32_t nvec,
                      int32_t reps, int32_t precision, double* wall_ms, double* kernel_ms, long* launches) {
  if (!ctx || !p || !arena || !c || !v || nvec <= 0 || reps <= 0 || !wall_ms || !kernel_ms || !launches)
    return fail(BSG_ERR_ARG, "bsg_sigma_profile: bad args");
  int rc = check_precision(p, arena, precision);
  if (rc) return rc;
  const bool split = precision == BSG_SPLIT_BF16;
  const size_t nch = p->chunks.size();
  const int ngroups = (nvec + p->batch - 1) / p->batch;
  constexpr size_t per = 5;  // events per chunk launch (enqueue_chunk)
  struct Events : std::vector<hipEvent_t> {
    using std::vector<hipEvent_t>::vector;
    ~Events() {
      for (hipEvent_t e : *this)
        if (e) (void)hipEventDestroy(e);
    }
  } ev((size_t)reps * ngroups * nch * per + 2, nullptr);
  for (auto& e : ev) HIPCHK(hipEventCreate(&e));
  long disp = 0;
  std::lock_guard<std::mutex> lk(ctx->apply);
  HIPCHK(hipEventRecord(ev[0], ctx->stream));
  for (int r = 0; r < reps; ++r)
    if ((rc = sigma_apply_with(ctx, p, arena, c, v, nvec, precision, p->part[precision == BSG_SPLIT_BF16], p->batch, &disp,
                               &ev[1 + (size_t)r * ngroups * nch * per])))
      return rc;
  const size_t q = 1 + (size_t)reps * ngroups * nch * per;
  HIPCHK(hipEventRecord(ev[q], ctx->stream));
  HIPCHK(hipEventSynchronize(ev[q]));
  float ms = 0.f;
  HIPCHK(hipEventElapsedTime(&ms, ev[0], ev[q]));
  *wall_ms = ms;
  for (int i = 0; i < 3; ++i) {
    kernel_ms[i] = 0.0;
    launches[i] = 0;
  }
  size_t k = 1;
  for (int r = 0; r < reps * ngroups; ++r)
    for (auto& ch : p->chunks) {
      const ModeLists& ml = ch.ml[split];
      // [0] fork to join of all fused kernels, [1] reduction, [2] the side
      // stream's kernels alone
      const int from[3] = {0, 3, 1}, to[3] = {3, 4, 2};
      const bool present[3] = {true, ml.n_red > 0, ml.side()};
      for (int i = 0; i < 3; ++i) {
        if (!present[i]) continue;
        HIPCHK(hipEventElapsedTime(&ms, ev[k + from[i]], ev[k + to[i]]));
        kernel_ms[i] += ms;
      }
      k += per;
    }
  // kernel dispatches of all applications (every kernel launch counted)
  launches[0] = disp;
  return BSG_OK;
}

int bsg_diag_apply(bsg_context* ctx, const bsg_diag_t* terms, int32_t n, const double* arena, double* diag) {
  if (!ctx || (n > 0 && (!terms || !diag))) return fail(BSG_ERR_ARG, "bsg_diag_apply: bad args");
  if (n == 0) return BSG_OK;
  // group terms by target block, keeping their order inside a group
  std::vector<int> idx(n);
  for (int i = 0; i < n; ++i) idx[i] = i;
  std::stable_sort(idx.begin(), idx.end(), [&](int a, int b) { return terms[a].v_off < terms[b].v_off; });
  std::vector<bsg_diag_t> sorted(n);
  std::vector<DiagGroup> groups;
  for (int i = 0; i < n; ++i) {
    sorted[i] = terms[idx[i]];
    if (i == 0 || sorted[i].v_off != sorted[i - 1].v_off) groups.push_back({i, 0});
    else if (sorted[i].m != sorted[i - 1].m || sorted[i].n != sorted[i - 1].n)
      return fail(BSG_ERR_ARG, "bsg_diag_apply: terms of one block disagree on its shape");
    groups.back().count++;
  }
  std::vector<DiagItem> items;
  for (size_t g = 0; g < groups.size(); ++g) {
    const int64_t mn = (int64_t)sorted[groups[g].first].m * sorted[groups[g].first].n;
    for (int64_t e0 = 0; e0 < mn; e0 += 256) items.push_back({(int32_t)g, (int32_t)e0});
  }
  if (items.empty()) return BSG_OK;
  bsg_diag_t* dt = nullptr;
  DiagGroup* dg = nullptr;
  DiagItem* di = nullptr;
  HIPCHK(hipMalloc(&dt, sizeof(bsg_diag_t) * n));
  HIPCHK(hipMalloc(&dg, sizeof(DiagGroup) * groups.size()));
  HIPCHK(hipMalloc(&di, sizeof(DiagItem) * items.size()));
  HIPCHK(hipMemcpyAsync(dt, sorted.data(), sizeof(bsg_diag_t) * n, hipMemcpyHostToDevice, ctx->stream));
  HIPCHK(hipMemcpyAsync(dg, groups.data(), sizeof(DiagGroup) * groups.size(), hipMemcpyHostToDevice, ctx->stream));
  HIPCHK(hipMemcpyAsync(di, items.data(), sizeof(DiagItem) * items.size(), hipMemcpyHostToDevice, ctx->stream));
  hipLaunchKernelGGL(k_diag, dim3(items.size()), dim3(256), 0, ctx->stream, dt, dg, di, arena, diag);
  HIPCHK(hipGetLastError());
  HIPCHK(hipStreamSynchronize(ctx->stream));
  HIPCHK(hipFree(dt));
  HIPCHK(hipFree(dg));
  HIPCHK(hipFree(di));
  return BSG_OK;
}

int bsg_dot(bsg_context* ctx, const double* x, const double* y, int64_t n, double* result) {
  if (!ctx || !x || !y || !result || n < 0) return fail(BSG_ERR_ARG, "bsg_dot: bad args");
  const int nb = reduce_grid(n);
  hipLaunchKernelGGL(k_dot_partial<false>, dim3(nb), dim3(RB), 0, ctx->stream, x, y, (const double*)nullptr, n, ctx->red);
  hipLaunchKernelGGL(k_sum_partial, dim3(1), dim3(RB), 0, ctx->stream, ctx->red, nb, ctx->res_pin);
  HIPCHK(hipGetLastError());
  HIPCHK(hipStreamSynchronize(ctx->stream));
  *result = ctx->res_pin[0];
  return BSG_OK;
}
int bsg_gs_orthonormalise(bsg_context* ctx, double* r, const double* B, int32_t m, int64_t ld, int64_t n,
                          int32_t normalise) {
  if (!ctx || !r || n < 0 || m < 0 || (m > 0 && (!B || ld < n))) return fail(BSG_ERR_ARG, "bsg_gs_orthonormalise: bad args");
  if (n == 0) return BSG_OK;
  const int nb = reduce_grid(n);
  double *pin = ctx->red, *pout = ctx->red + 2 * RMAXB;
  if (m > 0) {
    hipLaunchKernelGGL(k_dot_partial<true>, dim3(nb), dim3(RB), 0, ctx->stream, r, r, B, n, pin);
    for (int32_t j = 0; j < m; ++j) {
      const double* bj = B + (int64_t)j * ld;
      hipLaunchKernelGGL(k_gs_step, dim3(nb), dim3(RB), 0, ctx->stream, r, bj, j + 1 < m ? bj + ld : nullptr, n, pin, nb,
                         pout);
      std::swap(pin, pout);
    }
  } else if (normalise) {
    hipLaunchKernelGGL(k_dot_partial<false>, dim3(nb), dim3(RB), 0, ctx->stream, r, r, (const double*)nullptr, n, pin);
  }
  if (normalise) hipLaunchKernelGGL(k_scal_rsqrt, dim3(nb), dim3(RB), 0, ctx->stream, pin, nb, 1e-15, r, n);
  HIPCHK(hipGetLastError());
  return BSG_OK;
}
int bsg_axpy(bsg_context* ctx, double a, const double* x, double* y, int64_t n) {
  if (!ctx || !x || !y || n < 0) return fail(BSG_ERR_ARG, "bsg_axpy: bad args");
  if (n == 0) return BSG_OK;
  hipLaunchKernelGGL(k_axpy, dim3(grid_for(n)), dim3(256), 0, ctx->stream, a, x, y, n);
  HIPCHK(hipGetLastError());
  return BSG_OK;
}
int bsg_gram(bsg_context* ctx, const double* X, const double* Y, int32_t m, int64_t n, int64_t ld, double* out) {
  if (!ctx || !X || !Y || !out || m <= 0 || m > GRAM_MAX || n < 0 || ld < n)
    return fail(BSG_ERR_ARG, "bsg_gram: bad args");
  // about four 16-deep steps per wavefront at least
  const int nblk = (int)std::max<int64_t>(1, std::min<int64_t>(GBLK, (n + 255) / 256));
  double* part = ctx->gpart;
  // GMAX x GMAX tiles in stream order (the partials are reused tile by tile);
  // the sums go straight to page-locked host memory
  for (int i0 = 0; i0 < m; i0 += GMAX)
    for (int j0 = 0; j0 < m; j0 += GMAX) {
      const int mx = std::min(GMAX, m - i0), my = std::min(GMAX, m - j0);
      hipLaunchKernelGGL(k_gram_partial, dim3(nblk), dim3(256), 0, ctx->stream, X + (int64_t)i0 * ld,
                         Y + (int64_t)j0 * ld, mx, my, n, ld, part);
      hipLaunchKernelGGL(k_gram_sum, dim3((mx * my + 3) / 4), dim3(256), 0, ctx->stream, part, nblk, mx, my,
                         ctx->res_pin + (int64_t)i0 * m + j0, m);
    }
  HIPCHK(hipGetLastError());
  HIPCHK(hipStreamSynchronize(ctx->stream));
  std::memcpy(out, ctx->res_pin, sizeof(double) * m * m);
  return BSG_OK;
}
int bsg_lincomb(bsg_context* ctx, const double* X, int32_t m, int64_t n, int64_t ld, const double* coef, int32_t mo,
                double* Y, int64_t ldy) {
  if (!ctx || !X || !coef || !Y || m <= 0 || m > GRAM_MAX || mo <= 0 || mo > GRAM_MAX || n < 0 || ld < n || ldy < n)
    return fail(BSG_ERR_ARG, "bsg_lincomb: bad args");
  // coefficients through page-locked staging slots used in turn, so the call
  // returns without waiting for the kernels (a slot is reused once its last
  // copy is done; its device copy is behind that in stream order)
  const int slot = ctx->coef_next;
  ctx->coef_next = (slot + 1) % COEF_SLOTS;
  const size_t at = (size_t)slot * GRAM_MAX * GRAM_MAX;
  double* cd = ctx->gpart + (size_t)GBLK * GMAX * GMAX + at;
  HIPCHK(hipEventSynchronize(ctx->coef_done[slot]));
  for (int32_t i = 0; i < m; ++i)  // transposed: a result's coefficients contiguous
    for (int32_t j = 0; j < mo; ++j) ctx->coef_pin[at + (size_t)j * m + i] = coef[(size_t)i * mo + j];
  HIPCHK(hipMemcpyAsync(cd, ctx->coef_pin + at, sizeof(double) * m * mo, hipMemcpyHostToDevice, ctx->stream));
  HIPCHK(hipEventRecord(ctx->coef_done[slot], ctx->stream));
  // GMAX x GMAX coefficient tiles; the first row tile of each output tile
  // overwrites Y, the others add in order
  for (int j0 = 0; j0 < mo; j0 += GMAX)
    for (int i0 = 0; i0 < m; i0 += GMAX) {
      const int mt = std::min(GMAX, m - i0);
      auto run = [&](auto MB) {
        hipLaunchKernelGGL(k_lincomb<decltype(MB)::value>, dim3(grid_for((n + 1) / 2)), dim3(256), 0, ctx->stream,
                           X + (int64_t)i0 * ld, mt, n, ld, cd + (int64_t)j0 * m + i0, m, std::min(GMAX, mo - j0),
                           Y + (int64_t)j0 * ldy, ldy, i0 > 0 ? 1 : 0);
      };
      switch ((mt + 3) / 4) {
        case 1: run(std::integral_constant<int, 1>{}); break;
        case 2: run(std::integral_constant<int, 2>{}); break;
        case 3: run(std::integral_constant<int, 3>{}); break;
        case 4: run(std::integral_constant<int, 4>{}); break;
        case 5: run(std::integral_constant<int, 5>{}); break;
        case 6: run(std::integral_constant<int, 6>{}); break;
        case 7: run(std::integral_constant<int, 7>{}); break;
        default: run(std::integral_constant<int, 8>{}); break;
      }
    }
  HIPCHK(hipGetLastError());
  return BSG_OK;
}
int bsg_copy(bsg_context* ctx, const double* x, double* y, int64_t n) {
  if (!ctx || !x || !y || n < 0) return fail(BSG_ERR_ARG, "bsg_copy: bad args");
  if (n == 0) return BSG_OK;
  hipLaunchKernelGGL(k_copy, dim3(grid_for(n)), dim3(256), 0, ctx->stream, x, y, n);
  HIPCHK(hipGetLastError());
  return BSG_OK;
}
int bsg_copy_segments(bsg_context* ctx, const bsg_copy_seg_t* segs, int32_t n_segs) {
  if (!ctx || n_segs < 0 || (n_segs > 0 && !segs)) return fail(BSG_ERR_ARG, "bsg_copy_segments: bad args");
  std::vector<bsg_copy_seg_t> chunks;
  for (int32_t i = 0; i < n_segs; ++i) {
    const bsg_copy_seg_t& s = segs[i];
    if (s.n < 0 || (s.n > 0 && (!s.src || !s.dst))) return fail(BSG_ERR_ARG, "bsg_copy_segments: bad segment");
    for (int64_t x = 0; x < s.n; x += COPY_CHUNK) chunks.push_back({s.src + x, s.dst + x, std::min(COPY_CHUNK, s.n - x)});
  }
  if (chunks.empty()) return BSG_OK;
  if (chunks.size() > (size_t)0x7fffffff) return fail(BSG_ERR_ARG, "bsg_copy_segments: too many chunks");
  HIPCHK(hipSetDevice(ctx->device));
  // every call returns with its copies done, so no queued work reads the list
  if (ctx->copy_cap < chunks.size()) {
    if (ctx->copy_list) HIPCHK(hipFree(ctx->copy_list));
    ctx->copy_list = nullptr;
    ctx->copy_cap = 0;
    const size_t cap = chunks.size() + chunks.size() / 2;
    HIPCHK(hipMalloc((void**)&ctx->copy_list, sizeof(bsg_copy_seg_t) * cap));
    ctx->copy_cap = cap;
  }
  HIPCHK(hipMemcpyAsync(ctx->copy_list, chunks.data(), sizeof(bsg_copy_seg_t) * chunks.size(), hipMemcpyHostToDevice,
                        ctx->stream));
  hipLaunchKernelGGL(k_copy_chunks, dim3((unsigned)chunks.size()), dim3(256), 0, ctx->stream, ctx->copy_list);
  HIPCHK(hipGetLastError());
  HIPCHK(hipStreamSynchronize(ctx->stream));
  return BSG_OK;
}
int bsg_build_apply(bsg_context* ctx, const bsg_build_group_t* groups, int32_t ngroups, const bsg_build_src_t* srcs,
                    int32_t nsrcs) {
  if (!ctx || ngroups < 0 || nsrcs < 0 || (ngroups > 0 && (!groups || !srcs))) return fail(BSG_ERR_ARG, "bsg_build_apply: bad args");
  if (ngroups == 0) return BSG_OK;
  std::vector<int64_t> estart(ngroups);
  int64_t nelem = 0;
  for (int32_t g = 0; g < ngroups; ++g) {
    const bsg_build_group_t& gr = groups[g];
    if (!gr.dst || gr.rows <= 0 || gr.cols <= 0 || gr.ld < gr.cols || gr.first < 0 || gr.count < 0 ||
        gr.first + gr.count > nsrcs)
      return fail(BSG_ERR_ARG, "bsg_build_apply: bad group");
    estart[g] = nelem;
    nelem += (int64_t)gr.rows * gr.cols;
  }
  for (int32_t j = 0; j < nsrcs; ++j)
    if (!srcs[j].src || srcs[j].ld <= 0) return fail(BSG_ERR_ARG, "bsg_build_apply: bad source");
  if (nelem == 0) return BSG_OK;
  if ((nelem + 255) / 256 > 0x7fffffffLL) return fail(BSG_ERR_ARG, "bsg_build_apply: too many elements");
  HIPCHK(hipSetDevice(ctx->device));
  bsg_build_group_t* dg = nullptr;
  bsg_build_src_t* ds = nullptr;
  int64_t* de = nullptr;
  HIPCHK(hipMalloc(&dg, sizeof(bsg_build_group_t) * ngroups));
  HIPCHK(hipMalloc(&ds, sizeof(bsg_build_src_t) * std::max(1, nsrcs)));
  HIPCHK(hipMalloc(&de, sizeof(int64_t) * ngroups));
  HIPCHK(hipMemcpyAsync(dg, groups, sizeof(bsg_build_group_t) * ngroups, hipMemcpyHostToDevice, ctx->stream));
  if (nsrcs > 0) HIPCHK(hipMemcpyAsync(ds, srcs, sizeof(bsg_build_src_t) * nsrcs, hipMemcpyHostToDevice, ctx->stream));
  HIPCHK(hipMemcpyAsync(de, estart.data(), sizeof(int64_t) * ngroups, hipMemcpyHostToDevice, ctx->stream));
  hipLaunchKernelGGL(k_build, dim3((unsigned)((nelem + 255) / 256)), dim3(256), 0, ctx->stream, dg, de, ngroups, ds,
                     nelem);
  HIPCHK(hipGetLastError());
  HIPCHK(hipStreamSynchronize(ctx->stream));
  HIPCHK(hipFree(dg));
  HIPCHK(hipFree(ds));
  HIPCHK(hipFree(de));
  return BSG_OK;
}
int bsg_scal(bsg_context* ctx, double a, double* x, int64_t n) {
  if (!ctx || !x || n < 0) return fail(BSG_ERR_ARG, "bsg_scal: bad args");
  if (n == 0) return BSG_OK;
  hipLaunchKernelGGL(k_scal, dim3(grid_for(n)), dim3(256), 0, ctx->stream, a, x, n);
  HIPCHK(hipGetLastError());
  return BSG_OK;
}
int bsg_precondition(bsg_context* ctx, double* x, const double* d, double e, double shift, int64_t n) {
  if (!ctx || !x || !d || n < 0) return fail(BSG_ERR_ARG, "bsg_precondition: bad args");
  if (n == 0) return BSG_OK;
  hipLaunchKernelGGL(k_precond, dim3(grid_for(n)), dim3(256), 0, ctx->stream, x, d, e, shift, n);
  HIPCHK(hipGetLastError());
  return BSG_OK;
}
int bsg_olsen_precondition(bsg_context* ctx, double* r, const double* c, const double* d, double e, double shift,
                           double* work, int64_t n) {
  if (!ctx || !r || !c || !d || !work || n < 0) return fail(BSG_ERR_ARG, "bsg_olsen_precondition: bad args");
  if (n == 0) return BSG_OK;
  const int nb = reduce_grid(n);
  hipLaunchKernelGGL(k_olsen_dots, dim3(nb), dim3(RB), 0, ctx->stream, r, c, d, e, shift, work, n, ctx->red);
  hipLaunchKernelGGL(k_olsen_step, dim3(nb), dim3(RB), 0, ctx->stream, r, c, d, e, shift, n, ctx->red, nb);
  HIPCHK(hipGetLastError());
  return BSG_OK;
}

}  // extern "C"

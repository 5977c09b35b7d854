// FP64 product tiles of the large blocks (included by sigma.hip inside its
// anonymous namespace).
//
// A pair of a large V block runs as two products: W = alpha op(A) C into a
// scratch buffer, then V += W B'.  Both are the same kernel: a workgroup of
// four wavefronts owns a 64 x 64 tile of one product's result (32 x 32 per
// wavefront) and walks a list of segments, out += alpha L_s R_s, as one
// contraction: one segment for W, the unit's run of pairs for V.  A pair with
// an identity partner is a single segment of the second kind.
//
// Bound by the FP64 matrix pipes (busy 59% of the time by the counters; 8% of
// the MFMAs are padding, waves wait 40% of their time for chunks and barriers,
// LDS is busy 21%, HBM traffic 1.8 TB/s).  24 orbitals, C1, M = 500 (169
// GFLOP): 6.19 ms per application on 16-row tiles that kept W on chip and read
// C and B' per 16 rows, 3.94 so (43 TFLOP/s); 30 orbitals, M = 800, four roots:
// 114.4 -> 69.7 ms.  At the time of 4.59 ms, 128 x 64 tiles
// of four wavefronts took 5.57, five waves per SIMD instead of four 5.81.
typedef double dbl2 __attribute__((ext_vector_type(2)));
__device__ inline dbl2 bload128(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
  return __builtin_bit_cast(dbl2, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0));
}

// where a segment's operand lives
enum : int32_t { SP_ARENA = 0, SP_W = 1, SP_C = 2 };
// out (m x n) += alpha L (m x K) R (K x n).  L is stored m x K row-major
// (SEG_LT clear) or K x m (set), R K x n (SEG_RT clear) or n x K (set).
// Shifts: L's and R's space.
enum : int32_t { SEG_LT = 1, SEG_RT = 2, SEG_LSPACE = 2, SEG_RSPACE = 4 };
struct GemmSeg {
  int64_t l, r;
  double alpha;
  int32_t k, flags;
};
// V += alpha C added to a unit's result (identity A and B')
struct GemmAdd {
  int64_t c;
  double alpha;
};
// segments [first, first + count) into the m x n result at out: W (GU_W),
// the partial tile buffer (GU_PART) or added into v (GU_V)
enum : int32_t { GU_W = 0, GU_PART = 1, GU_V = 2 };
struct GemmUnit {
  int64_t out;
  double alpha;  // of the whole result
  int32_t first, count, add_first, add_count, m, n, kind, pad;
};

constexpr int GKC = 16;      // K depth of a staged chunk
// LDS layout of a chunk: 16 doubles per row, the eight 16-byte pairs of K of
// row r in the order (pair ^ (r & 7)): 8 lanes reading the same pair of 8 rows,
// or writing the 8 pairs of one row, meet every bank once without padding.
__device__ __forceinline__ int chunk_at(int row, int k) { return row * GKC + ((((k >> 1) ^ row) & 7) << 1) + (k & 1); }

// One operand of a segment as a thread stages it: 64 rows of the operand x 16
// K per chunk, two 16-byte loads.  K contiguous: lanes 0-7 take the 16 K of
// one row.  Rows contiguous: a half wave takes 16 rows x 4 K, so both the
// loads (128-byte runs) and the transposing LDS writes are conflict-free.
// The thread's offsets hold for the whole segment; a chunk's K goes in the
// uniform offset.  Rows past the operand's end read zero or another row's
// values, which only reach results that are not stored; K past its depth
// reads zero, or (K contiguous) the next row, cut in store().
// The LDS places of a thread's values are the same in every segment.
template <int ROWS, int NT>
struct Staged {
  static constexpr int N = ROWS * GKC / (2 * NT);  // 16-byte loads per thread and chunk
  static constexpr int RSTEP = NT / 8;             // K contiguous: rows between a thread's loads
  static constexpr int KSTEP = 2 * NT / ROWS;      // rows contiguous: K between a thread's loads
  static_assert(N * RSTEP == ROWS && N * KSTEP == GKC && RSTEP % 8 == 0, "whole chunk");
  const double* base;       // the operand
  uint32_t bytes;           // its size
  uint32_t soff, step;      // byte offset of the next chunk, bytes per chunk
  uint32_t off[N];          // the thread's loads in a chunk
  bool kc;                  // K contiguous
  int kp, at_k, at_r[2 * N];  // K of the thread's pair, LDS places (doubles) of the two layouts
  __device__ __forceinline__ void init(int tid) {
    kp = 2 * (tid & 7);
    at_k = chunk_at(tid >> 3, kp);  // RSTEP is a multiple of 8: the same order in every row
#pragma unroll
    for (int u = 0; u < N; ++u)
#pragma unroll
      for (int e = 0; e < 2; ++e) at_r[2 * u + e] = chunk_at(row_r(tid) + e, k_r(tid) + KSTEP * u);
  }
  // rows contiguous: bits of tid are row pair (0-2), K (3-4), then the other row pairs, then K
  static __device__ __forceinline__ int row_r(int tid) { return 2 * ((tid & 7) | (((tid >> 5) % (ROWS / 16)) << 3)); }
  static __device__ __forceinline__ int k_r(int tid) { return ((tid >> 3) & 3) | ((tid >> 5) / (ROWS / 16) << 2); }
  __device__ __forceinline__ void open(const double* p, bool k_contig, int rows, int depth, int row0, int tid) {
    base = p;
    bytes = (uint32_t)(rows * depth) * 8u;
    kc = k_contig;
    soff = 0;
    if (kc) {
      const uint32_t o = (uint32_t)((row0 + (tid >> 3)) * depth + kp) * 8u;
#pragma unroll
      for (int u = 0; u < N; ++u) off[u] = o + (uint32_t)(depth * RSTEP * u) * 8u;
      step = GKC * 8u;
    } else {
      const uint32_t o = (uint32_t)(k_r(tid) * rows + row0 + row_r(tid)) * 8u;
#pragma unroll
      for (int u = 0; u < N; ++u) off[u] = o + (uint32_t)(rows * KSTEP * u) * 8u;
      step = (uint32_t)rows * (GKC * 8u);
    }
  }
  __device__ __forceinline__ void load(dbl2 (&x)[N]) {
    const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc((void*)base, (short)0, (int)bytes, 0x00020000);
#pragma unroll
    for (int u = 0; u < N; ++u) x[u] = bload128(r, off[u], soff);
    soff += step;
  }
  // depth: K values of the chunk
  __device__ __forceinline__ void store(double* buf, int depth, dbl2 (&x)[N]) const {
    if (kc) {
      if (depth < GKC) {
        asm volatile("" ::: "memory");  // a branch: the cut is rare and would cost every chunk
#pragma unroll
        for (int u = 0; u < N; ++u) {
          if (kp + 1 >= depth) x[u][1] = 0.0;
          if (kp >= depth) x[u][0] = 0.0;
        }
      }
#pragma unroll
      for (int u = 0; u < N; ++u) *(dbl2*)(buf + at_k + u * RSTEP * GKC) = x[u];
    } else {
#pragma unroll
      for (int u = 0; u < N; ++u) {
        buf[at_r[2 * u]] = x[u][0];
        buf[at_r[2 * u + 1]] = x[u][1];
      }
    }
  }
};

// Tile shapes: WR x WC wavefronts of NR x NC 16 x 16 blocks each
template <int WR_, int WC_, int NR_, int NC_, int EU_>
struct GemmTile {
  static constexpr int EU = EU_;
  static constexpr int WR = WR_, WC = WC_, NR = NR_, NC = NC_, NT = 64 * WR * WC, TM = 16 * WR * NR, TN = 16 * WC * NC;
};

// The contraction of a wavefront's part of the tile over the unit's segments.
// FULL: all its 16 x 16 blocks exist; the waves of a workgroup may run
// different instances (the same barriers in each).
template <class T, bool FULL>
__device__ __forceinline__ void gemm_loop(const GemmUnit& un, const GemmSeg* __restrict__ segs,
                                          const double* __restrict__ arena, const double* __restrict__ c,
                                          const double* __restrict__ wbuf, double (*lds)[(T::TM + T::TN) * GKC], int row0,
                                          int col0, int wr, int wc, int nr, int nc, int tid, dbl4 (&acc)[T::NR][T::NC]) {
  const int lane = tid & 63, li = lane & 15, lk = lane >> 4;
  const int lo = ((lk ^ li) & 7) << 1, hi = (((4 + lk) ^ li) & 7) << 1;  // places of K pairs lk and 4 + lk in row li
  // The loader runs one chunk ahead of the products, across segments: the
  // next chunk's loads are in flight during the current chunk's MFMAs and go
  // to the other LDS buffer after them, one barrier per chunk.
  int s = 0, left = 0, cur = 0;  // left: K of the open segment to load; cur: K values in the current buffer (0: none yet)
  Staged<T::TM, T::NT> sl;
  Staged<T::TN, T::NT> sr;
  sl.init(tid);
  sr.init(tid);
  GemmSeg nx{};  // the next segment's descriptor, requested one segment ahead
  double alpha = 1.0;
  if (un.count > 0) nx = segs[un.first];
  // one chunk: the loads of the next, the products of buffer B, the next into
  // the other buffer; false after the last
  auto chunk = [&](auto B) __attribute__((always_inline)) -> bool {
    constexpr int b = decltype(B)::value;
    const bool more = left > 0 || s < un.count;
    dbl2 xl[sl.N], xr[sr.N];
    if (more) {
      if (left <= 0) {
        const GemmSeg sg = nx;
        ++s;
        if (s < un.count) nx = segs[un.first + s];
        const int ls = (sg.flags >> SEG_LSPACE) & 3, rsp = (sg.flags >> SEG_RSPACE) & 3;
        const double *lp = arena, *rp = rsp == SP_C ? c : arena;
        if (ls == SP_W) lp = wbuf;
        if (ls == SP_C) lp = c;
        sl.open(lp + sg.l, !(sg.flags & SEG_LT), un.m, sg.k, row0, tid);
        sr.open(rp + sg.r, (sg.flags & SEG_RT) != 0, un.n, sg.k, col0, tid);
        alpha = sg.alpha;
        left = sg.k;
      }
      sl.load(xl);
      sr.load(xr);
    }
    if (cur > 0 && (FULL || (nr > 0 && nc > 0))) {
      // lane (li, lk) holds K = 8 h + 2 lk + {0, 1} of both operands
      const double* L = lds[b] + (wr + li) * GKC;
      const double* R = lds[b] + (T::TM + wc + li) * GKC;
      constexpr int NH = FULL ? 2 : 1;  // halves of the chunk whose fragments are read ahead
      dbl2 a[NH][T::NR], bb[NH][T::NC];
      auto frags = [&](int h) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < T::NR; ++i) a[h % NH][i] = *(const dbl2*)(L + i * 16 * GKC + (h ? hi : lo));
#pragma unroll
        for (int j = 0; j < T::NC; ++j) bb[h % NH][j] = *(const dbl2*)(R + j * 16 * GKC + (h ? hi : lo));
      };
      frags(0);
      if (FULL) frags(1);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        if (8 * h >= cur) break;
        if (!FULL && h) frags(h);
#pragma unroll
        for (int e = 0; e < 2; ++e)
#pragma unroll
          for (int i = 0; i < T::NR; ++i)
            if (FULL || i < nr)
#pragma unroll
              for (int j = 0; j < T::NC; ++j)
                if (FULL || j < nc)
                  acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[h % NH][i][e], bb[h % NH][j][e], acc[i][j], 0, 0, 0);
      }
    }
    if (!more) return false;
    cur = min(left, GKC);
    left -= GKC;
    if (alpha != 1.0) {
      asm volatile("" ::: "memory");  // a branch, as in store()
#pragma unroll
      for (int u = 0; u < sl.N; ++u) xl[u] *= alpha;
    }
    sl.store(lds[b ^ 1], cur, xl);
    sr.store(lds[b ^ 1] + T::TM * GKC, cur, xr);
    __syncthreads();
    return true;
  };
  while (chunk(std::integral_constant<int, 0>{}) && chunk(std::integral_constant<int, 1>{})) {
  }
}

template <class T>
__global__ __launch_bounds__(T::NT) __attribute__((amdgpu_waves_per_eu(T::EU))) void k_gemm(
    const GemmUnit* __restrict__ units, const GemmSeg* __restrict__ segs, const GemmAdd* __restrict__ adds,
    const TileRef* __restrict__ tiles, int ntiles, const double* __restrict__ arena, const double* __restrict__ c,
    double* __restrict__ v, double* __restrict__ wbuf, double* __restrict__ part, RootSet rs) {
  __shared__ __attribute__((aligned(16))) double lds[2][(T::TM + T::TN) * GKC];  // L, then R
  int tile;
  const int root = root_of(blockIdx.x, rs.n, tile);
  if (tile >= ntiles) return;
  const TileRef tr = tiles[tile];
  if (tr.item < 0) return;  // padding of the XCD-interleaved order
  const GemmUnit un = units[tr.item];
  c += root * rs.wstride;
  v += root * rs.wstride;
  part += root * rs.pstride;
  wbuf += root * rs.tstride;
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, lk = lane >> 4;
  // a wavefront's part of the tile turns with the workgroup, so that the
  // short edge tiles of different workgroups load all four SIMDs alike
  const int w = (__builtin_amdgcn_readfirstlane(tid >> 6) + blockIdx.x / 8) % (T::WR * T::WC);
  const int row0 = tr.tm * T::TM, col0 = tr.tn * T::TN, wr = w / T::WC * 16 * T::NR, wc = w % T::WC * 16 * T::NC;
  const int nr = min(T::NR, max(0, (un.m - row0 - wr + 15) >> 4)), nc = min(T::NC, max(0, (un.n - col0 - wc + 15) >> 4));
  dbl4 acc[T::NR][T::NC];
#pragma unroll
  for (int i = 0; i < T::NR; ++i)
#pragma unroll
    for (int j = 0; j < T::NC; ++j) acc[i][j] = dbl4{0.0, 0.0, 0.0, 0.0};
  for (int q = 0; q < un.add_count; ++q) {
    const GemmAdd ad = adds[un.add_first + q];
    const __amdgpu_buffer_rsrc_t rc = block_rsrc(c + ad.c, (int64_t)un.m * un.n);
#pragma unroll
    for (int i = 0; i < T::NR; ++i)
#pragma unroll
      for (int j = 0; j < T::NC; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int row = row0 + wr + 16 * i + lk + 4 * e, col = col0 + wc + 16 * j + li;
          acc[i][j][e] += ad.alpha * bload(rc, row < un.m && col < un.n ? (uint32_t)(row * un.n + col) * 8u : OOB);
        }
  }
  if (nr == T::NR && nc == T::NC)
    gemm_loop<T, true>(un, segs, arena, c, wbuf, lds, row0, col0, wr, wc, nr, nc, tid, acc);
  else
    gemm_loop<T, false>(un, segs, arena, c, wbuf, lds, row0, col0, wr, wc, nr, nc, tid, acc);
  double* out = (un.kind == GU_V ? v : un.kind == GU_W ? wbuf : part) + un.out;
#pragma unroll
  for (int i = 0; i < T::NR; ++i)
#pragma unroll
    for (int j = 0; j < T::NC; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int row = row0 + wr + 16 * i + lk + 4 * e, col = col0 + wc + 16 * j + li;
        if (row < un.m && col < un.n) {
          double* o = out + (size_t)row * un.n + col;
          const double x = un.alpha * acc[i][j][e];
          *o = un.kind == GU_V ? *o + x : x;
        }
      }
}

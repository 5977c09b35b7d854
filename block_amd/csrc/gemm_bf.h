// Split-precision product tiles of the large blocks (included by sigma.hip
// inside its anonymous namespace): the two products of gemm_f64.h on BF16
// slices.  Every operand has its K contiguous, padded to 8 and zero there:
// op(A) and B' slices (made once per arena), C^T slices (per application) and
// W slices (written by the first product).  K groups of 32 start at multiples
// of 32 and are summed in FP32 by the six slice products in mma6's order,
// added into FP64, as in the grouped kernel.
//   W^T = alpha C^T op(A)^T: a lane holds 4 consecutive W columns of a W row,
//   which are scaled, split and stored as 8 bytes per slice;
//   V += alpha W B'.
// A slice element is 6 bytes for 32 / 6 of the FP64 kernel's product rate, so the
// tile is as large as the registers of two waves per SIMD hold (128 x 128: 12
// TB/s at full rate, half of a 64 x 64's).  Bound by the chunks' way from L2:
// waves wait half of their time, with only two per SIMD to cover it (counters:
// matrix pipes busy 18%, LDS 20% and 7% in bank conflicts, HBM 1.9 TB/s).
// 24 orbitals, C1, M = 500: 4.90 ms per application on 16-row tiles that read
// every slice fragment for 16 rows, 2.70 so.

// spaces of a segment's operands
enum : int32_t { BS_OPER = 0, BS_W = 1, BS_C = 2 };

template <int WR_, int WC_, int NR_, int NC_, int EU_>
struct SplitTile {
  static constexpr int WR = WR_, WC = WC_, NR = NR_, NC = NC_, EU = EU_, NT = 64 * WR * WC, T = 16 * WR * NR;
  static_assert(16 * WC * NC == T && NT == 4 * T, "square tile, four threads per staged row");
};

template <class T>
__global__ __launch_bounds__(T::NT) __attribute__((amdgpu_waves_per_eu(T::EU))) void k_gemm_bf(
    const GemmUnit* __restrict__ units, const GemmSeg* __restrict__ segs, const GemmAdd* __restrict__ adds,
    const TileRef* __restrict__ tiles, int ntiles, const __bf16* __restrict__ slices,
    const __bf16* __restrict__ cslices, const double* __restrict__ c, double* __restrict__ v,
    __bf16* __restrict__ wbuf, double* __restrict__ part, RootSet rs) {
  // [buffer][L, R][slice][row][4 x 8 K], the 16-byte pieces of row r in the
  // order piece ^ (r >> 2): 8 lanes reading one piece of 8 rows meet every
  // bank once
  __shared__ __attribute__((aligned(16))) __bf16 lds[2][6 * T::T * 32];
  int tile;
  const int root = root_of(blockIdx.x, rs.n, tile);
  if (tile >= ntiles) return;
  const TileRef tr = tiles[tile];
  if (tr.item < 0) return;  // padding of the XCD-interleaved order
  const GemmUnit un = units[tr.item];
  c += root * rs.wstride;
  v += root * rs.wstride;
  part += root * rs.pstride;
  cslices += root * rs.cstride;
  wbuf += root * rs.tstride * 4;  // tstride counts doubles
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, lk = lane >> 4;
  const int w = (__builtin_amdgcn_readfirstlane(tid >> 6) + blockIdx.x / 8) % (T::WR * T::WC);
  const int row0 = tr.tm * T::T, col0 = tr.tn * T::T, wr = w / T::WC * 16 * T::NR, wc = w % T::WC * 16 * T::NC;
  const int nr = min(T::NR, max(0, (un.m - row0 - wr + 15) >> 4)), nc = min(T::NC, max(0, (un.n - col0 - wc + 15) >> 4));
  dbl4 acc[T::NR][T::NC];  // register e: row 16 i + 4 lk + e, column 16 j + li
#pragma unroll
  for (int i = 0; i < T::NR; ++i)
#pragma unroll
    for (int j = 0; j < T::NC; ++j) acc[i][j] = dbl4{0.0, 0.0, 0.0, 0.0};
  // alpha C: into V, or (first product, identity A) as W^T
  for (int q = 0; q < un.add_count; ++q) {
    const GemmAdd ad = adds[un.add_first + q];
    const int sr = un.kind == GU_W ? 1 : un.n, sc = un.kind == GU_W ? un.m : 1;  // C strides of the tile's rows, columns
    const __amdgpu_buffer_rsrc_t rc = block_rsrc(c + ad.c, (int64_t)un.m * un.n);
#pragma unroll
    for (int i = 0; i < T::NR; ++i)
#pragma unroll
      for (int j = 0; j < T::NC; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int row = row0 + wr + 16 * i + 4 * lk + e, col = col0 + wc + 16 * j + li;
          acc[i][j][e] += ad.alpha * bload(rc, row < un.m && col < un.n ? (uint32_t)(row * sr + col * sc) * 8u : OOB);
        }
  }
  // staging: a thread takes one 16-byte piece of one row of every slice
  const int srow = tid >> 2, sq = tid & 3, at = srow * 32 + ((sq ^ (srow >> 2)) & 3) * 8;
  const int piece = ((lk ^ (li >> 2)) & 3) * 8;  // this lane's piece in row li
  int s = 0, left = 0, cur = 0;  // left: K of the open segment to load; cur: whether a chunk is staged
  GemmSeg nx{};
  if (un.count > 0) nx = segs[un.first];
  const __bf16 *lp = slices, *rp = slices;
  uint32_t lbytes = 0, rbytes = 0, loff = 0, roff = 0, soff = 0;  // bytes of a slice, the thread's offsets, K offset
  double alpha = 1.0, nalpha = 1.0;
  auto chunk = [&](auto B) __attribute__((always_inline)) -> bool {
    constexpr int b = decltype(B)::value;
    const bool more = left > 0 || s < un.count;
    i32x4 x[6];
    if (more) {
      if (left <= 0) {
        const GemmSeg sg = nx;
        ++s;
        if (s < un.count) nx = segs[un.first + s];
        const int ls = (sg.flags >> SEG_LSPACE) & 3, rsp = (sg.flags >> SEG_RSPACE) & 3;
        lp = slices;
        if (ls == BS_W) lp = wbuf;
        if (ls == BS_C) lp = cslices;
        lp += sg.l;
        rp = (rsp == BS_C ? cslices : slices) + sg.r;
        lbytes = (uint32_t)(un.m * sg.k) * 2u;
        rbytes = (uint32_t)(un.n * sg.k) * 2u;
        loff = row0 + srow < un.m ? (uint32_t)((row0 + srow) * sg.k + 8 * sq) * 2u : OOB;
        roff = col0 + srow < un.n ? (uint32_t)((col0 + srow) * sg.k + 8 * sq) * 2u : OOB;
        nalpha = sg.alpha;
        soff = 0;
        left = sg.k;
      }
      const __amdgpu_buffer_rsrc_t rl = __builtin_amdgcn_make_buffer_rsrc((void*)lp, (short)0, (int)(3 * lbytes), 0x00020000);
      const __amdgpu_buffer_rsrc_t rr = __builtin_amdgcn_make_buffer_rsrc((void*)rp, (short)0, (int)(3 * rbytes), 0x00020000);
      const bool in = 8 * sq < left;  // K past the padded depth reads zero
      const uint32_t lo = in ? loff : OOB, ro = in ? roff : OOB;
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        x[q] = __builtin_amdgcn_raw_buffer_load_b128(rl, lo, soff + q * lbytes, 0);
        x[3 + q] = __builtin_amdgcn_raw_buffer_load_b128(rr, ro, soff + q * rbytes, 0);
      }
      soff += 64;
    }
    if (cur && nr > 0 && nc > 0) {
      const __bf16* L = lds[b] + (wr + li) * 32 + piece;
      const __bf16* R = lds[b] + (3 * T::T + wc + li) * 32 + piece;
      Frag fl[T::NR], fr[T::NC];
#pragma unroll
      for (int i = 0; i < T::NR; ++i) {
        fl[i].h = *(const bf16x8*)(L + i * 512);
        fl[i].m = *(const bf16x8*)(L + T::T * 32 + i * 512);
        fl[i].l = *(const bf16x8*)(L + 2 * T::T * 32 + i * 512);
      }
#pragma unroll
      for (int j = 0; j < T::NC; ++j) {
        fr[j].h = *(const bf16x8*)(R + j * 512);
        fr[j].m = *(const bf16x8*)(R + T::T * 32 + j * 512);
        fr[j].l = *(const bf16x8*)(R + 2 * T::T * 32 + j * 512);
      }
      // mma6's products in its order, a row of blocks at a time (independent chains)
#pragma unroll
      for (int i = 0; i < T::NR; ++i) {
        if (i >= nr) break;
        f32x4 y[T::NC];
#pragma unroll
        for (int j = 0; j < T::NC; ++j)
          y[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fl[i].l, fr[j].h, f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
        for (int j = 0; j < T::NC; ++j) y[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fl[i].m, fr[j].m, y[j], 0, 0, 0);
#pragma unroll
        for (int j = 0; j < T::NC; ++j) y[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fl[i].h, fr[j].l, y[j], 0, 0, 0);
#pragma unroll
        for (int j = 0; j < T::NC; ++j) y[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fl[i].m, fr[j].h, y[j], 0, 0, 0);
#pragma unroll
        for (int j = 0; j < T::NC; ++j) y[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fl[i].h, fr[j].m, y[j], 0, 0, 0);
#pragma unroll
        for (int j = 0; j < T::NC; ++j) y[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fl[i].h, fr[j].h, y[j], 0, 0, 0);
#pragma unroll
        for (int j = 0; j < T::NC; ++j)
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[i][j][e] = __builtin_fma(alpha, (double)y[j][e], acc[i][j][e]);
      }
    }
    if (!more) return false;
    cur = 1;
    left -= 32;
    alpha = nalpha;
#pragma unroll
    for (int q = 0; q < 6; ++q) *(i32x4*)(lds[b ^ 1] + q * T::T * 32 + at) = x[q];
    __syncthreads();
    return true;
  };
  while (chunk(std::integral_constant<int, 0>{}) && chunk(std::integral_constant<int, 1>{})) {
  }
  if (un.kind == GU_W) {  // W slices, [W row][W columns padded to 8]
    const int pitch = (un.m + 7) & ~7;
    __bf16* out = wbuf + un.out;
    const int64_t slice = (int64_t)un.n * pitch;
#pragma unroll
    for (int i = 0; i < T::NR; ++i)
#pragma unroll
      for (int j = 0; j < T::NC; ++j) {
        const int wcol = row0 + wr + 16 * i + 4 * lk, wrow = col0 + wc + 16 * j + li;
        if (wcol >= pitch || wrow >= un.n) continue;
        typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
        bf16x4 h, m, l;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          __bf16 a, bb, cc;
          split_f32(un.alpha * acc[i][j][e], a, bb, cc);
          h[e] = a;
          m[e] = bb;
          l[e] = cc;
        }
        __bf16* o = out + (int64_t)wrow * pitch + wcol;
        *(bf16x4*)o = h;
        *(bf16x4*)(o + slice) = m;
        *(bf16x4*)(o + 2 * slice) = l;
      }
    return;
  }
  double* out = (un.kind == GU_V ? v : part) + un.out;
#pragma unroll
  for (int i = 0; i < T::NR; ++i)
#pragma unroll
    for (int j = 0; j < T::NC; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int row = row0 + wr + 16 * i + 4 * lk + e, col = col0 + wc + 16 * j + li;
        if (row < un.m && col < un.n) {
          double* o = out + (size_t)row * un.n + col;
          *o = un.kind == GU_V ? *o + acc[i][j][e] : acc[i][j][e];
        }
      }
}

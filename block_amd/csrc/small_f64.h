// FP64 kernel of the small blocks (included by sigma.hip inside its anonymous
// namespace).
//
// V blocks and contraction depths of at most 32: a pair is a few dozen MFMAs,
// so a pair's operand round trip to memory, not its arithmetic, sets the time.
// A wavefront walks the pairs of one work unit alone (no LDS, no barriers).
// The planner orders a block's pairs by C block; C^T stays in registers for a
// run of pairs on one C block, and the operands of the next D - 1 pairs are
// requested while a pair is multiplied, in D register sets used in turn.
// Loads need no masks and no branches: rows past the end of a block read zero
// (range check), columns past its width meet zeros of C^T or rows and columns
// of V that are not stored, and a transposed operand only changes strides.
//
// K order: step (o, e) of lane lk is 8 o + 2 lk + e in both products; W^T comes
// out of the first product with W columns 16 j + 8 (i >> 1) + 2 lk + (i & 1) in
// register i (the C^T rows are permuted for that), which is the second
// product's A operand.  Depths are padded to 8.
//
// Measured on 238,000 pairs of V blocks up to 24 wide (36 orbitals, D2h,
// M = 250, whole application): 452 us with four waves to a workgroup, C read
// for every pair and nothing requested ahead; 161 us now (1.1 TB/s of
// operands, MFMAs 60% busy in the 24-wide class).

// Loads of one pair: O 8-deep K groups, RB x NB 16-blocks of V
template <int RB, int NB, int O>
struct SmallOps {
  double a[RB][O][2];  // op(A)(16 r + li, 8 o + 2 lk + e)
  double b[O][2][NB];  // B'(8 o + 2 lk + e, 16 t + li)
  double alpha;
};

template <int RB, int NB, int O, int D>
__device__ __forceinline__ void small_run(const PanelPair* __restrict__ prs, int count, const double* __restrict__ arena,
                                          const double* __restrict__ cb, int m, int n, int k1, int k2, int li, int lk,
                                          dbl4 (&acc)[RB][NB]) {
  constexpr int NJ = (O + 1) / 2;
  double ct[NJ][O][2];  // C(8 o + 2 lk + e, W column of row li of group j)
  {
    const __amdgpu_buffer_rsrc_t r = block_rsrc(cb, (int64_t)k1 * k2);
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const int col = 16 * j + 8 * (li >> 3) + 2 * (li & 3) + ((li >> 2) & 1);
      const uint32_t off = col < k2 ? (uint32_t)(2 * lk * k2 + col) * 8u : OOB;
#pragma unroll
      for (int o = 0; o < O; ++o)
#pragma unroll
        for (int e = 0; e < 2; ++e) ct[j][o][e] = bload2(r, off, (uint32_t)((8 * o + e) * k2) * 8u);
    }
  }
  const uint32_t oa0 = (uint32_t)(li * k1 + 2 * lk) * 8u, oa1 = (uint32_t)(2 * lk * m + li) * 8u;
  const uint32_t ob0 = (uint32_t)(2 * lk * n + li) * 8u, ob1 = (uint32_t)(li * k2 + 2 * lk) * 8u;
  SmallOps<RB, NB, O> set[D];
  PanelPair nxt = prs[0];
  auto load = [&](SmallOps<RB, NB, O>& x, int q) __attribute__((always_inline)) {
    const PanelPair p = nxt;
    nxt = prs[min(q + 1, count - 1)];
    const bool in = q < count;  // past the run's end: empty ranges, nothing is read
    const bool ta = p.trans & 1, tb = p.trans & 2;
    const __amdgpu_buffer_rsrc_t ra = block_rsrc(arena + p.a, in ? m * k1 : 0);
    const __amdgpu_buffer_rsrc_t rb = block_rsrc(arena + p.b, in ? k2 * n : 0);
    x.alpha = p.alpha;
    const uint32_t oa = ta ? oa1 : oa0, ob = tb ? ob1 : ob0;
    const uint32_t ak = ta ? 8u * m : 8u, ar = ta ? 128u : 128u * k1;
    const uint32_t bk = tb ? 8u : 8u * n, bc = tb ? 128u * k2 : 128u;
#pragma unroll
    for (int o = 0; o < O; ++o)
#pragma unroll
      for (int e = 0; e < 2; ++e) {
#pragma unroll
        for (int r = 0; r < RB; ++r) x.a[r][o][e] = bload2(ra, oa, (8 * o + e) * ak + r * ar);
#pragma unroll
        for (int t = 0; t < NB; ++t) x.b[o][e][t] = bload2(rb, ob, (8 * o + e) * bk + t * bc);
      }
  };
  auto multiply = [&](const SmallOps<RB, NB, O>& x) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      dbl4 w[RB];
#pragma unroll
      for (int r = 0; r < RB; ++r) w[r] = dbl4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int o = 0; o < O; ++o)
#pragma unroll
        for (int e = 0; e < 2; ++e)
#pragma unroll
          for (int r = 0; r < RB; ++r)
            w[r] = __builtin_amdgcn_mfma_f64_16x16x4f64(ct[j][o][e], x.a[r][o][e], w[r], 0, 0, 0);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int o = 2 * j + (i >> 1);
        if (o < O) {
#pragma unroll
          for (int r = 0; r < RB; ++r) {
            const double wv = x.alpha * w[r][i];
#pragma unroll
            for (int t = 0; t < NB; ++t)
              acc[r][t] = __builtin_amdgcn_mfma_f64_16x16x4f64(wv, x.b[o][i & 1][t], acc[r][t], 0, 0, 0);
          }
        }
      }
    }
  };
#pragma unroll
  for (int d = 0; d < D - 1; ++d) load(set[d], d);
  for (int q = 0;; q += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      load(set[(d + D - 1) % D], q + d + D - 1);
      multiply(set[d]);
      if (q + d + 1 >= count) return;
    }
  }
}

// Pairs with an identity partner: V += alpha C, V += alpha op(A) C or
// V += alpha C B'
template <int RB, int NB>
__device__ __forceinline__ void small_identity(const PanelPair& pr, const double* __restrict__ arena,
                                               const double* __restrict__ cb, int m, int n, int li, int lk,
                                               dbl4 (&acc)[RB][NB]) {
  const __amdgpu_buffer_rsrc_t rc = block_rsrc(cb, (int64_t)pr.k1 * pr.k2);
  if (pr.a < 0 && pr.b < 0) {
#pragma unroll
    for (int r = 0; r < RB; ++r)
#pragma unroll
      for (int t = 0; t < NB; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int row = 16 * r + lk + 4 * i, col = 16 * t + li;
          acc[r][t][i] += pr.alpha * bload(rc, row < m && col < n ? (uint32_t)(row * pr.k2 + col) * 8u : OOB);
        }
    return;
  }
  // left (m x K, row and K strides) times right (K x n)
  const bool ia = pr.a < 0;
  const __amdgpu_buffer_rsrc_t ro = ia ? block_rsrc(arena + pr.b, (int64_t)pr.k2 * n) : block_rsrc(arena + pr.a, (int64_t)m * pr.k1);
  const int depth = ia ? pr.k2 : pr.k1;
  const int lr = ia ? pr.k2 : ((pr.trans & 1) ? 1 : pr.k1), ls = ia ? 1 : ((pr.trans & 1) ? m : 1);
  const int rs = ia ? ((pr.trans & 2) ? 1 : n) : pr.k2, rcol = ia && (pr.trans & 2) ? pr.k2 : 1;
  for (int k0 = 0; k0 < depth; k0 += 4) {
    const int k = k0 + lk;
    double x[NB];
#pragma unroll
    for (int t = 0; t < NB; ++t) {
      const int col = 16 * t + li;
      const uint32_t off = k < depth && col < n ? (uint32_t)(k * rs + col * rcol) * 8u : OOB;
      x[t] = ia ? bload(ro, off) : bload(rc, off);
    }
#pragma unroll
    for (int r = 0; r < RB; ++r) {
      const int row = 16 * r + li;
      const uint32_t off = k < depth && row < m ? (uint32_t)(row * lr + k * ls) * 8u : OOB;
      const double a = pr.alpha * (ia ? bload(rc, off) : bload(ro, off));
#pragma unroll
      for (int t = 0; t < NB; ++t) acc[r][t] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, x[t], acc[r][t], 0, 0, 0);
    }
  }
}

// One work unit: the runs of pairs on one C block, those with an identity
// partner first
template <int OM, int RB, int NB>
__device__ __forceinline__ void small_unit(const Seg& sg, const bsg_vblock_t& vb, const PanelPair* __restrict__ prs,
                                           const double* __restrict__ arena, const double* __restrict__ c,
                                           double* __restrict__ v, double* __restrict__ part, int li, int lk) {
  constexpr int D = OM == 2 ? 4 : 2;
  dbl4 acc[RB][NB];  // register i of lane (li, lk): V(16 r + lk + 4 i, 16 t + li)
#pragma unroll
  for (int r = 0; r < RB; ++r)
#pragma unroll
    for (int t = 0; t < NB; ++t) acc[r][t] = dbl4{0.0, 0.0, 0.0, 0.0};
  prs += sg.first;
  for (int q = 0; q < sg.count;) {
    const PanelPair p0 = prs[q];
    const double* cb = c + p0.c;
    if (p0.a < 0 || p0.b < 0) {
      small_identity<RB, NB>(p0, arena, cb, vb.m, vb.n, li, lk, acc);
      ++q;
      continue;
    }
    const int e = min(sg.count, q + p0.pad);  // pad: pairs of the block's list left in the run, this one included
    const int k = max(p0.k1, p0.k2);
    if (k <= 8)
      small_run<RB, NB, 1, D>(prs + q, e - q, arena, cb, vb.m, vb.n, p0.k1, p0.k2, li, lk, acc);
    else if (OM == 2 || k <= 16)
      small_run<RB, NB, 2, D>(prs + q, e - q, arena, cb, vb.m, vb.n, p0.k1, p0.k2, li, lk, acc);
    else
      small_run<RB, NB, OM, D>(prs + q, e - q, arena, cb, vb.m, vb.n, p0.k1, p0.k2, li, lk, acc);
    q = e;
  }
  const bool direct = sg.p_off < 0;
  double* out = direct ? v + vb.v_off : part + sg.p_off;
#pragma unroll
  for (int r = 0; r < RB; ++r)
#pragma unroll
    for (int t = 0; t < NB; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = 16 * r + lk + 4 * i, col = 16 * t + li;
        if (row < vb.m && col < vb.n) {
          double* o = out + row * vb.n + col;
          *o = direct ? *o + acc[r][t][i] : acc[r][t][i];
        }
      }
}

// OM: 8-wide groups of the largest dimension a unit holds (2: up to 16, 3: up
// to 24, 4: up to 32), so that the narrow pairs, which are over half of a
// point-group superblock's, get the registers of five waves per SIMD (the
// 24-wide ones: three) to cover their loads.  One wavefront per workgroup, so a finished unit makes
// room for the next at once.
template <int OM>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(OM == 2 ? 4 : (OM == 3 ? 3 : 2)))) void k_small(
    const bsg_vblock_t* __restrict__ vbs, const PanelPair* __restrict__ prs, const Seg* __restrict__ segs,
    const int32_t* __restrict__ units, int nunits, const double* __restrict__ arena, const double* __restrict__ c,
    double* __restrict__ v, double* __restrict__ part, RootSet rs) {
  int u;
  const int root = root_of(blockIdx.x, rs.n, u);
  if (u >= nunits) return;
  const Seg sg = segs[units[u]];
  const bsg_vblock_t vb = vbs[sg.vb];
  c += root * rs.wstride;
  v += root * rs.wstride;
  part += root * rs.pstride;
  const int li = threadIdx.x & 15, lk = threadIdx.x >> 4;
  if constexpr (OM == 2) {
    small_unit<OM, 1, 1>(sg, vb, prs, arena, c, v, part, li, lk);
  } else {
    if (vb.m <= 16 && vb.n <= 16)
      small_unit<OM, 1, 1>(sg, vb, prs, arena, c, v, part, li, lk);
    else if (vb.m <= 16)
      small_unit<OM, 1, 2>(sg, vb, prs, arena, c, v, part, li, lk);
    else if (vb.n <= 16)
      small_unit<OM, 2, 1>(sg, vb, prs, arena, c, v, part, li, lk);
    else
      small_unit<OM, 2, 2>(sg, vb, prs, arena, c, v, part, li, lk);
  }
}

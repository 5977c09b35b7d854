// FP64 panel kernel of the medium blocks (included by sigma.hip inside its
// anonymous namespace).
//
// Every pair of a V block that reads the same C block needs the same C
// operands, so the planner orders a block's pairs by C block and a workgroup
// keeps C in LDS (transposed, zero-padded to 16s) while it walks them.  A
// wavefront owns 16 rows of the V block (all its columns, up to 96): per pair
// it holds its rows of op(A) in registers, forms W^T = C^T op(A)^T 16 W columns
// at a time (C^T from LDS), and the result registers are at once the A operand
// of the product with B'.  What a wavefront streams per pair is op(A)'s rows
// and B'.  Each has one register set, requested as soon as the product that
// reads it is done and while the other product runs, which leaves room for
// three waves per SIMD up to 80.  The waves of a workgroup (the 16-row panels of one
// V block) meet only where the C block changes.
//
// K order: step (s, e) of lane lk is 8 s + 2 lk + e in both products, so that
// a 16-byte load takes two K of an operand whose K is contiguous (the C^T rows
// are permuted, so that W columns come out in that order).
//
// Bound by the MFMA chains of too few wavefronts (matrix pipes busy 50% by the
// counters; operands at 3.4 TB/s from HBM): C's 51 KB of LDS and 168
// registers allow ten to twelve per CU, blocks of 65 to 80 rows fill 7.5.  36
// orbitals, D2h, M = 1000 (330,000 pairs, blocks up to 79): 4.25 ms per
// application on the grouped and per-wave tiles, 2.3 with this kernel on two
// register sets of each operand and two waves per SIMD, 1.96 so.  Measured and
// not kept: five panels to a workgroup (2.68), a launch of its own for C up to
// 64 x 64 with the LDS for it (2.22 to 2.31 where one launch took 2.22).
struct PanelPair {
  int64_t a, c, b;       // offsets; a, b < 0: identity
  double alpha;
  int32_t k1, k2, trans, pad;  // trans: bit 0 op(A) stored k1 x m, bit 1 B' stored n x k2
};

constexpr int WAIT_VM0 = 0x0f70;  // s_waitcnt: no vector load under way
constexpr int PANEL_MAX = 96;  // rows, columns and contraction depths the kernel takes
// LDS place of C(k, col): 16-byte pairs of K, the eight pairs of 16 K in an
// order that lets the lanes of 8 successive columns meet every bank once
__device__ __forceinline__ int panel_at(int col, int k, int kp) {
  const int f = col & 7;
  return col * kp + (k & ~15) + ((((k >> 1) ^ f) & 7) << 1) + (k & 1);
}

// One run of pairs with the same C block, k1 <= 16 KB and n <= 16 NB (a whole
// wavefront: rows row0 .. row0 + 15 of the block).  stage() puts C into LDS
// (between barriers) once the first pair's loads are under way.
template <int KB, int NB, class F>
__device__ __forceinline__ void panel_run(const PanelPair* __restrict__ prs, int count,
                                          const double* __restrict__ arena, const double* cl, int kp, int m, int n,
                                          int k1, int k2, int row0, int li, int lk, dbl4 (&acc)[NB], F&& stage) {
  const int nk = (k1 + 7) >> 3, njb = (k2 + 15) >> 4;
  // byte offsets in a block, the same for every pair of the run: op(A)
  // (row row0 + li) and B' (column li of a 16-column group)
  const uint32_t oa0 = (uint32_t)((row0 + li) * k1 + 2 * lk) * 8u;   // m x k1, K contiguous
  const uint32_t oa1 = (uint32_t)(2 * lk * m + row0 + li) * 8u;      // k1 x m
  const uint32_t ob0 = (uint32_t)(2 * lk * n + li) * 8u;             // k2 x n
  const uint32_t ob1 = (uint32_t)(li * k2 + 2 * lk) * 8u;            // n x k2, K contiguous
  const double* cp[2];  // this lane's C^T row of a 16-column group (permuted), K pairs lk and 4 + lk
  {
    const int col = 8 * (li >> 3) + 2 * (li & 3) + ((li >> 2) & 1);
    cp[0] = cl + panel_at(col, 2 * lk, kp);
    cp[1] = cl + panel_at(col, 8 + 2 * lk, kp);
  }
  dbl2 a[2 * KB];
  dbl2 b[2][NB];
  auto load_a = [&](const PanelPair& p) __attribute__((always_inline)) {
    const __amdgpu_buffer_rsrc_t r = block_rsrc(arena + p.a, (int64_t)m * k1);
    const bool ta = p.trans & 1;
    const uint32_t oa = ta ? oa1 : oa0, ak = ta ? 8u * m : 8u;
#pragma unroll
    for (int s = 0; s < 2 * KB; ++s)
      if (s < nk) {
        a[s][0] = bload2(r, oa, (uint32_t)(8 * s) * ak);
        a[s][1] = bload2(r, oa, (uint32_t)(8 * s + 1) * ak);
      }
  };
  auto load_b = [&](const PanelPair& p, int jb) __attribute__((always_inline)) {
    const __amdgpu_buffer_rsrc_t r = block_rsrc(arena + p.b, (int64_t)n * k2);
    if (p.trans & 2) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int t = 0; t < NB; ++t) b[i][t] = bload128(r, ob1, (uint32_t)(16 * jb + 8 * i) * 8u + (uint32_t)(t * k2) * 128u);
    } else {
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int e = 0; e < 2; ++e)
#pragma unroll
          for (int t = 0; t < NB; ++t) b[i][t][e] = bload2(r, ob0, (uint32_t)((16 * jb + 8 * i + e) * n) * 8u + 128u * t);
    }
  };
  PanelPair cur = prs[0];
  PanelPair nxt = prs[count > 1 ? 1 : 0];
  load_a(cur);
  load_b(cur, 0);
  stage();
  // register i of lane (li, lk): W(row0 + li, 16 jb + 8 (i >> 1) + 2 lk + (i & 1))
  auto first = [&](int jb) __attribute__((always_inline)) {
    dbl4 w = dbl4{0.0, 0.0, 0.0, 0.0};
    const int o = jb * 16 * kp;
#pragma unroll
    for (int s = 0; s < 2 * KB; ++s)
      if (s < nk) {
        const dbl2 x = *(const dbl2*)(cp[s & 1] + o + (s >> 1) * 16);
        w = __builtin_amdgcn_mfma_f64_16x16x4f64(x[0], a[s][0], w, 0, 0, 0);
        w = __builtin_amdgcn_mfma_f64_16x16x4f64(x[1], a[s][1], w, 0, 0, 0);
      }
    return w;
  };
  auto second = [&](dbl4 w, double alpha, int i) __attribute__((always_inline)) {
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const double wv = alpha * w[2 * i + e];
#pragma unroll
      for (int t = 0; t < NB; ++t) acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(wv, b[i][t][e], acc[t], 0, 0, 0);
    }
  };
  const bool half = ((k2 - 1) & 15) < 8;  // the last 16 W columns' upper half is empty
  for (int q = 0; q < count; ++q) {
    const double alpha = cur.alpha;
    for (int jb = 0; jb + 1 < njb; ++jb) {
      const dbl4 w = first(jb);
      __builtin_amdgcn_s_waitcnt(WAIT_VM0);
      second(w, alpha, 0);
      second(w, alpha, 1);
      load_b(cur, jb + 1);
    }
    const dbl4 w = first(njb - 1);
    cur = nxt;
    if (q + 2 < count) nxt = prs[q + 2];
    // explicit waits for B', then for op(A): both were requested a product
    // earlier, and without them the compiler, which cannot count the loads of
    // a storage order it does not know, waits for the newest ones too
    __builtin_amdgcn_s_waitcnt(WAIT_VM0);
    if (q + 1 < count) load_a(cur);
    second(w, alpha, 0);
    if (!half) second(w, alpha, 1);
    __builtin_amdgcn_s_waitcnt(WAIT_VM0);
    if (q + 1 < count) load_b(cur, 0);
  }
}

// A pair with an identity partner (any sizes up to PANEL_MAX), C in LDS
template <int NB>
__device__ __forceinline__ void panel_identity(const PanelPair& pr, const double* __restrict__ arena, const double* cl,
                                               int kp, int m, int n, int row0, int li, int lk, dbl4 (&acc)[NB]) {
  if (pr.a < 0 && pr.b < 0) {  // V += alpha C
#pragma unroll
    for (int t = 0; t < NB; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = row0 + lk + 4 * i, col = 16 * t + li;
        if (row < m && col < n) acc[t][i] += pr.alpha * cl[panel_at(col, row, kp)];
      }
  } else if (pr.a < 0) {  // V += alpha C B': W(row0 + li, k) = alpha C(row0 + li, k)
    const __amdgpu_buffer_rsrc_t r = block_rsrc(arena + pr.b, (int64_t)n * pr.k2);
    const int ks = (pr.trans & 2) ? 1 : n, cs = (pr.trans & 2) ? pr.k2 : 1;
    for (int k0 = 0; k0 < pr.k2; k0 += 4) {
      const int k = k0 + lk;
      const double wv = k < pr.k2 && row0 + li < m ? pr.alpha * cl[panel_at(k, row0 + li, kp)] : 0.0;
#pragma unroll
      for (int t = 0; t < NB; ++t) {
        const int col = 16 * t + li;
        const double b = bload(r, k < pr.k2 && col < n ? (uint32_t)(k * ks + col * cs) * 8u : OOB);
        acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(wv, b, acc[t], 0, 0, 0);
      }
    }
  } else {  // V += alpha op(A) C
    const __amdgpu_buffer_rsrc_t r = block_rsrc(arena + pr.a, (int64_t)m * pr.k1);
    const int ks = (pr.trans & 1) ? m : 1, rs = (pr.trans & 1) ? 1 : pr.k1;
    for (int k0 = 0; k0 < pr.k1; k0 += 4) {
      const int k = k0 + lk;
      const double a = pr.alpha * bload(r, k < pr.k1 && row0 + li < m ? (uint32_t)((row0 + li) * rs + k * ks) * 8u : OOB);
#pragma unroll
      for (int t = 0; t < NB; ++t) {
        const int col = 16 * t + li;
        const double x = k < pr.k1 && col < n ? cl[panel_at(col, k, kp)] : 0.0;
        acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, x, acc[t], 0, 0, 0);
      }
    }
  }
}

// One work unit's rows: four wavefronts at most, one 16-row panel each
// (TileRef: item = segment, pad = panels of a workgroup, tm = which of them).
template <int KB, int NB>
__device__ __forceinline__ void panel_unit(const Seg& sg, const bsg_vblock_t& vb, const PanelPair* __restrict__ prs,
                                           const double* __restrict__ arena, const double* __restrict__ c,
                                           double* __restrict__ v, double* __restrict__ part, double* cl, int row0,
                                           int tid, int nthreads) {
  const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
  dbl4 acc[NB];  // register i of lane (li, lk): V(row0 + lk + 4 i, 16 t + li)
#pragma unroll
  for (int t = 0; t < NB; ++t) acc[t] = dbl4{0.0, 0.0, 0.0, 0.0};
  for (int q = 0; q < sg.count;) {
    const PanelPair p0 = prs[sg.first + q];
    const int k1 = p0.k1, k2 = p0.k2, kp = (k1 + 15) & ~15, np = (k2 + 15) & ~15;
    // the run of pairs on this C block: [q, f) with an identity partner, then [f, e)
    int f = q;
    while (f < sg.count) {
      const PanelPair& p = prs[sg.first + f];
      if (p.c != p0.c || p.k1 != k1 || p.k2 != k2 || (p.a >= 0 && p.b >= 0)) break;
      ++f;
    }
    int e = f;
    while (e < sg.count) {
      const PanelPair& p = prs[sg.first + e];
      if (p.c != p0.c || p.k1 != k1 || p.k2 != k2 || p.a < 0 || p.b < 0) break;
      ++e;
    }
    // C^T into LDS, zeros up to whole 16s: 8 lanes take 16 columns of a row, a
    // column group's loads of all rows before their stores
    auto stage = [&]() __attribute__((always_inline)) {
      __syncthreads();
      const __amdgpu_buffer_rsrc_t r = block_rsrc(c + p0.c, (int64_t)k1 * k2);
      const int col0 = 2 * (tid & 7), kstep = nthreads >> 3;
      for (int k = tid >> 3; k < kp; k += kstep) {
        dbl2 x[KB];
#pragma unroll
        for (int j = 0; j < KB; ++j) {
          const int col = 16 * j + col0;
          if (16 * j < np) x[j] = bload128(r, col < k2 ? (uint32_t)(k * k2 + col) * 8u : OOB, 0);
        }
#pragma unroll
        for (int j = 0; j < KB; ++j) {
          const int col = 16 * j + col0;
          if (16 * j < np) {
            cl[panel_at(col, k, kp)] = x[j][0];
            cl[panel_at(col + 1, k, kp)] = col + 1 < k2 ? x[j][1] : 0.0;
          }
        }
      }
      __syncthreads();
      for (; q < f; ++q)
        panel_identity<NB>(prs[sg.first + q], arena, cl, kp, vb.m, vb.n, row0, li, lk, acc);
    };
    if (f < e)
      panel_run<KB, NB>(prs + sg.first + f, e - f, arena, cl, kp, vb.m, vb.n, k1, k2, row0, li, lk, acc, stage);
    else
      stage();
    q = e;
  }
  const bool direct = sg.p_off < 0;
  double* out = direct ? v + vb.v_off : part + sg.p_off;
#pragma unroll
  for (int t = 0; t < NB; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = row0 + lk + 4 * i, col = 16 * t + li;
      if (row < vb.m && col < vb.n) {
        double* o = out + row * vb.n + col;
        *o = direct ? *o + acc[t][i] : acc[t][i];
      }
    }
}

// KB: 16-deep groups of k1 the registers hold, also the largest V column
// group count and C^T size: 3 (up to 48), 5 (up to 80) or 6 (up to 96, two
// waves per SIMD and two workgroups per CU: on blocks of 81 to 96 still faster
// than 64 x 64 product tiles, which pad them to 128: 24 orbitals, D2h, peak
// dimension 90 1.77 -> 1.44 ms, 100 2.70 -> 1.98; 112 would leave one
// workgroup per CU).
template <int KB>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(KB <= 5 ? 3 : 2))) void k_panel(
    const bsg_vblock_t* __restrict__ vbs, const PanelPair* __restrict__ prs, const Seg* __restrict__ segs,
    const TileRef* __restrict__ tiles, int ntiles, const double* __restrict__ arena, const double* __restrict__ c,
    double* __restrict__ v, double* __restrict__ part, RootSet rs) {
  __shared__ __attribute__((aligned(16))) double cl[256 * KB * KB];
  int tile;
  const int root = root_of(blockIdx.x, rs.n, tile);
  if (tile >= ntiles) return;
  const TileRef tr = tiles[tile];
  if (tr.item < 0) return;  // padding of the XCD-interleaved order
  const Seg sg = segs[tr.item];
  const bsg_vblock_t vb = vbs[sg.vb];
  c += root * rs.wstride;
  v += root * rs.wstride;
  part += root * rs.pstride;
  // a wavefront's panel turns with the workgroup, so that workgroups with
  // fewer than four panels load all SIMDs alike; a wave without one ends at
  // once and leaves its registers to another workgroup (barriers count the
  // waves that are left)
  const int w = (__builtin_amdgcn_readfirstlane(threadIdx.x >> 6) + blockIdx.x / 8) & 3;
  const int row0 = 16 * (tr.tm * tr.pad + w);
  const int np = min(tr.pad, (vb.m + 15) / 16 - tr.tm * tr.pad);  // panels of this workgroup
  if (w >= np) return;
  const int tid = 64 * w + (threadIdx.x & 63), nt = 64 * np;
  const int nb = (vb.n + 15) >> 4;
  if (nb <= 1)
    panel_unit<KB, 1>(sg, vb, prs, arena, c, v, part, cl, row0, tid, nt);
  else if (nb == 2)
    panel_unit<KB, 2>(sg, vb, prs, arena, c, v, part, cl, row0, tid, nt);
  else if (KB <= 3 || nb == 3)
    panel_unit<KB, 3>(sg, vb, prs, arena, c, v, part, cl, row0, tid, nt);
  else if constexpr (KB > 3) {
    if (nb == 4)
      panel_unit<KB, 4>(sg, vb, prs, arena, c, v, part, cl, row0, tid, nt);
    else if (KB <= 5 || nb == 5)
      panel_unit<KB, 5>(sg, vb, prs, arena, c, v, part, cl, row0, tid, nt);
    else if constexpr (KB > 5)
      panel_unit<KB, 6>(sg, vb, prs, arena, c, v, part, cl, row0, tid, nt);
  }
}

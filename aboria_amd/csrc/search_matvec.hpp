// The sparse operator evaluated on the fly, for work items of up to 64
// queries of one home cell (k_search_group serves the other queries).
// Included by search.hip inside its namespace.
//
// Bound by vector instructions: about 14 for a radius test of 64 lanes and 50
// to 70 for a round of kernel values.  A lane evaluates the kernel for its
// own hits only, so a block of candidates takes as many rounds as the lane
// with the most hits has.  The visited buckets are therefore read as one flat
// list, cut into 64 / kMix pieces, and a block takes kMix candidates of every
// piece: with blocks taken bucket by bucket a lane had either many hits in a
// block or none, and the rounds were four times the mean number of hits.  The
// profile is chosen outside the loop over hits, the number of right-hand
// sides is a template argument and a block serves one work item, which keeps
// the grid's and the kernel's parameters out of the loops (the compiler had
// moved 180 scalar registers into vector lanes and read 16 of them back in
// every round).  The tests and the rounds are compiled with and without
// periodic images (the rounds also for buckets visited more than once): chosen
// at run time, the choice was a branch in every test and round, which kept their
// dependent chains from overlapping.  An item of a crowded cell, alone on its
// SIMD, then took twice as long as one candidate block after another had.
// 4M-particle mixture, Wendland, eight right-hand sides: 38.2 -> 25.1 ms, now
// 21.5; one: 25.7 -> 20.8, 17.4 ms.  1,000,000 points at 60 a cell, Gaussian, one
// right-hand side: 3.40 -> 2.04, 1.69 ms.

constexpr int kMix = 4;

template <int V> struct Profile { static constexpr int value = V; };

// Right-hand sides of the pooled candidates in LDS, NR per candidate, as
// pieces of 16 bytes.  The pieces of a row are permuted by the row number, so
// that lanes reading one piece of different rows spread over all the banks
// (plain rows of 64 or 32 bytes put them in a quarter or half of them).
template <typename T, int NR> struct PoolRhs {
  static constexpr int kPer = 16 / int(sizeof(T)) < NR ? 16 / int(sizeof(T)) : NR;
  static constexpr int kPieces = NR / kPer;
  struct __align__(sizeof(T) * kPer) Piece { T v[kPer]; };
  static __device__ __forceinline__ Piece *piece(void *xs, int t, int c) {
    const int turn = kPieces == 4 ? (t >> 2) & 3 : (kPieces == 2 ? (t >> 3) & 1 : 0);
    return static_cast<Piece *>(xs) + t * kPieces + (c ^ turn);
  }
  static __device__ __forceinline__ void load(void *xs, int t, T (&x)[NR]) {
#pragma unroll
    for (int c = 0; c < kPieces; ++c) {
      const Piece p = *piece(xs, t, c);
#pragma unroll
      for (int e = 0; e < kPer; ++e) x[c * kPer + e] = p.v[e];
    }
  }
  static __device__ __forceinline__ void store(void *xs, int t, const T (&x)[NR]) {
#pragma unroll
    for (int c = 0; c < kPieces; ++c) {
      Piece p;
#pragma unroll
      for (int e = 0; e < kPer; ++e) p.v[e] = x[c * kPer + e];
      *piece(xs, t, c) = p;
    }
  }
};

// LDS of k_matvec: stencil, segments, pooled candidates, right-hand sides
inline size_t matvec_lds_bytes(int nslots, int nr, bool fp32) {
  const size_t slots = size_t(nslots) * (sizeof(Slot) + 4 + kGroup + 8);
  return ((slots + 15) & ~size_t(15)) + size_t(kGroup) * sizeof(StageRec) +
         size_t(kGroup) * nr * (fp32 ? 4 : 8);
}

// FP32: the FP32-compensated form.  nrhs <= NR right-hand sides.
template <int D, bool FP32, int NR>
__global__ __launch_bounds__(kGroup) __attribute__((amdgpu_waves_per_eu(3))) void k_matvec(
    SearchArgs a, GridParams g) {
  using T = typename std::conditional<FP32, float, double>::type;
  using Pool = PoolRhs<T, NR>;
  extern __shared__ __align__(16) unsigned char lds[];
  if (blockIdx.x >= *a.nwork) return;  // (the grid is an upper bound)
  const int S = a.nslots, lane = threadIdx.x;
  Slot *slots = reinterpret_cast<Slot *>(lds);
  int32_t *sorder = reinterpret_cast<int32_t *>(slots + S);
  uint8_t *mult = reinterpret_cast<uint8_t *>(sorder + S);  // [S][64]
  int32_t *seg_end = reinterpret_cast<int32_t *>(mult + size_t(S) * kGroup);
  int32_t *seg_slot = seg_end + S;
  StageRec *st = reinterpret_cast<StageRec *>(
      lds + ((size_t(S) * (sizeof(Slot) + 4 + kGroup + 8) + 15) & ~size_t(15)));
  void *xs = st + kGroup;

  const WorkItem it = a.work[blockIdx.x];
  const int qk = it.start + (lane < it.count ? lane : 0);
  double q[D];
  bool finite = true;
#pragma unroll
  for (int d = 0; d < D; ++d) {
    q[d] = a.qpos[int64_t(qk) * D + d];
    finite = finite && isfinite(q[d]);
  }
  const bool has_row = lane < it.count, active = has_row && finite;
  double qlo[D], qhi[D];
#pragma unroll
  for (int d = 0; d < D; ++d) {
    qlo[d] = uniform_f64(wave_min_f64(active ? q[d] : INFINITY));
    qhi[d] = uniform_f64(wave_max_f64(active ? q[d] : -INFINITY));
  }
  const int64_t row = a.qperm ? int64_t(a.qperm[qk]) : int64_t(qk);
  stencil_setup<D, false>(a, g, it, q, active, slots, sorder, mult);

  // visited buckets as segments of the flat candidate list
  int nseg = 0, total = 0;
  bool multi = false, images = false;  // buckets visited more than once, other images
  constexpr int kHomeImg = D == 1 ? 1 : (D == 2 ? 5 : 21);
  for (int s = 0; s < S; ++s) {
    const int m = mult[s * kGroup + lane];
    multi = multi || __ballot(m > 1) != 0;
    if (__ballot(m != 0) == 0 && lane == 0) slots[s].len = 0;  // no lane visits it
  }
  __syncthreads();
  for (int k0 = 0; k0 < S; k0 += kGroup) {
    int s = 0, len = 0;
    if (k0 + lane < S) {
      s = sorder[k0 + lane];
      len = slots[s].len;
    }
    const bool use = len > 0;
    const uint64_t um = __ballot(use);
    const int incl = abh::wave_incl_scan(len);
    if (use) {
      const int idx = nseg + __popcll(um & abh::lanemask_lt());
      seg_end[idx] = total + incl;
      seg_slot[idx] = s;
    }
    images = images || __ballot(use && slots[s].img != kHomeImg) != 0;
    nseg += __popcll(um);
    total += __shfl(incl, kGroup - 1, 64);
  }
  __syncthreads();
  total = abh::uniform_i32(total);
  constexpr int kPieces = kGroup / kMix;
  const int chunk = ((total + kPieces - 1) / kPieces + kMix - 1) / kMix * kMix;
  int f = (lane / kMix) * chunk + lane % kMix;  // this lane's next candidate
  int seg = 0, beg = 0, end = 0, info = 0;      // its segment, found when f >= end

  double acc64[NR];
  float acc32[NR], cmp32[NR];
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    acc64[r] = has_row && r < a.nrhs ? a.y[int64_t(r) * a.ldy + row] : 0.0;
    acc32[r] = 0.0f;
    cmp32[r] = 0.0f;
  }
  double wrow = 1.0;
  if (a.k.row_s || a.k.col_s) {
    wrow = a.k.w0;
    if (a.k.row_s && active) wrow = wrow + a.k.wr * a.k.row_s[row];
  }
  int np = 0;       // pooled candidates
  uint64_t hm = 0;  // this lane's hits among them, the latest candidate at bit 0
  double L[D];
#pragma unroll
  for (int d = 0; d < D; ++d) L[d] = g.L[d];
  // centre seen by a candidate of image digits img
  auto centre = [&](int img, int d) {
    return images ? image_of((img >> (2 * d)) & 3, q[d], L[d]) : q[d];
  };
  // kernel values of the hits, added in pool order, once per visit; a pool's
  // terms are summed before they join the row's sum, since rows of a crowded
  // cell have a thousand terms: against sums in extended precision 20,000 rows
  // of 500 to 2,500 terms are 2.7e-16 off, one running sum per row 1.4e-15.  A
  // plain 64-bit evaluation, which is such a running sum, therefore differs by
  // its own rounding (4M-particle mixture 1.7e-15, as from a row sum with full
  // compensation, which takes 15% longer).
  auto eval = [&](auto profile, auto plain) {
    double part[NR];
#pragma unroll
    for (int r = 0; r < NR; ++r) part[r] = 0.0;
    while (hm != 0) {
      const int p = 63 - __builtin_clzll(hm);
      hm ^= 1ull << p;
      const int t = np - 1 - p;
      double e1[3];
      int j1;
      load_stage(st[t], e1, j1);
      T x[NR];
      Pool::load(xs, t, x);
      const int pinfo = decltype(plain)::value ? 0 : st[t].pad;
      double acc = 0.0;
#pragma unroll
      for (int d = 0; d < D; ++d) {
        const double dx = e1[d] - (decltype(plain)::value ? q[d] : centre(pinfo >> 16, d));
        acc = acc + dx * dx;
      }
      double w = wrow;
      if (a.k.col_s) w = w + a.k.wc * a.k.col_s[j1];
      const int m = !decltype(plain)::value && multi
                        ? int(mult[(pinfo & 0xffff) * kGroup + lane]) : 1;
      if constexpr (FP32) {
        const float fv = abh::phi32t<decltype(profile)::value>(a.k, float(acc)) * float(w);
        for (int rep = 0; rep < m; ++rep)
#pragma unroll
          for (int r = 0; r < NR; ++r) kb_add(acc32[r], cmp32[r], fv * x[r]);
      } else {
        const double fv = abh::phi64t<decltype(profile)::value>(a.k, acc) * w;
        for (int rep = 0; rep < m; ++rep)
#pragma unroll
          for (int r = 0; r < NR; ++r) part[r] = fma(fv, x[r], part[r]);
      }
    }
    if constexpr (!FP32)
#pragma unroll
      for (int r = 0; r < NR; ++r) acc64[r] += part[r];
  };
  for (int b = 0; b <= chunk; b += kMix, f += kMix) {
    const bool last = b == chunk;  // only what is left in the pool
    bool keep = !last && f < total;
    double x[D];
#pragma unroll
    for (int d = 0; d < D; ++d) x[d] = 0.0;
    int jc = 0;
    if (keep) {
      if (f >= end) {
        while (f >= seg_end[seg]) ++seg;
        const Slot sl = slots[seg_slot[seg]];
        end = seg_end[seg];
        beg = sl.beg - (end - sl.len);
        info = seg_slot[seg] | (sl.img << 16);
      }
      jc = beg + f;
#pragma unroll
      for (int d = 0; d < D; ++d) x[d] = a.pos[int64_t(jc) * D + d];
    }
    // culled against the box of the item's centres, as in the list passes
    double dd = 0.0;
#pragma unroll
    for (int d = 0; d < D; ++d) {
      const int dg = (info >> (16 + 2 * d)) & 3;
      const double lo = images ? image_of(dg, qlo[d], L[d]) : qlo[d];
      const double hi = images ? image_of(dg, qhi[d], L[d]) : qhi[d];
      double e = 0.0;
      if (x[d] < lo) e = lo - x[d];
      else if (x[d] > hi) e = x[d] - hi;
      dd = dd + e * e;
    }
    keep = keep && dd <= a.r2;
    const uint64_t km = __ballot(keep);
    if (km == 0 && !last) continue;
    const int nk = __popcll(km);
    if (np + nk > kGroup || last) {
      auto evals = [&](auto plain) {
        switch (a.k.type) {
          case ABH_KERNEL_CONSTANT: eval(Profile<ABH_KERNEL_CONSTANT>{}, plain); break;
          case ABH_KERNEL_GAUSSIAN: eval(Profile<ABH_KERNEL_GAUSSIAN>{}, plain); break;
          case ABH_KERNEL_WENDLAND_C2: eval(Profile<ABH_KERNEL_WENDLAND_C2>{}, plain); break;
          case ABH_KERNEL_MULTIQUADRIC: eval(Profile<ABH_KERNEL_MULTIQUADRIC>{}, plain); break;
          case ABH_KERNEL_SMOOTH_INV_R: eval(Profile<ABH_KERNEL_SMOOTH_INV_R>{}, plain); break;
        }
      };
      if (images || multi) evals(std::false_type{});
      else evals(std::true_type{});
      if (last) break;
      np = 0;
      __syncthreads();  // the next block overwrites the pool
    }
    if (keep) {
      const int sl = np + __popcll(km & abh::lanemask_lt());
      st[sl] = StageRec{x[0], D > 1 ? x[D > 1 ? 1 : 0] : 0.0, D > 2 ? x[D > 2 ? 2 : 0] : 0.0, jc,
                        info};
      // (the FP32 form rounds its right-hand sides here, once)
      T xr[NR];
#pragma unroll
      for (int r = 0; r < NR; ++r)
        xr[r] = r < a.nrhs ? T(a.x[int64_t(r) * a.ldx + jc]) : T(0);
      Pool::store(xs, sl, xr);
    }
    __syncthreads();  // single-wave group: the pooled block is complete
    // radius tests of the new candidates; a lane that does not visit a
    // candidate's bucket has no hit there
    auto tests = [&](auto img) {
      auto test = [&](int t) {
        double e[3];
        int j;
        load_stage(st[t], e, j);
        const int pinfo = abh::uniform_i32(st[t].pad);
        const int mv = mult[(pinfo & 0xffff) * kGroup + lane];
        double acc = 0.0;
#pragma unroll
        for (int d = 0; d < D; ++d) {
          const double dx =
              e[d] - (decltype(img)::value ? image_of((pinfo >> (16 + 2 * d)) & 3, q[d], L[d])
                                           : q[d]);
          acc = acc + dx * dx;
        }
        return acc <= a.r2 && mv != 0;
      };
      int t = np;
      np += nk;
      for (; t + kStageUnroll <= np; t += kStageUnroll) {
        bool h[kStageUnroll];
#pragma unroll
        for (int u = 0; u < kStageUnroll; ++u) h[u] = test(t + u);
#pragma unroll
        for (int u = 0; u < kStageUnroll; ++u) hm = (hm << 1) + (h[u] ? 1ull : 0ull);
      }
      for (; t < np; ++t) hm = (hm << 1) + (test(t) ? 1ull : 0ull);
    };
    if (images) tests(std::true_type{});
    else tests(std::false_type{});
  }
  if (!has_row) return;
#pragma unroll
  for (int r = 0; r < NR; ++r)
    if (r < a.nrhs)
      a.y[int64_t(r) * a.ldy + row] =
          FP32 ? acc64[r] + (double(acc32[r]) + double(cmp32[r])) : acc64[r];
}

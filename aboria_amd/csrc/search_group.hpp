// Radius search and operator with eight lanes per query: the form for cells
// that hold few particles.  Included by search.hip inside its namespace.
//
// k_search gives a wavefront to the queries of one home cell and tests every
// candidate against all 64 lanes: with six queries in a cell 58 lanes idle,
// and the wave walks its stencil's buckets one after another (100,000 points,
// 6 per cell: 644 us to count; 2,003 points in 2D: 269 us).  Here a wave
// serves eight queries whatever their cells.  A query's eight lanes first
// evaluate its stencil buckets, eight at a time (visit multiplicity, offsets),
// and write the visited ones to LDS as segments of one flat candidate list in
// ascending bucket order; they then test that list eight candidates at a time,
// four loads in flight per lane.  Bound by the latency of those loads (small
// sets) and by the vector instructions of the tests (large ones).
// Count, before and now: 100,000 points in 3D, 6 per cell, 644 -> 69 us;
// 2,003 points in 2D, 269 -> 9 us.

constexpr int kGl = 8;                               // lanes per query
constexpr int kGlThreads = 256;
constexpr int kGlGroups = kGlThreads / kGl;          // queries per block
constexpr int kGlMaxSlots = 125;                     // stencils of up to 5^3 buckets
constexpr int kGlUnroll = 4;                         // candidate loads in flight per lane
constexpr int kGlHits = 32;                          // matvec: hits kept per query

// A hit waiting for its kernel value.
struct __align__(16) HitRec {
  double r2;
  int32_t j, m;
};

inline size_t group_lds_bytes(int nslots, bool matvec) {
  return ((size_t(nslots) * 12 * kGlGroups + 15) & ~size_t(15)) +
         (matvec ? sizeof(HitRec) * kGlHits * kGlGroups : 0);
}

// LDS written by lanes of this wave is visible to the others after it
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

__device__ __forceinline__ uint32_t group_ballot(bool p) {
  return uint32_t(__ballot(p) >> (threadIdx.x & 56)) & 0xffu;
}
template <class T> __device__ __forceinline__ T group_sum(T v) {
#pragma unroll
  for (int o = 1; o < kGl; o <<= 1) v += __shfl_xor(v, o, kGl);
  return v;
}

// quadrants Q (bit Q of the mask) whose bit d is set
__device__ __forceinline__ constexpr uint32_t up_mask(int d) {
  return d == 0 ? 0xaau : (d == 1 ? 0xccu : 0xf0u);
}

// One dimension of a stencil bucket b seen by the image coordinate q: the
// quadrants that contain b (in) or start at it (st), folded into the masks;
// the terms of the box distance of b and of the two quadrant starts.  The
// same FP64 expressions as quad_state / visit_count.
__device__ __forceinline__ void slot_dim(const GridParams &g, int d, double q, int b, uint32_t &in,
                                         uint32_t &st, double &term, double &gu, double &gd) {
  const int mu = int(floor((q + 0.5 * g.side[d] - g.lo[d]) * g.inv[d]));
  const int md = int(floor((q + (-0.5) * g.side[d] - g.lo[d]) * g.inv[d]));
  gu = box_term(g, d, mu, q);
  gd = box_term(g, d, md, q);
  term = box_term(g, d, b, q);
  const int su = mu < 0 ? 0 : mu;
  const int sd = md > g.end_bucket[d] ? g.end_bucket[d] : md;
  const bool uok = mu <= g.end_bucket[d], dok = md >= 0;
  const uint32_t up = up_mask(d), dn = ~up;
  in &= (uok && b >= su ? up : 0u) | (dok && b <= sd ? dn : 0u);
  st &= (uok && b == su ? up : 0u) | (dok && b == sd ? dn : 0u);
}

// Whether a query's visited buckets leave its stencil (escapes_stencil), one
// quadrant per lane, over the images that can reach the domain.
template <int D>
__device__ __forceinline__ bool group_escapes(const GridParams &g, const double *q, double r2,
                                              const int *home, const int *w, int l) {
  constexpr int NQ = 1 << D;
  const int Q = l & (NQ - 1);
  // images of one dimension that alone are within r of the domain
  uint32_t dig[3] = {2u, 2u, 2u};
  double od[3][3] = {};
#pragma unroll
  for (int d = 0; d < D; ++d) {
    dig[d] = 0;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      if (c != 1 && !g.periodic[d]) continue;
      const double qi = image_of(c, q[d], g.L[d]);
      const double mid = 0.5 * (g.lo[d] + g.hi[d]);
      double t = fabs(mid - qi) - 0.5 * g.L[d];
      t = t < 0.0 ? 0.0 : t;
      od[d][c] = t * t;
      if (!(od[d][c] > r2)) dig[d] |= 1u << c;
    }
  }
  bool esc = false;
#pragma unroll 1
  for (uint32_t m0 = dig[0]; m0; m0 &= m0 - 1) {
#pragma unroll 1
    for (uint32_t m1 = dig[1]; m1; m1 &= m1 - 1) {
#pragma unroll 1
      for (uint32_t m2 = dig[2]; m2; m2 &= m2 - 1) {
        const int c[3] = {__ffs(int(m0)) - 1, __ffs(int(m1)) - 1, __ffs(int(m2)) - 1};
        double acc = 0.0;
#pragma unroll
        for (int d = 0; d < D; ++d) acc = acc + pick3(c[d], od[d][0], od[d][1], od[d][2]);
        if (acc > r2) continue;  // the image point does not reach the domain
        double qi[D], gs[D];
        int s[D], ctr[D];
        bool ok = true;
        double start = 0.0;
#pragma unroll
        for (int d = 0; d < D; ++d) {
          qi[d] = image_of(c[d], q[d], g.L[d]);
          ctr[d] = home[d] + (c[d] - 1) * g.size[d];
          const bool up = (Q >> d) & 1;
          const int mm = up ? int(floor((qi[d] + 0.5 * g.side[d] - g.lo[d]) * g.inv[d]))
                            : int(floor((qi[d] + (-0.5) * g.side[d] - g.lo[d]) * g.inv[d]));
          start = start + box_term(g, d, mm, qi[d]);
          if (up) {
            s[d] = mm < 0 ? 0 : mm;
            if (mm > g.end_bucket[d]) ok = false;
          } else {
            s[d] = mm > g.end_bucket[d] ? g.end_bucket[d] : mm;
            if (mm < 0) ok = false;
          }
        }
        if (!ok || start > r2) continue;
#pragma unroll
        for (int d = 0; d < D; ++d) {
          gs[d] = box_term(g, d, s[d], qi[d]);
          if (s[d] < ctr[d] - w[d] || s[d] > ctr[d] + w[d]) esc = true;
        }
#pragma unroll
        for (int d = 0; d < D; ++d) {
          const bool up = (Q >> d) & 1;
          const int e = up ? ctr[d] + w[d] + 1 : ctr[d] - w[d] - 1;
          if (e < 0 || e > g.end_bucket[d]) continue;
          if (up ? e < s[d] : e > s[d]) continue;
          double dist = 0.0;
#pragma unroll
          for (int k = 0; k < D; ++k) dist = dist + (k == d ? box_term(g, k, e, qi[k]) : gs[k]);
          if (!(dist > r2)) esc = true;
        }
      }
    }
  }
  return esc;
}

// list / nlist: the queries (sorted order) to serve, or null for all nq
template <int D, int MODE>
__global__ __launch_bounds__(kGlThreads) void k_search_group(SearchArgs a, GridParams g,
                                                             const int32_t *__restrict__ list,
                                                             const uint32_t *__restrict__ nlist,
                                                             int64_t nq) {
  extern __shared__ __align__(16) unsigned char lds[];
  constexpr bool kMV = (MODE == kMatvec64 || MODE == kMatvec32);
  constexpr bool kList = (MODE == kFill || MODE == kAssemble || MODE == kFillPadded);
  const int S = a.nslots;
  const int l = threadIdx.x & (kGl - 1), grp = threadIdx.x / kGl;
  const int64_t gi = int64_t(blockIdx.x) * kGlGroups + grp;
  const int64_t count = nlist ? int64_t(*nlist) : nq;
  if (gi >= count) return;  // no block-wide barriers below
  const int64_t qk = list ? int64_t(list[gi]) : gi;
  int32_t *seg_end = reinterpret_cast<int32_t *>(lds) + grp * S;  // end in the flat list
  int32_t *seg_base = seg_end + kGlGroups * S;                    // container index - flat index
  int32_t *seg_info = seg_base + kGlGroups * S;                   // multiplicity | image << 8
  HitRec *hits = reinterpret_cast<HitRec *>(
                     lds + ((size_t(S) * 12 * kGlGroups + 15) & ~size_t(15))) + grp * kGlHits;

  double q[D];
  bool finite = true;
#pragma unroll
  for (int d = 0; d < D; ++d) {
    q[d] = a.qpos[qk * D + d];
    finite = finite && isfinite(q[d]);
  }
  const int64_t row = a.qperm ? int64_t(a.qperm[qk]) : qk;
  int home[3] = {0, 0, 0}, span[3] = {1, 1, 1}, rot[3] = {0, 0, 0};
#pragma unroll
  for (int d = 0; d < D; ++d) {
    home[d] = home_of<D>(g, q, d);
    span[d] = 2 * a.w[d] + 1;
    // the offset with the lowest bucket: virtual cells past a periodic face
    // come from the other end (a dimension has no bucket twice, see plan)
    const int v0 = home[d] - a.w[d];
    if (v0 < 0 && v0 + span[d] > 0) rot[d] = -v0;
    else if (v0 < g.size[d] && v0 + span[d] > g.size[d]) rot[d] = g.size[d] - v0;
  }
  constexpr int kHomeImg = D == 1 ? 1 : (D == 2 ? 5 : 21);  // digit 1 in every dimension

  // visited buckets, in ascending order, as segments of the candidate list
  int nseg = 0, total = 0;
  uint32_t seen = 0;  // multiplicities above 1 (bit 0), images other than home (bit 1)
  for (int s0 = 0; s0 < S; s0 += kGl) {
    const int s = s0 + l;
    int m = 0, beg = 0, len = 0, img = 0;
    if (s < S && finite) {
      int bv[3] = {0, 0, 0}, dg[3] = {1, 1, 1};
      bool ok = true;
      int rem = s;
#pragma unroll
      for (int d = D - 1; d >= 0; --d) {
        int o = rem % span[d] + rot[d];
        rem /= span[d];
        if (o >= span[d]) o -= span[d];
        const int v = home[d] - a.w[d] + o;
        const int n = g.size[d];
        int b = v, I = 0;
        if (v < 0) { b = v + n; I = 1; }
        else if (v >= n) { b = v - n; I = -1; }
        if (I != 0 && !g.periodic[d]) ok = false;
        if (b < 0 || b >= n) ok = false;  // would need an image beyond +-1
        bv[d] = b;
        dg[d] = I + 1;
        img |= (I + 1) << (2 * d);
      }
      if (ok) {
        uint32_t index = 0, mul = 1;
#pragma unroll
        for (int i = D - 1; i >= 0; --i) {
          if (i != D - 1) mul *= uint32_t(g.size[i + 1]);
          index += mul * uint32_t(bv[i]);
        }
        beg = int(a.bbeg[index]);
        len = int(a.bend[index]) - beg;
        uint32_t in = (1u << (1 << D)) - 1u, st = in;
        double dist = 0.0, outside = 0.0, gu[D], gd[D];
#pragma unroll
        for (int d = 0; d < D; ++d) {
          const double qi = image_of(dg[d], q[d], g.L[d]);
          double term;
          slot_dim(g, d, qi, bv[d], in, st, term, gu[d], gd[d]);
          dist = dist + term;
          const double mid = 0.5 * (g.lo[d] + g.hi[d]);
          double t = fabs(mid - qi) - 0.5 * g.L[d];
          t = t < 0.0 ? 0.0 : t;
          outside = outside + t * t;
        }
        if (!(outside > a.r2)) {
          const bool near = !(dist > a.r2);
          // usually one quadrant holds the bucket
          for (uint32_t f = near ? in : st; f; f &= f - 1) {
            const int Q = __ffs(int(f)) - 1;
            double acc = 0.0;
#pragma unroll
            for (int d = 0; d < D; ++d) acc = acc + ((Q >> d) & 1 ? gu[d] : gd[d]);
            m += acc > a.r2 ? 0 : 1;
          }
        }
      }
    }
    const bool use = m > 0 && len > 0;
    const uint32_t gb = group_ballot(use);
    int incl = use ? len : 0;
#pragma unroll
    for (int o = 1; o < kGl; o <<= 1) {
      const int t = __shfl_up(incl, o, kGl);
      if (l >= o) incl += t;
    }
    if (use) {
      const int idx = nseg + __popc(gb & ((1u << l) - 1u));
      seg_end[idx] = total + incl;
      seg_base[idx] = beg - (total + incl - len);
      seg_info[idx] = m | (img << 8);
      seen |= (m > 1 ? 1u : 0u) | (img != kHomeImg ? 2u : 0u);
      if (MODE == kCapacity) seg_base[idx] = len;
    }
    nseg += __popc(gb);
    total += __shfl(incl, kGl - 1, kGl);
  }
  if (MODE == kCount || MODE == kCapacity) {
    if (finite && group_escapes<D>(g, q, a.r2, home, a.w, l)) atomicOr(a.escape_flag, 1u);
  }
  wave_lds_sync();
  if (MODE == kCapacity) {
    // candidates of every visited bucket with multiplicity, rounded up to 16
    // entries as k_search rounds them
    int64_t cap = 0;
    for (int s = l; s < nseg; s += kGl) cap += int64_t(seg_info[s] & 255) * seg_base[s];
    cap = group_sum(cap);
    if (l == 0) a.counts[row] = (cap + 15) & ~int64_t(15);
    return;
  }
  const bool multi = __any(int(seen & 1u));
  const bool images = __any(int(seen & 2u));

  int64_t cnt = 0;
  const int64_t out = kList ? a.row_ptr[row] : 0;
  double wrow = 1.0;
  if ((kMV || MODE == kAssemble) && (a.k.row_s || a.k.col_s)) {
    wrow = a.k.w0;
    if (a.k.row_s && finite) wrow = wrow + a.k.wr * a.k.row_s[row];
  }
  // The sums, right-hand side l of this query in lane l (one right-hand side:
  // in every lane), in candidate order as k_search forms them.
  const bool one = a.nrhs == 1;
  const int rl = one ? 0 : (l < a.nrhs ? l : 0);
  double acc64 = 0.0;
  float acc32 = 0.0f, cmp32 = 0.0f;
  if (kMV) acc64 = a.y[int64_t(rl) * a.ldy + row];
  int nh = 0;
  // Kernel values of the hits kept so far, one hit per lane (a lane evaluates
  // hits only, not the candidates it missed; the loads of up to four rounds
  // are issued together), put back in LDS (with one right-hand side as the
  // finished term) and summed in order by every lane.
  auto flush = [&]() {
    if (nh == 0) return;
    wave_lds_sync();
    constexpr int kR = kGlHits / kGl;
    double r2[kR], x1[kR];
    int hj[kR];
#pragma unroll
    for (int u = 0; u < kR; ++u) {
      const HitRec h = hits[min(kGl * u + l, nh - 1)];
      r2[u] = h.r2;
      hj[u] = h.j;
      x1[u] = one ? a.x[h.j] : 1.0;
    }
#pragma unroll
    for (int u = 0; u < kR; ++u) {
      if (kGl * u >= nh) break;
      double w = wrow;
      if (a.k.col_s) w = w + a.k.wc * a.k.col_s[hj[u]];
      if (MODE == kMatvec64) {
        const double f = phi64(a.k, r2[u]) * w;
        r2[u] = one ? f * x1[u] : f;
      } else {
        const float f = phi32(a.k, float(r2[u])) * float(w);
        r2[u] = double(one ? f * float(x1[u]) : f);
      }
    }
    wave_lds_sync();
#pragma unroll
    for (int u = 0; u < kR; ++u)
      if (kGl * u + l < nh) hits[kGl * u + l].r2 = r2[u];
    wave_lds_sync();
    for (int e0 = 0; e0 < nh; e0 += kGl) {
      HitRec h[kGl];
      double x[kGl];
#pragma unroll
      for (int e = 0; e < kGl; ++e) h[e] = hits[min(e0 + e, nh - 1)];
      if (!one) {
#pragma unroll
        for (int e = 0; e < kGl; ++e) x[e] = a.x[int64_t(rl) * a.ldx + h[e].j];
      }
#pragma unroll
      for (int e = 0; e < kGl; ++e) {
        const int m = e0 + e < nh ? (multi ? h[e].m : 1) : 0;
        if (MODE == kMatvec64) {
          const double v = one ? h[e].r2 : h[e].r2 * x[e];
          if (multi) {
            for (int rep = 0; rep < m; ++rep) acc64 += v;
          } else {
            acc64 = m ? acc64 + v : acc64;
          }
        } else {
          const float v = one ? float(h[e].r2) : float(h[e].r2) * float(x[e]);
          for (int rep = 0; rep < m; ++rep) kb_add(acc32, cmp32, v);
        }
      }
    }
    wave_lds_sync();
    nh = 0;
  };

  int s = 0, send = 0, sbase = 0, sinfo = 0;
  if (total > 0) {
    send = seg_end[0];
    sbase = seg_base[0];
    sinfo = seg_info[0];
  }
  for (int t0 = 0; t0 < total; t0 += kGl * kGlUnroll) {
    double x[kGlUnroll][D];
    int j[kGlUnroll], info[kGlUnroll];
#pragma unroll
    for (int u = 0; u < kGlUnroll; ++u) {
      // past the end: the last candidate again (a valid address), no hit
      const int t = min(t0 + kGl * u + l, total - 1);
      while (t >= send) {
        ++s;
        send = seg_end[s];
        sbase = seg_base[s];
        sinfo = seg_info[s];
      }
      j[u] = sbase + t;
      info[u] = sinfo;
#pragma unroll
      for (int d = 0; d < D; ++d) x[u][d] = a.pos[int64_t(j[u]) * D + d];
    }
#pragma unroll
    for (int u = 0; u < kGlUnroll; ++u) {
      if (t0 + kGl * u >= total) break;
      double acc = 0.0;
#pragma unroll
      for (int d = 0; d < D; ++d) {
        const double qi = images ? image_of((info[u] >> (8 + 2 * d)) & 3, q[d], g.L[d]) : q[d];
        const double dx = x[u][d] - qi;
        acc = acc + dx * dx;
      }
      const bool hit = acc <= a.r2 && t0 + kGl * u + l < total;
      const int m = multi ? info[u] & 255 : 1;
      if (MODE == kCount) {
        cnt += hit ? m : 0;
      } else if (kList) {
        int before, all;
        if (multi) {
          int incl = hit ? m : 0;
#pragma unroll
          for (int o = 1; o < kGl; o <<= 1) {
            const int v = __shfl_up(incl, o, kGl);
            if (l >= o) incl += v;
          }
          before = incl - (hit ? m : 0);
          all = __shfl(incl, kGl - 1, kGl);
        } else {
          const uint32_t gb = group_ballot(hit);
          before = __popc(gb & ((1u << l) - 1u));
          all = __popc(gb);
        }
        if (hit) {
          const int64_t at = out + cnt + before;
          double f = 0.0;
          float f32 = 0.0f;
          if (MODE == kAssemble) {
            double w = wrow;
            if (a.k.col_s) w = w + a.k.wc * a.k.col_s[j[u]];
            f = phi64(a.k, acc) * w;
            f32 = phi32(a.k, float(acc)) * float(w);
          }
          for (int rep = 0; rep < m; ++rep) {
            a.col[at + rep] = j[u];
            if (MODE == kAssemble) {
              if (a.val) a.val[at + rep] = f;
              if (a.val32) a.val32[at + rep] = f32;
            }
          }
        }
        cnt += all;
      } else {
        const uint32_t gb = group_ballot(hit);
        if (hit) hits[nh + __popc(gb & ((1u << l) - 1u))] = HitRec{acc, j[u], m};
        nh += __popc(gb);
        if (nh > kGlHits - kGl) flush();
      }
    }
  }
  if (MODE == kCount) {
    cnt = group_sum(cnt);
    if (l == 0) a.counts[row] = cnt;
  }
  if (MODE == kFillPadded && l == 0) a.counts[row] = cnt;
  if (kMV) {
    flush();
    if (one ? l == 0 : l < a.nrhs)
      a.y[int64_t(rl) * a.ldy + row] =
          MODE == kMatvec64 ? acc64 : acc64 + (double(acc32) + double(cmp32));
  }
}

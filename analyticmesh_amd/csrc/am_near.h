// The polygon walk of one region on the few constraints near it, one wave64 per
// region.
//
// A region's polygon is small against the spread of its constraint planes
// (3.5 vertices among C = 1,024 planes on the 4x256 network), so nearly every
// plane is too far away to bound an edge or cut a vertex.  One pass over the
// constraints takes each plane's distance from the region's seed point p (the
// middle of an edge of the neighbour it was found from); the up to 64 nearest
// become one constraint per lane, and the walk runs on those alone.  Every
// excluded plane has p inside it by at least the radius r, so it holds at any
// vertex within 0.9 r of p by a margin above the rounding of its evaluation
// (near_covers): the walk takes a vertex only there.  A region it cannot settle
// (a seed, a vertex beyond that, a turn or sign that is not certain) goes on the
// list of the walks over all constraints, so the near walk never decides
// otherwise than they do.
//
// What bounds it: VALU issue and the planes' read (32 bytes per constraint).
// The walks over all constraints read every plane once per vertex, from LDS
// that leaves 4 to 6 regions per CU.  4x256 network, 1,022,340 regions, one
// MI355X: candidate scan 75.3 -> 9.3 ms, FP64 ray walk 21.4 -> 9.3 ms, FP32 ray
// walk 17.5 -> 10.2 ms; the trained 4x60 network (248,231 regions) 11.6 -> 3.5 ms.
// In small levels it is one region's serial chain: 21 us a level of 140 regions.
#pragma once
#include "am_device.h"
#include "am_kernels.h"
#include "am_walk.h"

namespace am {

#define AM_NEAR_MAX 64        // near constraints: one per lane
#define AM_NEAR_PL (4 * 66)   // their planes; before, the face plane's inputs [4][66] (a stride of 66: four
                              // components read together fall into different banks)

// Scratch of the near walk in dynamic LDS, ahead of the walk records.
template <typename T>
struct NearLds {
  T* stage;         // [4][66] the face plane's inputs
  T* pl;            // [64][4] the near constraints' planes, for broadcast reads (over stage); SET_LDS: [C][4] all
  uint16_t* key;    // [C] squared distance of p inside each constraint (0 where outside, +inf: never a
                    // bound), as the upper half of its FP32 bits, i.e. rounded down
  uint16_t* cand;   // [64] near constraints
  uint32_t* mask;   // [Wd]
  uint32_t* used;   // [C bits] (over key where that is not used)
  WalkRecs rec;
};
#define AM_ALL_MAX 256        // constraints up to which SET_LDS is taken
__host__ __device__ inline size_t near_lds_bytes(int C, int Wd, int vm, int tsize, bool jinv, bool all = false) {
  auto a16 = [](size_t x) { return (x + 15) & ~(size_t)15; };
  // (all: planes behind the face plane's inputs)
  return (size_t)AM_NEAR_PL * tsize + (all ? (size_t)C * 4 * tsize : 0) + a16((size_t)C * 2) +
         AM_NEAR_MAX * 2 + a16((size_t)Wd * 4) + walk_rec_bytes(vm, jinv);
}
template <typename T>
__device__ inline NearLds<T> carve_near(unsigned char* p, int C, int Wd, int vm, bool jinv, bool all = false) {
  auto a16 = [](size_t x) { return (x + 15) & ~(size_t)15; };
  NearLds<T> s;
  s.stage = reinterpret_cast<T*>(p);
  s.pl = s.stage;
  p += (size_t)AM_NEAR_PL * sizeof(T);
  if (all) {
    s.pl = reinterpret_cast<T*>(p);
    p += (size_t)C * 4 * sizeof(T);
  }
  s.key = reinterpret_cast<uint16_t*>(p);
  s.used = reinterpret_cast<uint32_t*>(p);
  p += a16((size_t)C * 2);
  s.cand = reinterpret_cast<uint16_t*>(p);
  p += AM_NEAR_MAX * 2;
  s.mask = reinterpret_cast<uint32_t*>(p);
  p += a16((size_t)Wd * 4);
  s.rec = carve_walk_recs(p, vm, jinv);
  return s;
}

template <int CTRL, int ROWS>
__device__ __forceinline__ float dpp_min_step(float x) {
  const int b = __float_as_int(x);
  return fminf(x, __int_as_float(__builtin_amdgcn_update_dpp(b, b, CTRL, ROWS, 0xf, false)));
}
// Minimum over the wave, in every lane (DPP moves, as wave_argmin).
__device__ __forceinline__ float wave_min(float x) {
  x = dpp_min_step<0x111, 0xf>(x);
  x = dpp_min_step<0x112, 0xf>(x);
  x = dpp_min_step<0x114, 0xf>(x);
  x = dpp_min_step<0x118, 0xf>(x);
  x = dpp_min_step<0x142, 0xa>(x);
  x = dpp_min_step<0x143, 0xc>(x);
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), 63));
}
__device__ __forceinline__ double lane_value(double x, int l) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(x), l),
                          __builtin_amdgcn_readlane(__double2loint(x), l));
}
__device__ __forceinline__ float lane_value(float x, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), l));
}

// The nearest crossing of a ray: each lane keeps its best quotient num / den
// (den > 0) in FP32 with a handle of its constraint, take() returns the wave's
// (-1: none).  A proposal only: the caller's tests at the vertex confirm it (a
// nearer plane would be violated there).
template <typename T>
struct Nearest {
  float t = __builtin_inff();
  int h = -1;
  __device__ __forceinline__ void add(T num, T den, bool on, int handle) {
    const float q = (float)num * __builtin_amdgcn_rcpf((float)den);
    if (on && q < t) { t = q; h = handle; }
  }
  __device__ __forceinline__ int take() const {
    const float m = wave_min(t);
    const unsigned long long b = __ballot(t == m && h >= 0);
    return b ? __builtin_amdgcn_readlane(h, __builtin_ctzll(b)) : -1;
  }
};

// Distances of p from all constraints and the nearest of them: cand[0, n), n
// <= 64, returned (0: not to be settled here).  r receives the radius: every
// finite plane that is not a candidate has p inside by more than r.  In
// squared distances T: the wave keeps each lane's nearest, takes the value that
// KT of the 64 are within (a search over the bits, one ballot each; with C /
// 64 constraints per lane about KT + KT^2 / 128 constraints are then within
// it), and compacts the constraints within it in index order.
// qmax: with per-plane estimates, the largest sigma_g / |a_g|.
// One wave's pass over distances, constraint by constraint.
template <typename T, bool SCAN>
struct NearScan {
  uint32_t best = 0x7f80u;              // upper halves of non-negative floats order as the values
  float qm = 0.f;
  bool bad = false, inf = false;
  // constraint g with (signed) plane q and estimate e
  __device__ __forceinline__ void add(const T* q, T e, const T* p, uint16_t* key, int g) {
    const float s = (float)plane_eval(q[0], q[1], q[2], q[3], p);
    const float nn = (float)plane_nn(q[0], q[1], q[2]);
    const float u = fmaxf(-(s * fabsf(s)) * __builtin_amdgcn_rcpf(nn), 0.f);
    const bool fine = nn > 1e-30f && nn < 1e30f && fabsf(s) < 1e15f;
    if (sizeof(T) == 4) qm = fmaxf(qm, (float)e * __builtin_amdgcn_rsqf(nn));
    // a plane without a normal holds or fails everywhere; others that are out
    // of range are left to the walks over all constraints
    const bool holds = sizeof(T) == 8 && q[0] == T(0) && q[1] == T(0) && q[2] == T(0) &&
                       (SCAN ? q[3] <= T(0) : q[3] < T(0));
    bad = bad || !(fine || holds);
    inf = inf || !fine;
    const uint32_t k = fine ? __float_as_uint(u) >> 16 : 0x7f80u;
    key[g] = (uint16_t)k;
    best = min(best, k);
  }
};

// Constraints j0, j0 + 64, ... (U of them) of part l.
template <typename T, bool SCAN, int U, typename Src>
__device__ __forceinline__ void near_batch(const Src& P, int l, int j0, int n, int g0, const T* p, uint16_t* key,
                                           NearScan<T, SCAN>& sc) {
  T q[U][4], e[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int j = min(j0 + 64 * u, n - 1);
    P.load(l, j, q[u]);
    e[u] = sizeof(T) == 4 ? T(P.err(g0 + j)) : T(0);
  }
#pragma unroll
  for (int u = 0; u < U; ++u)
    if (j0 + 64 * u < n) sc.add(q[u], e[u], p, key, g0 + j0 + 64 * u);
}

// sc, skip: the pass so far, and the part of the constraints it has done (-1: none).
template <typename T, bool SCAN, typename Src>
__device__ __forceinline__ int near_constraints(const Src& P, int C, const T* p, uint16_t* key, uint16_t* cand, T& r,
                                                T& qmax, NearScan<T, SCAN> sc, int skip) {
  const int lane = threadIdx.x;
  for (int l = 0; l < P.parts(); ++l) {
    if (l == skip) continue;
    const int n = P.size(l), g0 = P.first(l);
    // several constraints' loads in flight: up to four per lane, then their distances
    int j0 = lane;
    for (; j0 - lane + 128 < n; j0 += 256) near_batch<T, SCAN, 4>(P, l, j0, n, g0, p, key, sc);
    for (; j0 - lane < n; j0 += 128) near_batch<T, SCAN, 2>(P, l, j0, n, g0, p, key, sc);
  }
  if (__any(sc.bad)) return 0;
  __syncthreads();
  int nfin = C;
  if (__any(sc.inf))
    for (int g0 = 0; g0 < C; g0 += 64)
      nfin -= __popcll(__ballot(g0 + lane < C && key[g0 + lane] == 0x7f80u));
  const uint32_t best = sc.best;
  if (sizeof(T) == 4) qmax = T(-wave_min(-sc.qm));
  for (int KT = 34; KT >= 10; KT -= 12) {
    uint32_t lim = 0x7f7fu;                    // every finite one
    if (nfin > AM_NEAR_MAX) {
      uint32_t t = 0u;
#pragma unroll
      for (int b = 14; b >= 2; --b) {
        const uint32_t c = t | (1u << b);
        if (__popcll(__ballot(best < c)) < KT) t = c;
      }
      lim = min(t + 3u, 0x7f7fu);
    }
    int n = 0;
    for (int g0 = 0; g0 < C; g0 += 64) {
      const int g = g0 + lane;
      const bool keep = g < C && key[g] <= lim;
      const unsigned long long bal = __ballot(keep);
      const int pos = n + __builtin_amdgcn_mbcnt_hi((unsigned)(bal >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)bal, 0u));
      if (keep && pos < AM_NEAR_MAX) cand[pos] = (uint16_t)g;
      n += __popcll(bal);
    }
    __syncthreads();
    if (n <= AM_NEAR_MAX) {
      // 1e-5: the FP32 rounding of the squared distances
      r = n == nfin ? T(1e18) : T(__builtin_sqrtf(__uint_as_float((lim + 1u) << 16)) * (1.f - 1e-5f));
      return n;
    }
  }
  return 0;
}

// Whether every excluded constraint holds at v: |v - p| <= 0.9 r, and a tenth
// of r above the evaluation's error.  With D >= r the distance of p inside
// constraint g, its value at v is at most -|a| (D - |v - p|) <= -|a| D / 10.  The
// certified walks' bound for g is at most |a| (E (1 + |p|_1 + D) + F) (its largest
// coefficient is at most |a| (1 + |p|_1 + D); F: the share by |a| alone), below
// |a| D / 10 when E <= 0.01 and 20 (E (1 + |p|_1) + F) <= r.
template <typename T>
__device__ __forceinline__ bool near_covers(const T* v, const T* p, T r, T E, T F) {
  if (r >= T(1e18)) return E <= T(0.01) && v[0] == v[0] && v[1] == v[1] && v[2] == v[2];
  const T dx = v[0] - p[0], dy = v[1] - p[1], dz = v[2] - p[2];
  const T p1 = T(1) + absT(p[0]) + absT(p[1]) + absT(p[2]);
  const T u = sizeof(T) == 8 ? T(1e-13) : T(2e-5);   // the rounding of D
  return dx * dx + dy * dy + dz * dz <= T(0.81) * r * r && E <= T(0.01) && T(20) * (E * p1 + F) <= r && u * p1 <= r;
}

// The scan's order (distance_key).
template <typename T>
__device__ __forceinline__ T near_order_key(const T* x, const T* p) {
  const T s = plane_eval(x[0], x[1], x[2], x[3], p);
  const T nn = plane_nn(x[0], x[1], x[2]);
  T k = nn > T(0) ? s * absT(s) / nn : (s > T(0) ? T(__builtin_inf()) : T(-__builtin_inf()));
  if (k != k) k = -__builtin_inf();
  return k;
}
// Constraint g's plane into LDS for SET_LDS.
template <typename T>
__device__ __forceinline__ void near_stage(const NearLds<T>& S, int g, const T* x) {
  for (int q = 0; q < 4; ++q) S.pl[g * 4 + q] = x[q];
}

// SCAN: the candidate scan's decisions (walk_region<double, false>), bit for
// bit: the next edge plane is the first unused constraint in distance order
// whose vertex no constraint violates.  On the line of the current edge that is
// one of the two planes bounding the edge; the walk proposes it, tests its
// vertex against the constraints with the scan's own expressions, and requires
// that every unused constraint before it in the order is violated by one of the
// edge's two bounding planes -- so the scan would have passed it over too.
// Else: the checked ray walk's decisions (walk_ray), same proposals, vertices
// and bounds.
// SET_ALL: every constraint takes part and each pass reads all planes again, for
// a region whose polygon the near constraints do not cover: about one in a
// hundred on the geometric networks.
// SET_LDS: every constraint takes part, planes in LDS (up to AM_ALL_MAX
// constraints): no distances to sort out and nothing left over; on the trained
// network a third of the polygons (long thin faces) are not covered by 64 of its
// 240 constraints.
// Returns NEAR_DONE (settled, record written), NEAR_RETRY (the constraints at
// hand do not suffice), or the reason bits (AM_WHY_BIT) for which the checked ray
// walk would leave the region undecided.
#define NEAR_DONE 0
#define NEAR_RETRY (-1)
#define SET_NEAR 0
#define SET_ALL 1
#define SET_LDS 2
template <typename T, bool SCAN, int SET, typename Src>
__device__ __forceinline__ int near_walk(const NetDev& net, const RegionIO& io, const WalkParams& wp, int rid,
                                          int slot_region, const Src& P, const NearLds<T>& S, const T* eq, const T* p,
                                          int start, T eqe = T(0), NearScan<T, SCAN> sc = NearScan<T, SCAN>{},
                                          int skip = -1) {
  constexpr bool per_plane = sizeof(T) == 4;
  constexpr bool FULL = SET != SET_NEAR;
  const int lane = threadIdx.x;
  const int C = net.C, vm = net.vm;
  T r = T(1e18), qmax = T(0);
  // near: this lane's constraint; a constraint's handle is its lane (FULL: its index)
  int g = -1;
  T a[4] = {T(0), T(0), T(0), T(0)};
  T sig = T(0), key = T(0);
  bool have = false;
  int sl = start;
  auto order_key = [&](const T* x) { return near_order_key<T>(x, p); };
  if (!FULL) {
    const int n = near_constraints<T, SCAN>(P, C, p, S.key, S.cand, r, qmax, sc, skip);
    if (n < 3) return NEAR_RETRY;
    have = lane < n;
    g = have ? (int)S.cand[lane] : -1;
    if (have) {
      P.get(g, a);
      if (per_plane) sig = P.err(g);
      if (SCAN) key = order_key(a);
    }
    if constexpr (sizeof(T) == 8) {
      reinterpret_cast<double2*>(S.pl)[2 * lane] = double2{a[0], a[1]};
      reinterpret_cast<double2*>(S.pl)[2 * lane + 1] = double2{a[2], a[3]};
    } else {
      reinterpret_cast<float4*>(S.pl)[lane] = float4{a[0], a[1], a[2], a[3]};
    }
    const unsigned long long sb = __ballot(g == start && have);
    if (!sb) return NEAR_RETRY;
    sl = __builtin_ctzll(sb);
  } else {
    for (int w = lane; w < (C + 31) >> 5; w += 64) S.used[w] = 0u;
    if (SET == SET_LDS)
      for (int l = 0; l < P.parts(); ++l) {
        if (l == skip) continue;   // staged by the caller
        for (int j = lane; j < P.size(l); j += 64) {
          T x[4];
          P.load(l, j, x);
          near_stage<T>(S, P.first(l) + j, x);
        }
      }
  }
  __syncthreads();
  unsigned long long used = 0ull;      // near: lanes of the polygon's planes (FULL: S.used)
  auto is_used = [&](int h) { return FULL ? (bool)((S.used[h >> 5] >> (h & 31)) & 1u) : (bool)((used >> h) & 1ull); };
  auto use = [&](int h) {
    if (!FULL) used |= 1ull << h;
    else if (lane == 0) S.used[h >> 5] |= 1u << (h & 31);
  };
  auto plane = [&](int h, T* o) {
    if (SET == SET_ALL) P.get(h, o);
    else
      for (int q = 0; q < 4; ++q) o[q] = S.pl[h * 4 + q];
  };
  auto index_of = [&](int h) { return FULL ? h : __builtin_amdgcn_readlane(g, h); };
  auto err_of = [&](int h) { return !per_plane ? T(0) : FULL ? T(P.err(h)) : lane_value(sig, h); };
  // f(plane, handle, index, sigma) for each of this lane's constraints
  auto each = [&](auto&& f) {
    if (!FULL) {
      if (have) f(a, lane, g, sig);
    } else if (SET == SET_LDS) {
      for (int h = lane; h < C; h += 64) {
        T x[4];
        plane(h, x);
        f(x, h, h, T(0));
      }
    } else {
      for (int l = 0; l < P.parts(); ++l) {
        const int n = P.size(l), g0 = P.first(l);
#pragma unroll 1
        for (int j = lane; j < n; j += 64) {
          T x[4];
          P.load(l, j, x);
          f(x, g0 + j, g0 + j, per_plane ? T(P.err(g0 + j)) : T(0));
        }
      }
    }
  };

  // the start plane's edge: nearest planes both ways along its line
  int cl = sl, ql, rl;   // the plane walked along, the plane come from, the next plane
  T pc[4], pq[4];        // planes of cl and ql
  T d[3];                // along cl, towards rl
  plane(sl, pc);
  {
    const T(&ps)[4] = pc;
    for (int q = 0; q < 3; ++q) d[q] = ps[(q + 1) % 3] * eq[(q + 2) % 3] - ps[(q + 2) % 3] * eq[(q + 1) % 3];
    const T pd[4] = {d[0], d[1], d[2], -(d[0] * p[0] + d[1] * p[1] + d[2] * p[2])};
    T x0[3];
    solve3(ps, eq, pd, x0);
    Nearest<T> hi, lo;
    each([&](const T* x, int h, int, T) {
      const T al = fmaT(x[0], d[0], fmaT(x[1], d[1], x[2] * d[2]));
      const T num = -plane_eval(x[0], x[1], x[2], x[3], x0);
      hi.add(num, al, h != sl && al > T(0), h);
      lo.add(num, -al, h != sl && al < T(0), h);
    });
    rl = hi.take();
    ql = lo.take();
    if (rl < 0 || ql < 0) return FULL ? (int)AM_WHY_BIT(AM_WHY_START) : NEAR_RETRY;
    if (SCAN) {
      T kh, kl;
      if (FULL) {
        T x[4];
        plane(rl, x);
        kh = order_key(x);
        plane(ql, x);
        kl = order_key(x);
      } else {
        kh = lane_value(key, rl);
        kl = lane_value(key, ql);
      }
      if (key_before(kl, index_of(ql), kh, index_of(rl))) {
        const int t = rl;
        rl = ql;
        ql = t;
        for (int q = 0; q < 3; ++q) d[q] = -d[q];
      }
    }
  }
  plane(ql, pq);
  int ntab = 1, nv = 0;
  use(sl);
  double lastv[3] = {0.0, 0.0, 0.0};
  bool vinacc = false;
  if (lane == 0) S.rec.tab[0] = start;
  while (true) {
    // next edge plane rl: its vertex with the plane walked along and f = iso
    if (FULL) __syncthreads();        // S.used
    const bool in_tab = is_used(rl) && !(rl == sl && ntab >= 3);
    T pr[4], v[3];
    plane(rl, pr);
    double vd[3];
    VertexBound<T> vb{};
    // along the next edge plane, away from the one walked along
    T dn[3] = {pr[1] * eq[2] - pr[2] * eq[1], pr[2] * eq[0] - pr[0] * eq[2], pr[0] * eq[1] - pr[1] * eq[0]};
    if (pc[0] * dn[0] + pc[1] * dn[1] + pc[2] * dn[2] > T(0)) { dn[0] = -dn[0]; dn[1] = -dn[1]; dn[2] = -dn[2]; }
    Nearest<T> next;
    const T(&n1)[4] = pq;             // with two planes or more, the last two of the polygon (for the turn)
    const T(&n2)[4] = pc;
    if (SCAN) {
      solve3(pr, pc, eq, v);
      for (int q = 0; q < 3; ++q) vd[q] = (double)v[q];
      if (in_tab || !near_covers<T>(v, p, r, T(0), T(0)) || (nv > 0 && same_vertex(lastv, vd)) ||
          (ntab >= 2 && !pivot_valid(eq, n1, n2, pr)))
        return NEAR_RETRY;
      // An unused constraint before rl in the scan's order must have been passed
      // over: its vertex on this edge's line is outside rl or ql.  Along the line
      // from v, x crosses at t = -x(v) / (x . d); a crossing that lies outside rl
      // or ql by far more than v, the scan's vertex and their evaluation can be off
      // settles it without the order or the vertex: with the condition numbers Kx =
      // |x| |pc| |eq| / |x . d| and Kv = |pr| |pc| |eq| / |pr . d| that is below 200 u Kx Kv (1 +
      // |v| + |t d|) per unit normal (1e-11 here is 90,000 u), and 1e-5 covers the
      // FP32 arithmetic.  The others, few, take the scan's own expressions.  The planes
      // of a network scaled by 2^k are all scaled by it, so a product of norms is taken
      // in FP32 together with the quotient that undoes its scale (1e-11 |pc|^2 |eq|^2 |pr| on its
      // own is 0 from 2^-23 on), and normals of 1e-15 or less settle nothing here.  (The
      // instruction's square root, within an ulp: a rounded one takes 15 in its place.)
      const T apr = pr[0] * d[0] + pr[1] * d[1] + pr[2] * d[2], apq = pq[0] * d[0] + pq[1] * d[1] + pq[2] * d[2];
      const float nnr = (float)plane_nn(pr[0], pr[1], pr[2]), nnq = (float)plane_nn(pq[0], pq[1], pq[2]);
      const float nnc = (float)plane_nn(pc[0], pc[1], pc[2]), nne = (float)plane_nn(eq[0], eq[1], eq[2]);
      const float npr = __builtin_amdgcn_sqrtf(nnr), npq = __builtin_amdgcn_sqrtf(nnq);
      const float nce = __builtin_amdgcn_sqrtf(nnc) * __builtin_amdgcn_sqrtf(nne);
      const float fr = (float)apr, fq = (float)apq, vq = (float)plane_eval(pq[0], pq[1], pq[2], pq[3], v);
      const float ince = __builtin_amdgcn_rcpf(nce);
      const float dx = (float)d[0] * ince, dy = (float)d[1] * ince, dz = (float)d[2] * ince;
      const float dl = nce * __builtin_amdgcn_sqrtf(dx * dx + dy * dy + dz * dz);
      const float v1 = 1.f + (float)(absT(v[0]) + absT(v[1]) + absT(v[2]));
      const float kv = fminf(fminf(nnr, nnq), fminf(nnc, nne)) > 1e-30f
                           ? (1e-11f * nce) * ((nce * npr) * __builtin_amdgcn_rcpf(fabsf(fr)))
                           : __builtin_inff();
      const int gw = index_of(rl);
      bool fail = false;
      each([&](const T* x, int h, int gi, T) {
        if (h == cl || h == rl) return;
        const T sv = plane_eval(x[0], x[1], x[2], x[3], v);
        const T nn = plane_nn(x[0], x[1], x[2]);
        fail = fail || (sv > T(0) && sv * sv > (Tol<T>::EPS * Tol<T>::EPS) * nn);
        const T al = fmaT(x[0], dn[0], fmaT(x[1], dn[1], x[2] * dn[2]));
        next.add(-sv, al, al > T(0), h);
        const T ax = fmaT(x[0], d[0], fmaT(x[1], d[1], x[2] * d[2]));
        const float ra = __builtin_amdgcn_rcpf((float)ax), t = -(float)sv * ra;
        const float fn = (float)nn;
        const float far = 1e-17f + kv * (__builtin_amdgcn_sqrtf(fn) * fabsf(ra)) * (v1 + fabsf(t) * dl);
        const float tr = fr * t, tq = fq * t;
        const bool passed =
            fn > 1e-30f && (tr > npr * far || vq + tq > npq * far + 1e-5f * (fabsf(vq) + fabsf(tq)));
        if (!passed && (!is_used(h) || (h == sl && ntab >= 3)) &&
            key_before(FULL ? order_key(x) : key, gi, order_key(pr), gw)) {
          T vt[3];
          solve3(x, pc, eq, vt);
          fail = fail || !(violates(pr[0], pr[1], pr[2], pr[3], vt) ||
                           (h != ql && violates(pq[0], pq[1], pq[2], pq[3], vt)));
        }
      });
      if (__any(fail)) return NEAR_RETRY;
    } else {
      if constexpr (sizeof(T) == 4) {
        const double a4[4] = {pr[0], pr[1], pr[2], pr[3]};
        const double b4[4] = {pc[0], pc[1], pc[2], pc[3]};
        const double e4[4] = {eq[0], eq[1], eq[2], eq[3]};
        solve3(a4, b4, e4, vd);
        for (int q = 0; q < 3; ++q) v[q] = T(vd[q]);
      } else {
        solve3_rcp(pr, pc, eq, v);
        for (int q = 0; q < 3; ++q) vd[q] = (double)v[q];
      }
      const T lam = per_plane ? T(wp.lam) : T(0);
      vb = vertex_bound_unit<T>(pr, pc, eq, lam * err_of(rl), lam * err_of(cl), lam * eqe, T(wp.eps), T(wp.h_max), lam,
                                T(wp.lam_v));
      scale_bound<T>(vb, T(1) + absT(v[0]) + absT(v[1]) + absT(v[2]));
      T E = vb.E, F = T(0);
      if constexpr (sizeof(T) == 4) {
        // |lambda_i . a| <= |n_i| |a|; twice, for the FP32 rounding of either side
        const T l1 = __builtin_sqrtf(plane_nn(vb.n1[0], vb.n1[1], vb.n1[2]));
        const T l2 = __builtin_sqrtf(plane_nn(vb.n2[0], vb.n2[1], vb.n2[2]));
        const T l3 = __builtin_sqrtf(plane_nn(vb.n3[0], vb.n3[1], vb.n3[2]));
        E = T(2) * vb.e0;
        F = T(2) * (vb.w1 * l1 + vb.w2 * l2 + vb.w3 * l3 + vb.eg * qmax);
      }
      // (a system that is not trusted decides nothing: only its place counts)
      if (!FULL && !near_covers<T>(v, p, r, vb.ok ? E : T(0), vb.ok ? F : T(0))) return NEAR_RETRY;
      if (in_tab) return (int)AM_WHY_BIT(AM_WHY_TAB);
      if (ntab >= 2) {   // the turn (walk_ray's test)
        const T A12 = AM_DOT3(n1, n2), A23 = AM_DOT3(n2, pr), A13 = AM_DOT3(n1, pr), A22 = AM_DOT3(n2, n2);
        const T C1 = AM_DOT3(n1, eq), C2 = AM_DOT3(n2, eq), C3 = AM_DOT3(pr, eq), B = AM_DOT3(eq, eq);
        const T val = (A12 * A23 - A22 * A13) * B - (A12 * C2 * C3 + A23 * C1 * C2 - A13 * C2 * C2 - A22 * C1 * C3);
        const T mag = (absT(A12 * A23) + absT(A22 * A13)) * B +
                      (absT(A12 * C2 * C3) + absT(A23 * C1 * C2) + absT(A13 * C2 * C2) + absT(A22 * C1 * C3));
        if (!(val > T(wp.eps_turn) * mag)) return (int)AM_WHY_BIT(AM_WHY_TURN);
      }
      int bits = 0;
      each([&](const T* x, int h, int, T e) {
        if (h == cl || h == rl) return;
        const T sv = plane_eval(x[0], x[1], x[2], x[3], v);
        bits |= checked_verdict_at<T>(sv, x[0], x[1], x[2], x[3], e, vb);
        const T al = fmaT(x[0], dn[0], fmaT(x[1], dn[1], x[2] * dn[2]));
        next.add(-sv, al, al > T(0), h);
      });
      if (__any(bits & 1)) return (int)AM_WHY_BIT(AM_WHY_VIOL);
      if (__any(bits & 2)) return (int)AM_WHY_BIT(AM_WHY_UNSURE);
      if (!vb.ok) return (int)AM_WHY_BIT(AM_WHY_HMAX);
      if (nv > 0) {
        const double l1 = fabs(vd[0] - lastv[0]) + fabs(vd[1] - lastv[1]) + fabs(vd[2] - lastv[2]);
        if (!(l1 > 4.0 * Tol<double>::SAME_EPS)) return (int)AM_WHY_BIT(AM_WHY_SAME);
      }
    }
    // record the vertex
    const int gr = index_of(rl), gc = index_of(cl);
    const bool vacc = per_plane && wp.lam_v > 0.f && vertex_accurate(vb, v);
    if (per_plane && (wp.lam_v < 0.f || (wp.lam_v > 0.f && !wp.vsel && !vacc))) vinacc = true;
    if (lane == 0) {
      for (int q = 0; q < 3; ++q) S.rec.verts[nv * 3 + q] = vd[q];
      S.rec.vpair[nv * 2 + 0] = gr;
      S.rec.vpair[nv * 2 + 1] = gc;
      S.rec.tab[ntab] = gr;
      if (per_plane) {
        for (int x = 0; x < 3; ++x) {
          S.rec.jinv[nv * 9 + x] = float(vb.n1[x]);
          S.rec.jinv[nv * 9 + 3 + x] = float(vb.n2[x]);
          S.rec.jinv[nv * 9 + 6 + x] = float(vb.n3[x]);
        }
        if (wp.vsel && vacc) S.rec.jinv[nv * 9] = __builtin_nanf("");   // no Newton step needed
      }
    }
    for (int q = 0; q < 3; ++q) lastv[q] = vd[q];
    nv += 1;
    ntab += 1;
    use(rl);
    if (ntab >= 4 && rl == sl) break;       // closed
    if (ntab >= vm + 1) return SCAN ? NEAR_RETRY : (int)AM_WHY_BIT(AM_WHY_TRUNC);
    const int nx = next.take();
    if (nx < 0) return FULL ? (int)AM_WHY_BIT(AM_WHY_NEXT) : NEAR_RETRY;
    ql = cl;
    cl = rl;
    rl = nx;
    for (int q = 0; q < 4; ++q) {
      pq[q] = pc[q];
      pc[q] = pr[q];
    }
    for (int q = 0; q < 3; ++q) d[q] = dn[q];
  }
  __syncthreads();
  if constexpr (SCAN)
    finish_region<double, false, double>(net, io, wp, rid, slot_region, S.mask, eq, S.rec.tab, S.rec.verts,
                                         S.rec.vpair, ntab, nv, start, start, AM_ST_OK, false);
  else
    finish_region<T, true, double>(net, io, wp, rid, slot_region, S.mask, eq, S.rec.tab, S.rec.verts, S.rec.vpair,
                                   ntab, nv, start, start, AM_ST_OK, false, 0u, vinacc,
                                   per_plane ? S.rec.jinv : nullptr);
  return NEAR_DONE;
}

// The walk of one region on its near constraints, else on all of them.  FP64
// forms retry on all constraints whatever the reason; the FP32 form leaves a
// fifth of its regions undecided, for reasons all constraints would confirm.
template <typename T, bool SCAN, typename Src>
__device__ __forceinline__ int near_or_full_walk(const NetDev& net, const RegionIO& io, const WalkParams& wp, int rid,
                                                 int slot_region, const Src& P, const NearLds<T>& S, const T* eq,
                                                 const T* p, int start, T eqe = T(0)) {
  if (start < 0 || start >= net.C) return NEAR_RETRY;
  const int w = near_walk<T, SCAN, SET_NEAR>(net, io, wp, rid, slot_region, P, S, eq, p, start, eqe);
  if (w == NEAR_DONE || (sizeof(T) == 4 && w != NEAR_RETRY)) return w;
  __syncthreads();
  return near_walk<T, SCAN, SET_ALL>(net, io, wp, rid, slot_region, P, S, eq, p, start, eqe);
}

// Puts a region the near walk left (slot b of its launch) on the list.
__device__ __forceinline__ void near_left(const NearList& left, int b) {
  if (threadIdx.x == 0) left.slots[atomicAdd(left.cnt, 1)] = b;
}

}  // namespace am

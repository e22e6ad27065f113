// Constraint planes shared by activation prefix (am_prefix.h): the table, the
// layer products, and the FP64 walks that read those planes.
#include "am_prefix.h"

#include "am_device.h"
#include "am_kernels.h"
#include "am_near.h"
#include "am_walk.h"

namespace am {

// Prefix of depth d of a mask: its first off[d] bits.
__device__ __forceinline__ int prefix_words(const NetDev& net, int d) { return (net.off[d] + 31) >> 5; }
__device__ __forceinline__ uint32_t prefix_word(const NetDev& net, const uint32_t* m, int d, int w) {
  const uint32_t x = m[w];
  const int rest = net.off[d] - 32 * w;
  return rest >= 32 ? x : x & ((1u << rest) - 1u);
}

// High word of a table entry: 27 bits of the hash and the depth, so that a slot
// with another prefix is passed over without a look at that one's words.
__device__ __forceinline__ uint32_t prefix_key(uint64_t hm, int d) { return (uint32_t)(hm >> 37) << 5 | (uint32_t)d; }
static_assert(AM_MAX_LINEAR < 32, "five bits for the depth");

// A wave takes 16 regions at one depth, four lanes per prefix: they hash and
// compare its words and look at four slots at a time.  What bounds it is the
// longest chain of dependent reads in a block; slot by slot, with the words
// compared at each, that was 15.6 us for a level of 2,000 regions of a 4x128
// network, now 8.  A region
// that claims an empty slot makes a new id: its prefix's region is this one,
// whose mask is already in the store, so others that meet the slot compare with
// it at once and nothing waits.  One atomic per block and depth numbers the new
// ids (their order does not matter: planes do not depend on the id).
__global__ __launch_bounds__(4 * AM_PFX_REGIONS) void k_prefix(NetDev net, PrefixDev pf, PrefixRegions rg) {
  __shared__ int s_cnt, s_base;
  const int tid = threadIdx.x, lane = tid & 63;
  const int d = blockIdx.y + 1;
  const int cnt = launch_count(rg);
  stage_mark(pf.clk, T_CHAIN64);
  if ((int)blockIdx.x * AM_PFX_REGIONS >= cnt) return;
  if (tid == 0) s_cnt = 0;
  __syncthreads();
  const int j = lane & 3, lead = lane & ~3;
  const int nw = prefix_words(net, d);
  const int i = blockIdx.x * AM_PFX_REGIONS + (tid >> 2);
  const bool act = i < cnt;
  const int rid = act ? (rg.ids ? rg.ids[i] : launch_first(rg, rg.first) + i) : 0;
  const uint32_t* m = rg.reg_mask + (size_t)rid * net.Wd;
  uint64_t h = 0;
  if (act)
    for (int w = j; w < nw; w += 4) h += word_hash(prefix_word(net, m, d, w), w);
#pragma unroll
  for (int x = 1; x < 4; x <<= 1) {
    const uint32_t lo = (uint32_t)__shfl_xor((int)(uint32_t)h, x, 64);
    const uint32_t hi = (uint32_t)__shfl_xor((int)(uint32_t)(h >> 32), x, 64);
    h += ((uint64_t)hi << 32) | lo;
  }
  const uint64_t hm = mix64(h + (uint64_t)d);
  uint32_t s = (uint32_t)hm & pf.cap_mask;
  const uint32_t key = prefix_key(hm, d);
  bool done = !act, won = false;
  const unsigned long long mine = ((unsigned long long)key << 32) | (uint32_t)rid;
  for (uint32_t probes = 0; __ballot(!done) != 0ull;) {
    // four slots at once, one per lane: the first that is empty or has the key
    unsigned long long e = 0ull;
    if (!done) e = __hip_atomic_load(&pf.tab[(s + j) & pf.cap_mask], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const unsigned long long hits = __ballot(!done && (e == AM_PFX_EMPTY || (uint32_t)(e >> 32) == key));
    const uint32_t grp = (uint32_t)(hits >> lead) & 0xfu;
    const int at = grp ? __builtin_ctz(grp) : 4;
    bool claimed = false;
    if (!done && j == at && e == AM_PFX_EMPTY) {
      e = atomicCAS(&pf.tab[(s + at) & pf.cap_mask], AM_PFX_EMPTY, mine);
      claimed = e == AM_PFX_EMPTY;
    }
    const bool got = (__ballot(claimed) >> lead) & 0xfull;
    const uint32_t elo = (uint32_t)__shfl((int)(uint32_t)e, lead + (at & 3), 64);
    const uint32_t ehi = (uint32_t)__shfl((int)(uint32_t)(e >> 32), lead + (at & 3), 64);
    const bool cmp = !done && at < 4 && !got && ehi == key;
    uint32_t diff = 0;
    if (cmp) {
      const uint32_t* o = rg.reg_mask + (size_t)elo * net.Wd;
      for (int w = j; w < nw; w += 4) diff |= prefix_word(net, m, d, w) ^ prefix_word(net, o, d, w);
    }
    const unsigned long long bal = __ballot(diff != 0);
    if (!done) {
      if (got || (cmp && ((bal >> lead) & 0xfull) == 0ull)) {
        won = got;
        done = true;
        s = (s + at) & pf.cap_mask;
      } else {
        const uint32_t step = at < 4 ? at + 1 : 4;
        probes += step;
        if (probes > pf.cap_mask) done = true;   // table full: the host sizes it so that this never happens
        s = (s + (done ? 0u : step)) & pf.cap_mask;
      }
    }
  }
  const bool claim = won && j == 0;
  if (act && j == 0) pf.rslot[(size_t)i * pf.nd + d - 1] = (int)s;
  const unsigned long long bal = __ballot(claim);
  int at = 0;
  if (bal && lane == 0) at = atomicAdd(&s_cnt, __popcll(bal));
  at = __builtin_amdgcn_readfirstlane(at);
  __syncthreads();
  if (tid == 0 && s_cnt) s_base = atomicAdd(&pf.total[d * AM_PFX_TS], s_cnt);
  __syncthreads();
  if (claim) {
    const int id = s_base + at +
                   __builtin_amdgcn_mbcnt_hi((unsigned)(bal >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)bal, 0u));
    pf.tab_id[s] = id;
    *prefix_region(pf, net, d, id) = rid;
    pf.fresh[(size_t)d * pf.fresh_stride + id - pf.done[d]] = make_int2(rid, i);
  }
}

__global__ void k_prefix_clear(PrefixDev pf, size_t cap) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < cap) pf.tab[i] = AM_PFX_EMPTY;
  if (i <= (size_t)pf.nd) {
    pf.total[i * AM_PFX_TS] = 0;
    pf.done[i] = 0;
  }
}

// Re-inserts the ids of depth d into an empty (larger) table; n: at least their number.
__global__ void k_prefix_rehash(NetDev net, PrefixDev pf, const uint32_t* reg_mask, int d, int n) {
  const int id = blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= n || id >= pf.total[d * AM_PFX_TS]) return;
  const int rid = *prefix_region(pf, net, d, id);
  const uint32_t* m = reg_mask + (size_t)rid * net.Wd;
  uint64_t h = 0;
  for (int w = 0; w < prefix_words(net, d); ++w) h += word_hash(prefix_word(net, m, d, w), w);
  const uint64_t hm = mix64(h + (uint64_t)d);
  uint32_t s = (uint32_t)hm & pf.cap_mask;
  const unsigned long long mine = ((unsigned long long)prefix_key(hm, d) << 32) | (uint32_t)rid;
  for (uint32_t probes = 0; probes <= pf.cap_mask; ++probes) {
    if (atomicCAS(&pf.tab[s], AM_PFX_EMPTY, mine) == AM_PFX_EMPTY) {
      pf.tab_id[s] = id;
      return;
    }
    s = (s + 1) & pf.cap_mask;
  }
}

__global__ void k_prefix_ptrs(char** blk, PrefixPtrs ptrs) {
  const int i = threadIdx.x;
  if (i < ptrs.n) blk[ptrs.at[i]] = ptrs.p[i];
}

__global__ void k_pack_pairs(const double* xyz, const double* c, int n, double2* out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  out[i] = double2{xyz[i * 3 + 0], xyz[i * 3 + 1]};
  out[n + i] = double2{xyz[i * 3 + 2], c[i]};
}

typedef double am_f64x4 __attribute__((ext_vector_type(4)));
typedef double am_f64x2 __attribute__((ext_vector_type(2)));
typedef const __attribute__((address_space(1))) am_f64x2* gplanes;
typedef const __attribute__((address_space(1))) double* gdoubles;

// One layer's planes of AM_PT new prefixes: Y = W X + b with X = diag(m) P, 32
// columns; block (x, y) takes tile x and rows 128 y ..., 32 rows per wave as two
// 16-row blocks by two 16-column blocks, so that one fragment of W feeds two
// products and one of X two.  The k loop runs over the inputs active in some
// prefix of the tile, in ascending order: entries k | active prefixes << 16,
// padded to a multiple of 16 with the +0 row.  W streams from L2 four steps
// ahead; X goes through LDS, 64 list positions at a time, the next ones in
// registers meanwhile.  17 KB of LDS leave five blocks per CU, so that one's
// dependent first reads (region, slot, id, planes) hide behind the others'
// products; with all of X in LDS (68 KB, two blocks of eight waves) they took
// half the time, and with X read from memory by every wave L1 was the limit (80
// accesses per step).  Result element v of lane l is row l / 16 + 4 v, column l %
// 16.  Transform skips continue the same accumulation over their own inputs.
// Bound: the FP64 matrix cores (78.6 TFLOP/s).
template <bool SKIPS>
__global__ __launch_bounds__(256, SKIPS ? 4 : 5) void k_layer(NetDev net, PrefixDev pf, PrefixRegions rg, int d) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int id0 = pf.done[d] + (int)blockIdx.x * AM_PT;
  const int np = min(AM_PT, pf.total[d * AM_PFX_TS] - id0);
  if (np <= 0) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nout = net.nodes[d + 1];
  uint32_t* kl = reinterpret_cast<uint32_t*>(smem_raw);   // [widest input + 32]
  __shared__ double Xs[AM_PKC * AM_PXS];
  __shared__ gplanes s_src[AM_PT];
  __shared__ int s_cnt[4];
  // the tile's regions: every lane t % AM_PT knows prefix t's
  const int2 reg = pf.fresh[(size_t)d * pf.fresh_stride + blockIdx.x * AM_PT + min(lane & (AM_PT - 1), np - 1)];
  const int l16 = lane & 15, l4 = lane >> 4, q_l = l16 & 3;
  // rows per wave: 32, or 16 where that leaves no wave idle (layers up to 64 wide) or
  // where the tiles do not fill half the chip (a grid of 64-row blocks then; the
  // second half of it exits when they do)
  const int tiles = (pf.total[d * AM_PFX_TS] - pf.done[d] + AM_PT - 1) / AM_PT, rows128 = (nout + 127) >> 7;
  const int rpw = nout <= 64 || ((int)gridDim.y > rows128 && tiles * rows128 <= 128) ? 16 : 32;
  if ((int)blockIdx.y * 4 * rpw >= nout) return;
  const int row0 = (int)blockIdx.y * 4 * rpw + wave * rpw;
  const int nrb = row0 >= nout ? 0 : (rpw == 16 || row0 + 16 >= nout ? 1 : 2);   // the wave's row blocks with rows
  am_f64x4 acc[2][2];
#pragma unroll
  for (int rb = 0; rb < 2; ++rb)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int row = row0 + 16 * rb + l4 + 4 * v;
      const double b = q_l == 3 && row < nout ? pf.bp[d][row] + 0.0 : 0.0;   // -0 bias -> +0
      acc[rb][0][v] = b;
      acc[rb][1][v] = b;
    }
  // planes of hidden node `from` for the tile's prefixes
  auto sources = [&](int from) {
    if (tid < AM_PT) {
      const double2* p = pf.layer1;
      if (from > 1)
        p = prefix_planes(pf, net, from - 1, pf.tab_id[pf.rslot[(size_t)reg.y * pf.nd + from - 2]]);
      s_src[tid] = (gplanes)p;
    }
  };
  // acc += W X over the inputs of hidden node `from` (planes masked by its
  // activations); W^T has rows of ld, and row n_from is +0
  auto product = [&](int from, const double* W, int ld) {
    const int nin = net.nodes[from], in0 = net.off[from - 1];
    sources(from);
    // inputs active in some prefix of the tile, ascending: 64 inputs per wave
    int base = 0;
    for (int kb = 0; kb < nin; kb += 256) {
      const int k = kb + tid;
      uint32_t on = 0u;
      if (k < nin) {
        const int w = (in0 + k) >> 5, bit = (in0 + k) & 31;
#pragma unroll
        for (int t = 0; t < AM_PT; ++t) {
          const int rid = __builtin_amdgcn_readlane(reg.x, t);
          const uint32_t m = rg.reg_mask[(size_t)rid * net.Wd + w];
          on |= (t < np ? (m >> bit) & 1u : 0u) << t;
        }
      }
      const unsigned long long bal = __ballot(on != 0u);
      if (lane == 0) s_cnt[wave] = __popcll(bal);
      __syncthreads();
      int at = base;
      for (int w = 0; w < wave; ++w) at += s_cnt[w];
      if (on) kl[at + __builtin_amdgcn_mbcnt_hi((unsigned)(bal >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)bal, 0u))] = (uint32_t)k | (on << 16);
      base += s_cnt[0] + s_cnt[1] + s_cnt[2] + s_cnt[3];
      __syncthreads();
    }
    const int nk = (base + 15) & ~15;
    if (tid < nk + 16 - base) kl[base + tid] = (uint32_t)nin;
    __syncthreads();
    typedef const __attribute__((address_space(1))) char* gbytes;
    const uint32_t wrow = (uint32_t)(row0 + l16) * 8u, wld = (uint32_t)ld * 8u;   // byte offsets (below 2^32)
    const uint32_t rb1 = nrb > 1 ? 16u : 0u;   // (re-reads the first block when there is no second)
    // inputs of AM_PKC list positions: lane i of wave w reads position i's planes
    // of prefixes w and w + 4 (consecutive lanes, ascending k), zero where inactive
    am_f64x2 xr[2][2];
    auto fetch = [&](int c0) {
      const uint32_t e = c0 + lane < nk ? kl[c0 + lane] : 0u;
      const int k = min((int)(e & 0xffffu), nin - 1);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const gplanes src = s_src[wave + 4 * h];
        const bool on = (e >> (16 + wave + 4 * h)) & 1u;
        const am_f64x2 u = src[k], v = src[nin + k];
        xr[h][0] = on ? u : am_f64x2{0.0, 0.0};
        xr[h][1] = on ? v : am_f64x2{0.0, 0.0};
      }
    };
    double a0[4], a1[4];
    auto weights = [&](int u, uint32_t e) {
      const gdoubles w = (gdoubles)((gbytes)W + (wrow + (e & 0xffffu) * wld));
      a0[u] = w[0];
      a1[u] = w[rb1];
    };
    fetch(0);
    if (nrb > 0)
#pragma unroll
      for (int u = 0; u < 4; ++u) weights(u, kl[4 * u + l4]);
    for (int c0 = 0; c0 < nk; c0 += AM_PKC) {
      __syncthreads();                   // the previous inputs are read
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        double* o = Xs + lane * AM_PXS + 4 * (wave + 4 * h);
        o[0] = xr[h][0].x;
        o[1] = xr[h][0].y;
        o[2] = xr[h][1].x;
        o[3] = xr[h][1].y;
      }
      __syncthreads();
      if (c0 + AM_PKC < nk) fetch(c0 + AM_PKC);
      if (nrb == 0) continue;
      const int n = min(AM_PKC, nk - c0);
      for (int i0 = 0; i0 < n; i0 += 16) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int ii = i0 + 4 * u + l4;
          const double x0 = Xs[ii * AM_PXS + l16], x1 = Xs[ii * AM_PXS + 16 + l16];
          const double p0 = a0[u], p1 = a1[u];
          weights(u, kl[c0 + ii + 16]);
          acc[0][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(p0, x0, acc[0][0], 0, 0, 0);
          acc[0][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(p0, x1, acc[0][1], 0, 0, 0);
          if (nrb > 1) {
            acc[1][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(p1, x0, acc[1][0], 0, 0, 0);
            acc[1][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(p1, x1, acc[1][1], 0, 0, 0);
          }
        }
      }
    }
    __syncthreads();                     // list and sources are free
  };
  // element (rb, cb, v) of this lane: row, column's prefix 4 cb + l16 / 4, component q_l
  auto each = [&](auto&& f) {
#pragma unroll
    for (int rb = 0; rb < 2; ++rb)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int row = row0 + 16 * rb + l4 + 4 * v;
        if (rb < nrb && row < nout) {
          acc[rb][0][v] = f(acc[rb][0][v], row, l16 >> 2);
          acc[rb][1][v] = f(acc[rb][1][v], row, 4 + (l16 >> 2));
        }
      }
  };
  product(d, pf.Wp[d], pf.noutp[d]);
  // additive skips into this layer, in connection order (backend/inc/process.h:73-146)
  for (int s = 0; SKIPS && s < net.nskip[d]; ++s) {
    const int from = net.skip_from[d][s], tm = net.skip_tm[d][s];
    const bool ident = net.tm_h[tm] == 0 && net.tm_w[tm] == 0;
    if (from == 0) {
      const double* T = net.tm[tm];
      each([&](double a, int row, int) {
        return (ident ? row == q_l && row < 3 : q_l < 3) ? a + (ident ? 1.0 : T[row * 3 + q_l]) : a;
      });
    } else if (ident) {
      sources(from);
      __syncthreads();
      const int os = net.off[from - 1], nf = net.nodes[from];
      each([&](double a, int row, int t) {
        const int rid = __shfl(reg.x, t, 64);
        if (!(t < np && row < nf && mbit(rg.reg_mask + (size_t)rid * net.Wd, os + row))) return a;
        const am_f64x2 x = s_src[t][(q_l >> 1) * nf + row];
        return a + ((q_l & 1) ? x.y : x.x);
      });
      __syncthreads();
    } else {
      product(from, pf.tmp[tm], pf.tmpo[tm]);
    }
  }
  double* o0 = reinterpret_cast<double*>(prefix_planes(pf, net, d, id0 + min(l16 >> 2, np - 1)));
  double* o1 = reinterpret_cast<double*>(prefix_planes(pf, net, d, id0 + min(4 + (l16 >> 2), np - 1)));
  each([&](double a, int row, int t) {
    if (t < np) (t < 4 ? o0 : o1)[2 * ((size_t)(q_l >> 1) * nout + row) + (q_l & 1)] = a;
    return a;
  });
}
template __global__ void k_layer<false>(NetDev, PrefixDev, PrefixRegions, int);
template __global__ void k_layer<true>(NetDev, PrefixDev, PrefixRegions, int);

// A region's planes: base pointer of each hidden layer's (and the extras')
// planes, in LDS (as global-memory pointers, so that reads through them are not
// flat loads, which would also wait for LDS).
__device__ __forceinline__ void prefix_bases(const NetDev& net, const PrefixDev& pf, int place, gplanes* bases, int t0,
                                             int nt) {
  for (int l = t0; l <= net.D; l += nt) {
    const double2* p = l == 0 ? pf.layer1 : pf.extra;
    if (l > 0 && l < net.D) p = prefix_planes(pf, net, l, pf.tab_id[pf.rslot[(size_t)place * pf.nd + l - 1]]);
    bases[l] = (gplanes)p;
  }
}

// Signed constraint planes of one region, in parts: hidden layer l + 1 for l <
// D, then the extra planes.
struct PrefixPlanes {
  const NetDev& net;
  const gplanes* bases;          // [D + 1], LDS
  const uint32_t* mask;          // LDS
  __device__ __forceinline__ int parts() const { return net.E ? net.D + 1 : net.D; }
  __device__ __forceinline__ int first(int l) const { return net.off[l]; }
  __device__ __forceinline__ int size(int l) const { return l < net.D ? net.nodes[l + 1] : net.E; }
  __device__ __forceinline__ double err(int) const { return 0.0; }
  __device__ __forceinline__ void load(int l, int j, double* p) const { at(bases[l], size(l), l < net.D, first(l), j, p); }
  __device__ __forceinline__ void at(gplanes b, int n, bool hidden, int g0, int j, double* p) const {
    const am_f64x2 u = b[j], v = b[n + j];
    const uint32_t sm = hidden && mbit(mask, g0 + j) ? 0x80000000u : 0u;
    p[0] = flip_sign(u.x, sm);
    p[1] = flip_sign(u.y, sm);
    p[2] = flip_sign(v.x, sm);
    p[3] = flip_sign(v.y, sm);
  }
  __device__ __forceinline__ void get(int g, double* p) const {
    int l = 0;
    for (int i = 1; i <= net.D; ++i) l += g >= net.off[i] ? 1 : 0;
    load(l, g - first(l), p);
  }
};

// fma chain of 16 terms in ascending order: acc = fma(w of lane u of this
// lane's 16-lane row, x_u, acc), the weight through a DPP row broadcast.
__device__ __forceinline__ double fma_chain16(double acc, double w, const double (&x)[16]) {
  asm volatile(
      "s_nop 1\n"
      "v_fmac_f64_dpp %0, %1, %2 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %1, %3 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %1, %4 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %1, %5 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %1, %6 row_newbcast:4 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %1, %7 row_newbcast:5 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %1, %8 row_newbcast:6 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %1, %9 row_newbcast:7 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %1, %10 row_newbcast:8 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %1, %11 row_newbcast:9 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %1, %12 row_newbcast:10 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %1, %13 row_newbcast:11 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %1, %14 row_newbcast:12 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %1, %15 row_newbcast:13 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %1, %16 row_newbcast:14 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %1, %17 row_newbcast:15 row_mask:0xf bank_mask:0xf\n"
      : "+&v"(acc)
      : "v"(w), "v"(x[0]), "v"(x[1]), "v"(x[2]), "v"(x[3]), "v"(x[4]), "v"(x[5]), "v"(x[6]), "v"(x[7]), "v"(x[8]),
        "v"(x[9]), "v"(x[10]), "v"(x[11]), "v"(x[12]), "v"(x[13]), "v"(x[14]), "v"(x[15]));
  return acc;
}

// The region's face plane f = iso: the output row's chain over layer D's
// masked planes, 64 inputs at a time through LDS (stage: [4][66]); lane l runs
// component l % 4.  Each plane is read once: visit(plane (signed), constraint)
// sees it too.
template <typename F>
__device__ __forceinline__ void face_plane(const NetDev& net, const PrefixDev& pf, const PrefixPlanes& P, double* stage,
                                           double* eq, F&& visit) {
  const int lane = threadIdx.x, q = lane & 3, li = net.D, n = net.nodes[li], g0 = net.off[li - 1];
  const gplanes base = P.bases[li - 1];
  const double* W = pf.Wp[li];
  const int ld = pf.noutp[li];
  double acc = q == 3 ? pf.bp[li][0] + 0.0 : 0.0;
  am_f64x2 a{0.0, 0.0}, b{0.0, 0.0};
  if (lane < n) {
    a = base[lane];
    b = base[n + lane];
  }
  for (int k0 = 0; k0 < n; k0 += 64) {
    const int k = k0 + lane;
    const bool on = k < n && mbit(P.mask, g0 + min(k, n - 1));
    // (weight row n is +0; the inputs past n are +0)
    double w[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) w[c] = W[(size_t)min(k0 + 16 * c + (lane & 15), n) * ld];
    const am_f64x2 ca = a, cb = b;
    if (k + 64 < n) {
      a = base[k + 64];
      b = base[n + k + 64];
    }
    stage[lane] = on ? ca.x : 0.0;
    stage[66 + lane] = on ? ca.y : 0.0;
    stage[132 + lane] = on ? cb.x : 0.0;
    stage[198 + lane] = on ? cb.y : 0.0;
    if (k < n) {
      const uint32_t sm = on ? 0x80000000u : 0u;
      const double x[4] = {flip_sign(ca.x, sm), flip_sign(ca.y, sm), flip_sign(cb.x, sm), flip_sign(cb.y, sm)};
      visit(x, g0 + k);
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      if (k0 + 16 * c < n) {
        double x[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) x[u] = stage[q * 66 + 16 * c + u];
        acc = fma_chain16(acc, w[c], x);
      }
    }
    __syncthreads();
  }
  for (int c = 0; c < 4; ++c) eq[c] = lane_value(acc, c);
  eq[3] = eq[3] - net.iso;
}

// The candidate scan of one region, all its planes into LDS.
__device__ __forceinline__ void scan_prefix_region(const NetDev& net, const RegionIO& io, int rid, const gplanes* bases,
                                                   unsigned char* smem, const double* eq, const double* p) {
  const int C = net.C, Cs = io.Cs, N2 = io.Csort, lane = threadIdx.x;
  double* Px = reinterpret_cast<double*>(smem);
  double* Py = Px + Cs;
  double* Pz = Py + Cs;
  double* Pc = Pz + Cs;
  double* keys = Pc + Cs;
  int* order = reinterpret_cast<int*>(keys + N2);
  uint32_t* used = reinterpret_cast<uint32_t*>(order + N2);
  uint32_t* smask = used + ((C + 31) >> 5);
  for (int w = lane; w < net.Wd; w += 64) smask[w] = io.reg_mask[(size_t)rid * net.Wd + w];
  for (int w = lane; w < ((C + 31) >> 5); w += 64) used[w] = 0u;
  __syncthreads();
  const PrefixPlanes P{net, bases, smask};
  for (int l = 0; l < P.parts(); ++l)
    for (int j = lane; j < P.size(l); j += 64) {
      double x[4];
      P.load(l, j, x);
      const int g = P.first(l) + j;
      Px[g] = x[0];
      Py[g] = x[1];
      Pz[g] = x[2];
      Pc[g] = x[3];
    }
  __syncthreads();
  const WalkParams wp{0.f, 0.f, 0.f};
  const WalkRecs rec = carve_walk_recs(smem + scan_lds_head(C, N2, net.Wd), net.vm, false);
  walk_region<double, false>(net, io, wp, rid, rid - level_first(io), Px, Py, Pz, Pc, keys, order, used, smask, eq, p, rec.tab,
                             rec.verts, rec.vpair);
  __syncthreads();   // this region's LDS is free for the next
}

// Consecutive blocks go to the eight XCDs in turn; this gives each XCD a run of
// consecutive regions instead: neighbours share prefixes, and with them the
// planes in the XCD's L2.
__device__ __forceinline__ int xcd_run(int b, int n) {
  const int q = n >> 3, rem = n & 7, x = b & 7, k = b >> 3;
  return x * q + min(x, rem) + k;
}

template <bool SCAN, bool ALL>
__global__ __launch_bounds__(64, 4) void k_near64(NetDev net, PrefixDev pf, RegionIO io, int rid0, WalkParams wp,
                                                  double* eqb, int only_undecided, NearList left) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  __shared__ gplanes s_bases[AM_MAX_LINEAR + 1];
  stage_mark(io.clk, SCAN ? T_SCAN64 : T_RAY64);
  // the launch's layer products are done: their ids are no longer new
  if (blockIdx.x == 0 && (int)threadIdx.x <= pf.nd) pf.done[threadIdx.x] = pf.total[threadIdx.x * AM_PFX_TS];
  const int n = launch_count(io);
  if ((int)blockIdx.x >= n) return;
  const int b = xcd_run(blockIdx.x, n);
  const int rid = io.ids ? io.ids[b] : launch_first(io, rid0) + b;
  // a region an earlier walk decided keeps its records (its flag is 0 and stays 0)
  if (only_undecided && !(io.flags[rid - level_first(io)] & AM_UNDECIDED)) return;
  const NearLds<double> S = carve_near<double>(smem_raw, net.C, net.Wd, net.vm, false, ALL);
  const int start = io.reg_start[rid];
  prefix_bases(net, pf, b, s_bases, threadIdx.x, 64);
  for (int w = threadIdx.x; w < net.Wd; w += 64) S.mask[w] = io.reg_mask[(size_t)rid * net.Wd + w];
  double p[3], eq[4];
  for (int q = 0; q < 3; ++q) p[q] = io.reg_point[(size_t)rid * 3 + q];
  __syncthreads();
  const PrefixPlanes P{net, s_bases, S.mask};
  NearScan<double, SCAN> sc;
  face_plane(net, pf, P, S.stage, eq, [&](const double* x, int g) {
    if (ALL) near_stage<double>(S, g, x);
    else sc.add(x, 0.0, p, S.key, g);
  });
  bool done = false;
  if (start >= 0 && start < net.C)
    done = near_walk<double, SCAN, ALL ? SET_LDS : SET_NEAR>(net, io, wp, rid, rid - level_first(io), P, S, eq, p, start,
                                                             0.0, sc, net.D - 1) == NEAR_DONE;
  if (SCAN && ALL) {
    // (a launch of its own for the seeds and the few others took 4.6 us a level)
    if (!done) {
      __syncthreads();
      scan_prefix_region(net, io, rid, s_bases, smem_raw, eq, p);
    }
    return;
  }
  // (thread 0 wrote the flag in finish_region: the orientation may be undecided)
  if (threadIdx.x == 0 && (!done || (!SCAN && (io.flags[rid - level_first(io)] & AM_UNDECIDED)))) {
    for (int q = 0; q < 4; ++q) eqb[(size_t)b * 4 + q] = eq[q];
    near_left(left, b);
  }
}
template __global__ void k_near64<true, false>(NetDev, PrefixDev, RegionIO, int, WalkParams, double*, int, NearList);
template __global__ void k_near64<false, false>(NetDev, PrefixDev, RegionIO, int, WalkParams, double*, int, NearList);
template __global__ void k_near64<true, true>(NetDev, PrefixDev, RegionIO, int, WalkParams, double*, int, NearList);
template __global__ void k_near64<false, true>(NetDev, PrefixDev, RegionIO, int, WalkParams, double*, int, NearList);

// The listed regions (blocks stride over the list) on all constraints: with
// `quick` the walk that reads the planes once per vertex, then, for seeds and
// what that does not settle, the candidate scan.  The planes' pointers lie where
// the scan keeps its records, which it writes once the planes are in LDS (past
// all of the other walk's scratch): 136 bytes more would leave no room for them at
// the largest constraint counts.
__global__ __launch_bounds__(64, 4) void k_walk_fp64(NetDev net, PrefixDev pf, RegionIO io, int rid0, const int* count,
                                                  const int* slots, const double* eqb, int quick) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  gplanes* const bases = reinterpret_cast<gplanes*>(smem_raw + scan_lds_head(net.C, io.Csort, net.Wd));
  if (!quick) stage_mark(io.clk, T_SCAN64);
  const int lane = threadIdx.x;
  const int total = min(*count, io.count);
  for (int i = blockIdx.x; i < total; i += gridDim.x) {
    const int b = slots[i];
    const int rid = io.ids ? io.ids[b] : launch_first(io, rid0) + b;
    const int start = io.reg_start[rid];
    prefix_bases(net, pf, b, bases, lane, 64);
    double p[3], eq[4];
    for (int q = 0; q < 3; ++q) p[q] = io.reg_point[(size_t)rid * 3 + q];
    for (int q = 0; q < 4; ++q) eq[q] = eqb[(size_t)b * 4 + q];
    if (quick && start >= 0 && start < net.C) {
      const WalkParams wp{0.f, 0.f, 0.f};
      const NearLds<double> S = carve_near<double>(smem_raw, net.C, net.Wd, net.vm, false);
      for (int w = lane; w < net.Wd; w += 64) S.mask[w] = io.reg_mask[(size_t)rid * net.Wd + w];
      __syncthreads();
      const PrefixPlanes P{net, bases, S.mask};
      const int done = near_walk<double, true, SET_ALL>(net, io, wp, rid, rid - level_first(io), P, S, eq, p, start);
      __syncthreads();
      if (done == NEAR_DONE) continue;
    }
    scan_prefix_region(net, io, rid, bases, smem_raw, eq, p);
  }
}

// The checked ray walk over all constraints of the listed regions: planes in
// LDS past hidden layer 1's (rebuilt from its weights where read, PlaneView),
// NW waves per region (the records do not depend on NW: every reduction breaks
// ties by constraint index and each serial step runs on one wave).  A region
// it leaves undecided goes on the candidate scan's list (its counter zeroed
// before) and counts itself and its reasons in left.run (as k_collect_slots
// would).
template <int NW>
__global__ __launch_bounds__(64 * NW, 24 / NW) void k_walk_ray64(NetDev net, PrefixDev pf, RegionIO io, int rid0,
                                                                 WalkParams wp, const double* eqb, NearList list,
                                                                 SlotList left) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  __shared__ gplanes s_bases[AM_MAX_LINEAR + 1];
  const int n1 = net.nodes[1], Cl = net.C - n1, tid = threadIdx.x;
  double2* Q = reinterpret_cast<double2*>(smem_raw);   // (x, y) pairs, then (z, c) pairs
  uint32_t* smask = reinterpret_cast<uint32_t*>(Q + 2 * Cl);
  const WalkRecs rec = carve_walk_recs(reinterpret_cast<unsigned char*>(Q + 2 * Cl) + ((net.Wd * 4 + 15) & ~15),
                                       net.vm, false);
  const int total = min(*list.cnt, io.count);
  for (int i = blockIdx.x; i < total; i += gridDim.x) {
    const int b = list.slots[i];
    const int rid = io.ids ? io.ids[b] : launch_first(io, rid0) + b;
    const int start_in = io.reg_start[rid];
    prefix_bases(net, pf, b, s_bases, tid, 64 * NW);
    for (int w = tid; w < net.Wd; w += 64 * NW) smask[w] = io.reg_mask[(size_t)rid * net.Wd + w];
    __syncthreads();
    const PrefixPlanes S{net, s_bases, smask};
    for (int l = 1; l < S.parts(); ++l)
      for (int j = tid; j < S.size(l); j += 64 * NW) {
        double x[4];
        S.load(l, j, x);
        Q[S.first(l) - n1 + j] = double2{x[0], x[1]};
        Q[Cl + S.first(l) - n1 + j] = double2{x[2], x[3]};
      }
    double p[3], eq[4];
    for (int q = 0; q < 3; ++q) p[q] = io.reg_point[(size_t)rid * 3 + q];
    for (int q = 0; q < 4; ++q) eq[q] = eqb[(size_t)b * 4 + q];
    __syncthreads();
    const PlaneView<double> P{reinterpret_cast<const double*>(Q), Cl, n1, net.W0, net.b[0], smask};
    walk_ray<double, NW>(net, io, wp, rid, rid - level_first(io), P, smask, eq, p, rec, start_in);
    // thread 0 wrote the region's flag (finish_region)
    if (tid == 0) {
      const unsigned f = io.flags[rid - level_first(io)];
      if (f & AM_UNDECIDED) {
        left.slots[atomicAdd(left.cnt, 1)] = b;
        atomicAdd(left.run, 1);
        for (int w = 0; w < AM_WHY_COUNT; ++w)
          if (f & AM_WHY_BIT(w)) atomicAdd(left.run + 1 + w, 1);
      }
    }
    __syncthreads();   // this region's LDS is free for the next
  }
}
template __global__ void k_walk_ray64<2>(NetDev, PrefixDev, RegionIO, int, WalkParams, const double*, NearList, SlotList);
template __global__ void k_walk_ray64<4>(NetDev, PrefixDev, RegionIO, int, WalkParams, const double*, NearList, SlotList);
template __global__ void k_walk_ray64<8>(NetDev, PrefixDev, RegionIO, int, WalkParams, const double*, NearList, SlotList);

// Vertices of a region whose polygon (the tight-constraint pair of every
// vertex, its order and orientation) a reduced-precision walk certified: each
// is the intersection of the FP64 planes of its pair with the face plane,
// solved as the FP64 ray walk solves it (new constraint, constraint walked
// along, face plane), so the coordinates carry FP64 rounding only.
__global__ __launch_bounds__(64) void k_vertex_fp64(NetDev net, PrefixDev pf, RegionIO io, int rid0) {
  __shared__ gplanes s_bases[AM_MAX_LINEAR + 1];
  __shared__ uint32_t s_mask[AM_MAX_WORDS];
  __shared__ __align__(16) double s_stage[AM_NEAR_PL];
  const int b = blockIdx.x;
  stage_mark(io.clk, T_VERT64);
  if (b >= launch_count(io)) return;
  const int rid = io.ids ? io.ids[b] : launch_first(io, rid0) + b;
  if (io.flags && (io.flags[rid - level_first(io)] & AM_UNDECIDED)) return;   // left to the FP64 walk
  const int vm = net.vm;
  const int nv = io.reg_info[(size_t)rid * AM_INFO_STRIDE + 2];
  prefix_bases(net, pf, b, s_bases, threadIdx.x, 64);
  for (int w = threadIdx.x; w < net.Wd; w += 64) s_mask[w] = io.reg_mask[(size_t)rid * net.Wd + w];
  __syncthreads();
  const PrefixPlanes P{net, s_bases, s_mask};
  double eq[4];
  face_plane(net, pf, P, s_stage, eq, [](const double*, int) {});
  for (int i = threadIdx.x; i < nv && i < vm; i += 64) {
    const int r = io.reg_vpair[((size_t)rid * vm + i) * 2 + 0];
    const int s = io.reg_vpair[((size_t)rid * vm + i) * 2 + 1];
    if (r < 0 || r >= net.C || s < 0 || s >= net.C) continue;
    double pr[4], ps[4];
    P.get(r, pr);
    P.get(s, ps);
    double v[3];
    solve3_rcp(pr, ps, eq, v);
    double* out = io.reg_verts + ((size_t)rid * vm + i) * 3;
    out[0] = v[0];
    out[1] = v[1];
    out[2] = v[2];
  }
}

}  // namespace am

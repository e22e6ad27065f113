// FP64 planes of many regions at once, bit-identical to the one-region chain.
//
// The masked affine chain (backend/inc/process.h:18-193) is a GEMM per layer:
// Y = W_li * X with X = diag(m) P_{li-1}, one column per plane component (x, y,
// z, c) of each region.  A workgroup takes AM_CT regions = 32 columns through all
// layers, its activations staying in LDS: four waves of up to 32 rows each (eight
// for layers over 128 wide), v_mfma_f64_16x16x4f64 on 16 x 16 blocks (A: lane l
// holds W[row0 + l % 16][list entry i0 + l / 16], B: X[i0 + l / 16][16 cb + l % 16];
// result element v of lane l is row row0 + l / 16 + 4 v, column 16 cb + l % 16).
// That instruction is one fma per term in ascending k, so with the accumulators
// starting at (0, 0, 0, b_j + 0) and the list of active inputs ascending each output
// is the same sequence of roundings as the canonical chain.  An inactive k adds
// fma(w, +0, acc) = acc exactly (no accumulator is ever -0: each starts at +0 or a
// nonzero bias, and a sum of opposite-signed zeros rounds to +0), so zero-filling
// the inputs that only other regions of the tile have active reproduces skipping them.
//
// What bounds it is latency: a layer is a dependent chain (list, products, mask),
// and a level of a few thousand small regions gives each CU one or two tiles.  Eight
// regions a tile instead of 16 give twice the tiles, and four waves cover layers up
// to 128 wide without idle ones.  Eight networks 3x16..4x64 (85 levels of up to 5,800
// regions): 48 us a level with 16-region tiles of 16 waves, 36 so; the planes of a 4x128
// network's 241,000 regions for its gradients 3.5 -> 2.2 ms.
//
// The regions' walks on those planes (am_near.h, am_walk.h) follow.
#include "am_device.h"
#include "am_kernels.h"
#include "am_near.h"
#include "am_walk.h"

namespace am {


// Plane g of a region (x, y, z, c) as the chain defines it.  Hidden layer 1's
// planes are the rows of (W0 | b0), negated where the neuron is active; the
// chain does not store them, they are rebuilt here from the weights and the
// region's mask.  The others come from the chain's record at src.
__device__ __forceinline__ void plane64(const NetDev& net, const uint32_t* mask, const double* src, int Cs_hbm, int g,
                                        double* p) {
  if (g < net.nodes[1]) {
    const bool on = mbit(mask, g);
    const double v[4] = {net.W0[g * 3 + 0], net.W0[g * 3 + 1], net.W0[g * 3 + 2], net.b[0][g]};
    for (int q = 0; q < 4; ++q) p[q] = on ? -v[q] : v[q];
  } else {
    for (int q = 0; q < 4; ++q) p[q] = src[(size_t)q * Cs_hbm + g];
  }
}

// One region's planes into LDS, threads t0, t0 + nt, ...
__device__ __forceinline__ void load_planes64(const NetDev& net, const uint32_t* mask, const double* src, int Cs_hbm,
                                              double* Px, double* Py, double* Pz, double* Pc, int t0, int nt) {
  for (int g = t0; g < net.C; g += nt) {
    double p[4];
    plane64(net, mask, src, Cs_hbm, g, p);
    Px[g] = p[0];
    Py[g] = p[1];
    Pz[g] = p[2];
    Pc[g] = p[3];
  }
}

typedef double am_f64x4 __attribute__((ext_vector_type(4)));

// The planes of one tile: regions first + r0 .. + nreg - 1 of lv, written at planes
// slots r0 + t.  io supplies the plane stride
// and the layer operands; maxw >= the network's layer widths (LDS layout).
template <int NW>
__device__ __forceinline__ void chain_tile(const NetDev& net, const ChainIO& io, const ChainLevel& lv, int r0, int nreg,
                                           int maxw) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  constexpr int NT = 64 * NW;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  double* Xs = reinterpret_cast<double*>(smem_raw);                            // [maxw + 1][AM_CXS] the layer's inputs
  uint32_t* kl = reinterpret_cast<uint32_t*>(Xs + (size_t)(maxw + 1) * AM_CXS);   // [maxw + 32] the active ones
  uint32_t* mk = kl + maxw + 32;                                               // [AM_CT][Wd]
  __shared__ int s_cnt[NW];
  const int Wd = net.Wd, Cs = io.Cs;
  for (int idx = tid; idx < AM_CT * Wd; idx += NT) {
    const int t = idx / Wd, w = idx - t * Wd, r = r0 + min(t, nreg - 1);
    mk[idx] = lv.reg_mask[(size_t)(lv.first + r) * Wd + w];
  }
  for (int idx = tid; idx < AM_CN * net.E; idx += NT) {
    const int col = idx / net.E, e = idx - col * net.E, t = col >> 2, q = col & 3;
    if (t < nreg) lv.planes[((size_t)(r0 + t) * 4 + q) * Cs + net.L + e] = q < 3 ? net.ew[e * 3 + q] : net.eb[e];
  }
  __syncthreads();
  // layer 1's planes: rows of (W0 | b0), masked (readers rebuild them: not written out)
  const int n1 = net.nodes[1];
  for (int k = tid >> 3; k < n1; k += NT / 8) {
    const int t = tid & 7;
    const bool on = mbit(mk + t * Wd, k);
    double* o = Xs + k * AM_CXS + 4 * t;
    for (int q = 0; q < 3; ++q) o[q] = on ? net.W0[k * 3 + q] : 0.0;
    o[3] = on ? net.b[0][k] : 0.0;
  }
  if (tid < AM_CN) Xs[n1 * AM_CXS + tid] = 0.0;
  const int l16 = lane & 15, l4 = lane >> 4, q_l = l16 & 3;
  for (int li = 1; li <= net.D; ++li) {
    const int nin = net.nodes[li], nout = net.nodes[li + 1], in0 = net.off[li - 1];
    // inputs active in some region of the tile, ascending (nin <= NT)
    bool on = false;
    if (tid < nin) {
      const int w = (in0 + tid) >> 5, bit = (in0 + tid) & 31;
      uint32_t m = 0u;
#pragma unroll
      for (int t = 0; t < AM_CT; ++t) m |= mk[t * Wd + w];
      on = (m >> bit) & 1u;
    }
    const unsigned long long bal = __ballot(on);
    if (lane == 0) s_cnt[wave] = __popcll(bal);
    __syncthreads();                     // (and the inputs are staged)
    int at = 0, base = 0;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      at += w < wave ? s_cnt[w] : 0;
      base += s_cnt[w];
    }
    if (on) kl[at + __builtin_amdgcn_mbcnt_hi((unsigned)(bal >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)bal, 0u))] = (uint32_t)tid;
    const int nk = (base + 15) & ~15;
    if (tid < nk + 16 - base) kl[base + tid] = (uint32_t)nin;   // (weight row and input row nin are +0)
    __syncthreads();
    const int rpw = nout <= 16 * NW ? 16 : 32, row0 = wave * rpw;
    const int nrb = row0 >= nout ? 0 : (rpw == 32 && row0 + 16 < nout ? 2 : 1);   // the wave's row blocks
    am_f64x4 acc[2][2];
    if (nrb > 0) {
#pragma unroll
      for (int rb = 0; rb < 2; ++rb)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int row = row0 + 16 * rb + l4 + 4 * v;
          const double b = q_l == 3 && row < nout ? io.bp[li][row] + 0.0 : 0.0;   // -0 bias -> +0
          acc[rb][0][v] = b;
          acc[rb][1][v] = b;
        }
      typedef const __attribute__((address_space(1))) double* gdoubles;
      const gdoubles W = (gdoubles)(io.Wp[li] + row0 + l16);
      const uint32_t ld = (uint32_t)io.noutp[li], rb1 = nrb > 1 ? 16u : 0u;
      double a0[4], a1[4];
      uint32_t e[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        e[u] = kl[4 * u + l4];
        a0[u] = W[e[u] * ld];
        a1[u] = W[e[u] * ld + rb1];
      }
      for (int i0 = 0; i0 < nk; i0 += 16) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const double x0 = Xs[e[u] * AM_CXS + l16], x1 = Xs[e[u] * AM_CXS + 16 + l16];
          const double p0 = a0[u], p1 = a1[u];
          e[u] = kl[i0 + 16 + 4 * u + l4];
          a0[u] = W[e[u] * ld];
          a1[u] = W[e[u] * ld + rb1];
          acc[0][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(p0, x0, acc[0][0], 0, 0, 0);
          acc[0][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(p0, x1, acc[0][1], 0, 0, 0);
          if (nrb > 1) {
            acc[1][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(p1, x0, acc[1][0], 0, 0, 0);
            acc[1][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(p1, x1, acc[1][1], 0, 0, 0);
          }
        }
      }
    }
    __syncthreads();                     // the inputs are read
#pragma unroll
    for (int rb = 0; rb < 2; ++rb)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int row = row0 + 16 * rb + l4 + 4 * v;
        if (rb < nrb && row < nout) {
          Xs[row * AM_CXS + l16] = acc[rb][0][v];
          Xs[row * AM_CXS + 16 + l16] = acc[rb][1][v];
        }
      }
    if (li < net.D && tid < AM_CN) Xs[nout * AM_CXS + tid] = 0.0;
    __syncthreads();
    if (li == net.D) {
      if (tid < AM_CN && (tid >> 2) < nreg)
        lv.eq[(size_t)(r0 + (tid >> 2)) * 4 + (tid & 3)] = (tid & 3) == 3 ? Xs[tid] - net.iso : Xs[tid];
      break;
    }
    // signed to HBM (consecutive lanes on consecutive constraints), masked in place
    const int g0 = net.off[li];
    for (int col = wave; col < AM_CN; col += NW) {
      const int t = col >> 2;
      double* dst = lv.planes + ((size_t)(r0 + t) * 4 + (col & 3)) * Cs + g0;
      for (int row = lane; row < nout; row += 64) {
        const double y = Xs[row * AM_CXS + col];
        const bool act = mbit(mk + t * Wd, g0 + row);
        if (t < nreg) dst[row] = act ? -y : y;
        if (!act) Xs[row * AM_CXS + col] = 0.0;
      }
    }
  }
}

template <int NW>
__global__ __launch_bounds__(64 * NW) void k_chain_tile_fp64(NetDev net, ChainIO io, int maxw) {
  const int r0 = blockIdx.x * AM_CT;
  if (r0 >= io.count) return;
  const ChainLevel lv{io.first, io.count, io.planes, io.eq, io.reg_mask, nullptr};
  chain_tile<NW>(net, io, lv, r0, min(AM_CT, io.count - r0), maxw);
}
template __global__ void k_chain_tile_fp64<4>(NetDev, ChainIO, int);
template __global__ void k_chain_tile_fp64<8>(NetDev, ChainIO, int);

// Many networks in one launch: block b takes tiles[b] = (network, r0, regions);
// the tile's regions are lv.first + r0 + t, all of one network.
template <int NW>
__global__ __launch_bounds__(64 * NW) void k_chain_tile_fp64_multi(const NetDev* nets, const ChainIO* cios, ChainLevel lv,
                                                                   const int4* tiles, int maxw) {
  stage_mark(lv.clk, T_CHAIN64);
  const int4 tl = tiles[blockIdx.x];
  if (tl.z <= 0) return;
  chain_tile<NW>(nets[tl.x], cios[tl.x], lv, tl.y, tl.z, maxw);
}
template __global__ void k_chain_tile_fp64_multi<4>(const NetDev*, const ChainIO*, ChainLevel, const int4*, int);
template __global__ void k_chain_tile_fp64_multi<8>(const NetDev*, const ChainIO*, ChainLevel, const int4*, int);

// The candidate scan of one region (rid) on the planes at slot sl.
__device__ __forceinline__ void walk_fp64_body(const NetDev& net, const RegionIO& io, int rid, int sl,
                                               const double* planes, const double* eqb, int Cs_hbm) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int C = net.C;
  const int Cs = io.Cs;
  const int N2 = io.Csort;
  double* Px = reinterpret_cast<double*>(smem_raw);
  double* Py = Px + Cs;
  double* Pz = Py + Cs;
  double* Pc = Pz + Cs;
  double* keys = Pc + Cs;
  int* order = reinterpret_cast<int*>(keys + N2);
  uint32_t* used = reinterpret_cast<uint32_t*>(order + N2);
  uint32_t* smask = used + ((C + 31) >> 5);

  const int lane = threadIdx.x;
  for (int w = lane; w < net.Wd; w += 64) smask[w] = io.reg_mask[(size_t)rid * net.Wd + w];
  for (int w = lane; w < ((C + 31) >> 5); w += 64) used[w] = 0u;
  load_planes64(net, io.reg_mask + (size_t)rid * net.Wd, planes + (size_t)sl * 4 * Cs_hbm, Cs_hbm, Px, Py, Pz,
                Pc, lane, 64);
  double p[3];
  p[0] = io.reg_point[(size_t)rid * 3 + 0];
  p[1] = io.reg_point[(size_t)rid * 3 + 1];
  p[2] = io.reg_point[(size_t)rid * 3 + 2];
  const double eq[4] = {eqb[(size_t)sl * 4 + 0], eqb[(size_t)sl * 4 + 1], eqb[(size_t)sl * 4 + 2],
                        eqb[(size_t)sl * 4 + 3]};
  __syncthreads();
  const WalkParams wp{0.f, 0.f, 0.f};
  const WalkRecs rec = carve_walk_recs(smem_raw + scan_lds_head(C, N2, net.Wd), net.vm, false);
  walk_region<double, false>(net, io, wp, rid, rid - io.first, Px, Py, Pz, Pc, keys, order, used, smask, eq, p, rec.tab,
                             rec.verts, rec.vpair);
  __syncthreads();   // this region's LDS is free for the next
}

// Network of a region in a batch of networks: the last word of its mask.
__device__ __forceinline__ int region_net(const RegionIO& io, int Wd, int rid) {
  return (int)io.reg_mask[(size_t)rid * Wd + Wd - 1];
}

// LDS layout of the candidate scan for a network of C constraints (the host
// sizes the launch for the widest network of the batch).
__device__ __forceinline__ RegionIO scan_layout(const RegionIO& io, int C) {
  RegionIO r = io;
  int n2 = AM_TOPK;
  while (n2 < C) n2 <<= 1;
  r.Cs = C;
  r.Csort = n2;
  return r;
}

// Planes of one region of a batch: the chain's record, hidden layer 1's from the
// weights (plane64).
struct TilePlanes {
  const NetDev& net;
  const double* src;
  int Cs;
  const uint32_t* mask;   // LDS
  __device__ __forceinline__ int parts() const { return net.D; }
  __device__ __forceinline__ int first(int l) const { return net.off[l]; }
  __device__ __forceinline__ int size(int l) const { return net.nodes[l + 1]; }
  __device__ __forceinline__ double err(int) const { return 0.0; }
  __device__ __forceinline__ void get(int g, double* p) const { plane64(net, mask, src, Cs, g, p); }
  __device__ __forceinline__ void load(int l, int j, double* p) const { get(first(l) + j, p); }
};

// The candidate scan of the listed slots (blocks stride over the list).
__global__ __launch_bounds__(64) void k_walk_fp64_multi(const NetDev* nets, RegionIO io, int Wd, int rid0,
                                                        const int* count, const int* slots, const double* planes,
                                                        const double* eqb, int Cs_hbm) {
  stage_mark(io.clk, T_SCAN64);
  const int total = min(*count, io.count);
  for (int b = blockIdx.x; b < total; b += gridDim.x) {
    const int sl = slots[b];
    const int rid = rid0 + sl;
    const NetDev& net = nets[region_net(io, Wd, rid)];
    walk_fp64_body(net, scan_layout(io, net.C), rid, sl, planes, eqb, Cs_hbm);
  }
}

// Checked ray-shooting walk on the FP64 planes of k_chain_tile_fp64.  The
// planes are the canonical FP64 planes, so the only uncertainty is the
// rounding of the walk's own evaluations; regions it cannot certify are
// flagged (io.flags, level-relative) for the candidate scan.
template <int NW>
__device__ __forceinline__ void walk_ray64_body(const NetDev& net, const RegionIO& io, int rid, int b,
                                                const WalkParams& wp, const double* planes, const double* eqb,
                                                int Cs_hbm) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  // LDS holds the planes past hidden layer 1 (index g - n1); layer 1's are
  // rebuilt from W0 and b0 where read (PlaneView), which leaves LDS for more
  // regions per CU
  const int n1 = net.nodes[1], Cl = net.C - n1;
  double2* Q = reinterpret_cast<double2*>(smem_raw);   // (x, y) pairs, then (z, c) pairs
  uint32_t* smask = reinterpret_cast<uint32_t*>(Q + 2 * Cl);
  const WalkRecs rec = carve_walk_recs(reinterpret_cast<unsigned char*>(Q + 2 * Cl) + ((net.Wd * 4 + 15) & ~15),
                                       net.vm, false);
  const int lane = threadIdx.x;
  const int start_in = io.reg_start[rid];
  for (int w = lane; w < net.Wd; w += 64 * NW) smask[w] = io.reg_mask[(size_t)rid * net.Wd + w];
  const double* src = planes + (size_t)b * 4 * Cs_hbm + n1;
  for (int i = lane; i < Cl; i += 64 * NW) {
    Q[i] = double2{src[i], src[Cs_hbm + i]};
    Q[Cl + i] = double2{src[2 * (size_t)Cs_hbm + i], src[3 * (size_t)Cs_hbm + i]};
  }
  double p[3];
  p[0] = io.reg_point[(size_t)rid * 3 + 0];
  p[1] = io.reg_point[(size_t)rid * 3 + 1];
  p[2] = io.reg_point[(size_t)rid * 3 + 2];
  const double eq[4] = {eqb[(size_t)b * 4 + 0], eqb[(size_t)b * 4 + 1], eqb[(size_t)b * 4 + 2],
                        eqb[(size_t)b * 4 + 3]};
  __syncthreads();
  const PlaneView<double> P{reinterpret_cast<const double*>(Q), Cl, n1, net.W0, net.b[0], smask};
  walk_ray<double, NW>(net, io, wp, rid, rid - io.first, P, smask, eq, p, rec, start_in);
}

// The near walk of a batch's regions (am_near.h), one wave per region; ALL
// (every network of the batch has up to AM_ALL_MAX constraints): on all of them, and
// the few regions it leaves, and seeds, take the walks over all constraints in the
// same wave (two launches for them took 9.6 us a level).  Else they go on a list.  Eight networks of 48 to 256 constraints
// (85 levels of up to 5,800 regions): 47 us a level with two-wave ray walks over all
// constraints, 36 so.
template <bool SCAN, bool ALL>
__global__ __launch_bounds__(64, 4) void k_near64_multi(const NetDev* nets, RegionIO io, int Wd, int rid0, WalkParams wp,
                                                     const double* planes, const double* eqb, int Cs_hbm,
                                                     NearList left, int* run) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  stage_mark(io.clk, SCAN ? T_SCAN64 : T_RAY64);
  const int b = blockIdx.x;
  if (b >= io.count) return;
  const int rid = rid0 + b;
  const NetDev& net = nets[region_net(io, Wd, rid)];
  const NearLds<double> S = carve_near<double>(smem_raw, net.C, Wd, net.vm, false, ALL);
  const int start = io.reg_start[rid];
  for (int w = threadIdx.x; w < Wd; w += 64) S.mask[w] = io.reg_mask[(size_t)rid * Wd + w];
  double p[3], eq[4];
  for (int q = 0; q < 3; ++q) p[q] = io.reg_point[(size_t)rid * 3 + q];
  for (int q = 0; q < 4; ++q) eq[q] = eqb[(size_t)b * 4 + q];
  __syncthreads();
  const TilePlanes P{net, planes + (size_t)b * 4 * Cs_hbm, Cs_hbm, S.mask};
  bool done = false;
  if (start >= 0 && start < net.C) {
    if (ALL) done = near_walk<double, SCAN, SET_LDS>(net, io, wp, rid, rid - io.first, P, S, eq, p, start) == NEAR_DONE;
    else if (SCAN) done = near_or_full_walk<double, true>(net, io, wp, rid, rid - io.first, P, S, eq, p, start) == NEAR_DONE;
    else done = near_walk<double, false, SET_NEAR>(net, io, wp, rid, rid - io.first, P, S, eq, p, start) == NEAR_DONE;
  }
  if (ALL) {
    if (done && (SCAN || !(__builtin_amdgcn_readfirstlane(io.flags[rid - io.first]) & AM_UNDECIDED))) return;
    __syncthreads();
    if (!SCAN) {
      walk_ray64_body<1>(net, io, rid, b, wp, planes, eqb, Cs_hbm);
      const unsigned f = __builtin_amdgcn_readfirstlane(io.flags[rid - io.first]);
      if (!(f & AM_UNDECIDED)) return;
      if (threadIdx.x == 0) {
        atomicAdd(run, 1);
        for (int w = 0; w < AM_WHY_COUNT; ++w)
          if (f & AM_WHY_BIT(w)) atomicAdd(run + 1 + w, 1);
      }
      __syncthreads();
    }
    walk_fp64_body(net, scan_layout(io, net.C), rid, b, planes, eqb, Cs_hbm);
    return;
  }
  // (thread 0 wrote the flag in finish_region: the orientation may be undecided)
  if (threadIdx.x == 0 && (!done || (!SCAN && (io.flags[rid - io.first] & AM_UNDECIDED)))) near_left(left, b);
}
template __global__ void k_near64_multi<true, false>(const NetDev*, RegionIO, int, int, WalkParams, const double*, const double*, int, NearList, int*);
template __global__ void k_near64_multi<false, false>(const NetDev*, RegionIO, int, int, WalkParams, const double*, const double*, int, NearList, int*);
template __global__ void k_near64_multi<true, true>(const NetDev*, RegionIO, int, int, WalkParams, const double*, const double*, int, NearList, int*);
template __global__ void k_near64_multi<false, true>(const NetDev*, RegionIO, int, int, WalkParams, const double*, const double*, int, NearList, int*);

// ... of the listed slots (blocks stride over the list); a region it leaves
// undecided goes on the candidate scan's list and counts itself and its reasons.
template <int NW>
__global__ __launch_bounds__(64 * NW, 24 / NW) void k_walk_ray64_multi(const NetDev* nets, RegionIO io, int Wd, int rid0,
                                                              WalkParams wp, const double* planes, const double* eqb,
                                                              int Cs_hbm, NearList list, SlotList left) {
  const int total = min(*list.cnt, io.count);
  for (int i = blockIdx.x; i < total; i += gridDim.x) {
    const int b = list.slots[i], rid = rid0 + b;
    walk_ray64_body<NW>(nets[region_net(io, Wd, rid)], io, rid, b, wp, planes, eqb, Cs_hbm);
    // thread 0 wrote the region's flag (finish_region)
    if (threadIdx.x == 0) {
      const unsigned f = io.flags[rid - io.first];
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
template __global__ void k_walk_ray64_multi<2>(const NetDev*, RegionIO, int, int, WalkParams, const double*,
                                               const double*, int, NearList, SlotList);
template __global__ void k_walk_ray64_multi<4>(const NetDev*, RegionIO, int, int, WalkParams, const double*,
                                               const double*, int, NearList, SlotList);
template __global__ void k_walk_ray64_multi<8>(const NetDev*, RegionIO, int, int, WalkParams, const double*,
                                               const double*, int, NearList, SlotList);

}  // namespace am

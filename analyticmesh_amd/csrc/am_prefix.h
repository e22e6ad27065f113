// Constraint planes shared by activation prefix.
//
// The planes of hidden layer l + 1 depend on the activations of layers 1 .. l
// only, so regions whose masks agree there have them in common: on a network
// of D equal layers the surface meets about (l / D)^2 as many patterns of the
// first l layers as it has regions.  Instead of one masked affine chain per
// region, each distinct pattern ("prefix" of depth l) gets its layer l + 1
// planes once per march: a hash table maps prefixes to ids, one GEMM per layer
// computes the planes of the ids that are new, and the walks find a region's
// planes through the ids of its prefixes.  On the 4x256 network that is 29% of
// the chain's arithmetic (1/16 + 4/16 + 9/16 of a layer's product per region
// instead of 3), and a third of it with what is done again: its 7.2 GB of planes
// fill the storage, and the table starts over once or twice a march.
//
// The products run on the FP64 matrix cores in the canonical order:
// v_mfma_f64_16x16x4f64 rounds like four fused multiply-adds in ascending k
// (measured against the four-term fma chain on random operands, 51,200 of
// 51,200 results equal; no other order of the four is), and an inactive input
// adds fma(w, +0, acc) = acc.  With the bias as the initial accumulator the
// planes therefore equal the sequential chain's bit for bit, whatever tile a
// prefix falls into.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "am_kernels.h"

namespace am {

#define AM_PFX_SHIFT 12                 // ids per block of plane storage: 4096
#define AM_PFX_IDS (1 << AM_PFX_SHIFT)
#define AM_PFX_BLOCKS 1024              // blocks per depth
#define AM_PFX_EMPTY (~0ull)
#define AM_PT 8                         // prefixes per GEMM workgroup
#define AM_PKC 64                       // inputs in LDS at a time
#define AM_PXS (4 * AM_PT + 1)          // LDS row stride (doubles): x, y, z, c of each prefix

// Depth d = 1 .. nd = D - 1: prefixes of layers 1 .. d and the planes of layer
// d + 1.  Planes of an id: n (x, y) pairs, then n (z, c) pairs, unsigned.
struct PrefixDev {
  int nd;
  uint32_t cap_mask;
  unsigned long long* tab;      // [cap] prefix_key << 32 | a region with that prefix, or empty
  int* tab_id;                  // [cap] its id
  int* total;                   // [nd + 1] ids given per depth, AM_PFX_TS apart
  int* done;                    // [nd + 1] ids whose planes are there
  char* const* blk;             // [nd + 1][AM_PFX_BLOCKS] storage: AM_PFX_IDS records of planes, then of prefix_region
  StageClock* clk;
  int2* fresh;                  // [nd + 1][fresh_stride] the launch's new ids in order: (region, its place in the launch)
  int fresh_stride;
  int* rslot;                   // [regions of the launch][nd] table slots of a region's prefixes
  const double2* layer1;        // hidden layer 1's planes: n1 (x, y) pairs, n1 (z, c) pairs
  const double2* extra;         // the extra planes, likewise
  const double* Wp[AM_MAX_LINEAR];   // li >= 1: W_li^T padded, [>= n_li + 1][noutp[li]], zero past n_li, n_li+1
  const double* bp[AM_MAX_LINEAR];   // li >= 1: b_li padded
  int noutp[AM_MAX_LINEAR];
  const double* tmp[AM_MAX_TMS];     // transforms of skips, transposed and padded likewise
  int tmpo[AM_MAX_TMS];              // their padded row lengths
};

// Regions of one launch: ids, or first + i.
struct PrefixRegions {
  const uint32_t* reg_mask;
  const int* ids;
  int first, count;
  const int* dcount = nullptr;  // as in RegionIO
  int dbase = 0;
  const int2* lvl = nullptr;
  int lvl_bound = 0;
};

__device__ __forceinline__ double2* prefix_planes(const PrefixDev& pf, const NetDev& net, int d, int id) {
  char* b = pf.blk[(size_t)d * AM_PFX_BLOCKS + (id >> AM_PFX_SHIFT)];
  return reinterpret_cast<double2*>(b) + (size_t)(id & (AM_PFX_IDS - 1)) * 2 * net.nodes[d + 1];
}
// the region that added the id
__device__ __forceinline__ int* prefix_region(const PrefixDev& pf, const NetDev& net, int d, int id) {
  char* b = pf.blk[(size_t)d * AM_PFX_BLOCKS + (id >> AM_PFX_SHIFT)];
  return reinterpret_cast<int*>(b + (size_t)AM_PFX_IDS * 32 * net.nodes[d + 1]) + (id & (AM_PFX_IDS - 1));
}
inline size_t prefix_block_bytes(int n) { return (size_t)AM_PFX_IDS * (32 * (size_t)n + 4); }   // (a multiple of 16 KiB)

#define AM_PFX_TS 32                    // ints between two depths' totals (their own lines)
#define AM_PFX_REGIONS 256              // regions per block of k_prefix
// Finds or adds the prefixes of the launch's regions (grid: ceil(count / AM_PFX_REGIONS) x nd).
__global__ void k_prefix(NetDev net, PrefixDev pf, PrefixRegions rg);
// Planes of layer d + 1 for the new ids of depth d (grid: ceil(count / AM_PT) x ceil(n_out / 128) or ceil(n_out / 64),
// 256 threads, layer_lds bytes).  SKIPS: additive skips lead into the layer.
template <bool SKIPS>
__global__ void k_layer(NetDev net, PrefixDev pf, PrefixRegions rg, int d);
inline size_t layer_lds(int nin_max) { return ((size_t)nin_max + 32) * 4; }
__global__ void k_prefix_clear(PrefixDev pf, size_t cap);
__global__ void k_prefix_rehash(NetDev net, PrefixDev pf, const uint32_t* reg_mask, int d, int n);
struct PrefixPtrs {
  int n;
  int at[24];
  char* p[24];
};
__global__ void k_prefix_ptrs(char** blk, PrefixPtrs ptrs);
__global__ void k_pack_pairs(const double* xyz, const double* c, int n, double2* out);

// The near walk, and the walks over all constraints of what it leaves, on
// prefix planes.  ALL: the near walk takes every constraint (C <= AM_ALL_MAX).
// The near walk computes each region's face plane from layer
// D's planes (the output row's fma chain) and stores those of the regions it
// leaves in eq.
template <bool SCAN, bool ALL>
__global__ void k_near64(NetDev net, PrefixDev pf, RegionIO io, int rid0, WalkParams wp, double* eq,
                         int only_undecided, NearList left);
template <int NW>
__global__ void k_walk_ray64(NetDev net, PrefixDev pf, RegionIO io, int rid0, WalkParams wp, const double* eq,
                             NearList list, SlotList left);
__global__ void k_walk_fp64(NetDev net, PrefixDev pf, RegionIO io, int rid0, const int* count, const int* slots,
                            const double* eq, int quick);
__global__ void k_vertex_fp64(NetDev net, PrefixDev pf, RegionIO io, int rid0);

}  // namespace am

// Kernel interfaces of the marching engine (device side).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "am_limits.h"
#include "am_timer.h"

namespace am {

// Region store + the current level's candidate slots.
struct RegionIO {
  const uint32_t* reg_mask;   // [R][Wd]
  const int* reg_start;       // [R]   start plane (-1: seed)
  const double* reg_point;    // [R][3] seed point of the region
  int* reg_info;              // [R][AM_INFO_STRIDE]
  int* reg_tab;               // [R][vm + 1]
  double* reg_verts;          // [R][vm][3]
  int* reg_vpair;             // [R][vm][2]
  uint32_t* cand_mask;        // [count * vm][Wd]
  int* cand_start;            // [count * vm]   -2: no candidate in this slot
  double* cand_point;         // [count * vm][3]
  uint64_t* cand_hash;        // [count * vm] key hash sum of the candidate's mask (key_hash_sum)
  int first;                  // region id of blockIdx.x == 0
  int count;                  // regions in this launch
  int Cs;                     // stride of one SoA plane array in LDS
  int Csort;                  // power of two >= C (sort width)
  unsigned* flags;            // [count] per-region flags (bit 0: undecided in reduced precision)
  const int* ids;             // optional: region ids to process (FP64 re-decision); else first + blockIdx.x
  const int* dcount = nullptr;  // optional: ids past *dcount - dbase are not valid (a launch sized on
  int dbase = 0;                // the host for the worst case; blocks past the device count exit)
  const int2* lvl = nullptr;    // the level's first region and count on the device (first is not valid then)
  int lvl_bound = 0;            // largest count the launch is sized for
  StageClock* clk = nullptr;    // the march's stage times, if taken
  uint16_t* reg_jinv = nullptr; // optional [R][vm][9] bf16: per vertex the inverse of its 3x3 system
                                // from the reduced planes (columns for the new, walked and face plane),
                                // for the FP64 Newton step (a record with it has info[7] = 1)
};

// Regions of a launch whose count may be known on the device only: a level
// launched ahead of its size (lvl: first region and count, none when the count
// passes the bound it was launched for), or a list (dcount).
template <typename IO>
__device__ __forceinline__ int launch_count(const IO& io) {
  if (io.dcount) return min(io.count, *io.dcount - io.dbase);
  if (io.lvl) {
    const int n = io.lvl->y;
    return n <= io.lvl_bound ? min(io.count, n - io.dbase) : 0;
  }
  return io.count;
}
// First region of the launch (host: the value known there), and of its level.
template <typename IO>
__device__ __forceinline__ int launch_first(const IO& io, int host) {
  return io.lvl ? io.lvl->x + io.dbase : host;
}
__device__ __forceinline__ int level_first(const RegionIO& io) { return io.lvl ? io.lvl->x : io.first; }

// Regions of a level known on the device (as launch_count).
__device__ __forceinline__ int level_count(const int2* lvl, int bound) { return lvl->y <= bound ? lvl->y : 0; }

// Visited-set insertion of one level's candidates.
struct InsertIO {
  const uint32_t* cand_mask;  // [n][Wd]
  const uint64_t* cand_hash;  // [n] key_hash_sum of each candidate's mask
  const int* cand_start;      // [n]  -2 = empty slot
  const uint32_t* reg_mask;   // [R][Wd]
  uint32_t* table;            // [cap]  0xFFFFFFFF empty, 0x80000000|cand pending, else region id
  int* slot;                  // [n]  table slot of a pending candidate, -1: empty or already visited
  int n;
  int Wd;
  uint32_t cap_mask;
  unsigned long long* scan_state;  // [scan_words] tile states of the level's one-pass scan, cleared here
  int scan_words;
  const int2* lvl = nullptr;       // as in RegionIO: n is then vm slots per region of the level
  int lvl_bound = 0, vm = 0;
  int* zero = nullptr;             // two counters of the walks, cleared for the next level
  StageClock* clk = nullptr;
};

// Tiled FP64 chain: the planes of a tile of regions in HBM, for the walk kernel.
#define AM_CT 8                 // regions per chain workgroup
#define AM_CN (4 * AM_CT)       // chain columns: x, y, z, c of each region
#define AM_CXS (AM_CN + 1)      // LDS row stride (doubles) of the chain's layer buffer
#define AM_CR 16                // rows the operands are padded to
#define AM_CHAIN_MAXW 256       // widest layer the tiled chain takes
#define AM_RAY_WAVES 4          // waves per region in the ray-shooting walks
inline size_t chain_tile_lds(int maxw, int Wd) {
  return (size_t)(maxw + 1) * AM_CXS * 8 + (size_t)(maxw + 32) * 4 + (size_t)AM_CT * Wd * 4;
}
struct ChainIO {
  const uint32_t* reg_mask;   // [R][Wd]
  int first, count;           // regions of this launch
  int Cs;                     // stride of one component array in `planes` (>= C)
  double* planes;             // [count][4][Cs]: signed constraint planes, extras appended; entries of
                              // hidden layer 1 are not written (readers rebuild them from W0, b0, mask)
  double* eq;                 // [count][4]: output plane with iso subtracted
  const double* Wp[AM_MAX_LINEAR];  // li >= 1: W_li^T padded, [n_li][noutp[li]] (zero rows past n_out)
  const double* bp[AM_MAX_LINEAR];  // li >= 1: b_li padded to noutp[li]
  int noutp[AM_MAX_LINEAR];         // n_out rounded up to AM_CR
};

// A list of chunk-local slots filled by atomics (cnt zeroed before), with
// counters of what was listed: run[0] the entries, run[1 + w] those with
// reason bit w.
struct SlotList {
  int* cnt = nullptr;
  int* slots = nullptr;
  int* run = nullptr;
};

// Launch slots of the regions a near walk leaves, in no particular order.
struct NearList {
  int* cnt = nullptr;
  int* slots = nullptr;
};

// The regions and plane buffers of one tiled-chain launch.
struct ChainLevel {
  int first, count;           // regions first .. first + count - 1
  double* planes;             // [count][4][Cs]
  double* eq;                 // [count][4]
  const uint32_t* reg_mask;   // [R][Wd]
  StageClock* clk;
};

// NW waves: 4 for layers up to 128 wide (maxw), 8 up to 256.
template <int NW>
__global__ void k_chain_tile_fp64(NetDev net, ChainIO io, int maxw);
// A batch of networks (each region's network is the last word of its mask):
// tiles[b] = (network, first slot, regions, -) of one network.
template <int NW>
__global__ void k_chain_tile_fp64_multi(const NetDev* nets, const ChainIO* cios, ChainLevel lv, const int4* tiles,
                                        int maxw);
struct WalkParams;
// Batch-of-networks forms (region rid0 + b; its network is mask word Wd - 1;
// the scan's LDS layout follows each network's C, the launch is sized for the
// widest network).
__global__ void k_walk_fp64_multi(const NetDev* nets, RegionIO io, int Wd, int rid0, const int* count,
                                  const int* slots, const double* planes, const double* eq, int Cs_hbm);
template <bool SCAN, bool ALL>
__global__ void k_near64_multi(const NetDev* nets, RegionIO io, int Wd, int rid0, WalkParams wp, const double* planes,
                               const double* eq, int Cs_hbm, NearList left, int* run);
template <int NW>
__global__ void k_walk_ray64_multi(const NetDev* nets, RegionIO io, int Wd, int rid0, WalkParams wp,
                                   const double* planes, const double* eq, int Cs_hbm, NearList list, SlotList left);
__global__ void k_fill_i32(int* p, size_t n, int v);

// Weight layouts on the device (am_layout.hip): dst[j * ni + i] = src[i * cols + j]
// for i < rows, j < cols, +0 elsewhere (i < ni, j < nj); src float or double
// (f64), device-readable.  A copy with padding is cols = nj = 1.
void launch_transpose_pad(const void* src, int f64, int rows, int cols, double* dst, int ni, int nj, hipStream_t st);
void launch_transpose_pad(const void* src, int f64, int rows, int cols, float* dst, int ni, int nj, hipStream_t st);

}  // namespace am

// Back projection by image tiles, projection-data runs staged in LDS.
//
// What bounds it, and why it is built this way. A back projection gathers one
// projection-data run (up to 127 floats) per table entry and adds it to one
// image column. Read straight from memory (bp_kernel) nearly every gather
// misses L1 and, starting at any 4-byte address, moves three 128-byte lines:
// 7.2 cycles of a CU's L2 path for 64 lanes, against 2.3 for a run read from
// LDS at any alignment. So one workgroup owns a tile of 8 x 8 columns, copies
// the runs that cross it into LDS once and lets all 64 columns read them
// there (each staged run is used by about nine entries at mMR size).
//
// Measured at mMR size (4.2e8 entries, 837 x 252 x 344 bins, 344 x 344 x 127
// voxels): 10.8 ms with the column kernel, 5.65 ms with this one: three
// workgroups of 8 waves and 53 KB of LDS per CU. Two of 16 waves and 80 KB:
// 6.15 ms (5.97 with the reads of a group kept together); of 8 waves and
// 80 KB: 6.7; four of 8 waves and 40 KB: 6.3 (shorter lists, more padding);
// tiles of 12 x 8 columns: 5.75, of 16 x 8: 6.2. With the copies left out it
// takes 4.1 ms, without copies and barriers 3.6 (the LDS reads alone 3.2).
//
// In OSEM a subset's pass takes 0.32 ms, 21 of them 6.8: of that, 0.05 go to
// reading sensitivities and the estimate and writing it.
//
// Work: phases. The (segment, view) viewgrams of a subset are taken in family
// order; consecutive ones form a phase as long as the tangential positions
// that cross the tile fill no more than `rows` LDS rows. Per phase the
// workgroup copies the rows (loads that write LDS directly, all in flight at
// once), then every wave walks its columns' entries. Three workgroups share a
// CU, so two compute while one waits for its rows.
//
// LDS rows: `stride` floats per run, the run spread to one value per image
// plane (ppa planes per axial position: zeros between) and followed by zeros.
// An entry holds the byte offset of plane 0 in its run's row, so lane l of
// slot q reads plane 64 q + l; the stride is chosen so that planes the run
// does not reach fall on zeros (of its own row, or of the end of the row
// before it): no test, clamp or select, and the sum is the column table's,
// term by term and bit for bit.
//
// Entries: per (phase, column) a list padded to groups of 4 with entries that
// read the leading zeros with weight 0. Offsets and weights are two arrays;
// each row of 16 lanes loads the same 16 consecutive entries and a group
// takes its four by DPP broadcast inside the add and the multiply-add, so an
// entry costs one address add, one two-slot LDS read and a multiply-add per
// slot: 3 vector instructions for 128 planes, no scalar ones.
//
// TOF: every (element, TOF bin it reaches) is an entry of its own, and every
// TOF bin of a (segment, view) a viewgram with rows of its own: 2.1e9 terms at
// mMR size with 11 TOF bins (up to 5 per element). 24.4 ms, against 45.7 with
// the stored back records, whose five gathers per element also went to L2; per
// term it costs what the non-TOF kernel does. The table is 17 GB where the
// records were 13.5, and takes 0.12 s more to make.
//
// One workgroup takes its time however few there are: images of few tiles (60 x
// 60 columns: 0.25 to 0.8 times as fast) stay with the column kernels
// (mi_ctx::min_tiles in pmrt_capi.cpp).
#include <hip/hip_runtime.h>

#include <cstdint>

#include "pmrt_device.hpp"
#include "pmrt_kernels.hpp"

namespace mi {

namespace {

using namespace dev;

constexpr int kTileCpw = kTileCols / kTileWaves;  // columns per wave

// The matrix element of a family as the tile table sees it: tile, line of the
// tile, the line's plane of axial position 0; false when it reaches no image
// plane.
struct TileElem {
  int t, c, k;
};
__device__ inline bool tile_elem(const Family& f, int coords, const ImageDims& d, const TileShape& S, TileElem& E) {
  int x, y, z, xo, yo;
  decode(coords, x, y, z);
  inplane_any_op(f.inplane, x, y, xo, yo);
  const int cx = xo - d.min_x, cy = yo - d.min_y;
  E.k = f.zsign * z + f.zadd0 - d.min_z;
  const int last = E.k + f.ppa * (f.nax - 1);
  if (cx < 0 || cx >= d.nx || cy < 0 || cy >= d.ny || last < 0 || E.k >= d.nz) return false;
  E.t = (cy / S.ty) * S.ntx + cx / S.tx;
  E.c = (cy % S.ty) * S.tx + cx % S.tx;
  if (S.par == 2) {
    E.c = 2 * E.c + (E.k & 1);
    E.k >>= 1;
  }
  return true;
}

// The terms of a family's element e: its weight (non-TOF), or its weight in
// each TOF bin it reaches, from the stored forward record (fp_rec, W weights
// from bin c on; TOF families have rows of their own). fn(bin, weight).
template <class F>
__device__ inline void element_terms(const int32_t* __restrict__ fp_rec, int W, int64_t pool_index, int weight, F&& fn) {
  if (!fp_rec) {
    fn(0, weight);
    return;
  }
  const int32_t* r = fp_rec + pool_index * (2 + W);
  const int c = r[0] >> 20;
  for (int j = 0; j < W; ++j)
    if (__int_as_float(r[2 + j]) != 0.F) fn(c + j, r[2 + j]);
}

// pass 1, one wave per family: the tangential positions of every (tile, view,
// TOF bin) and, over all elements, the most planes a row needs after a run's
// start (need[0]: nz - k) and before its end (need[1]: run length + k)
__global__ void __launch_bounds__(kWave) tile_range_kernel(const Family* __restrict__ fams,
                                                           const int2* __restrict__ fam_pos, int nfam,
                                                           const int2* __restrict__ pool,
                                                           const int32_t* __restrict__ fp_rec, int W, ImageDims d,
                                                           TileShape S, int nviews, int ntof, int2* __restrict__ rng,
                                                           int* __restrict__ need) {
  const int fi = blockIdx.x;
  if (fi >= nfam) return;
  const Family f = fams[fi];
  const int2 pos = fam_pos[fi];  // view, tangential index
  const int lane = static_cast<int>(threadIdx.x);
  int after = 0, before = 0;
  for (int e0 = 0; e0 < f.row_len; e0 += kWave) {
    const int e = e0 + lane;
    TileElem E;
    const int64_t pi = static_cast<int64_t>(f.row_start) + (e < f.row_len ? e : 0);
    const bool ok = e < f.row_len && tile_elem(f, pool[pi].x, d, S, E);
    uint32_t bins = 0;  // the element's TOF bins
    if (ok) {
      after = max(after, (d.nz + S.par - 1) / S.par - E.k);
      before = max(before, f.ppa / S.par * (f.nax - 1) + 1 + E.k);
      element_terms(fp_rec, W, pi, 0, [&](int bin, int) { bins |= 1U << bin; });
    }
    // neighbouring elements of a row lie mostly in one tile and the same bins:
    // one update per run of them
    const int t = ok ? E.t : -1;
    const int prev_t = __shfl_up(t, 1, kWave);
    const uint32_t prev_b = __shfl_up(bins, 1, kWave);
    if (ok && (lane == 0 || prev_t != t || (bins & ~prev_b))) {
      for (int k = 0; k < ntof; ++k) {
        if (!(bins >> k & 1)) continue;
        int2* r = rng + (static_cast<int64_t>(t) * nviews + pos.x) * ntof + k;
        // (a stale value read here only costs the atomic)
        if (pos.y < __hip_atomic_load(&r->x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMin(&r->x, pos.y);
        if (pos.y > __hip_atomic_load(&r->y, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(&r->y, pos.y);
      }
    }
  }
  for (int o = kWave / 2; o > 0; o >>= 1) {
    after = max(after, __shfl_xor(after, o, kWave));
    before = max(before, __shfl_xor(before, o, kWave));
  }
  // most families do not raise the maxima: read them first, or every wave
  // would queue on one address
  if (lane == 0 && before > 0) {
    if (after > __hip_atomic_load(need, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(need, after);
    if (before > __hip_atomic_load(need + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(need + 1, before);
  }
}

// pass 2, one thread per (tile, subset): its units dealt to phases. FILL 0:
// slot[tile][unit] = phase within (tile, subset) << 16 | first row, and the
// numbers of phases and rows; 1: the rows and the first row of every phase. A
// run's planes before its start fall on the end of the row before it: after a
// longer run (of another segment) a row of zeros lies between.
template <bool FILL>
__global__ void tile_phase_kernel(const int4* __restrict__ units, const int32_t* __restrict__ unit_off, int nsub,
                                  int ntiles, int nunits, int nrng, const int2* __restrict__ rng, int rows,
                                  uint32_t* __restrict__ slot, uint32_t* __restrict__ nphase,
                                  uint32_t* __restrict__ nrow, const uint32_t* __restrict__ phase_off,
                                  const uint32_t* __restrict__ row_off, int2* __restrict__ row,
                                  uint32_t* __restrict__ phase_row, int* __restrict__ bad) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nsub * ntiles) return;
  const int t = i / nsub, s = i - t * nsub;
  int ph = -1, used = 0, prev = 0;
  uint32_t n = 0;
  for (int u = unit_off[s]; u < unit_off[s + 1]; ++u) {
    const int4 U = units[u];  // device offset, nax, ppa (of a line), index among the tile's ranges
    const int2 r = rng[static_cast<int64_t>(t) * nrng + U.w];
    const int T = r.y - r.x + 1;
    if (r.y < r.x) continue;
    const int len = U.z * (U.y - 1) + 1;
    int gap = prev > len;
    if (T > rows) *bad = 1;
    if (ph < 0 || used + gap + T > rows) {
      ++ph;
      used = gap = 0;
      if (FILL) phase_row[phase_off[i] + ph] = row_off[i] + n;
    }
    prev = len;
    if (FILL) {
      int2* o = row + row_off[i] + n;
      if (gap) *o++ = make_int2(0, 1 << 16);  // an empty run
      for (int k = 0; k < T; ++k) o[k] = make_int2(U.x + (r.x + k) * U.y, U.y | U.z << 16);
    } else {
      slot[static_cast<int64_t>(t) * nunits + u] = static_cast<uint32_t>(ph) << 16 | (used + gap);
    }
    used += gap + T;
    n += gap + T;
  }
  if (!FILL) {
    nphase[i] = ph + 1;
    nrow[i] = n;
    if (ph + 1 > 65535) *bad = 1;
  }
}

// passes 3 and 4, one wave per family of subset s: the number of entries of
// every (phase, column), then every term's key and entry at slot
// (element offset - first) * span + its rank, in family order, element order,
// bin order (slots without a term get the last key)
template <bool COUNT>
__global__ void __launch_bounds__(kWave) tile_entries_kernel(const Family* __restrict__ fams,
                                                             const int2* __restrict__ fam_pos, int fam_begin,
                                                             int fam_end, int ntang, const int2* __restrict__ pool,
                                                             const int32_t* __restrict__ fp_rec, int W, int ntof,
                                                             int subset, ImageDims d, TileArgs A, int nunits,
                                                             const uint32_t* __restrict__ slot,
                                                             uint32_t* __restrict__ counts, uint32_t none, int span,
                                                             const int64_t* __restrict__ fam_entry_off, int64_t first,
                                                             uint32_t* __restrict__ keys, int2* __restrict__ raw) {
  const int fi = fam_begin + blockIdx.x;
  if (fi >= fam_end) return;
  const Family f = fams[fi];
  const int2 pos = fam_pos[fi];
  const int unit = fi / ntang * ntof;
  const int64_t base = COUNT ? 0 : fam_entry_off[fi] - first;
  for (int e = threadIdx.x; e < f.row_len; e += kWave) {
    const int64_t pi = static_cast<int64_t>(f.row_start) + e;
    const int2 el = pool[pi];
    TileElem E;
    int n = 0;
    if (tile_elem(f, el.x, d, A.shape, E))
      element_terms(fp_rec, W, pi, el.y, [&](int bin, int weight) {
        const uint32_t sl = slot[static_cast<int64_t>(E.t) * nunits + unit + bin];
        const uint32_t ph = A.phase_off[static_cast<int64_t>(E.t) * A.nsub + subset] + (sl >> 16);
        const uint32_t key = ph * A.shape.lines() + E.c;
        if (COUNT) {
          atomicAdd(&counts[key], 1U);
        } else {
          const int2 r = A.rng[(static_cast<int64_t>(E.t) * A.nviews + pos.x) * ntof + bin];
          const int row = static_cast<int>(sl & 0xffff) + pos.y - r.x;
          keys[(base + e) * span + n] = key;
          raw[(base + e) * span + n] = make_int2(4 * (A.lead + row * A.stride - E.k), weight);
        }
        ++n;
      });
    if (!COUNT)
      for (; n < span; ++n) keys[(base + e) * span + n] = none;
  }
}

// groups of 4 entries of every list: of lists in lockstep the most of them
__global__ void tile_groups_kernel(const uint32_t* __restrict__ counts, int64_t n, int lockstep,
                                   uint32_t* __restrict__ groups, int* __restrict__ bad) {
  for (int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; i < n;
       i += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    uint32_t g = (counts[i] + 3) / 4;
    if (lockstep > 1) {
      const int64_t first = i / lockstep * lockstep;
      for (int64_t j = first; j < first + lockstep && j < n; ++j) g = max(g, (counts[j] + 3) / 4);
    }
    groups[i] = g;
    if (g > 255 && lockstep == 1) *bad = 1;
  }
}

// per (phase, wave): first group, the group counts of its columns (one byte
// each) or of its lines in lockstep, and the phase's first row; `slack` more
// phases without groups close the list
__global__ void tile_headers_kernel(const uint32_t* __restrict__ groups, const uint32_t* __restrict__ group_off,
                                    const uint32_t* __restrict__ phase_row, uint32_t total_rows, int64_t nphase,
                                    int64_t slack, TileShape S, uint4* __restrict__ hdr) {
  const int lw = S.lines_of_wave();
  for (int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; i < (nphase + slack) * kTileWaves;
       i += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const int64_t p = i / kTileWaves;
    if (p >= nphase) {
      hdr[i] = make_uint4(0, 0, 0, total_rows);
      continue;
    }
    uint32_t c[2] = {0, 0};
    if (S.lockstep() > 1) c[0] = groups[i * lw];
    else
      for (int j = 0; j < kTileCpw; ++j) c[j / 4] |= groups[i * lw + j] << (8 * (j % 4));
    hdr[i] = make_uint4(group_off[i * lw], c[0], c[1], phase_row[p]);
  }
}

// groups of every tile (its work)
__global__ void tile_work_kernel(const uint32_t* __restrict__ group_off, const uint32_t* __restrict__ phase_off, int nsub,
                                 int ntiles, int lines, uint32_t* __restrict__ work) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= ntiles) return;
  const int64_t a = phase_off[static_cast<int64_t>(t) * nsub], b = phase_off[static_cast<int64_t>(t + 1) * nsub];
  work[t] = group_off[b * lines] - group_off[a * lines];
}

// sorted term r -> its place: the groups of a list follow one another, those
// of lists in lockstep alternate (a list has a few tens of entries)
__global__ void tile_place_kernel(const uint32_t* __restrict__ keys, const uint32_t* __restrict__ idx,
                                  const int2* __restrict__ raw, const uint32_t* __restrict__ group_off, uint32_t none,
                                  int lockstep, int64_t n, int32_t* __restrict__ off, float* __restrict__ w) {
  for (int64_t r = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; r < n;
       r += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const uint32_t key = keys[r];
    if (key == none) continue;
    // the list's first term among the wave's, or else by bisection before them
    const int lane = static_cast<int>(threadIdx.x % kWave);
    const bool head = r == 0 || keys[r - 1] != key;
    const uint64_t heads = __ballot(head) & (~0ull >> (kWave - 1 - lane));
    int64_t rank;
    if (heads) {
      rank = lane - (63 - __builtin_clzll(heads));
    } else {
      int64_t lo = 0, hi = r - lane - 1;  // keys[hi] == key
      for (int64_t step = 64; hi > 0; step *= 2) {
        const int64_t at = hi > step ? hi - step : 0;
        if (keys[at] != key) { lo = at + 1; break; }
        hi = at;
      }
      while (lo < hi) {
        const int64_t mid = (lo + hi) / 2;
        if (keys[mid] == key) hi = mid;
        else lo = mid + 1;
      }
      rank = r - hi;
    }
    const int2 E = raw[idx[r]];
    const uint32_t line = key % lockstep;
    const int64_t at = 4 * (group_off[key - line] + rank / 4 * lockstep + line) + rank % 4;
    off[at] = E.x;
    w[at] = __int_as_float(E.y);
  }
}

// lane j of the row of 16 lanes, in every lane of the row
template <int J>
__device__ inline int row_bcast(int v) {
  return __builtin_amdgcn_update_dpp(0, v, 0x150 + J, 0xf, 0xf, true);
}
// lane (i + 4) % 16 of the row of 16 lanes
__device__ inline int row_next4(int v) { return __builtin_amdgcn_update_dpp(0, v, 0x120 + 12, 0xf, 0xf, true); }

// acc + lane J's w of the row times p, in one rounding; the instruction takes
// the broadcast itself (the compiler moves it to a register first when two
// slots share the weight). A DPP read needs two wait states after a VALU write
// of w, which the compiler does not count across asm: the first of a group
// brings them.
template <int J>
__device__ inline void add_bcast(float& acc, int w, float p) {
  if constexpr (J == 0)
    asm("s_nop 1\n\tv_fmac_f32_dpp %0, %1, %2 row_newbcast:0 row_mask:0xf bank_mask:0xf" : "+v"(acc) : "v"(w), "v"(p));
  else if constexpr (J == 1)
    asm("v_fmac_f32_dpp %0, %1, %2 row_newbcast:1 row_mask:0xf bank_mask:0xf" : "+v"(acc) : "v"(w), "v"(p));
  else if constexpr (J == 2)
    asm("v_fmac_f32_dpp %0, %1, %2 row_newbcast:2 row_mask:0xf bank_mask:0xf" : "+v"(acc) : "v"(w), "v"(p));
  else
    asm("v_fmac_f32_dpp %0, %1, %2 row_newbcast:3 row_mask:0xf bank_mask:0xf" : "+v"(acc) : "v"(w), "v"(p));
}

// an ordered (not invariant) load: it stays behind the copy of the registers it overwrites
__device__ inline int entry_word(const char* base, unsigned off) {
  return *(const MI_AS_GLOBAL int*)((const MI_AS_GLOBAL char*)base + off);
}

// the next four entries (lanes 0-3 of every row hold them) added to one column
template <int NSLOT>
__device__ inline void tile_group(int off, int w, const char* lds, int lane4, float (&acc)[NSLOT]) {
  const int o[4] = {row_bcast<0>(off), row_bcast<1>(off), row_bcast<2>(off), row_bcast<3>(off)};
  float v[4][NSLOT];
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int q = 0; q < NSLOT; ++q) v[j][q] = *reinterpret_cast<const float*>(lds + (lane4 + o[j]) + 256 * q);
  __builtin_amdgcn_sched_barrier(0);  // all reads of the group in flight before the first is waited for
#pragma unroll
  for (int q = 0; q < NSLOT; ++q) add_bcast<0>(acc[q], w, v[0][q]);
#pragma unroll
  for (int q = 0; q < NSLOT; ++q) add_bcast<1>(acc[q], w, v[1][q]);
#pragma unroll
  for (int q = 0; q < NSLOT; ++q) add_bcast<2>(acc[q], w, v[2][q]);
#pragma unroll
  for (int q = 0; q < NSLOT; ++q) add_bcast<3>(acc[q], w, v[3][q]);
}

// TOF: the sums of kTileSumPhases phases are added to the voxel's sum
// together. An element has a term per TOF bin here, so that one chain of
// additions would be as many times longer than the elements' (and its rounding
// error larger) as an element reaches bins.
constexpr uint32_t kTileSumPhases = 8;

template <int MODE, int NSLOT, bool TOF>
__device__ __forceinline__ void tile_sums(const TileArgs& A, int t, int sb, int se, const float* __restrict__ proj,
                                          float* __restrict__ img, const ImageDims& d, const BpData& data) {
  extern __shared__ float tile_lds[];
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) / kWave);
  const int lane = static_cast<int>(threadIdx.x % kWave);
  const int lane4 = 4 * lane;
  for (int i = threadIdx.x; i < A.lds_floats; i += kWave * kTileWaves) tile_lds[i] = 0.F;
  float acc[kTileCpw][NSLOT], sum[kTileCpw][NSLOT];
#pragma unroll
  for (int c = 0; c < kTileCpw; ++c)
#pragma unroll
    for (int q = 0; q < NSLOT; ++q) acc[c][q] = sum[c][q] = 0.F;
#if defined(__HIP_DEVICE_COMPILE__)
  const char* lds = reinterpret_cast<const char*>(tile_lds);
  const int l16 = lane % 16;
  const uint32_t p0 = as_const(A.phase_off)[static_cast<int64_t>(t) * A.nsub + sb];
  const uint32_t p1 = as_const(A.phase_off)[static_cast<int64_t>(t) * A.nsub + se];
  // headers two phases ahead and rows one phase ahead, by vector loads (scalar
  // loads in flight would make every LDS wait a full wait); lane l has the
  // wave's row l
  int zero = 0;
  asm volatile("" : "+v"(zero));
  const uint4* hp = A.hdr + static_cast<int64_t>(p0) * kTileWaves + wave + zero;
  uint4 h = hp[0], h1 = hp[kTileWaves];
  int2 rw = A.row[h.w + wave + kTileWaves * lane];
  for (uint32_t p = p0; p < p1; ++p) {
    const uint32_t group0 = __builtin_amdgcn_readfirstlane(h.x);
    const uint32_t cnt[2] = {static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(h.y)),
                             static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(h.z))};
    const int nrow = static_cast<int>(__builtin_amdgcn_readfirstlane(h1.w) - __builtin_amdgcn_readfirstlane(h.w));
    const int2 cur = rw;
    const char* po = reinterpret_cast<const char*>(A.off + 4 * static_cast<int64_t>(group0));
    const char* pw = reinterpret_cast<const char*>(A.w + 4 * static_cast<int64_t>(group0));
    unsigned at = 4 * l16;  // byte offset of this lane's entry
    __syncthreads();        // the previous phase's rows have been read
    float* dst = tile_lds + A.lead + wave * A.stride;
    for (int l = 0, r = wave; r < nrow; ++l, r += kTileWaves, dst += kTileWaves * A.stride) {
      const int np = __builtin_amdgcn_readlane(cur.y, l);
      const __amdgpu_buffer_rsrc_t run =
          run_buffer(as_const(proj), static_cast<unsigned>(__builtin_amdgcn_readlane(cur.x, l)), np & 0xffff);
#pragma unroll
      for (int q = 0; q < NSLOT; ++q) {
        // this lane's plane in the run; outside [0, 4 nax) the buffer reads 0
        const int z = kWave * q + lane;
        int v = 4 * z;
        if ((np >> 16) == 2) v = z & 1 ? -4 : 2 * z;
        else if ((np >> 16) > 2) v = z % (np >> 16) ? -4 : z / (np >> 16) * 4;
        if (kWave * q < A.longest)
          __builtin_amdgcn_raw_ptr_buffer_load_lds(run, (__attribute__((address_space(3))) void*)(dst + kWave * q), 4,
                                                   whole_offset(v), 0, 0, 0);
      }
    }
    h = h1;
    hp += kTileWaves;
    h1 = hp[kTileWaves];
    rw = A.row[h.w + wave + kTileWaves * lane];
    int off = entry_word(po, at), w = entry_word(pw, at);
    at += 64;
    int off1 = entry_word(po, at), w1 = entry_word(pw, at);
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): this wave's rows are in LDS
    __syncthreads();
    int left = 4;  // groups left in the current chunk
#pragma unroll
    for (int c = 0; c < kTileCpw; ++c) {
      for (uint32_t n = (cnt[c / 4] >> (8 * (c % 4))) & 255; n > 0; --n) {
        tile_group<NSLOT>(off, w, lds, lane4, acc[c]);
        if (--left == 0) {
          // copied by hand, so that the next chunk's loads, requested after it,
          // can write off1 and w1 themselves (a copy that the compiler places
          // comes after the loads and waits for them)
          asm volatile("v_mov_b32 %0, %2\n\tv_mov_b32 %1, %3\n\ts_nop 1"
                       : "=&v"(off), "=&v"(w)
                       : "v"(off1), "v"(w1)
                       : "memory");
          at += 64;
          off1 = entry_word(po, at);
          w1 = entry_word(pw, at);
          left = 4;
        } else {
          off = row_next4(off);
          w = row_next4(w);
        }
      }
    }
    if constexpr (TOF) {
      if ((p - p0) % kTileSumPhases == kTileSumPhases - 1) {
#pragma unroll
        for (int c = 0; c < kTileCpw; ++c)
#pragma unroll
          for (int q = 0; q < NSLOT; ++q) {
            sum[c][q] += acc[c][q];
            acc[c][q] = 0.F;
          }
      }
    }
  }
  if constexpr (TOF) {
#pragma unroll
    for (int c = 0; c < kTileCpw; ++c)
#pragma unroll
      for (int q = 0; q < NSLOT; ++q) acc[c][q] += sum[c][q];
  }
#endif
  const TileShape& S = A.shape;
  const int x0 = (t % S.ntx) * S.tx, y0 = (t / S.ntx) * S.ty;
#pragma unroll
  for (int c = 0; c < kTileCpw; ++c) {
    const int cc = wave * kTileCpw + c;
    const int cx = x0 + cc % S.tx, cy = y0 + cc / S.tx;
    if (cx >= d.nx || cy >= d.ny) continue;
    const int col = cy * d.nx + cx;
#pragma unroll
    for (int q = 0; q < NSLOT; ++q) {
      const int z = lane + kWave * q;
      if (z >= d.nzp) continue;
      const int64_t idx = static_cast<int64_t>(col) * d.nzp + z;
      if constexpr (MODE == BP_PLAIN) {
        as_global(img)[idx] = z < d.nz ? acc[c][q] : 0.F;
      } else {
        if (z < d.nz) {
          const float u = osem_factor(acc[c][q], as_const(data.sens)[idx], data.threshold, data.thr_lo, data.thr_hi);
          as_global(data.estimate)[idx] = as_global(data.estimate)[idx] * u;
          if (data.update) as_global(data.update)[idx] = u;
        }
      }
    }
  }
}

template <int MODE, int NSLOT, bool TOF>
__global__ void __launch_bounds__(kWave* kTileWaves) bp_tile_kernel(TileArgs A, int sb, int se,
                                                                    const float* __restrict__ proj,
                                                                    float* __restrict__ img, ImageDims d, BpData data,
                                                                    int chunk) {
  const int b = xcd_chunk_remap(static_cast<int>(blockIdx.x), chunk);
  if (b >= A.ntiles) return;
  tile_sums<MODE, NSLOT, TOF>(A, as_const(A.order)[b], sb, se, proj, img, d, data);
}

// tiles of several problems, heaviest first, one subset
template <int MODE, int NSLOT>
__global__ void __launch_bounds__(kWave* kTileWaves) bp_tile_batch_kernel(const ProblemDesc* __restrict__ descs,
                                                                          const TileArgs* __restrict__ tiles,
                                                                          const WorkItem* __restrict__ work, int nwork,
                                                                          int subset, int threshold) {
  const int b = xcd_chunk_remap(static_cast<int>(blockIdx.x), kTileXcdChunk);
  if (b >= nwork) return;
  const int p = __builtin_amdgcn_readfirstlane(work[b].problem);
  const int t = __builtin_amdgcn_readfirstlane(work[b].index);
  const ProblemDesc& P = descs[p];
  BpData bd{};
  bd.sens = P.sens ? as_const(P.sens)[subset] : nullptr;
  bd.estimate = P.estimate;
  bd.update = nullptr;
  bd.threshold = threshold;
  bd.thr_lo = P.thr_lo;
  bd.thr_hi = P.thr_hi;
  const TileArgs A = tiles[p];
  tile_sums<MODE, NSLOT, false>(A, t, subset, subset + 1, P.bp_in, P.bp_out, P.d, bd);
}

// ---- short images
//
// A wave holds 64 / LPC lines of LPC lanes, LPC >= the planes of a line: an
// image of up to 16 or 32 planes. With two planes per axial position (span 1)
// an entry reaches the planes of one parity, so each parity is a line of its
// own, its planes l of [0, LPC) the image's PAR l + parity, and the rows need
// no zeros between. One wave has one set of lines, whose lists are padded to
// the same length.
//
// What bounds it: with short lines the rows are short too (8 floats for 8
// rings) and a phase has hundreds of them, so that copying them takes about as
// long as adding the entries. Copy waves fill one buffer while the others read
// the other; a copy wave's lanes cover the rows end to end (64 lanes write 64
// consecutive floats), each with its own address from the row list.
//
// Measured, all subsets, against the column kernels: 8 rings, span 1, 128^2
// columns 182 -> 34 us, 256^2 and all ring differences 2670 -> 475; 8 rings,
// span 3, 69 -> 28; 16 rings, span 1, 1755 -> 460; span 3, 734 -> 443; 4 rings,
// 64^2, 48 -> 17 us. Without the additions it takes as long: requests to memory
// bound it (copies by 4-byte lanes, entries of 8 bytes). Lists of lines in
// lockstep alternate by groups, so that one load covers 128 bytes of entries
// and not pieces of 16 (8 rings, 256^2: 585 -> 507 us); the steps from copy to
// copy by a carry instead of a division: 507 -> 475. 8 copy waves: the same.

template <int CTRL>
__device__ inline int dpp_all(int v) { return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xf, 0xf, true); }

// acc + lane J's w of the quad times p (see add_bcast)
template <int J>
__device__ inline void add_quad(float& acc, int w, float p) {
  if constexpr (J == 0)
    asm("s_nop 1\n\tv_fmac_f32_dpp %0, %1, %2 quad_perm:[0,0,0,0] row_mask:0xf bank_mask:0xf" : "+v"(acc) : "v"(w), "v"(p));
  else if constexpr (J == 1)
    asm("v_fmac_f32_dpp %0, %1, %2 quad_perm:[1,1,1,1] row_mask:0xf bank_mask:0xf" : "+v"(acc) : "v"(w), "v"(p));
  else if constexpr (J == 2)
    asm("v_fmac_f32_dpp %0, %1, %2 quad_perm:[2,2,2,2] row_mask:0xf bank_mask:0xf" : "+v"(acc) : "v"(w), "v"(p));
  else
    asm("v_fmac_f32_dpp %0, %1, %2 quad_perm:[3,3,3,3] row_mask:0xf bank_mask:0xf" : "+v"(acc) : "v"(w), "v"(p));
}

// N groups of four entries of every line of the wave (each quad of lanes holds
// its line's), all reads in flight before the first is waited for
template <int N>
__device__ inline void short_groups(const int* off, const int* w, const char* lds, int lane4, float& acc) {
  float v[N][4];
#pragma unroll
  for (int j = 0; j < N; ++j) {
    v[j][0] = *reinterpret_cast<const float*>(lds + (lane4 + dpp_all<0x00>(off[j])));
    v[j][1] = *reinterpret_cast<const float*>(lds + (lane4 + dpp_all<0x55>(off[j])));
    v[j][2] = *reinterpret_cast<const float*>(lds + (lane4 + dpp_all<0xaa>(off[j])));
    v[j][3] = *reinterpret_cast<const float*>(lds + (lane4 + dpp_all<0xff>(off[j])));
  }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int j = 0; j < N; ++j) {
    add_quad<0>(acc, w[j], v[j][0]);
    add_quad<1>(acc, w[j], v[j][1]);
    add_quad<2>(acc, w[j], v[j][2]);
    add_quad<3>(acc, w[j], v[j][3]);
  }
}

constexpr int kShortThreads = kWave * (kTileWaves + kShortCopyWaves);

// SUM2: the sum of a phase is added to the voxel's sum as a whole (shorter
// chains of additions); otherwise all terms one by one, as the column kernel
// for one plane per axial position.
template <int MODE, int LPC, int PAR, bool SUM2, int NSET>  // NSET: sets of lines of a wave
__global__ void __launch_bounds__(kShortThreads, 6) bp_tile_short_kernel(TileArgs A, int sb, int se,
                                                                      const float* __restrict__ proj,
                                                                      float* __restrict__ img, ImageDims d, BpData data,
                                                                      int chunk) {
  extern __shared__ float tile_lds[];
  const int b = xcd_chunk_remap(static_cast<int>(blockIdx.x), chunk);
  if (b >= A.ntiles) return;
  const int t = as_const(A.order)[b];
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) / kWave);
  const int lane = static_cast<int>(threadIdx.x % kWave);
  for (int i = threadIdx.x; i < 2 * A.lead; i += kShortThreads)
    tile_lds[i < A.lead ? i : A.buffer + i - A.lead] = 0.F;
  float acc[NSET], sum[NSET];
#pragma unroll
  for (int s = 0; s < NSET; ++s) acc[s] = sum[s] = 0.F;
#if defined(__HIP_DEVICE_COMPILE__)
  const uint32_t p0 = as_const(A.phase_off)[static_cast<int64_t>(t) * A.nsub + sb];
  const uint32_t p1 = as_const(A.phase_off)[static_cast<int64_t>(t) * A.nsub + se];
  int zero = 0;
  asm volatile("" : "+v"(zero));
  const int cw = wave - kTileWaves;
  const uint4* hp = A.hdr + static_cast<int64_t>(p0) * kTileWaves + zero;
  if (cw >= 0) {
    const __amdgpu_buffer_rsrc_t all =
        __builtin_amdgcn_make_buffer_rsrc((void*)proj, static_cast<short>(0), static_cast<int>(A.proj_bytes), 0x00020000);
    // (past the phase's last row a copy writes the next phase's floats into the
    // buffer's slack)
    const ShortCopyWalk walk(cw, lane, A.stride, A.div_stride);
    int2 ra[kShortBatch], rb[kShortBatch];
    int row = 0, row_at = 0, at = 0;  // of the next request, of the next copy
    auto request = [&](int2 (&r)[kShortBatch], uint32_t base) {
      const int2* list = A.row + base;
#pragma unroll
      for (int j = 0; j < kShortBatch; ++j) {
        r[j] = list[row];
        row += walk.row_step + walk.carry(row_at);
      }
    };
    auto copy = [&](const int2 (&r)[kShortBatch], int first, int n, float* buf) {
#pragma unroll
      for (int j = 0; j < kShortBatch; ++j) {
        const int f = (cw + kShortCopyWaves * (first + j)) * kWave;
        if (f < n) {
          const int nax = r[j].y & 0xffff, ppa = r[j].y >> 16;
          int a = at;
          bool ok = true;
          if (PAR == 1 && ppa > 1) {
            a = at / ppa;
            ok = a * ppa == at;
          }
          ok = ok && a < nax;
          const int v = ok ? static_cast<int>(4U * static_cast<unsigned>(r[j].x + a)) : -4;  // -4: reads 0
          __builtin_amdgcn_raw_ptr_buffer_load_lds(all, (__attribute__((address_space(3))) void*)(buf + f), 4,
                                                   whole_offset(v), 0, 0, 0);
          walk.carry(at);
        }
      }
    };
    uint32_t row0 = hp[0].w, row1 = hp[kTileWaves].w;
    int nrow = static_cast<int>(__builtin_amdgcn_readfirstlane(row1) - __builtin_amdgcn_readfirstlane(row0));
    row = walk.row_first;
    row_at = walk.at_first;
    request(ra, row0);
    int which = 0;
    for (uint32_t p = p0; p <= p1; ++p) {
      if (p < p1) {
        float* buf = tile_lds + A.lead + which * A.buffer;
        which ^= 1;
        const int n = nrow * A.stride;
        auto any = [&](int first) { return (cw + kShortCopyWaves * first) * kWave < n; };
        at = walk.at_first;
        for (int first = 0; any(first); first += 2 * kShortBatch) {
          const bool second = any(first + kShortBatch);
          if (second) request(rb, row0);
          copy(ra, first, n, buf);
          if (any(first + 2 * kShortBatch)) request(ra, row0);
          if (second) copy(rb, first + kShortBatch, n, buf);
        }
        // the next phase's first batch
        hp += kTileWaves;
        row0 = row1;
        row1 = hp[kTileWaves].w;
        nrow = static_cast<int>(__builtin_amdgcn_readfirstlane(row1) - __builtin_amdgcn_readfirstlane(row0));
        row = walk.row_first;
        row_at = walk.at_first;
        request(ra, row0);
        __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): this wave's rows are in LDS
      }
      __syncthreads();
    }
    return;
  }
  const char* lds = reinterpret_cast<const char*>(tile_lds);
  const int lane4 = 4 * (lane % LPC);
  // The wave's entries are one stream over the phases, requested kRing chunks
  // of four groups ahead (they come from memory, and a phase has only a few
  // chunks). Lane i holds the header of phase q0 + i. The loop below has no
  // load behind a branch: the compiler counts the loads in flight, and would
  // wait for all of them where it cannot.
  constexpr int kRing = 2, kLast = 8, kEnd = 16;
  constexpr int kStep = 16 * NSET * kWave / LPC;  // bytes of a group of all the wave's lines
  struct Chunk {
    int o[NSET][4], w[NSET][4], info;  // info: groups, last of its phase, end of the stream
  } ring[kRing];
  int which = 0;
  bool first_block = true;
  for (uint32_t q0 = p0; q0 < p1; q0 += kWave) {
    const uint32_t q1 = min(q0 + kWave, p1);
    // (the header of phase p1 exists, of the next tile or the table's slack)
    const uint4 hq = A.hdr[static_cast<int64_t>(min(q0 + lane, q1)) * kTileWaves + wave + zero];
    uint32_t fp = q0;
    int fleft = 0;
    const char *po = nullptr, *pw = nullptr;
    unsigned at[NSET];
    auto phase = [&] {  // the phase fp: its first group and groups left
      const uint32_t first = __builtin_amdgcn_readlane(hq.x, fp - q0);
      fleft = __builtin_amdgcn_readlane(hq.y, fp - q0);
      po = reinterpret_cast<const char*>(A.off + 4 * static_cast<int64_t>(first));
      pw = reinterpret_cast<const char*>(A.w + 4 * static_cast<int64_t>(first));
#pragma unroll
      for (int s = 0; s < NSET; ++s) at[s] = 16 * (s * (kWave / LPC) + lane / LPC) + 4 * (lane % 4);
    };
    auto fetch = [&](Chunk& c) {
      c.info = fp >= q1 ? kEnd : min(fleft, 4);
#pragma unroll
      for (int s = 0; s < NSET; ++s)
#pragma unroll
        for (int j = 0; j < 4; ++j) {  // past the stream's end its last chunk again
          c.o[s][j] = entry_word(po, at[s] + kStep * j);
          c.w[s][j] = entry_word(pw, at[s] + kStep * j);
        }
      if (fp < q1) {
        fleft -= 4;
        if (fleft <= 0) {
          c.info |= kLast;
          if (++fp < q1) phase();
        } else {
#pragma unroll
          for (int s = 0; s < NSET; ++s) at[s] += 4 * kStep;
        }
      }
    };
    phase();
#pragma unroll
    for (int r = 0; r < kRing; ++r) fetch(ring[r]);
    if (first_block) __syncthreads();  // the first phase's rows are there (and the leading zeros)
    first_block = false;
    while (ring[0].info != kEnd) {  // (chunks past the end: no groups)
#pragma unroll
      for (int r = 0; r < kRing; ++r) {
        Chunk& c = ring[r];
        const int n = c.info & 7;
        if (n == 4) {
#pragma unroll
          for (int s = 0; s < NSET; ++s) short_groups<4>(c.o[s], c.w[s], lds, lane4, acc[s]);
        } else {
#pragma unroll
          for (int j = 0; j < 3; ++j)
            if (n > j) {
#pragma unroll
              for (int s = 0; s < NSET; ++s) short_groups<1>(c.o[s] + j, c.w[s] + j, lds, lane4, acc[s]);
            }
        }
        if (c.info & kLast) {
          if constexpr (SUM2) {
#pragma unroll
            for (int s = 0; s < NSET; ++s) {
              sum[s] += acc[s];
              acc[s] = 0.F;
            }
          }
          which ^= 1;
          lds = reinterpret_cast<const char*>(tile_lds + which * A.buffer);
          __syncthreads();
        }
        fetch(c);
      }
    }
  }
  if (first_block) __syncthreads();
#endif
  const TileShape& S = A.shape;
#pragma unroll
  for (int s = 0; s < NSET; ++s) {
    const int ln = (wave * NSET + s) * (kWave / LPC) + lane / LPC;
    const int cc = ln / PAR, z = PAR * (lane % LPC) + ln % PAR;
    const int cx = (t % S.ntx) * S.tx + cc % S.tx, cy = (t / S.ntx) * S.ty + cc / S.tx;
    if (cx >= d.nx || cy >= d.ny || z >= d.nzp) continue;
    const int64_t idx = static_cast<int64_t>(cy * d.nx + cx) * d.nzp + z;
    const float v = SUM2 ? sum[s] : acc[s];
    if constexpr (MODE == BP_PLAIN) {
      as_global(img)[idx] = z < d.nz ? v : 0.F;
    } else if (z < d.nz) {
      const float u = osem_factor(v, as_const(data.sens)[idx], data.threshold, data.thr_lo, data.thr_hi);
      as_global(data.estimate)[idx] = as_global(data.estimate)[idx] * u;
      if (data.update) as_global(data.update)[idx] = u;
    }
  }
}

unsigned grid_of(int64_t n) {
  int64_t b = (n + 255) / 256;
  if (b > 65536) b = 65536;
  if (b < 1) b = 1;
  return static_cast<unsigned>(b);
}

}  // namespace

void launch_tile_range(const Family* d_fams, const int2* d_fam_pos, int nfam, const int2* d_pool,
                       const int32_t* d_fp_rec, int w, const ImageDims& dims, const TileShape& shape, int nviews, int ntof,
                       int2* d_rng, int* d_need, hipStream_t stream) {
  if (nfam <= 0) return;
  hipLaunchKernelGGL(tile_range_kernel, dim3(nfam), dim3(kWave), 0, stream, d_fams, d_fam_pos, nfam, d_pool, d_fp_rec, w,
                     dims, shape, nviews, ntof, d_rng, d_need);
}

void launch_tile_phases(const int4* d_units, const int32_t* d_unit_off, int nsub, int ntiles, int nunits, int nrng,
                        const int2* d_rng, int rows, uint32_t* d_slot, uint32_t* d_nphase, uint32_t* d_nrow,
                        int* d_bad, hipStream_t stream) {
  hipLaunchKernelGGL(tile_phase_kernel<false>, dim3((nsub * ntiles + 63) / 64), dim3(64), 0, stream, d_units, d_unit_off,
                     nsub, ntiles, nunits, nrng, d_rng, rows, d_slot, d_nphase, d_nrow, nullptr, nullptr,
                     nullptr, nullptr, d_bad);
}

void launch_tile_rows(const int4* d_units, const int32_t* d_unit_off, int nsub, int ntiles, int nunits, int nrng,
                      const int2* d_rng, int rows, const uint32_t* d_phase_off, const uint32_t* d_row_off,
                      int2* d_row, uint32_t* d_phase_row, int* d_bad, hipStream_t stream) {
  hipLaunchKernelGGL(tile_phase_kernel<true>, dim3((nsub * ntiles + 63) / 64), dim3(64), 0, stream, d_units, d_unit_off,
                     nsub, ntiles, nunits, nrng, d_rng, rows, nullptr, nullptr, nullptr, d_phase_off, d_row_off,
                     d_row, d_phase_row, d_bad);
}

void launch_tile_count(const Family* d_fams, const int2* d_fam_pos, int fam_begin, int fam_end, int ntang,
                       const int2* d_pool, const int32_t* d_fp_rec, int w, int ntof, int subset, const ImageDims& dims,
                       const TileArgs& A, int nunits, const uint32_t* d_slot, uint32_t* d_counts, hipStream_t stream) {
  if (fam_end <= fam_begin) return;
  hipLaunchKernelGGL(tile_entries_kernel<true>, dim3(fam_end - fam_begin), dim3(kWave), 0, stream, d_fams, d_fam_pos,
                     fam_begin, fam_end, ntang, d_pool, d_fp_rec, w, ntof, subset, dims, A, nunits, d_slot, d_counts, 0U,
                     0, nullptr, int64_t{0}, nullptr, nullptr);
}

void launch_tile_make(const Family* d_fams, const int2* d_fam_pos, int fam_begin, int fam_end, int ntang,
                      const int2* d_pool, const int32_t* d_fp_rec, int w, int ntof, int subset, const ImageDims& dims,
                      const TileArgs& A, int nunits, const uint32_t* d_slot, uint32_t none, int span,
                      const int64_t* d_fam_entry_off, int64_t first, uint32_t* d_keys, int2* d_raw, hipStream_t stream) {
  if (fam_end <= fam_begin) return;
  hipLaunchKernelGGL(tile_entries_kernel<false>, dim3(fam_end - fam_begin), dim3(kWave), 0, stream, d_fams, d_fam_pos,
                     fam_begin, fam_end, ntang, d_pool, d_fp_rec, w, ntof, subset, dims, A, nunits, d_slot, nullptr, none,
                     span, d_fam_entry_off, first, d_keys, d_raw);
}

void launch_tile_groups(const uint32_t* d_counts, int64_t n, int lockstep, uint32_t* d_groups, int* d_bad,
                        hipStream_t stream) {
  hipLaunchKernelGGL(tile_groups_kernel, dim3(grid_of(n)), dim3(256), 0, stream, d_counts, n, lockstep, d_groups, d_bad);
}

void launch_tile_headers(const uint32_t* d_groups, const uint32_t* d_group_off, const uint32_t* d_phase_row,
                         uint32_t total_rows, int64_t nphase, const TileShape& shape, uint4* d_hdr, hipStream_t stream) {
  const int64_t n = (nphase + kTileHdrSlack) * kTileWaves;
  hipLaunchKernelGGL(tile_headers_kernel, dim3(grid_of(n)), dim3(256), 0, stream, d_groups, d_group_off, d_phase_row,
                     total_rows, nphase, int64_t{kTileHdrSlack}, shape, d_hdr);
}

void launch_tile_work(const uint32_t* d_group_off, const uint32_t* d_phase_off, int nsub, int ntiles, int lines,
                      uint32_t* d_work, hipStream_t stream) {
  hipLaunchKernelGGL(tile_work_kernel, dim3((ntiles + 255) / 256), dim3(256), 0, stream, d_group_off, d_phase_off, nsub,
                     ntiles, lines, d_work);
}

void launch_tile_place(const uint32_t* d_keys, const uint32_t* d_idx, const int2* d_raw, const uint32_t* d_group_off,
                       uint32_t none, int lockstep, int64_t n, int32_t* d_off, float* d_w, hipStream_t stream) {
  if (n <= 0) return;
  hipLaunchKernelGGL(tile_place_kernel, dim3(grid_of(n)), dim3(256), 0, stream, d_keys, d_idx, d_raw, d_group_off, none,
                     lockstep, n, d_off, d_w);
}

void launch_back_project_tile(BpMode mode, const TileArgs& A, int subset_begin, int subset_end, const float* d_proj,
                              float* d_img, const ImageDims& dims, const BpData& data, hipStream_t stream) {
  const int nslot = (dims.nz + kWave - 1) / kWave;
  const int chunk = kTileXcdChunk, round = kNumXcd * chunk;
  const dim3 grid((A.ntiles + round - 1) / round * round), block(kWave * kTileWaves);
  const size_t lds = static_cast<size_t>(A.lds_floats) * sizeof(float);
  if (A.shape.lanes < kWave) {
    // one plane per axial position (and mixed ones): the column kernel's order
    // of additions, bit for bit
#define MI_SHORT(M, L, P, S2, N)                                                                                       \
  hipLaunchKernelGGL((bp_tile_short_kernel<M, L, P, S2, N>), grid, dim3(kShortThreads), lds, stream, A, subset_begin,  \
                     subset_end, d_proj, d_img, dims, data, chunk)
#define MI_SHORT_N(M, L, P, S2)               \
  if (A.shape.tx == 8) MI_SHORT(M, L, P, S2, 2); \
  else MI_SHORT(M, L, P, S2, 1);
#define MI_SHORT_S(M)                                        \
  if (A.shape.par == 2) {                                    \
    if (A.shape.lanes == 8) MI_SHORT(M, 8, 2, true, 1);      \
    else { MI_SHORT_N(M, 16, 2, true) }                      \
  } else if (A.tof) {                                        \
    if (A.shape.lanes == 16) MI_SHORT(M, 16, 1, true, 1);    \
    else { MI_SHORT_N(M, 32, 1, true) }                      \
  } else {                                                   \
    if (A.shape.lanes == 16) MI_SHORT(M, 16, 1, false, 1);   \
    else { MI_SHORT_N(M, 32, 1, false) }                     \
  }
    if (mode == BP_PLAIN) { MI_SHORT_S(BP_PLAIN) }
    else { MI_SHORT_S(BP_OSEM_UPDATE) }
#undef MI_SHORT_S
#undef MI_SHORT_N
#undef MI_SHORT
    return;
  }
#define MI_TILE(M, S, T)                                                                                          \
  hipLaunchKernelGGL((bp_tile_kernel<M, S, T>), grid, block, lds, stream, A, subset_begin, subset_end, d_proj, d_img, \
                     dims, data, chunk)
#define MI_TILE_S(M, T)              \
  switch (nslot) {                  \
    case 1: MI_TILE(M, 1, T); break; \
    case 2: MI_TILE(M, 2, T); break; \
    case 3: MI_TILE(M, 3, T); break; \
    default: MI_TILE(M, 4, T); break; \
  }
  if (A.tof) {
    if (mode == BP_PLAIN) { MI_TILE_S(BP_PLAIN, true) }
    else { MI_TILE_S(BP_OSEM_UPDATE, true) }
  } else {
    if (mode == BP_PLAIN) { MI_TILE_S(BP_PLAIN, false) }
    else { MI_TILE_S(BP_OSEM_UPDATE, false) }
  }
#undef MI_TILE_S
#undef MI_TILE
}

void launch_back_project_tile_batch(BpMode mode, int nslot, const ProblemDesc* d_descs, const TileArgs* d_tiles,
                                    const WorkItem* d_work, int nwork, int subset, int threshold, hipStream_t stream) {
  if (nwork <= 0) return;
  const int round = kNumXcd * kTileXcdChunk;
  const dim3 grid((nwork + round - 1) / round * round), block(kWave * kTileWaves);
#define MI_TILE(M, S) \
  hipLaunchKernelGGL((bp_tile_batch_kernel<M, S>), grid, block, kTileLdsBytes, stream, d_descs, d_tiles, d_work, nwork, \
                     subset, threshold)
#define MI_TILE_S(M)               \
  switch (nslot) {                 \
    case 1: MI_TILE(M, 1); break;  \
    case 2: MI_TILE(M, 2); break;  \
    case 3: MI_TILE(M, 3); break;  \
    default: MI_TILE(M, 4); break; \
  }
  if (mode == BP_OSEM_UPDATE) { MI_TILE_S(BP_OSEM_UPDATE) }
  else { MI_TILE_S(BP_PLAIN) }
#undef MI_TILE_S
#undef MI_TILE
}

}  // namespace mi

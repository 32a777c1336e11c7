// Forward projection by row groups: the short families of small scanners.
//
// What bounds it, and why it is built this way. fp_kernel gives a family (or a
// +-segment pair) a wave, lanes over its axial positions. A scanner of 8 rings
// has families of 5 to 8 of them, so 7 lanes of 8 idle through the same loads
// and adds. Here the lanes of a wave take the bins of all families that share
// one basic row (its symmetry-related views, tangential positions and
// segments; up to 16 families, all of one subset and one length), family after
// family and cut every 64 bins, so only a group's last wave has idle lanes.
// The row's elements stay wave-uniform (scalar loads, decoded by scalar
// instructions); the in-plane operation, the z sign and the axial shift of a
// lane's bin are folded into one linear form of the element's coordinates,
//     byte offset = A x + B y + Z z + K,
// three 24-bit multiply-adds per element, then a multiply and an add. The
// image is one range-checked buffer. Planes outside the image are read as the
// zeros that pad every column; a group whose rows reach further than the pad
// (flag `inside` 0) tests the plane.
// Each bin sums its row in row order, as fp_kernel does: the same values bit
// for bit.
// Measured, tasks against row groups: 8 rings x 192 crystals (5.4e5 bins of 116
// elements) 0.356 -> 0.063 ms, 16 rings x 288 (span 1, 128 x 128 columns) 1.21 ->
// 0.43, 24 rings x 288 (span 3) 0.265 -> 0.207. They lose where families are
// longer, images larger or a subset small (rows_pay in pmrt_capi.cpp has the
// line): their waves read two or three image columns per element, tasks one.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "pmrt_device.hpp"
#include "pmrt_kernels.hpp"

namespace mi {

namespace {

using namespace dev;

constexpr int kRowUnroll = 16;  // gathers in flight per wave
static_assert(kRowUnroll <= kRowSlack, "read-ahead beyond the rows' slack");

// xo = ca x + cb y, yo = cc x + ce y for the in-plane operation codes
__device__ inline void inplane_coeffs(int ip, int& ca, int& cb, int& cc, int& ce) {
  int x1, y1, x2, y2;
  inplane_any_op(ip, 1, 0, x1, y1);
  inplane_any_op(ip, 0, 1, x2, y2);
  ca = x1;
  cc = y1;
  cb = x2;
  ce = y2;
}

// groups[i].inside = 1 when every plane that an element of the group's row
// reaches, for every bin of the group, is at most nzp - nz planes outside the
// image (one wave per group)
__global__ void __launch_bounds__(kWave) row_group_reach_kernel(RowGroup* __restrict__ groups, int ngroups,
                                                                const int32_t* __restrict__ fam_list,
                                                                const Family* __restrict__ fams,
                                                                const int2* __restrict__ pool, ImageDims d) {
  const int g = blockIdx.x;
  if (g >= ngroups) return;
  const RowGroup G = groups[g];
  int lo = 4096, hi = -4096;
  for (int e = threadIdx.x; e < G.row_len; e += kWave) {
    int x, y, z;
    decode(pool[G.row_start + e].x, x, y, z);
    lo = min(lo, z);
    hi = max(hi, z);
  }
  for (int o = kWave / 2; o > 0; o >>= 1) {
    lo = min(lo, __shfl_xor(lo, o, kWave));
    hi = max(hi, __shfl_xor(hi, o, kWave));
  }
  const int pad = d.nzp - d.nz;
  bool inside = true;
  for (int k = threadIdx.x; k < G.nfam; k += kWave) {  // (the empty rows' group has thousands)
    const Family f = fams[fam_list[G.first + k]];
    const int z0 = f.zadd0 - d.min_z + (f.zsign > 0 ? lo : -hi), z1 = f.zadd0 - d.min_z + (f.zsign > 0 ? hi : -lo);
    inside = inside && z0 >= -pad && z1 + f.ppa * (f.nax - 1) < d.nz + pad;
  }
  inside = __all(inside);
  if (threadIdx.x != 0) return;
  groups[g].inside = inside;
}

// item it (group, first bin): 64 bins of a group; log-likelihood sum to place w
template <int MODE>
__device__ __forceinline__ void rows_item(int w, const int2 it, const RowGroup* __restrict__ groups,
                                          const int32_t* __restrict__ fam_list, const Family* __restrict__ fams,
                                          const int2* __restrict__ pool, const float* __restrict__ img,
                                          float* __restrict__ out, const ImageDims& d, const FpData& data) {
  const int lane = static_cast<int>(threadIdx.x % kWave);
  const RowGroup G = as_const(groups)[it.x];
  const int j = it.y + lane, last = G.nfam * G.nax - 1;
  const bool valid = j <= last;
  const int jj = min(j, last), k = jj / G.nax, a = jj - k * G.nax;
  const Family f = fams[fam_list[G.first + k]];
  int ca, cb, cc, ce;
  inplane_coeffs(f.inplane, ca, cb, cc, ce);
  const int nzp4 = 4 * d.nzp;
  const int A = (cc * d.nx + ca) * nzp4, B = (ce * d.nx + cb) * nzp4, Z = 4 * f.zsign;
  const int zb = f.zadd0 + f.ppa * a - d.min_z;
  // coordinates enter as packed: x + 512, y + 512, z + 2048
  const int K = (-d.min_y * d.nx - d.min_x) * nzp4 + 4 * zb - 512 * (A + B) - 2048 * Z;
  const int zq = zb - 2048 * f.zsign;
  float acc = 0.F;
#if defined(__HIP_DEVICE_COMPILE__)
  const __amdgpu_buffer_rsrc_t image = run_buffer(as_const(img), 0, d.ncols * d.nzp);
  cptr<int2> row = as_const(pool) + G.row_start;
  const int n = G.row_len;
  auto offset = [&](int c, bool check) {
    const int x = c & 1023, y = (c >> 10) & 1023, z = static_cast<int>(static_cast<unsigned>(c) >> 20);
    int off = whole_offset(__mul24(A, x) + K);  // kept apart, so that each step is one multiply-add
    off = whole_offset(__mul24(B, y) + off);
    off = __mul24(Z, z) + off;
    if (check && static_cast<unsigned>(__mul24(f.zsign, z) + zq) >= static_cast<unsigned>(d.nz)) off = -4;
    return off;
  };
  auto sum = [&](bool check) {
    int e = 0;
    if (n >= kRowUnroll) {
      int2 cur[kRowUnroll];
#pragma unroll
      for (int u = 0; u < kRowUnroll; ++u) cur[u] = row[u];
      for (; e + kRowUnroll <= n; e += kRowUnroll) {
        int2 nxt[kRowUnroll];
#pragma unroll
        for (int u = 0; u < kRowUnroll; ++u) nxt[u] = row[e + kRowUnroll + u];  // the pool ends in slack
        float v[kRowUnroll], wt[kRowUnroll];
#pragma unroll
        for (int u = 0; u < kRowUnroll; ++u) {
          wt[u] = __int_as_float(cur[u].y);
          v[u] = load_run(image, whole_offset(offset(cur[u].x, check)));
        }
#pragma unroll
        for (int u = 0; u < kRowUnroll; ++u) acc = acc + v[u] * wt[u];
#pragma unroll
        for (int u = 0; u < kRowUnroll; ++u) cur[u] = nxt[u];
      }
    }
    for (; e < n; ++e) {
      const int2 el = row[e];
      acc = acc + load_run(image, whole_offset(offset(el.x, check))) * __int_as_float(el.y);
    }
  };
  if (G.inside) sum(false);
  else sum(true);
#endif
  double ll = 0.0;
  if (valid) fp_epilogue<MODE>(acc, static_cast<int64_t>(f.sino_base) + a, f.viewgram, data, out, ll);
  if constexpr (fp_accumulates_loglik(MODE)) {
    for (int off = kWave / 2; off > 0; off >>= 1) ll += __shfl_xor(ll, off, kWave);
    if (lane == 0) as_global(data.partial)[w] = ll;
  }
}

template <int MODE>
__global__ void __launch_bounds__(kWave* kWavesPerBlock) fp_rows_kernel(const int2* __restrict__ items, int nitems,
                                                                        const RowGroup* __restrict__ groups,
                                                                        const int32_t* __restrict__ fam_list,
                                                                        const Family* __restrict__ fams,
                                                                        const int2* __restrict__ pool,
                                                                        const float* __restrict__ img,
                                                                        float* __restrict__ out, ImageDims d,
                                                                        FpData data) {
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) / kWave);
  const int w = xcd_chunk_remap(static_cast<int>(blockIdx.x), kRowsXcdChunk) * kWavesPerBlock + wave;
  if (w >= nitems) return;
  rows_item<MODE>(w, as_const(items)[w], groups, fam_list, fams, pool, img, out, d, data);
}

// work: (problem, group, first bin)
template <int MODE>
__global__ void __launch_bounds__(kWave* kWavesPerBlock) fp_rows_batch_kernel(const ProblemDesc* __restrict__ descs,
                                                                              const RowProblem* __restrict__ rows,
                                                                              const int4* __restrict__ work,
                                                                              int nwork) {
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) / kWave);
  const int w = xcd_chunk_remap(static_cast<int>(blockIdx.x), kRowsXcdChunk) * kWavesPerBlock + wave;
  if (w >= nwork) return;
  const int4 it = as_const(work)[w];
  const ProblemDesc P = as_const(descs)[it.x];
  const RowProblem R = as_const(rows)[it.x];
  rows_item<MODE>(w, make_int2(it.y, it.z), R.groups, R.fam_list, P.fams, P.pool, P.fp_in, P.fp_out, P.d, P.fd);
}

}  // namespace

void launch_row_group_reach(RowGroup* d_groups, int ngroups, const int32_t* d_fam_list, const Family* d_fams,
                            const int2* d_pool, const ImageDims& dims, hipStream_t stream) {
  if (ngroups <= 0) return;
  hipLaunchKernelGGL(row_group_reach_kernel, dim3(ngroups), dim3(kWave), 0, stream, d_groups, ngroups, d_fam_list,
                     d_fams, d_pool, dims);
}

void launch_forward_project_rows(FpMode mode, const int2* d_items, int nitems, const RowGroup* d_groups,
                                 const int32_t* d_fam_list, const Family* d_fams, const int2* d_pool,
                                 const float* d_img, float* d_out, const ImageDims& dims, const FpData& data,
                                 hipStream_t stream) {
  if (nitems <= 0) return;
  const int blocks = (nitems + kWavesPerBlock - 1) / kWavesPerBlock, round = kNumXcd * kRowsXcdChunk;
  const dim3 grid((blocks + round - 1) / round * round), block(kWave * kWavesPerBlock);
  switch (mode) {
#define MI_ROWS(M)                                                                                                  \
  case M:                                                                                                           \
    hipLaunchKernelGGL(fp_rows_kernel<M>, grid, block, 0, stream, d_items, nitems, d_groups, d_fam_list, d_fams,    \
                       d_pool, d_img, d_out, dims, data);                                                           \
    break;
    MI_ROWS(FP_PLAIN)
    MI_ROWS(FP_RATIO)
    MI_ROWS(FP_GRADIENT)
    MI_ROWS(FP_LOGLIK)
    MI_ROWS(FP_GRADIENT_LOGLIK)
    MI_ROWS(FP_RATIO_LOGLIK)
    MI_ROWS(FP_DRATIO)
    MI_ROWS(FP_SCALE)
    MI_ROWS(FP_LM_RATIO)
    MI_ROWS(FP_LM_VALUE)
#undef MI_ROWS
  }
}

void launch_forward_project_rows_batch(FpMode mode, const ProblemDesc* d_descs, const RowProblem* d_rows,
                                       const int4* d_work, int nwork, hipStream_t stream) {
  if (nwork <= 0) return;
  const int blocks = (nwork + kWavesPerBlock - 1) / kWavesPerBlock, round = kNumXcd * kRowsXcdChunk;
  const dim3 grid((blocks + round - 1) / round * round), block(kWave * kWavesPerBlock);
  if (mode == FP_RATIO)
    hipLaunchKernelGGL(fp_rows_batch_kernel<FP_RATIO>, grid, block, 0, stream, d_descs, d_rows, d_work, nwork);
  else
    hipLaunchKernelGGL(fp_rows_batch_kernel<FP_PLAIN>, grid, block, 0, stream, d_descs, d_rows, d_work, nwork);
}

}  // namespace mi

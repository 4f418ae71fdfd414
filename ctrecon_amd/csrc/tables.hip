// The plan's large geometry tables, computed on the device from the small ones that the host
// uploads: a view's boundary lines and column constants, the row tables, and the mask's
// multiplier and per-slice extents.  FP64 arithmetic in the host's order without contraction
// (the divisions and square roots of both are correctly rounded), FP32 storage.
//
// A host-buffer call of 64^3 voxels and 72 views of 256 x 16, forward or back: 0.66 ms with host
// loops over (view, column) and a copy per table (16 of 13 us), 0.24 ms with one packed copy and
// this kernel (and no stream for the call's plan).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "ctr_internal.hpp"

namespace ctr {
namespace {

constexpr int kTB = 256;  // threads of a workgroup

// Workgroups [0, n0): (view, boundary) pairs; [n0, n0 + n1): the mask as floats; the next n2:
// mask extents, a wave per slice; the last: the rows.
struct TableBlocks {
  int n0, n1, n2;
};

__global__ __launch_bounds__(kTB) void plan_tables_kernel(PlanTables T, TableBlocks nb) {
#pragma clang fp contract(off)
  const int DNU = T.DNU, XN = T.XN, YN = T.YN;
  int blk = blockIdx.x;
  if (blk < nb.n0) {
    const long long n = (long long)T.PN * (DNU + 1);
    for (long long i = (long long)blk * kTB + threadIdx.x; i < n; i += (long long)nb.n0 * kTB) {
      const int p = (int)(i / (DNU + 1)), b = (int)(i - (long long)p * (DNU + 1));
      const double2 cs = T.rot64[p], src = T.src64[p], e = T.edge64[b];
      const double c = cs.x, s = cs.y, sx = src.x, sy = src.y, dx = T.dx;
      const bool xmarch = T.views[p].xmarch != 0;
      const double2 l = boundary_line(e, c, s, sx, sy, xmarch, T.ocx, T.ocy, dx, T.half);
      T.bnd64[i] = l;
      T.bnd[i] = make_float2((float)l.x, (float)l.y);
      if (b < DNU) {
        const double2 det = T.det64[b];
        const double ex = (det.x * c - det.y * s) - sx, ey = (det.x * s + det.y * c) - sy;
        const double ea = xmarch ? ex : ey;
        const double r0 = xmarch ? (-T.ocx * dx - sx) / ex : (-T.ocy * dx - sy) / ey;
        T.cols[(long long)p * DNU + b] = make_float4((float)r0, (float)(dx / ea),
                                                     (float)(ex * ex + ey * ey),
                                                     (float)(dx / fabs(ea)));
      }
    }
    return;
  }
  blk -= nb.n0;
  if (blk < nb.n1) {
    const long long n = (long long)XN * YN;
    for (long long i = (long long)blk * kTB + threadIdx.x; i < n; i += (long long)nb.n1 * kTB)
      T.maskf[i] = (float)T.mask[i];
    return;
  }
  blk -= nb.n1;
  if (blk < nb.n2) {
    // x-slices (cells along y), then y-slices; no cell: an empty interval
    const int lane = threadIdx.x & 63, k = blk * (kTB / 64) + (threadIdx.x >> 6);
    if (k >= XN + YN) return;
    const bool xs = k < XN;
    const int n = xs ? YN : XN;
    const size_t at = xs ? (size_t)k : (size_t)(k - XN) * XN, step = xs ? (size_t)XN : 1;
    int lo = n, hi = -1;
    for (int j = lane; j < n; j += 64)
      if (T.mask[at + j * step]) {
        lo = min(lo, j);
        hi = max(hi, j);
      }
    for (int off = 32; off > 0; off >>= 1) {
      lo = min(lo, __shfl_xor(lo, off, 64));
      hi = max(hi, __shfl_xor(hi, off, 64));
    }
    if (lane == 0)
      T.mext[k] = hi >= lo ? make_float2((float)lo - 0.5f, (float)hi + 0.5f)
                           : make_float2(0.f, -1.f);
    return;
  }
  for (int v = threadIdx.x; v <= T.DNV; v += kTB) {
    T.Bz[v] = (float)((T.bz64[v] - T.z0) / T.dz);
    if (v == T.DNV) break;
    const double h = T.zds64[v] - T.z0, step = T.bz64[v + 1] - T.bz64[v];
    T.h2[v] = (float)(h * h);
    T.zc[v] = (float)(h / T.dz);
    T.invdB[v] = (float)(T.dz / step);
  }
}

}  // namespace

int launch_plan_tables(const PlanTables& T, hipStream_t st) {
  auto blocks = [](long long n) { return (int)std::min<long long>((n + kTB - 1) / kTB, 16384); };
  const TableBlocks nb{blocks((long long)T.PN * (T.DNU + 1)), blocks((long long)T.XN * T.YN),
                       (T.XN + T.YN + kTB / 64 - 1) / (kTB / 64)};
  hipLaunchKernelGGL(plan_tables_kernel, dim3(nb.n0 + nb.n1 + nb.n2 + 1), dim3(kTB), 0, st, T, nb);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess)
    return fail(CTR_ERR_HIP, std::string("plan_tables_kernel: ") + hipGetErrorString(e));
  return CTR_OK;
}

}  // namespace ctr

// gfx950 kernels of the DD3 projector pair and the solver loops.
//
// Work mapping ("z-column waves"): every wave64 owns one column of 64 consecutive
// z-cells -- in the forward projector the 64 detector rows of one (view, column),
// in the back projectors 64 voxels along z of one (x, y) column.  All in-plane
// geometry is then the same for the wave and only the z part is per lane; reads
// of vol[...][z] and prj[...][v] are contiguous across the lanes.
//
// The reference samples 2-D summed-area tables through linear-filtered, clamped
// textures.  With exact weights that sample equals the integral of the
// piecewise-constant volume (sinogram) over the footprint rectangle clipped to
// the array, so the kernels integrate the footprint directly: the same operator,
// without the FP32 cancellation of whole-plane integral images and without the
// integral-image build pass.
#include <algorithm>
#include <type_traits>

#include "ctr_internal.hpp"
#include "device_common.hpp"

namespace ctr {
namespace {

// A lane's float as a wave-uniform value (v_readlane_b32 into a scalar register).
__device__ __forceinline__ float rdl(float v, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// A wave-uniform value in scalar registers that the compiler takes for a new one: what is computed
// or loaded from it in a loop is not hoisted out of the loop into registers.
template <typename V>
__device__ __forceinline__ V held(V v) {
  constexpr int N = sizeof(V) / 4;
  uint32_t w[N];
  __builtin_memcpy(w, &v, sizeof(V));
#pragma unroll
  for (int i = 0; i < N; ++i) {
    w[i] = __builtin_amdgcn_readfirstlane(w[i]);
    asm volatile("" : "+s"(w[i]));
  }
  __builtin_memcpy(&v, w, sizeof(V));
  return v;
}

// Block-wide sum of two doubles into slot[0], slot[1].
__device__ __forceinline__ void block_sum2(double a, double b, double* slot) {
  __shared__ double red[2][kWaves];
  for (int off = 32; off > 0; off >>= 1) {
    a += __shfl_xor(a, off, 64);
    b += __shfl_xor(b, off, 64);
  }
  const int w = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) {
    red[0][w] = a;
    red[1][w] = b;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    double sa = 0, sb = 0;
    for (int i = 0; i < kWaves; ++i) {
      sa += red[0][i];
      sb += red[1][i];
    }
    gp(slot)[0] = sa;
    gp(slot)[1] = sb;
  }
  __syncthreads();  // red[] is reused by the next work item of a persistent block
}

// ---------------------------------------------------------------------------
// Forward projector (mode 0 distance-driven), one lane per ray (p, u, v).
// Reference: DD3_gpu_proj_branchless_sat2d_ker, iterativeRecon/DD3_GPU.cu:844-990.
// Per slice ii the ray's footprint is [tl, tr] (in-plane) x [zl, zh] (z) in
// cell-centre index units; its mean over the footprint, summed over slices and
// scaled by dx/|dir| (K), is the ray sum.
// FUSED: out = (b - A x) * invRow (os_sart.m:24,30-31; b indexed by global view,
// invRow by the launch's compact view index, NULL for 1; out NULL: not written) and
// per-block sums of (b - A x)^2 and b^2.
// T: storage type of vol and out (float, or uint16_t for BF16); b and invRow are FP32
// and the ray sum is accumulated in FP32.
// ---------------------------------------------------------------------------

// In-plane part of slice ii of one detector column's footprint: the boundary lines
// t_b(ii) = a_b + ii f_b of its two boundaries (FP64: positions run to the slice width,
// where FP32 keeps only ~3e-5 of a cell), the footprint [ylo, yhi] clipped to the mask's
// extent e on the slice, its cells j0 .. j0 + nj - 1 with first / last overlap weights
// (FP64 differences, rounded once), the z magnification r and 1 / ((yhi - ylo) r).
// False when the clipped footprint is empty.
struct SliceIP {
  float r, inv, wj0, wjl;
  int j0, nj;
};
__device__ __forceinline__ bool fp_inplane(const double2& bl, const double2& br, const float4& ct,
                                           const float2& e, int ii, int NI, SliceIP& o) {
  const double fi = (double)ii;
  const double tl = fma(fi, bl.y, bl.x), tr = fma(fi, br.y, br.x);
  const double ylo = fmin(tl, tr), yhi = fmax(tl, tr);
  const double clo = fmax(ylo, (double)e.x), chi = fmin(yhi, (double)e.y);
  if (!(clo < chi)) return false;
  o.r = fmaf((float)ii, ct.y, ct.x);
  o.inv = __builtin_amdgcn_rcpf((float)(yhi - ylo) * o.r);
  o.j0 = (int)floor(clo + 0.5);
  o.nj = min((int)floor(chi + 0.5), NI - 1) - o.j0 + 1;
  o.wj0 = (float)(o.nj == 1 ? chi - clo : ((double)o.j0 + 0.5) - clo);
  o.wjl = (float)(chi - ((double)(o.j0 + o.nj - 1) - 0.5));
  return true;
}

// floor(x) as an integer (v_cvt_flr_i32_f32, one instruction).
__device__ __forceinline__ int floor_i(float x) {
  int k;
  asm("v_cvt_flr_i32_f32 %0, %1" : "=v"(k) : "v"(x));
  return k;
}

__device__ __forceinline__ float sat(float x) { return __builtin_amdgcn_fmed3f(x, 0.f, 1.f); }

// Infinities and NaNs.  Taps of zero weight may read a cell outside a footprint, and 0 * x is
// not 0 for these.  A wave whose sums are not all finite computes them again in the general form,
// which reads the footprint's cells only ("exact").
__device__ __forceinline__ bool not_finite(float x) { return __builtin_amdgcn_classf(x, 0x207); }

// Overlaps of [t, t + h] (cell edges at integers, h <= 2) with the cells k = floor(t),
// k + 1, k + 2.
struct Overlap3 {
  float w0, w1, w2;
  int k;
};
template <int NT>
__device__ __forceinline__ Overlap3 overlap3(float t, float h) {
#pragma clang fp contract(off)
  Overlap3 o;
  const float fr = __builtin_amdgcn_fractf(t);
  const float a = 1.f - fr;
  o.k = floor_i(t);
  o.w0 = __builtin_elementwise_minimum(h, a);
  o.w1 = sat(h - a);
  o.w2 = NT == 3 ? sat((h - 2.f) + fr) : 0.f;
  return o;
}

// The overlaps with five cells (h <= 4).
struct Overlap5 {
  float w[5];
  int k;
};
__device__ __forceinline__ Overlap5 overlap5(float t, float h) {
#pragma clang fp contract(off)
  Overlap5 o;
  const float a = 1.f - __builtin_amdgcn_fractf(t);
  o.k = floor_i(t);
  o.w[0] = __builtin_elementwise_minimum(h, a);
#pragma unroll
  for (int i = 1; i < 5; ++i) o.w[i] = sat((h - (float)(i - 1)) - a);
  return o;
}

// The run of NT (2 or 3) z taps from element e of the volume on.  FP32: one range-checked
// 2- or 3-dword load (an element past the array reads 0).  BF16: one 4- or 8-byte load at
// 2-byte alignment, so that the taps need no shifting by the element's parity; the caller
// keeps elements e .. e + 3 inside the array.
template <int NT>
__device__ __forceinline__ void z_run(const Buf<float>& V, const float*, uint32_t e,
                                      float (&a)[3]) {
  a[0] = V[e];
  a[1] = V[e + 1];
  if constexpr (NT == 3) a[2] = V[e + 2];
}
typedef uint32_t u32a2 __attribute__((aligned(2)));
typedef uint64_t u64a2 __attribute__((aligned(2)));
template <int NT>
__device__ __forceinline__ void z_run(const Buf<uint16_t>&, const uint16_t* vol, uint32_t e,
                                      float (&a)[3]) {
  const CTR_GLOBAL char* p = (const CTR_GLOBAL char*)vol + e * 2u;
  if constexpr (NT == 3) {
    const uint64_t q = *(const CTR_GLOBAL u64a2*)p;
    a[0] = __uint_as_float((uint32_t)q << 16);
    a[1] = __uint_as_float((uint32_t)q & 0xffff0000u);
    a[2] = __uint_as_float((uint32_t)(q >> 32) << 16);
  } else {
    const uint32_t q = *(const CTR_GLOBAL u32a2*)p;
    a[0] = __uint_as_float(q << 16);
    a[1] = __uint_as_float(q & 0xffff0000u);
  }
}

__device__ __forceinline__ float widened(float v) { return v; }
__device__ __forceinline__ float widened(uint16_t v) { return __uint_as_float((uint32_t)v << 16); }

// Four z taps from element e of a volume of n (at least four) elements on; past its end 0.
__device__ __forceinline__ void z_run4(const Buf<float>& V, const float*, int e, int,
                                       float (&a)[4]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) a[i] = V[e + i];
}
__device__ __forceinline__ void z_run4(const Buf<uint16_t>&, const uint16_t* vol, int e, int n,
                                       float (&a)[4]) {
  const int b = min(e, n - 4);
  const uint64_t q = *(const CTR_GLOBAL u64a2*)((const CTR_GLOBAL char*)vol + (uint32_t)b * 2u) >>
                     (16 * (e - b));
  a[0] = __uint_as_float((uint32_t)q << 16);
  a[1] = __uint_as_float((uint32_t)q & 0xffff0000u);
  a[2] = __uint_as_float((uint32_t)(q >> 32) << 16);
  a[3] = __uint_as_float((uint32_t)(q >> 32) & 0xffff0000u);
}

// Work mapping.  A wave's lanes are 64 / L groups of L = 2^lg lanes (lg = A.lg, 3 .. 6);
// group g takes item g of the wave, an item being L consecutive detector rows of one
// (view, column).  COLW: lg = 6, one column per wave, so that everything in-plane is
// uniform and lives in scalar registers.
//
// Slices are taken L at a time: lane i of a group first evaluates slice ii0 + i of its
// column (FP64 footprint, each cell's edge weight times its mask byte over the footprint's
// area, the magnification r) into the wave's LDS table and sorts the slice into a class by
// its number of cells and of z taps.  Each class then runs its slices in a loop of
// straight-line code, without a branch on counts: the magnification gives the row's z
// footprint [t, t + h] (cell edges at integers, relative to azi) and overlap3 its weights.  h is
// the difference of the rounded edges, so that neighbouring rows share an edge to the bit.
//
// COLW reads a slice's cells as z runs, one element per lane (a dword load of 64
// neighbouring elements costs the texture unit about a quarter of a 2- or 3-dword gather per
// lane, which bound this kernel at 97% of that unit), combines the cells per z into LDS,
// and every row takes its two or three taps there; the next slice's runs load meanwhile.
// What bounds it then is VALU issue (0.97 of the chip's rate, about 22 instructions per
// wave and slice).  512^2 x 256, 197 views of 888 x 64: 4.06 ms with a gather per cell and
// lane, 3.00 ms with slices in classes, 2.28 ms with runs and the deal of
// xcd_chunked_block; BF16 4.19 ms, 3.32 ms, 1.99 ms.
//
// Groups (fewer than 64 rows to a column) gather each cell's taps as one load per lane:
// 64^3, 720 views of 256 x 16, 212 us one thread per ray with its own FP64 footprints,
// 87 us with four columns per wave.
//
// FINE (Dims::fine, fine voxels or wide detector columns): slices of more than four cells take
// one pass per four, and those whose rows are more than two cells high four taps to a load,
// all in the classes' loops over the LDS table.  Without it such slices are rare and take the
// general form, which evaluates a footprint in every lane; a slice that both forms take rounds
// the same, so that a batch may run FINE for all of its scans.  128^2 x 64, 100 views of 400 or
// 888 columns, general form and FINE: 0.3 mm voxels, 64 rows 344 us, 125 us; 0.1 mm slices, 16
// rows 318 us, 124 us; 64^2 x 64 of 0.1 mm, 64 rows 163 us, 65 us; 4 mm columns, 16 rows 205 us,
// 83 us.  FINE keeps 5 to 25 more registers (five to eight waves per SIMD) and is slower where
// no slice needs it.
//
// ONES: the projection of a volume of ones (the row sums of OS-SART), read from no volume.
// A slice wholly inside the volume's z range adds its height times its cells' weights; the
// others take the weights of the projection itself, so that a ray that grazes the volume by
// a rounding error has a row sum that matches its projection (no contraction: the
// instantiations must not round a footprint differently).  FINE adds up a slice's weights first,
// in one pass: sums of 20 x 20 views of 888 x 64, 128^2 x 64 of 0.1 mm, with the columns' sums
// 7.7 ms in the general form, 1.5 ms with a pass per four cells, 1.05 ms.
template <bool FUSED, bool COLW, typename TV, typename TO, bool FINE, bool ONES = false>
__device__ __forceinline__ void fp_body(const FpArgs<TV, TO>& A, int k, int ublk, double* slot) {
#pragma clang fp contract(off)
  const Dims& d = A.d;
  const int p = A.vb + k * A.vs;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int lg = COLW ? 6 : A.lg;
  const int L = 1 << lg;
  const int nch = (d.DNV + L - 1) >> lg;  // items (row chunks) per column
  const int item = ((ublk * kWaves + wid) << (6 - lg)) + (COLW ? 0 : lane >> lg);
  const int ui = item / nch;
  const int li = lane & (L - 1);
  const bool uok = ui < d.DNU;
  double res = 0.0, bsq = 0.0;
  if (!COLW || uok) {
    const int u = COLW ? ui : min(ui, d.DNU - 1);
    const int v0 = (item - ui * nch) << lg;  // first row of the item
    const int v = v0 + li;
    const bool vok = uok && v < d.DNV;
    const int vr = min(v, d.DNV - 1);
    const ViewP vp = gload(A.views, p);
    const double2 bl = gload(A.bnd64, (size_t)p * (d.DNU + 1) + u);
    const double2 br = gload(A.bnd64, (size_t)p * (d.DNU + 1) + u + 1);
    const float4 ct = gload(A.cols, (size_t)p * d.DNU + u);
    // the row's lower and upper edge (of no height past the last row)
    const float Bv = gp(A.Bz)[vr], Bv1 = gp(A.Bz)[vok ? vr + 1 : vr];
    const float Blo = gp(A.Bz)[v0], Bhi = gp(A.Bz)[min(v0 + L, d.DNV)];
    const float Btop = gp(A.Bz)[min(v0 + L, d.DNV) - 1];  // lower edge of the last row
    int NS, NI, sS, cS, mS, mC;
    if (vp.xmarch) {
      NS = d.XN; NI = d.YN; sS = d.ZN; cS = d.XN * d.ZN; mS = 1; mC = d.XN;
    } else {
      NS = d.YN; NI = d.XN; sS = d.XN * d.ZN; cS = d.ZN; mS = d.XN; mC = 1;
    }
    // z in cell units relative to azi, cell edges at integers
    const float azf = vp.azf + 0.5f;
    const float tmin = -(float)vp.azi, tmax = (float)(d.ZN - vp.azi);
    const int kmax = d.ZN - 1 - vp.azi;
    const float2* me = A.mext + (vp.xmarch ? 0 : d.XN);
    const int NV = d.XN * d.YN * d.ZN;
    const Buf<TV> V(A.vol, (uint32_t)NV);
    // a volume past the buffer loads' 32-bit byte offsets (with room for a run before its first
    // element, which their range check has to reject): the general form throughout, by address
    // (as rows of infinite height)
    const bool far = !FINE && (uint32_t)NV > 0xffffffffu / (uint32_t)sizeof(TV) - kFarRun;
    const float dBmax = far ? __builtin_inff() : d.dBmax;
    const CTR_GLOBAL float* maskf = gp(A.maskf);
    float acc = 0.f;
    // one slice in the general form (any number of cells and taps; reads the footprint's cells
    // only), all quantities per lane
    auto general = [&](int ii) {
      SliceIP o;
      if (!vok || !fp_inplane(bl, br, ct, gload(me, ii), ii, NI, o)) return;
      const float t0 = fmaf(o.r, Bv, azf);
      const float t = fmaxf(t0, tmin), te = fminf(fmaf(o.r, Bv1, azf), tmax);
      if (!(t < te)) return;
      const int k0 = min((int)floorf(t), kmax);
      const int nk = min((int)ceilf(te) - 1, kmax) - k0 + 1;
      int e = ii * sS + o.j0 * cS + vp.azi + k0, mo = ii * mS + o.j0 * mC;
      for (int ij = 0; ij < o.nj; ++ij) {
        const float wy =
            o.inv * (((ij == 0) ? o.wj0 : (ij == o.nj - 1 ? o.wjl : 1.f)) * maskf[mo]);
        float g = 0.f;
        if constexpr (ONES) g = te - t;
        else
          for (int ik = 0; ik < nk; ++ik)
            g = fmaf(fminf(te, (float)(k0 + ik + 1)) - fmaxf(t, (float)(k0 + ik)),
                     widened(gp(A.vol)[e + ik]), g);
        acc = fmaf(wy, g, acc);
        e += cS;
        mo += mC;
      }
    };
    // FINE: the same for all lanes of a slice of up to NJ cells (r, wy, nc cells from element e, z
    // index azi, on; a cell past a group's own re-reads its last with weight 0), four taps of a
    // cell to a load (taps past the lane's own have weight 0, past the array's end they are 0)
    auto tall = [&](auto NJ_, float r, const float(&wy)[4], int e, int nc) {
      constexpr int NJ = decltype(NJ_)::value;
      const float t = fmaxf(fmaf(r, Bv, azf), tmin), te = fminf(fmaf(r, Bv1, azf), tmax);
      if (!(vok && t < te)) return;
      if constexpr (ONES) {
#pragma unroll
        for (int c = 0; c < NJ; ++c) acc = fmaf(wy[c], te - t, acc);
        return;
      }
      const int k0 = min((int)floorf(t), kmax);
      float g[NJ] = {};
      for (int k = k0; (float)k < te; k += 4) {
        float w[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float z = (float)(k + i);
          w[i] = fmaxf(fminf(te, z + 1.f) - fmaxf(t, z), 0.f);
        }
#pragma unroll
        for (int c = 0; c < NJ; ++c) {
          float a[4];
          z_run4(V, A.vol, e + k + min(c, nc - 1) * cS, NV, a);
#pragma unroll
          for (int i = 0; i < 4; ++i) g[c] = fmaf(w[i], a[i], g[c]);
        }
      }
#pragma unroll
      for (int c = 0; c < NJ; ++c) acc = fmaf(wy[c], g[c], acc);
    };
    // per wave: (r, wy0, wy1, wy2) of each slice, and for groups (element, cells, wy3)
    __shared__ float4 s_rec[kWaves * 64];
    __shared__ int4 s_off[COLW ? 1 : kWaves * 64];
    __shared__ float s_run[COLW ? kWaves * 128 : 1];
    float4* rec = s_rec + wid * 64;
    int4* off = s_off + (COLW ? 0 : wid * 64);
    float* zrun = s_run + (COLW ? wid * 128 : 0);
    const int gbase = lane & ~(L - 1);  // first record of the lane's group
    // FINE: slices of more than four cells are evaluated again from the next four cells (c0) on
    for (int ii0 = 0, c0 = 0, next; ii0 < NS; ii0 = next) {
      const int il = ii0 + li;
      float q_r = 0.f, wy0 = 0.f, wy1 = 0.f, wy2 = 0.f, wy3 = 0.f;
      int q_e = 0, q_nj = 0, q_kb = 0, q_last = 0;
      // bits of cls: 1 a third z tap, 2 more than 64 cells of z (COLW), 4 reaches past the
      // volume's ends, 8 the general form, 16 more cells
      int cls = 0;
      SliceIP o;
      // clipped to the mask's extent on the slice (inside [-0.5, NI - 0.5]): cells
      // outside it are zero
      if (il < NS && uok && fp_inplane(bl, br, ct, gload(me, il), il, NI, o)) {
        // z range of the item's rows; r > 0 beyond the source
        const float tl = fmaf(o.r, Blo, azf), th = fmaf(o.r, Bhi, azf);
        const int n = FINE ? o.nj - c0 : o.nj;  // cells from c0 on
        if (o.r > 0.f && th > tmin && tl < tmax && (!FINE || n > 0)) {
          q_r = o.r;
          q_nj = FINE ? (ONES ? 1 : min(n, 4)) : n;
          const float h = o.r * dBmax;
          const int j0 = FINE ? o.j0 + c0 : o.j0, mo = il * mS + j0 * mC;
          if constexpr (ONES && FINE) {  // all of the slice's cells as one
            float W = o.wj0 * maskf[mo];
            for (int j = 1; j < n; ++j) W += (j == n - 1 ? o.wjl : 1.f) * maskf[mo + j * mC];
            wy0 = o.inv * W;
          } else {
            wy0 = o.inv * ((!FINE || c0 == 0 ? o.wj0 : (n == 1 ? o.wjl : 1.f)) * maskf[mo]);
            if (n >= 2) wy1 = o.inv * ((n == 2 ? o.wjl : 1.f) * maskf[mo + mC]);
            if (n >= 3) wy2 = o.inv * ((n == 3 ? o.wjl : 1.f) * maskf[mo + 2 * mC]);
            if (n >= 4) wy3 = o.inv * ((!FINE || n == 4 ? o.wjl : 1.f) * maskf[mo + 3 * mC]);
          }
          const int e = il * sS + j0 * cS;
          q_e = e + vp.azi;
          bool gen = (!FINE && n > 4) || h > 2.f;
          cls = (h > 1.f ? 1 : 0) | (tl < tmin + 0.01f || th > tmax - 0.01f ? 4 : 0);
          if (FINE && !ONES && n > 4) cls |= 16;
          if constexpr (COLW) {
            // the z run of the item: cells from the first row's on, read up to the last
            // row's third tap; its 64 or 128 elements stay inside the array
            q_kb = floor_i(tl);
            if constexpr (!FINE) q_e += q_kb;
            q_last = floor_i(fmaf(o.r, Btop, azf)) - q_kb + 2;
            if (q_last > 63) cls |= 2;
            gen = gen || q_last > 127 ||
                  q_e + (FINE ? q_kb : 0) > NV - 128 - (max(q_nj, 2) - 1) * cS;
            if (FINE && !gen) q_e += q_kb;
          } else {
            // a run's elements stay inside the array: not on its last column
            gen = gen || e > NV - (d.ZN + 4) - (q_nj - 1) * cS;
          }
          // ones inside the volume's z range read nothing and take no taps
          if (ONES && FINE && !(cls & 4)) gen = false;
          cls |= gen ? 8 : 0;
        }
      }
      rec[lane] = make_float4(q_r, wy0, wy1, wy2);
      next = ii0 + L;
      int mj = q_nj;  // most cells of the slice over the wave's groups
      if constexpr (!COLW) {
        off[lane] = make_int4(q_e, q_nj, __float_as_int(wy3), 0);
        for (int x = L; x < 64; x <<= 1) {
          cls |= __shfl_xor(cls, x, 64);
          mj = max(mj, __shfl_xor(mj, x, 64));
        }
      }
      if constexpr (FINE) {
        const bool more = __any(cls & 16);
        cls &= 15;
        next = more ? ii0 : ii0 + L;
        c0 = more ? c0 + 4 : 0;
      }
      if (!__any(mj)) continue;
      // the class as a number: cells (one counts as two, the second of weight 0: the two are mixed
      // along a ray, and one class keeps more loads in flight; 512^2 x 256, 2.37 ms with classes of
      // their own, 2.27 ms) * 8 + 0 two taps, 1 three taps, 2 three taps of more than
      // 64 cells, 3 past the volume's ends; 7 the general form, 0 no footprint
      const int id = cls >= 4 ? 3 : min(cls, 2);
      const int key = cls >= 8 ? 7 : (mj == 0 ? 0 : id + 8 * max(mj, 2));
      const uint64_t low = ~0ull >> (64 - L);
      using std::integral_constant;
      using I2 = integral_constant<int, 2>;
      using I3 = integral_constant<int, 3>;
      using I4 = integral_constant<int, 4>;
      using F = std::false_type;
      using T = std::true_type;
      if constexpr (COLW) {
        // a class: NJ cells, NT z taps, TAIL more than 64 cells of z, EDGE cells outside
        // the volume's z range read as 0
        auto run = [&](auto NJ_, auto NT_, auto TAIL_, auto EDGE_, int id) {
          constexpr int NJ = decltype(NJ_)::value, NT = decltype(NT_)::value;
          constexpr bool TAIL = decltype(TAIL_)::value, EDGE = decltype(EDGE_)::value;
          constexpr int NZ = TAIL ? 2 : 1;
          uint64_t m = __ballot(key == 8 * NJ + id);
          if (!m) return;
          // the slice's z run of every cell, one element per lane (stored bits)
          auto fetch = [&](int j, uint32_t(&a)[NJ][NZ]) {
            if constexpr (ONES) return;
            const int e = __builtin_amdgcn_readlane(q_e, j);
            // lanes past the last cell re-read it, so that they touch no further cache lines
            // (FP32, 512^2 x 256: 2.37 ms against 2.50 ms unclamped; the first 64 BF16 cells
            // are two lines at most: 1.99 ms unclamped against 2.10 ms)
            const int last = __builtin_amdgcn_readlane(q_last, j);
#pragma unroll
            for (int h = 0; h < NZ; ++h) {
              const int i = sizeof(TV) == 2 && h == 0 ? lane : min(lane + 64 * h, last);
#pragma unroll
              for (int ij = 0; ij < NJ; ++ij)
                a[ij][h] = EDGE ? V.at_bits(e + i, ij * cS) : V.at_bits(i, e + ij * cS);
            }
          };
          // cells combined per z (R = sum_j wy_j V[j][z]) into LDS, then every row's taps
          auto use = [&](int j, const uint32_t(&a)[NJ][NZ]) {
            const float4 q = rec[j];
            const int kb = __builtin_amdgcn_readlane(q_kb, j);
            float wy[4] = {q.y, q.z, q.w, 0.f};
            if constexpr (NJ == 4) wy[3] = rdl(wy3, j);
            if constexpr (ONES && !EDGE) {
              float W = wy[0];
#pragma unroll
              for (int ij = 1; ij < NJ; ++ij) W += wy[ij];
              acc = fmaf(fmaf(q.x, Bv1, azf) - fmaf(q.x, Bv, azf), W, acc);
              return;
            }
#pragma unroll
            for (int h = 0; h < NZ; ++h) {
              float R = wy[0] * (ONES ? 1.f : Buf<TV>::widen(a[0][h]));
#pragma unroll
              for (int ij = 1; ij < NJ; ++ij)
                R = fmaf(wy[ij], ONES ? 1.f : Buf<TV>::widen(a[ij][h]), R);
              if constexpr (EDGE)
                R = (uint32_t)(kb + vp.azi + lane + 64 * h) < (uint32_t)d.ZN ? R : 0.f;
              zrun[lane + 64 * h] = R;
            }
            const float t = fmaf(q.x, Bv, azf), h = fmaf(q.x, Bv1, azf) - t;
            const Overlap3 w = overlap3<NT>(t, h);
            const float* z = zrun + (w.k - kb);
            float s = w.w0 * z[0];
            s = fmaf(w.w1, z[1], s);
            if constexpr (NT == 3) s = fmaf(w.w2, z[2], s);
            acc += s;
          };
          // the next slice's runs load while this one's are used (two sets in turn)
          uint32_t x0[NJ][NZ], x1[NJ][NZ];
          int j0 = __builtin_ctzll(m), j1;
          m &= m - 1;
          fetch(j0, x0);
          while (true) {
            if (!m) {
              use(j0, x0);
              break;
            }
            j1 = __builtin_ctzll(m);
            m &= m - 1;
            fetch(j1, x1);
            use(j0, x0);
            if (!m) {
              use(j1, x1);
              break;
            }
            j0 = __builtin_ctzll(m);
            m &= m - 1;
            fetch(j0, x0);
            use(j1, x1);
          }
        };
        auto cells = [&](auto NJ_) {
          run(NJ_, I2{}, F{}, F{}, 0);
          run(NJ_, I3{}, F{}, F{}, 1);
          run(NJ_, I3{}, T{}, F{}, 2);
          run(NJ_, I3{}, T{}, T{}, 3);
        };
        cells(I2{});
        cells(I3{});
        cells(I4{});
      } else {
        // one slice of a class: NJ cells (a cell past the group's own re-reads its last with
        // weight 0), NT z taps, EDGE footprints clamped to the volume's z range
        auto run = [&](auto NJ_, auto NT_, auto EDGE_, int id) {
          constexpr int NJ = decltype(NJ_)::value, NT = decltype(NT_)::value;
          constexpr bool EDGE = decltype(EDGE_)::value;
          uint64_t m = __ballot(key == 8 * NJ + id) & low;
          while (m) {
            const int j = __builtin_ctzll(m);
            m &= m - 1;
            const float4 q = rec[gbase + j];
            const int4 f = off[gbase + j];
            float t = fmaf(q.x, Bv, azf), h = fmaf(q.x, Bv1, azf) - t;
            if constexpr (ONES && !EDGE) {
              acc = fmaf(h, (q.y + q.z) + (q.w + __int_as_float(f.z)), acc);
              continue;
            }
            if constexpr (EDGE) {
              const float te = __builtin_elementwise_minimum(t + h, tmax);
              t = __builtin_elementwise_maximum(t, tmin);
              h = __builtin_elementwise_maximum(te - t, 0.f);
            }
            Overlap3 w = overlap3<NT>(t, h);
            if constexpr (EDGE) w.k = min(w.k, kmax);
            float a[NJ][3];
            const float wy[4] = {q.y, q.z, q.w, __int_as_float(f.z)};
            uint32_t e = (uint32_t)(w.k + f.x);
            // a group that the slice misses reads the array's first elements with weight 0
            if (f.y == 0) e = 0;
#pragma unroll
            for (int ij = 0; ij < NJ; ++ij) {
              if constexpr (ONES) a[ij][0] = a[ij][1] = a[ij][2] = 1.f;
              else z_run<NT>(V, A.vol, e, a[ij]);
              if (ij + 1 < f.y) e += cS;
            }
            float s = 0.f;
#pragma unroll
            for (int ij = 0; ij < NJ; ++ij) {
              float g = w.w0 * a[ij][0];
              g = fmaf(w.w1, a[ij][1], g);
              if constexpr (NT == 3) g = fmaf(w.w2, a[ij][2], g);
              s = ij == 0 ? wy[0] * g : fmaf(wy[ij], g, s);
            }
            acc += s;
          }
        };
        run(I2{}, I2{}, F{}, 0);
        run(I2{}, I3{}, F{}, 1);
        run(I2{}, I3{}, T{}, 3);
        run(I3{}, I2{}, F{}, 0);
        run(I3{}, I3{}, F{}, 1);
        run(I3{}, I3{}, T{}, 3);
        run(I4{}, I2{}, F{}, 0);
        run(I4{}, I3{}, F{}, 1);
        run(I4{}, I3{}, T{}, 3);
      }
      auto generals = [&](auto NJ_) {
        constexpr int NJ = decltype(NJ_)::value;
        uint64_t m = __ballot(key == 7 && (!FINE || mj == NJ)) & low;
        while (m) {
          const int j = __builtin_ctzll(m);
          m &= m - 1;
          if constexpr (!FINE) {
            general(ii0 + j);
          } else {
            const float4 q = rec[gbase + j];
            const int4 f = off[COLW ? 0 : gbase + j];
            const float wy[4] = {q.y, q.z, q.w, COLW ? rdl(wy3, j) : __int_as_float(f.z)};
            tall(NJ_, q.x, wy, COLW ? __builtin_amdgcn_readlane(q_e, j) : f.x,
                 COLW ? __builtin_amdgcn_readlane(q_nj, j) : f.y);
          }
        }
      };
      if constexpr (FINE) {
        generals(integral_constant<int, 1>{});
        generals(I2{});
        generals(I3{});
      }
      generals(I4{});
    }
    if constexpr (!ONES) {
      if (__builtin_expect(__any(vok && not_finite(acc)), 0)) {
        acc = 0.f;
        for (int ii = 0; ii < NS; ++ii) general(ii);
      }
    }
    if (vok) {
      const float K = ct.w * __builtin_amdgcn_sqrtf(ct.z + gp(A.h2)[v]) * gp(A.invdB)[v];
      const float val = acc * K;
      const size_t o = ((size_t)k * d.DNU + u) * d.DNV + v;
      if constexpr (FUSED) {
        const size_t og = ((size_t)p * d.DNU + u) * d.DNV + v;
        const float bb = gp(A.b)[og];
        const float diff = bb - val;
        if (A.out) st(gp(A.out), o, A.invRow ? diff * gp(A.invRow)[o] : diff);
        res = (double)diff * (double)diff;
        bsq = (double)bb * (double)bb;
      } else {
        st(gp(A.out), o, val);
      }
    }
  }
  if constexpr (FUSED) block_sum2(res, bsq, slot);
}

template <bool FUSED, bool COLW, typename TV, typename TO, bool FINE>
__global__ __launch_bounds__(kBlock) void fp_kernel(FpArgs<TV, TO> A, int bpv, int views) {
  const int hw = blockIdx.x;
  const int lb = xcd_chunked_block(hw);
  const int k = lb / bpv;
  if (k >= views) return;
  fp_body<FUSED, COLW, TV, TO, FINE>(A, k, lb - k * bpv, A.partials + 2 * lb);
}

// Forward projection of a volume of ones (A.vol unused).
template <bool COLW, bool FINE>
__global__ __launch_bounds__(kBlock) void fp_ones_kernel(FpArgs<float, float> A, int bpv,
                                                         int views) {
  const int lb = xcd_chunked_block(blockIdx.x);
  const int k = lb / bpv;
  if (k >= views) return;
  fp_body<false, COLW, float, float, FINE, true>(A, k, lb - k * bpv, nullptr);
}

// Batched persistent forward projection: each workgroup takes a range of the flat work list,
// items of one scan being consecutive (view-major, then column blocks).
// Work assignment of the batched kernels (sched): the workgroup's first item, the item
// step and the end.
//  0 contiguous: one range per workgroup, ranges ordered per XCD (neighbouring items
//    share an L2);
//  1 strided: items lb, lb + G, ... (every workgroup samples the whole list, which
//    balances uneven item costs);
//  2 one workgroup per item (G == total): workgroups are dispatched in order, so the
//    items of one scan run together on all XCDs, and within a scan's range every XCD takes one
//    contiguous part.
// The forward projector's own launches deal chunks to the XCDs in turn (xcd_chunked_block);
// the batched one does not, and falls behind them where the scans are large: sweeps of three
// scans of 512^2 x 256 86 ms, 74 ms scan by scan, of eight scans of 128^2 x 64 6.2 ms, 8.3 ms.
template <typename Item>
__device__ __forceinline__ void batch_range(const Item* __restrict__ D, int nscan, int total,
                                            int sched, int& i0, int& step, int& i1) {
  if (sched == 2) {
    const int hw = blockIdx.x;
    int s = 0;
    while (s + 1 < nscan && D[s + 1].begin <= hw) ++s;
    const int b0 = D[s].begin;
    const int n = (s + 1 < nscan ? D[s + 1].begin : total) - b0;
    i0 = b0 + xcd_logical_block(hw - b0, n);
    step = 1;
    i1 = i0 + 1;
    return;
  }
  const int lb = xcd_logical_block(blockIdx.x, gridDim.x);
  if (sched == 1) {
    i0 = lb;
    step = gridDim.x;
    i1 = total;
  } else {
    const int per = (total + gridDim.x - 1) / gridDim.x;
    i0 = lb * per;
    step = 1;
    i1 = min(total, i0 + per);
  }
}

template <bool FUSED, bool COLW, typename T, bool FINE>
__global__ __launch_bounds__(kBlock) void fp_batch_kernel(const FpBatchItem<T>* __restrict__ D,
                                                          int nscan, int total, int sched) {
  int i0, step, i1;
  batch_range(D, nscan, total, sched, i0, step, i1);
  int s = 0;
  for (int item = i0; item < i1; item += step) {
    if (sched == 1) s = 0;
    while (s + 1 < nscan && D[s + 1].begin <= item) ++s;
    const FpBatchItem<T>& B = D[s];
    const int local = item - B.begin;
    const int k = local / B.upv;
    fp_body<FUSED, COLW, T, T, FINE>(B.a, k, local - k * B.upv, B.a.partials + 2 * local);
  }
}


// fp_batch_kernel for the one-workgroup-per-item schedule (grid = total): no item loop.
template <bool FUSED, bool COLW, typename T, bool FINE>
__global__ __launch_bounds__(kBlock) void fp_batch1_kernel(const FpBatchItem<T>* __restrict__ D,
                                                           int nscan, int total) {
  int i0, step, i1;
  batch_range(D, nscan, total, 2, i0, step, i1);
  int s = 0;
  while (s + 1 < nscan && D[s + 1].begin <= i0) ++s;
  const FpBatchItem<T>& B = D[s];
  const int local = i0 - B.begin;
  const int k = local / B.upv;
  fp_body<FUSED, COLW, T, T, FINE>(B.a, k, local - k * B.upv, B.a.partials + 2 * local);
}

// ---------------------------------------------------------------------------
// Reference back projector: one wave per (x, y) column, each lane owning ZG
// voxels z = z0 + lane + 64 g (g < ZG), views looped inside.
// Reference: DD3_gpu_back_ker<_BRANCHLESS>, iterativeRecon/DD3_GPU.cu:1397-1475.
// The voxel's shadow in (fan-angle index, row index) space is integrated over the
// piecewise-constant sinogram and weighted by cosVal.  The fan-angle coordinate is
// the same for the whole column and is resolved in FP64 once per (column, view);
// the row coordinates are per lane in FP32.  A view whose row shadow misses the
// detector for every lane of a group is skipped for that group.
// UPDATE: vol += acc * invCol (os_sart.m:32,37-40), and shadow (when not NULL) gets
// the updated value rounded to BF16; otherwise vol = acc.
// T: storage type of prj (float, or uint16_t for BF16); vol is FP32.
// ---------------------------------------------------------------------------
// Per-(column, view) constants of the reference back projector, uniform over a wave:
// the fan-angle shadow (FP64) as first cell u0, cell count nu and first / last column
// weights, the cell-width factor with the sign of the corner difference folded in, and
// the row-shadow constants (rows of a voxel at dZ = Pz - sz: [dZ rlS + cA, dZ rlS + cB]).
struct BpView {
  float rlS, cA, cB, sz, l2, cws, wu0, fh;
  double rl;
  int u0, nu;
  bool uvis;
};

template <typename T>
__device__ __forceinline__ BpView bp_view(const BpArgs<T>& A, int p, double Px_, double Py_) {
  const Dims& d = A.d;
  const BpConsts& c = A.c;
  // (constants in scalar registers: hoisted out of a wave's loop over its views they would stand
  // in vector registers, which spilled)
  BpConsts64 c64 = A.c64;
  c64.inv_sid = held(c64.inv_sid);
  c64.dx = held(c64.dx);
  c64.ib = held(c64.ib);
  c64.cU = held(c64.cU);
  c64.S = held(c64.S);
  const double Px = held(Px_), Py = held(Py_);
  BpView r{};
  const ViewP vp = gload(A.views, p);
  // fan-angle shadow, FP64 (DD3_GPU.cu:1447-1464); sy*dX - sx*dY == sy*Px - sx*Py
  const double2 s64 = gload(A.src64, p);
  const double dX = Px - s64.x, dY = Py - s64.y;
  const double l2 = dX * dX + dY * dY;
  const double rl = rsqrt(l2);
  r.rl = rl;
  // row shadow (DD3_GPU.cu:1446-1450): t = (dZ +- hz) * S / l + cV
  const float rlS = (float)(rl * c64.S);
  const bool rneg = rlS < 0.f;  // rows then run backwards: swap the bounds
  const double alpha = asin_fan((s64.y * Px - s64.x * Py) * c64.inv_sid * rl);
  const double w = vp.wx ? dX : dY;
  const double dA = w * (rl * rl) * (c64.dx * 0.5);
  const double tL = (alpha - dA) * c64.ib + c64.cU;
  const double tR = (alpha + dA) * c64.ib + c64.cU;
  const double ulo = fmax(fmin(tL, tR), -0.5);
  const double uhi = fmin(fmax(tL, tR), (double)d.DNU - 0.5);
  r.uvis = ulo < uhi;
  if (r.uvis) {
    const int u0 = (int)floor(ulo + 0.5);
    const int nu = min((int)floor(uhi + 0.5), d.DNU - 1) - u0 + 1;
    // column weights: first / last partial, interior 1 (fractions taken in FP64)
    const float fl = (float)(((double)u0 + 0.5) - ulo);
    r.fh = (float)(uhi - ((double)(u0 + nu - 1) - 0.5));
    r.wu0 = (nu == 1) ? (float)(uhi - ulo) : fl;
    // sign of the reference's corner difference, (tR - tL) and (tU - tD), folded
    // into the cell-width factor (a sign flip is exact)
    const float sgn = ((tR < tL) != rneg) ? -1.f : 1.f;
    r.cws = sgn * (c.dx * __builtin_amdgcn_rcpf((float)w));
    r.u0 = u0;
    r.nu = nu;
  }
  const float cUp = fmaf(c.hz, rlS, c.cV), cDp = fmaf(-c.hz, rlS, c.cV);
  r.cA = rneg ? cUp : cDp;  // lower row bound
  r.cB = rneg ? cDp : cUp;  // upper row bound
  r.rlS = rlS;
  r.sz = vp.sz;
  r.l2 = (float)l2;
  return r;
}

// NU columns x 3 row taps of a shadow: all 3 NU loads are issued before the first is
// used (NU is the uniform column count, so every case is straight-line code), then the
// taps are combined in the order of the general loop below.
// NT = 2 when no lane of the wave needs a third row (wv2 == 0 everywhere: the term it
// drops is an exact zero).
template <int NU, int NT, typename T>
__device__ __forceinline__ float bp_cells(const Buf<T>& pp, int o, int DNV, int t1, int t2,
                                          float wv0, float wv1, float wv2, float wu0, float fh) {
  // no contraction: an interior column's weight 1 would otherwise fuse its add with the
  // first column's product, which the staged rows of bp_win_body (a run-time weight)
  // round separately
#pragma clang fp contract(off)
  float a[NU][3];
#pragma unroll
  for (int iu = 0; iu < NU; ++iu) {
    if constexpr (NT == 3) {
      pp.tap3(o + iu * DNV, t1, t2, a[iu][0], a[iu][1], a[iu][2]);
    } else {
      a[iu][0] = pp[o + iu * DNV];
      a[iu][1] = pp[o + iu * DNV + t1];
    }
  }
  // rows first combined over the columns (R_t = sum_u wu y[u][v0 + t]), then over the rows
  float R[3];
#pragma unroll
  for (int t = 0; t < NT; ++t) R[t] = wu0 * a[0][t];
#pragma unroll
  for (int iu = 1; iu < NU; ++iu) {
    const float wu = (iu == NU - 1) ? fh : 1.f;
#pragma unroll
    for (int t = 0; t < NT; ++t) R[t] = fmaf(wu, a[iu][t], R[t]);
  }
  float s = wv0 * R[0];
  s = fmaf(wv1, R[1], s);
  if constexpr (NT == 3) s = fmaf(wv2, R[2], s);
  return s;
}

// The voxel's shadow [vlo, vhi] (rows) x nu columns from offset o0 on integrated over the
// piecewise-constant view pp (first / last column weights wu0, fh).
template <typename T>
__device__ __forceinline__ float bp_cell_sum(const Buf<T>& pp, int o0, int nu, float wu0,
                                             float fh, float vlo, float vhi, int DNV) {
#pragma clang fp contract(off)
  // first row v0 = floor(vlo + .5) and its upper edge e; with d = vhi - e the overlaps of
  // rows v0, v0 + 1, v0 + 2 are min(vhi, e) - vlo, clamp(d, 0, 1), clamp(d - 1, 0, 1)
  // (the first / interior / last weights of edge_weights, without the row count)
  const float fv = floorf(vlo + 0.5f);
  const float e = fv + 0.5f;
  const int v0 = (int)fv;
  const float d = vhi - e;
  float s = 0.f;
  if (nu <= 4 && d <= 2.f) {
    const float wv0 = fminf(vhi, e) - vlo;
    const float wv1 = __builtin_amdgcn_fmed3f(d, 0.f, 1.f);
    const float wv2 = __builtin_amdgcn_fmed3f(d - 1.f, 0.f, 1.f);
    // taps of zero weight re-read the first row (never a row outside the shadow)
    const int t1 = d > 0.f ? 1 : 0, t2 = d > 1.f ? 2 : 0;
    const int o = o0 + v0;
    if (!__any(d > 1.f)) {  // at most two rows in every lane's shadow
      switch (nu) {  // uniform over the wave
        case 1: s = bp_cells<1, 2>(pp, o, DNV, t1, t2, wv0, wv1, wv2, wu0, fh); break;
        case 2: s = bp_cells<2, 2>(pp, o, DNV, t1, t2, wv0, wv1, wv2, wu0, fh); break;
        case 3: s = bp_cells<3, 2>(pp, o, DNV, t1, t2, wv0, wv1, wv2, wu0, fh); break;
        default: s = bp_cells<4, 2>(pp, o, DNV, t1, t2, wv0, wv1, wv2, wu0, fh); break;
      }
    } else {
      switch (nu) {
        case 1: s = bp_cells<1, 3>(pp, o, DNV, t1, t2, wv0, wv1, wv2, wu0, fh); break;
        case 2: s = bp_cells<2, 3>(pp, o, DNV, t1, t2, wv0, wv1, wv2, wu0, fh); break;
        case 3: s = bp_cells<3, 3>(pp, o, DNV, t1, t2, wv0, wv1, wv2, wu0, fh); break;
        default: s = bp_cells<4, 3>(pp, o, DNV, t1, t2, wv0, wv1, wv2, wu0, fh); break;
      }
    }
  } else {
    const int nv = min((int)floorf(vhi + 0.5f), DNV - 1) - v0 + 1;
    float wv0, wvl;
    edge_weights(vlo, vhi, v0, nv, wv0, wvl);
    for (int iv = 0; iv < nv; ++iv) {
      const float wv = (iv == 0) ? wv0 : (iv == nv - 1 ? wvl : 1.f);
      const int o = o0 + v0 + iv;
      float R = wu0 * pp[o];
      for (int iu = 1; iu < nu; ++iu) R = fmaf((iu == nu - 1) ? fh : 1.f, pp[o + iu * DNV], R);
      s = fmaf(wv, R, s);
    }
  }
  return s;
}

// Final value of voxel z of a column: vol = acc, or the OS-SART update
// vol += acc * invCol (and its BF16 shadow).
template <bool UPDATE, typename T>
__device__ __forceinline__ void bp_store(const BpArgs<T>& A, CTR_GLOBAL float* vcol, int col,
                                         int z, float acc) {
  if constexpr (UPDATE) {
    const size_t i = (size_t)col * A.d.ZN + z;
    const float nx = fmaf(acc, gp(A.invCol)[i], vcol[z]);
    vcol[z] = nx;
    if (A.shadow) gp(A.shadow)[i] = to_bf16_dither(nx, i);
  } else {
    vcol[z] = acc;
  }
}

template <bool UPDATE, int ZG, typename T>
__device__ __forceinline__ void bp_ref_body(const BpArgs<T>& A, int col, int zblk) {
  const Dims& d = A.d;
  const BpConsts64& c64 = A.c64;
  const int lane = threadIdx.x & 63;
  if (col >= d.XN * d.YN) return;
  const int zb0 = zblk * (64 * ZG);  // first z of the wave (uniform)
  const int zb = zb0 + lane;
  const int y = col / d.XN, x = col - y * d.XN;
  CTR_GLOBAL float* vcol = gp(A.vol) + (size_t)col * d.ZN;
  if (gp(A.mask)[col] != 1) {
    if constexpr (!UPDATE) {
#pragma unroll
      for (int g = 0; g < ZG; ++g)
        if (zb + 64 * g < d.ZN) vcol[zb + 64 * g] = 0.f;
    }
    return;
  }
  const double Px = held(((double)x - c64.ocx) * c64.dx);
  const double Py = held(((double)y - c64.ocy) * c64.dx);
  // z extent of the wave's voxel centres (uniform), for the whole-column view test
  const float Zlo = ((float)zb0 - d.ocz) * d.dz;
  const float Zhi = ((float)min(zb0 + 64 * ZG, d.ZN) - 1.f - d.ocz) * d.dz;
  float acc[ZG];
#pragma unroll
  for (int g = 0; g < ZG; ++g) acc[g] = 0.f;
  const float DNVh = (float)d.DNV - 0.5f;
  const int DNV = d.DNV;
  const uint32_t frame = (uint32_t)(d.DNU * d.DNV);
  // Views are taken 64 at a time: lane l first evaluates everything of view k0 + l that
  // is uniform over the column (visibility, fan-angle shadow in FP64, column weights,
  // row-shadow constants); the loop over the visible views then reads them with
  // readlane into scalar registers.  The arithmetic per view is unchanged.
  for (int k0 = 0; k0 < A.vc; k0 += 64) {
    const int kl = k0 + lane;
    BpView q{};
    bool vis = false;
    if (kl < A.vc) {
      q = bp_view(A, A.vb + kl * A.vs, Px, Py);
      // the whole group range of rows, to skip views the wave's voxels do not meet
      const float ta = fmaf(Zlo - q.sz, q.rlS, q.cA), tb = fmaf(Zhi - q.sz, q.rlS, q.cB);
      vis = q.uvis && fmaxf(ta, tb) > -0.5f && fminf(ta, tb) < DNVh;
    }
    uint64_t live = __ballot(vis);
    while (live) {
      const int j = __builtin_ctzll(live);
      live &= live - 1;
      const int k = k0 + j;
      const float rlS = rdl(q.rlS, j), cA = rdl(q.cA, j), cB = rdl(q.cB, j);
      const float vsz = rdl(q.sz, j), l2f = rdl(q.l2, j), cws = rdl(q.cws, j);
      const float wu0 = rdl(q.wu0, j), fh = rdl(q.fh, j);
      const int u0 = __builtin_amdgcn_readlane(q.u0, j), nu = __builtin_amdgcn_readlane(q.nu, j);
      const Buf<T> pp(A.prj + (size_t)k * frame, frame);
#pragma unroll
      for (int g = 0; g < ZG; ++g) {
        // voxel centre offset as in bp_win_body: one explicit fma, so that neither body
        // can round it differently (a hoisted product would be rounded on its own)
        const float dZ = fmaf((float)(zb + 64 * g) - d.ocz, d.dz, -vsz);
        const float vlo = fmaxf(fmaf(dZ, rlS, cA), -0.5f);
        const float vhi = fminf(fmaf(dZ, rlS, cB), DNVh);
        const bool vok = zb + 64 * g < d.ZN && vlo < vhi;
        if (!__any(vok)) continue;
        if (!vok) continue;
        const float cosVal = cws * __builtin_amdgcn_sqrtf(fmaf(dZ, dZ, l2f));
        acc[g] = fmaf(cosVal, bp_cell_sum(pp, u0 * DNV, nu, wu0, fh, vlo, vhi, DNV), acc[g]);
      }
    }
  }
#pragma unroll
  for (int g = 0; g < ZG; ++g) {
    const int z = zb + 64 * g;
    if (z < d.ZN) bp_store<UPDATE>(A, vcol, col, z, acc[g]);
  }
}

// Voxels of a column that view q's row shadow can reach: those with
// fmaf(dZ, rlS, cB) > -0.5 and fmaf(dZ, rlS, cA) < DNV - 0.5 lie in an open interval of
// voxel indices whose FP32 ends are within ~1e-4 of it, so the integers inside it widened
// by 1e-2 include every one of them.
__device__ __forceinline__ void bp_window(const Dims& d, const BpView& q, int& z0, int& z1) {
  const float DNVh = (float)held(d.DNV) - 0.5f, ZNf = (float)held(d.ZN), idz = held(d.idz);
  const float ocz = held(d.ocz);
  const float ea = (-0.5f - q.cB) / q.rlS, eb = (DNVh - q.cA) / q.rlS;
  const float za = fminf(fmaxf((fminf(ea, eb) + q.sz) * idz + ocz, -4.f), ZNf + 4.f);
  const float zb = fminf(fmaxf((fmaxf(ea, eb) + q.sz) * idz + ocz, -4.f), ZNf + 4.f);
  z0 = max((int)floorf(za - 1e-2f) + 1, 0);
  z1 = min((int)ceilf(zb + 1e-2f) - 1, d.ZN - 1);
}

// fetch(j, set), use(j, set) over the set bits j of m, one after the other.
template <typename Set, typename Fetch, typename Use>
__device__ __forceinline__ void in_turn(uint64_t m, Fetch fetch, Use use) {
  for (; m; m &= m - 1) {
    const int j = __builtin_ctzll(m);
    Set x;
    fetch(j, x);
    use(j, x);
  }
}

// Runs f(slot, j) ... over the set bits j of m with the fetches of the next bit in flight:
// fetch(j, set) loads into one of two register sets, use(j, set) consumes it.
template <typename Set, typename Fetch, typename Use>
__device__ __forceinline__ void pipelined(uint64_t m, Fetch fetch, Use use) {
  Set x0, x1;
  int j0 = __builtin_ctzll(m), j1;
  m &= m - 1;
  fetch(j0, x0);
  while (true) {
    if (!m) {
      use(j0, x0);
      break;
    }
    j1 = __builtin_ctzll(m);
    m &= m - 1;
    fetch(j1, x1);
    use(j0, x0);
    if (!m) {
      use(j1, x1);
      break;
    }
    j0 = __builtin_ctzll(m);
    m &= m - 1;
    fetch(j0, x0);
    use(j1, x1);
  }
}

// The same over i = 0 ... n - 1 (n > 0).
template <typename Set, typename Fetch, typename Use>
__device__ __forceinline__ void pipelined_n(int n, Fetch fetch, Use use) {
  Set x0, x1;
  fetch(0, x0);
  for (int i = 0;; i += 2) {
    if (i + 1 < n) fetch(i + 1, x1);
    use(i, x0);
    if (i + 1 >= n) break;
    if (i + 2 < n) fetch(i + 2, x0);
    use(i + 1, x1);
    if (i + 2 >= n) break;
  }
}

// Windowed form of bp_ref_body: one wave per voxel column over all of its z.  On a
// helical scan a view's cone covers a window of a few dozen voxels of a column, which
// fixed lane -> z groups cover with one 64-lane pass per group it touches (about half the
// lanes idle).  Here the lanes take the view's own window, z0 + lane, z0 + 64 + lane, ...,
// and the column's sums live in LDS.
//
// Staged rows (DNV <= 64 RC, RC = 1, 2, 4): 64 views at a time, lane l evaluates view
// k0 + l (fan-angle shadow in FP64, column weights times cosVal's width factor, the row
// shadow T(z) = T0 + (z - z0) s of its window in units of rows, row edges at integers) into
// the wave's LDS records and sorts the view into a class by its number of columns and of
// 64-voxel passes.  Each class runs its views in a loop of straight-line code: every lane
// loads its row of the view's columns (the next view's rows load meanwhile) and combines
// them (R[v] = sum_u w_u y[u][v]) into LDS, four rows of zeros on either side, and a voxel
// takes the three rows that its shadow [T, T + s] can overlap, without clamps.
// Views of more than four columns, or whose shadows are taller than two rows (key 1), follow in
// a second loop: any number of columns, five rows, or the shadow's own rows.
// Bound by VALU issue (0.98 of the chip's rate).  512^2 x 256, 197 views of 888 x 64:
// 3.76 ms with the views in order, four column loads and two-row clamps for each, 2.40 ms
// (BF16 sinogram 3.85 ms, 2.43 ms); 256^2 x 128 of 1 mm 0.92 ms, 0.61 ms; 277^2 x 165, 164 views
// of 611 x 80 in BF16, without staged rows 1.78 ms, with two chunks of rows 0.67 ms.  Grids where
// most views are of the second kind run view by view (bp_plain_body, bp_shape).
constexpr int kPadRows = 4, kPadEnd = 5;
template <int RC>
constexpr int kRowsLds = 64 * RC + 12;  // zeros, rows, zeros, a slot for idle lanes
template <int RC>
constexpr int kStagedF = kRowsLds<RC> + 64 * 8;   // floats of a staged wave before its sums

// Rows of a staged wave: the zero rows written once, and each lane's slot for row
// lane + 64 c (idle lanes write to a slot that is never read).
template <int RC>
__device__ __forceinline__ void stage_rows(float* rows, int DNV, int lane, int (&row)[RC],
                                           int (&slot)[RC]) {
  if (lane < kPadRows) rows[lane] = 0.f;
  if (lane < kPadEnd) rows[kPadRows + DNV + lane] = 0.f;
#pragma unroll
  for (int c = 0; c < RC; ++c) {
    const int v = lane + 64 * c;
    row[c] = min(v, DNV - 1);
    slot[c] = v < DNV ? v + kPadRows : 64 * RC + kPadRows + kPadEnd;
  }
}

// View kl's record: the window z0 ... z1; r = (T0, s, dZ of voxel z0, l^2); the weights w of up
// to four columns; the offset o of the first; its class key = columns * 2 + (more than `lanes`
// voxels), 0 when nothing is visible.  key = 1: more than four columns, or shadows of more than
// two rows, or `exact`; then w = (width factor, first, last partial weight, number of columns).
struct BpRecord {
  float4 r, w;
  int z0, z1, o, key;
};
template <typename T>
__device__ __forceinline__ BpRecord bp_record(const BpArgs<T>& A, int kl, double Px, double Py,
                                              int lanes, bool exact) {
#pragma clang fp contract(off)
  const Dims& d = A.d;
  BpConsts64 c64 = A.c64;
  c64.S = held(c64.S);
  c64.cV = held(c64.cV);
  c64.ocz = held(c64.ocz);
  BpRecord v{};
  v.z1 = -1;
  const BpView q = bp_view(A, A.vb + kl * A.vs, Px, Py);
  bp_window(d, q, v.z0, v.z1);
  if (q.uvis && v.z0 <= v.z1) {
    // row shadow of the window's first voxel and its step, dZ of that voxel
    const double rlS = q.rl * c64.S, dz = (double)d.dz;
    const double dZ = ((double)v.z0 - c64.ocz) * dz - (double)q.sz;
    const float s = (float)(dz * rlS);
    const float T0 = (float)((dZ - 0.5 * dz) * rlS + (c64.cV + 0.5));
    const int nu = q.nu;
    v.r = make_float4(T0, s, (float)dZ, q.l2);
    v.w = make_float4(q.cws * q.wu0, nu > 1 ? q.cws * (nu == 2 ? q.fh : 1.f) : 0.f,
                      nu > 2 ? q.cws * (nu == 3 ? q.fh : 1.f) : 0.f, nu > 3 ? q.cws * q.fh : 0.f);
    v.o = q.u0 * d.DNV;
    v.key = 2 * nu + (v.z1 - v.z0 >= lanes ? 1 : 0);
    if (exact || nu > 4 || s > 2.f) {
      v.key = 1;
      v.w = make_float4(q.cws, q.wu0, q.fh, __int_as_float(nu));
    }
  }
  return v;
}

// Column c's weight of a record of key 1.
__device__ __forceinline__ float rest_weight(const float4& w, int c, int n) {
#pragma clang fp contract(off)
  return w.x * (c == 0 ? w.y : c == n - 1 ? w.z : 1.f);
}

// Shadows of five taps: under four rows by more than the window's margin, so that the first tap
// lies on the row set's zeros (the last does for any).
constexpr float kTaps5 = 3.9f;

// Sum of the rows R[0 ... DNV) that [t, t + s] overlaps, for shadows of any height.
__device__ __forceinline__ float tall_rows(const float* R, float t, float s, float DNVf) {
#pragma clang fp contract(off)
  const float lo = fmaxf(t, 0.f), hi = fminf(t + s, DNVf);
  if (!(lo < hi)) return 0.f;
  const int v0 = (int)lo, v1 = (int)ceilf(hi) - 1;
  const float first = R[v0], last = R[v1];
  float mid = 0.f;
  // the rows between, four reads at a time (past the end: the last row, not added)
  for (int v = v0 + 1; v < v1; v += 4) {
    float a[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) a[i] = R[min(v + i, v1)];
#pragma unroll
    for (int i = 0; i < 4; ++i) mid += v + i < v1 ? a[i] : 0.f;
  }
  const float sum = fmaf(fminf(hi, (float)(v0 + 1)) - lo, first, mid);
  return v1 > v0 ? fmaf(hi - (float)v1, last, sum) : sum;
}

// A voxel's share of a view: its shadow's overlaps with the rows (R0: the row set's first row)
// times cosVal, in TAPS rows (3: shadows of up to two rows, 5: of up to kTaps5) or, 0, only the
// rows that it overlaps.
template <int TAPS>
__device__ __forceinline__ float bp_voxel(const Dims& d, const float4& r, float zi,
                                          const float* R0, float acc) {
#pragma clang fp contract(off)
  const float t = fmaf(zi, r.y, r.x);
  float sum;
  if constexpr (TAPS == 0) {
    sum = tall_rows(R0, t, r.y, (float)d.DNV);
  } else if constexpr (TAPS == 5) {
    const Overlap5 o = overlap5(t, r.y);
    const float* R = R0 + o.k;
    sum = o.w[0] * R[0];
#pragma unroll
    for (int i = 1; i < 5; ++i) sum = fmaf(o.w[i], R[i], sum);
  } else {
    const Overlap3 o = overlap3<3>(t, r.y);
    const float* R = R0 + o.k;
    sum = o.w0 * R[0];
    sum = fmaf(o.w1, R[1], sum);
    sum = fmaf(o.w2, R[2], sum);
  }
  const float dZ = fmaf(zi, d.dz, r.z);
  return fmaf(__builtin_amdgcn_sqrtf(fmaf(dZ, dZ, r.w)), sum, acc);
}

// f(columns, more than one pass) for every class of up to four columns.
template <typename F>
__device__ __forceinline__ void for_classes(F f) {
  using std::integral_constant;
  using N = std::false_type;
  using Y = std::true_type;
  f(integral_constant<int, 1>{}, N{});
  f(integral_constant<int, 1>{}, Y{});
  f(integral_constant<int, 2>{}, N{});
  f(integral_constant<int, 2>{}, Y{});
  f(integral_constant<int, 3>{}, N{});
  f(integral_constant<int, 3>{}, Y{});
  f(integral_constant<int, 4>{}, N{});
  f(integral_constant<int, 4>{}, Y{});
}

// Whether any of a wave's n sums is not finite; they are zeroed then.
__device__ __forceinline__ bool reset_not_finite(float* lacc, int n) {
  const int lane = threadIdx.x & 63;
  bool bad = false;
  for (int i = lane; i < n; i += 64) bad = bad || not_finite(lacc[i]);
  if (!__any(bad)) return false;
  for (int i = lane; i < n; i += 64) lacc[i] = 0.f;
  return true;
}

// ONES: the back projection of a sinogram of ones (the column sums of OS-SART), read from no
// sinogram, with the weights of the back projection itself: a voxel that a shadow grazes by a
// rounding error then has a column sum that matches its update.
template <bool UPDATE, typename T, int RC, bool ONES = false>
__device__ __forceinline__ void bp_staged_body(const BpArgs<T>& A, int col, float* lds) {
#pragma clang fp contract(off)
  const Dims& d = A.d;
  const BpConsts64& c64 = A.c64;
  const int lane = threadIdx.x & 63;
  if (col >= d.XN * d.YN) return;
  const int y = col / d.XN, x = col - y * d.XN;
  CTR_GLOBAL float* vcol = gp(A.vol) + (size_t)col * d.ZN;
  if (gp(A.mask)[col] != 1) {
    if constexpr (!UPDATE) {
      for (int z = lane; z < d.ZN; z += 64) vcol[z] = 0.f;
    }
    return;
  }
  float* rows = lds;
  float4* rec = reinterpret_cast<float4*>(lds + kRowsLds<RC>);  // [64][2]
  float* lacc = lds + kStagedF<RC>;
  for (int z = lane; z < d.ZN; z += 64) lacc[z] = 0.f;
  const int DNV = d.DNV;
  int row[RC], slot[RC];
  stage_rows<RC>(rows, DNV, lane, row, slot);
  const double Px = held(((double)x - c64.ocx) * c64.dx);
  const double Py = held(((double)y - c64.ocy) * c64.dx);
  const int frame = d.DNU * DNV;
  const float lanef = (float)lane;
  bool rest = false;
  for (int k0 = 0; k0 < A.vc; k0 += 64) {
    const int kl = k0 + lane;
    BpRecord v{};
    if (kl < A.vc) v = bp_record(A, kl, Px, Py, 64, false);
    const int z0 = v.z0, z1 = v.z1, q_o = lane * frame + v.o, key = v.key;
    if (!__any(key)) continue;
    rest = rest || __any(key == 1);
    if (key) {
      rec[2 * lane] = v.r;
      rec[2 * lane + 1] = v.w;
    }
    const Buf<T> P(A.prj + (size_t)k0 * frame, (uint32_t)min(64, A.vc - k0) * (uint32_t)frame);
    for_classes([&](auto NU_, auto MULTI_) {
      constexpr int NU = decltype(NU_)::value;
      constexpr bool MULTI = decltype(MULTI_)::value;
      const uint64_t m = __ballot(key == 2 * NU + (MULTI ? 1 : 0));
      if (!m) return;
      struct Set {
        uint32_t y[NU][RC];
      };
      pipelined<Set>(
          m,
          [&](int j, Set& f) {
            if constexpr (ONES) return;
            const int o = __builtin_amdgcn_readlane(q_o, j);
#pragma unroll
            for (int iu = 0; iu < NU; ++iu)
#pragma unroll
              for (int c = 0; c < RC; ++c) f.y[iu][c] = P.at_bits(row[c], o + iu * DNV);
          },
          [&](int j, const Set& f) {
            const float4 r = rec[2 * j], w = rec[2 * j + 1];
            const float wu[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
            for (int c = 0; c < RC; ++c) {
              float R = wu[0] * (ONES ? 1.f : Buf<T>::widen(f.y[0][c]));
#pragma unroll
              for (int iu = 1; iu < NU; ++iu)
                R = fmaf(wu[iu], ONES ? 1.f : Buf<T>::widen(f.y[iu][c]), R);
              rows[slot[c]] = R;
            }
            const int zf = __builtin_amdgcn_readlane(z0, j);
            const int n = __builtin_amdgcn_readlane(z1, j) - zf;
            auto pass = [&](float zi, int zz) {
              float* a = lacc + zf + zz + lane;
              *a = bp_voxel<3>(d, r, zi, rows + kPadRows, *a);
            };
            if constexpr (MULTI) {
              float zi = lanef;
              for (int zz = 0; zz <= n; zz += 64, zi += 64.f)
                if (lane <= n - zz) pass(zi, zz);
            } else {
              if (lane <= n) pass(lanef, 0);
            }
          });
    });
  }
  // the views of key 1; all of them where a sum is not finite
  bool exact = false;
  if constexpr (!ONES) exact = reset_not_finite(lacc, d.ZN);
  if (rest || exact)
    for (int k0 = 0; k0 < A.vc; k0 += 64) {
      const int kl = k0 + lane;
      BpRecord v{};
      if (kl < A.vc) v = bp_record(A, kl, Px, Py, 64, exact);
      const uint64_t m = __ballot(v.key == 1);
      if (!m) continue;
      rec[2 * lane] = v.r;
      rec[2 * lane + 1] = v.w;
      const int q_o = lane * frame + v.o;
      const Buf<T> P(A.prj + (size_t)k0 * frame, (uint32_t)min(64, A.vc - k0) * (uint32_t)frame);
      struct Set {
        uint32_t y[4][RC];
      };
      auto load = [&](int o, int c0, int n, Set& f) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int c = 0; c < RC; ++c)
            f.y[i][c] = ONES ? 0u : P.at_bits(row[c], o + min(c0 + i, n - 1) * DNV);
      };
      pipelined<Set>(
          m,
          [&](int j, Set& f) {
            load(__builtin_amdgcn_readlane(q_o, j), 0, __float_as_int(rdl(v.w.w, j)), f);
          },
          [&](int j, const Set& f0) {
            const float4 r = rec[2 * j], w = rec[2 * j + 1];
            const int o = __builtin_amdgcn_readlane(q_o, j);
            const int n = __float_as_int(rdl(v.w.w, j));
            float R[RC] = {};
            Set f = f0;
            for (int c0 = 0;;) {
#pragma unroll
              for (int i = 0; i < 4; ++i)
                if (c0 + i < n) {
                  const float wc = rest_weight(w, c0 + i, n);
#pragma unroll
                  for (int c = 0; c < RC; ++c)
                    R[c] = fmaf(wc, ONES ? 1.f : Buf<T>::widen(f.y[i][c]), R[c]);
                }
              if ((c0 += 4) >= n) break;
              load(o, c0, n, f);
            }
#pragma unroll
            for (int c = 0; c < RC; ++c) rows[slot[c]] = R[c];
            bool own = exact || rdl(v.r.y, j) > kTaps5;  // read the shadow's own rows only
#pragma unroll
            for (int c = 0; c < RC; ++c) own = own || not_finite(R[c]);
            const int zf = __builtin_amdgcn_readlane(v.z0, j);
            const int zn = __builtin_amdgcn_readlane(v.z1, j) - zf;
            const float* R0 = rows + kPadRows;
            float* a = lacc + zf;
            if (__any(own)) {
              for (int zz = lane; zz <= zn; zz += 64)
                a[zz] = bp_voxel<0>(d, r, (float)zz, R0, a[zz]);
            } else {
              for (int zz = lane; zz <= zn; zz += 64)
                a[zz] = bp_voxel<5>(d, r, (float)zz, R0, a[zz]);
            }
          });
    }
  for (int z = lane; z < d.ZN; z += 64) bp_store<UPDATE>(A, vcol, col, z, lacc[z]);
}

// Staged rows view by view, in one loop for any number of columns and rows: short, for where the
// classes do not pay (bp_shape).  Otherwise as bp_staged_body; rows that are not finite are read
// only by the shadows that they lie in.
template <bool UPDATE, typename T, int RC, bool ONES = false>
__device__ __forceinline__ void bp_plain_body(const BpArgs<T>& A, int col, float* lds) {
#pragma clang fp contract(off)
  const Dims& d = A.d;
  const BpConsts64& c64 = A.c64;
  const int lane = threadIdx.x & 63;
  if (col >= d.XN * d.YN) return;
  const int y = col / d.XN, x = col - y * d.XN;
  CTR_GLOBAL float* vcol = gp(A.vol) + (size_t)col * d.ZN;
  if (gp(A.mask)[col] != 1) {
    if constexpr (!UPDATE) {
      for (int z = lane; z < d.ZN; z += 64) vcol[z] = 0.f;
    }
    return;
  }
  float* rows = lds;
  float4* rec = reinterpret_cast<float4*>(lds + kRowsLds<RC>);  // [64][2]
  float* lacc = lds + kStagedF<RC>;
  for (int z = lane; z < d.ZN; z += 64) lacc[z] = 0.f;
  const int DNV = d.DNV;
  int row[RC], slot[RC];
  stage_rows<RC>(rows, DNV, lane, row, slot);
  const double Px = held(((double)x - c64.ocx) * c64.dx);
  const double Py = held(((double)y - c64.ocy) * c64.dx);
  const int frame = d.DNU * DNV;
  for (int k0 = 0; k0 < A.vc; k0 += 64) {
    const int kl = k0 + lane;
    BpRecord v{};
    if (kl < A.vc) v = bp_record(A, kl, Px, Py, 64, true);
    const uint64_t m = __ballot(v.key != 0);
    if (!m) continue;
    const int nu = __float_as_int(v.w.w);
    const float wx = v.w.x, wl = v.w.x * v.w.z;
    if (v.key) {
      rec[2 * lane] = v.r;
      rec[2 * lane + 1] = make_float4(v.w.x * v.w.y, nu > 1 ? (nu == 2 ? wl : wx) : 0.f,
                                      nu > 2 ? (nu == 3 ? wl : wx) : 0.f,
                                      nu > 3 ? (nu == 4 ? wl : wx) : 0.f);
    }
    const int q_o = lane * frame + v.o;
    const Buf<T> P(A.prj + (size_t)k0 * frame, (uint32_t)min(64, A.vc - k0) * (uint32_t)frame);
    struct Set {
      uint32_t y[4][RC];
    };
    auto fetch = [&](int j, Set& f) {
      if constexpr (ONES) return;
      const int o = __builtin_amdgcn_readlane(q_o, j), n = __builtin_amdgcn_readlane(nu, j);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int c = 0; c < RC; ++c) f.y[i][c] = P.at_bits(row[c], o + min(i, n - 1) * DNV);
    };
    auto use = [&](int j, const Set& f) {
      const float4 r = rec[2 * j], w = rec[2 * j + 1];
      const int n = __builtin_amdgcn_readlane(nu, j);
      const float wu[4] = {w.x, w.y, w.z, w.w};
      float R[RC];
#pragma unroll
      for (int c = 0; c < RC; ++c) {
        R[c] = wu[0] * (ONES ? 1.f : Buf<T>::widen(f.y[0][c]));
#pragma unroll
        for (int i = 1; i < 4; ++i)
          R[c] = fmaf(wu[i], ONES ? 1.f : Buf<T>::widen(f.y[i][c]), R[c]);
      }
      if (n > 4) {
        const int o = __builtin_amdgcn_readlane(q_o, j);
        const float wj = rdl(wx, j), lj = rdl(wl, j);
#pragma unroll 4
        for (int i = 4; i < n; ++i)
#pragma unroll
          for (int c = 0; c < RC; ++c)
            R[c] = fmaf(i == n - 1 ? lj : wj,
                        ONES ? 1.f : Buf<T>::widen(P.at_bits(row[c], o + i * DNV)), R[c]);
      }
      bool bad = false;
#pragma unroll
      for (int c = 0; c < RC; ++c) {
        rows[slot[c]] = R[c];
        bad = bad || not_finite(R[c]);
      }
      const float s = rdl(v.r.y, j);
      const int zf = __builtin_amdgcn_readlane(v.z0, j);
      const int zn = __builtin_amdgcn_readlane(v.z1, j) - zf;
      const float* R0 = rows + kPadRows;
      float* a = lacc + zf;
      if (s > kTaps5 || __any(bad)) {
        for (int zz = lane; zz <= zn; zz += 64) {
          if constexpr (ONES) {
            // every row of the shadow holds R
            const float t = fmaf((float)zz, r.y, r.x), dZ = fmaf((float)zz, d.dz, r.z);
            const float h = fmaxf(fminf(t + r.y, (float)DNV) - fmaxf(t, 0.f), 0.f);
            a[zz] = fmaf(__builtin_amdgcn_sqrtf(fmaf(dZ, dZ, r.w)), R[0] * h, a[zz]);
          } else {
            a[zz] = bp_voxel<0>(d, r, (float)zz, R0, a[zz]);
          }
        }
      } else if (s > 2.f) {
        for (int zz = lane; zz <= zn; zz += 64)
          a[zz] = bp_voxel<5>(d, r, (float)zz, R0, a[zz]);
      } else {
        for (int zz = lane; zz <= zn; zz += 64)
          a[zz] = bp_voxel<3>(d, r, (float)zz, R0, a[zz]);
      }
    };
    // (more row chunks run for a view or two only, and take the registers of one set)
    if constexpr (RC == 1) pipelined<Set>(m, fetch, use);
    else in_turn<Set>(m, fetch, use);
  }
  for (int z = lane; z < d.ZN; z += 64) bp_store<UPDATE>(A, vcol, col, z, lacc[z]);
}

// Staged rows with several views at a time, for detectors of few rows (bp_pack_lanes): the wave
// is split into G = 64 / L groups of L lanes, as many as a view's rows and its window of a
// column take, and each group takes its own view of a class, with its own rows and column sums
// in LDS (added up at the end, groups in order).  The records are sorted by class, so that a
// group reads its view's next to its neighbour's.  Otherwise as bp_staged_body.
// 197 views of 888 columns, one view at a time and packed: 64^3, 16 rows 71 us, 30 us (3 groups);
// 256^2 x 128, 16 rows 573 us, 327 us, 8 rows 567 us, 236 us (6 groups).
constexpr int kPackRowsLds = 64 + 8 * (kPadRows + kPadEnd + 1);  // up to 8 groups of rows
constexpr int kPackF = kPackRowsLds + 64 * 12;  // floats of a wave before its sums
struct Groups {
  int L, G, inv, grp, gl, row, slot, rows, sums;
  // rows, sums: offsets of the group's rows and column sums (ZN4 floats each)
  __device__ __forceinline__ Groups(int L_, int DNV, int ZN4)
      : L(L_), G(64 / L_), inv((65536 + G - 1) / G) {
    const int lane = threadIdx.x & 63;
    grp = min(lane / L, G - 1);
    gl = lane - grp * L;  // (lanes past the last group: >= L, never active)
    row = min(gl, DNV - 1);
    rows = grp * (L + kPadRows + kPadEnd + 1);
    slot = gl < DNV ? gl + kPadRows : L + kPadRows + kPadEnd;
    sums = grp * ZN4;
  }
  // ceil(n / G), n <= 64
  __device__ __forceinline__ int rounds(int n) const { return ((n + G - 1) * inv) >> 16; }
  __device__ __forceinline__ void zero_pads(float* set, int DNV) const {
    if (gl < kPadRows) set[rows + gl] = 0.f;
    if (gl < kPadEnd) set[rows + kPadRows + DNV + gl] = 0.f;
  }
};
// Sorts the lanes by class: returns this lane's position, first[k] that of class k's first lane
// (k = 1 ... 9, first[10] the total).  Lanes of key 0 have none.
__device__ __forceinline__ int sort_classes(int key, int (&first)[11]) {
  int pos = 0, base = 0;
#pragma unroll
  for (int k = 1; k <= 9; ++k) {
    const uint64_t m = __ballot(key == k);
    first[k] = base;
    if (key == k)
      pos = base + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                                  __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0));
    base += __builtin_popcountll(m);
  }
  first[10] = base;
  return pos;
}

template <bool UPDATE, typename T, bool ONES = false>
__device__ __forceinline__ void bp_packed_body(const BpArgs<T>& A, int col, float* lds) {
#pragma clang fp contract(off)
  const Dims& d = A.d;
  const BpConsts64& c64 = A.c64;
  const int lane = threadIdx.x & 63;
  if (col >= d.XN * d.YN) return;
  const int y = col / d.XN, x = col - y * d.XN;
  CTR_GLOBAL float* vcol = gp(A.vol) + (size_t)col * d.ZN;
  if (gp(A.mask)[col] != 1) {
    if constexpr (!UPDATE) {
      for (int z = lane; z < d.ZN; z += 64) vcol[z] = 0.f;
    }
    return;
  }
  const int DNV = d.DNV, ZN4 = (d.ZN + 3) & ~3;
  const Groups g(A.lanes, DNV, ZN4);
  float4* rec = reinterpret_cast<float4*>(lds + kPackRowsLds);  // [64][3]
  float* lacc = lds + kPackF;
  for (int i = lane; i < g.G * ZN4; i += 64) lacc[i] = 0.f;
  g.zero_pads(lds, DNV);
  float* rows = lds + g.rows;
  float* gacc = lacc + g.sums;
  const double Px = held(((double)x - c64.ocx) * c64.dx);
  const double Py = held(((double)y - c64.ocy) * c64.dx);
  const int frame = d.DNU * DNV;
  const float glf = (float)g.gl;
  bool rest = false;
  // a view's (offset of its first column, z0, z1 - z0)
  auto ints = [&](const BpRecord& v) {
    return make_float4(__int_as_float(lane * frame + v.o), __int_as_float(v.z0),
                       __int_as_float(v.z1 - v.z0), 0.f);
  };
  for (int k0 = 0; k0 < A.vc; k0 += 64) {
    const int kl = k0 + lane;
    BpRecord v{};
    if (kl < A.vc) v = bp_record(A, kl, Px, Py, g.L, false);
    if (!__any(v.key)) continue;
    rest = rest || __any(v.key == 1);
    int first[11];
    const int pos = sort_classes(v.key, first);
    if (v.key) {
      rec[3 * pos] = v.r;
      rec[3 * pos + 1] = v.w;
      rec[3 * pos + 2] = ints(v);
    }
    const Buf<T> P(A.prj + (size_t)k0 * frame, (uint32_t)min(64, A.vc - k0) * (uint32_t)frame);
    for_classes([&](auto NU_, auto MULTI_) {
      constexpr int NU = decltype(NU_)::value;
      constexpr bool MULTI = decltype(MULTI_)::value;
      constexpr int K = 2 * NU + (MULTI ? 1 : 0);
      const int n = first[K + 1] - first[K];
      if (!n) return;
      const float4* rc = rec + 3 * first[K];
      struct Set {
        uint32_t y[NU];
      };
      pipelined_n<Set>(
          g.rounds(n),
          [&](int i, Set& f) {
            if constexpr (ONES) return;
            const int e = min(i * g.G + g.grp, n - 1);
            const int o = __float_as_int(rc[3 * e + 2].x) + g.row;
#pragma unroll
            for (int iu = 0; iu < NU; ++iu) f.y[iu] = P.at_bits(o, iu * DNV);
          },
          [&](int i, const Set& f) {
            const int e = i * g.G + g.grp;
            const float4* re = rc + 3 * min(e, n - 1);
            const float4 r = re[0], w = re[1], oz = re[2];
            const float wu[4] = {w.x, w.y, w.z, w.w};
            float R = wu[0] * (ONES ? 1.f : Buf<T>::widen(f.y[0]));
#pragma unroll
            for (int iu = 1; iu < NU; ++iu)
              R = fmaf(wu[iu], ONES ? 1.f : Buf<T>::widen(f.y[iu]), R);
            rows[g.slot] = R;
            const int last = e < n && g.gl < g.L ? __float_as_int(oz.z) : -1;
            float* a = gacc + __float_as_int(oz.y) + g.gl;
            if constexpr (MULTI) {
              float zi = glf;
              for (int zz = 0; __any(zz <= last); zz += g.L, zi += (float)g.L)
                if (g.gl <= last - zz) a[zz] = bp_voxel<3>(d, r, zi, rows + kPadRows, a[zz]);
            } else {
              if (g.gl <= last) *a = bp_voxel<3>(d, r, glf, rows + kPadRows, *a);
            }
          });
    });
  }
  // the views of key 1; all of them where a sum is not finite
  bool exact = false;
  if constexpr (!ONES) exact = reset_not_finite(lacc, g.G * ZN4);
  if (rest || exact)
    for (int k0 = 0; k0 < A.vc; k0 += 64) {
      const int kl = k0 + lane;
      BpRecord v{};
      if (kl < A.vc) v = bp_record(A, kl, Px, Py, g.L, exact);
      int first[11];
      const int pos = sort_classes(v.key, first), n = first[2];
      if (!n) continue;
      if (v.key == 1) {
        rec[3 * pos] = v.r;
        rec[3 * pos + 1] = v.w;
        rec[3 * pos + 2] = ints(v);
      }
      const Buf<T> P(A.prj + (size_t)k0 * frame, (uint32_t)min(64, A.vc - k0) * (uint32_t)frame);
      struct Set {
        uint32_t y[4];
      };
      auto load = [&](int o, int c0, int nc, Set& f) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          f.y[i] = ONES ? 0u : P.at_bits(o + min(c0 + i, nc - 1) * DNV, 0);
      };
      pipelined_n<Set>(
          g.rounds(n),
          [&](int i, Set& f) {
            const float4* re = rec + 3 * min(i * g.G + g.grp, n - 1);
            load(__float_as_int(re[2].x) + g.row, 0, __float_as_int(re[1].w), f);
          },
          [&](int i, const Set& f0) {
            const int e = i * g.G + g.grp;
            const float4* re = rec + 3 * min(e, n - 1);
            const float4 r = re[0], w = re[1], oz = re[2];
            const int nc = __float_as_int(w.w);
            float R = 0.f;
            Set f = f0;
            for (int c0 = 0;;) {
#pragma unroll
              for (int i = 0; i < 4; ++i) {
                const float t = fmaf(rest_weight(w, c0 + i, nc),
                                     ONES ? 1.f : Buf<T>::widen(f.y[i]), R);
                R = c0 + i < nc ? t : R;
              }
              c0 += 4;
              if (!__any(c0 < nc)) break;
              load(__float_as_int(oz.x) + g.row, c0, nc, f);
            }
            rows[g.slot] = R;
            const int last = e < n && g.gl < g.L ? __float_as_int(oz.z) : -1;
            float* a = gacc + __float_as_int(oz.y);
            const float* R0 = rows + kPadRows;
            if (exact || __any(r.y > kTaps5 || not_finite(R))) {
              for (int zz = g.gl; zz <= last; zz += g.L)
                a[zz] = bp_voxel<0>(d, r, (float)zz, R0, a[zz]);
            } else {
              for (int zz = g.gl; zz <= last; zz += g.L)
                a[zz] = bp_voxel<5>(d, r, (float)zz, R0, a[zz]);
            }
          });
    }
  for (int z = lane; z < d.ZN; z += 64) {
    float a = lacc[z];
    for (int k = 1; k < g.G; ++k) a += lacc[k * ZN4 + z];
    bp_store<UPDATE>(A, vcol, col, z, a);
  }
}

// The windowed form without staged rows (more than 256 detector rows, or frames too large
// for the staged loads' 32-bit offsets), gathering each voxel's rows from memory; lacc: ZN
// floats of this wave, each updated by one lane per view, views in order.  Per-voxel
// arithmetic as bp_ref_body.
// ONES: the back projection of a sinogram of ones, read from no sinogram: the row weights of
// a shadow sum to its clipped height vhi - vlo and the column weights to Wu = wu0 + (nu - 2)
// + fh (wu0 alone for one column), so a voxel adds cosVal * Wu * (vhi - vlo).
template <bool UPDATE, typename T, bool ONES = false>
__device__ __forceinline__ void bp_win_body(const BpArgs<T>& A, int col, float* lacc) {
  const Dims& d = A.d;
  const BpConsts64& c64 = A.c64;
  const int lane = threadIdx.x & 63;
  if (col >= d.XN * d.YN) return;
  const int y = col / d.XN, x = col - y * d.XN;
  CTR_GLOBAL float* vcol = gp(A.vol) + (size_t)col * d.ZN;
  if (gp(A.mask)[col] != 1) {
    if constexpr (!UPDATE) {
      for (int z = lane; z < d.ZN; z += 64) vcol[z] = 0.f;
    }
    return;
  }
  for (int z = lane; z < d.ZN; z += 64) lacc[z] = 0.f;
  const double Px = held(((double)x - c64.ocx) * c64.dx);
  const double Py = held(((double)y - c64.ocy) * c64.dx);
  const float DNVh = (float)d.DNV - 0.5f;
  const int DNV = d.DNV;
  const uint32_t frame = (uint32_t)(d.DNU * d.DNV);
  for (int k0 = 0; k0 < A.vc; k0 += 64) {
    const int kl = k0 + lane;
    BpView q{};
    int q_z0 = 0, q_z1 = -1;
    if (kl < A.vc) {
      q = bp_view(A, A.vb + kl * A.vs, Px, Py);
      bp_window(d, q, q_z0, q_z1);
    }
    uint64_t live = __ballot(q.uvis && q_z0 <= q_z1);
    while (live) {
      const int j = __builtin_ctzll(live);
      live &= live - 1;
      const int k = k0 + j;
      const float rlS = rdl(q.rlS, j), cA = rdl(q.cA, j), cB = rdl(q.cB, j);
      const float vsz = rdl(q.sz, j), l2f = rdl(q.l2, j), cws = rdl(q.cws, j);
      const float wu0 = rdl(q.wu0, j), fh = rdl(q.fh, j);
      const int u0 = __builtin_amdgcn_readlane(q.u0, j), nu = __builtin_amdgcn_readlane(q.nu, j);
      const int z0 = __builtin_amdgcn_readlane(q_z0, j), z1 = __builtin_amdgcn_readlane(q_z1, j);
      const Buf<T> pp(A.prj + (size_t)k * frame, frame);
      for (int zz = z0; zz <= z1; zz += 64) {
        const int z = zz + lane;
        const float dZ = fmaf((float)z - d.ocz, d.dz, -vsz);
        const float vlo = fmaxf(fmaf(dZ, rlS, cA), -0.5f);
        const float vhi = fminf(fmaf(dZ, rlS, cB), DNVh);
        const bool vok = z <= z1 && vlo < vhi;
        if (!vok) continue;
        const float cosVal = cws * __builtin_amdgcn_sqrtf(fmaf(dZ, dZ, l2f));
        if constexpr (ONES) {
          const float Wu = nu == 1 ? wu0 : wu0 + (float)(nu - 2) + fh;
          lacc[z] = fmaf(cosVal, Wu * (vhi - vlo), lacc[z]);
        } else {
          lacc[z] = fmaf(cosVal, bp_cell_sum(pp, u0 * DNV, nu, wu0, fh, vlo, vhi, DNV), lacc[z]);
        }
      }
    }
  }
  for (int z = lane; z < d.ZN; z += 64) bp_store<UPDATE>(A, vcol, col, z, lacc[z]);
}

// The windowed body with staged rows (RC = 1, 2, 4), of packed views (kPacked), of rows staged
// view by view (kPlain, kPlain - 1, kPlain - 2: 1, 2, 4 row chunks) or without any (0);
// lds: bp_win_floats of this wave, sums = the floats of its column sums.
__host__ __device__ constexpr int bp_win_floats(int RC, int sums) {
  return (RC == kPacked ? kPackF
          : RC == 1 || RC == kPlain     ? kStagedF<1>
          : RC == 2 || RC == kPlain - 1 ? kStagedF<2>
          : RC == 4 || RC == kPlain - 2 ? kStagedF<4>
                        : 0) +
         ((sums + 3) & ~3);
}
// Waves per SIMD that a body is compiled for.  One row chunk takes one more in its own kernel (8
// waves, 64 registers, 8 values spilled; 512^2 x 256: 2.40 ms, 2.47 ms with 7 waves and none);
// two chunks spill up to 4 values, four 12.  While the FP64 constants of a view's evaluation stood
// in vector registers (held) they spilled 26, 12 and 24: 2.44 ms, and 14 us for 11 us where one
// view of 128^2 x 64 is projected.
constexpr int bp_waves(int RC) {
  return RC == 4 ? 5 : RC == 2 || RC == kPacked ? 6 : 7;
}
template <bool UPDATE, typename T, int RC, bool ONES = false>
__device__ __forceinline__ void bp_any_win_body(const BpArgs<T>& A, int col, float* lds) {
  if constexpr (RC == kPlain) bp_plain_body<UPDATE, T, 1, ONES>(A, col, lds);
  else if constexpr (RC == kPlain - 1) bp_plain_body<UPDATE, T, 2, ONES>(A, col, lds);
  else if constexpr (RC == kPlain - 2) bp_plain_body<UPDATE, T, 4, ONES>(A, col, lds);
  else if constexpr (RC == kPacked) bp_packed_body<UPDATE, T, ONES>(A, col, lds);
  else if constexpr (RC > 0) bp_staged_body<UPDATE, T, RC, ONES>(A, col, lds);
  else bp_win_body<UPDATE, T, ONES>(A, col, lds);
}

template <bool UPDATE, int ZG, typename T>
__global__ __launch_bounds__(kBlock) void bp_ref_kernel(BpArgs<T> A) {
  const int col = blockIdx.x * kWaves + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  bp_ref_body<UPDATE, ZG, T>(A, col, blockIdx.y);
}

// Windowed reference back projection; dynamic LDS: kWaves * bp_win_floats(RC, sums) floats.
template <bool UPDATE, typename T, int RC>
__global__ __launch_bounds__(kBlock, RC == 1 ? 8 : bp_waves(RC)) void bp_win_kernel(
    BpArgs<T> A, int sums) {
  extern __shared__ float4 lds_win[];
  float* lds = reinterpret_cast<float*>(lds_win);
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  bp_any_win_body<UPDATE, T, RC>(A, blockIdx.x * kWaves + wid,
                                 lds + wid * bp_win_floats(RC, sums));
}

// Back projection of a sinogram of ones (A.prj unused); dynamic LDS as bp_win_kernel.
template <int RC>
__global__ __launch_bounds__(kBlock, bp_waves(RC)) void bp_win_ones_kernel(BpArgs<float> A,
                                                                          int sums) {
  extern __shared__ float4 lds_win[];
  float* lds = reinterpret_cast<float*>(lds_win);
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  bp_any_win_body<false, float, RC, true>(A, blockIdx.x * kWaves + wid,
                                          lds + wid * bp_win_floats(RC, sums));
}

// Batched windowed reference back projection: flat work list of (scan, block of 4
// columns); RC as the scan of most rows needs it (packed scans have a list of their own),
// dynamic LDS: kWaves * bp_win_floats(RC, sums) floats (sums: the most of any scan).
template <typename T, int RC>
__global__ __launch_bounds__(kBlock, bp_waves(RC)) void bp_batch_win_kernel(
    const BpBatchItem<T>* __restrict__ D, int nscan, int total, int sched, int sums) {
  extern __shared__ float4 lds_win[];
  int i0, step, i1;
  batch_range(D, nscan, total, sched, i0, step, i1);
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  float* lds = reinterpret_cast<float*>(lds_win) + wid * bp_win_floats(RC, sums);
  int s = 0;
  for (int item = i0; item < i1; item += step) {
    if (sched == 1) s = 0;
    while (s + 1 < nscan && D[s + 1].begin <= item) ++s;
    const BpBatchItem<T>& B = D[s];
    bp_any_win_body<true, T, RC>(B.a, (item - B.begin) * kWaves + wid, lds);
  }
}

// bp_batch_win_kernel for the one-workgroup-per-item schedule (grid = total): no item
// loop, so nothing stays live around the column body.
template <typename T, int RC>
__global__ __launch_bounds__(kBlock, bp_waves(RC)) void bp_batch_win1_kernel(
    const BpBatchItem<T>* __restrict__ D, int nscan, int total, int sums) {
  extern __shared__ float4 lds_win[];
  int i0, step, i1;
  batch_range(D, nscan, total, 2, i0, step, i1);
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  float* lds = reinterpret_cast<float*>(lds_win) + wid * bp_win_floats(RC, sums);
  int s = 0;
  while (s + 1 < nscan && D[s + 1].begin <= i0) ++s;
  const BpBatchItem<T>& B = D[s];
  bp_any_win_body<true, T, RC>(B.a, (i0 - B.begin) * kWaves + wid, lds);
}

// Batched persistent reference back projection: flat work list of (scan, z block,
// block of 4 columns), contiguous ranges per workgroup as in fp_batch_kernel.
template <bool UPDATE, int ZG, typename T>
__global__ __launch_bounds__(kBlock) void bp_batch_kernel(const BpBatchItem<T>* __restrict__ D,
                                                          int nscan, int total, int sched) {
  int i0, step, i1;
  batch_range(D, nscan, total, sched, i0, step, i1);
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int s = 0;
  for (int item = i0; item < i1; item += step) {
    if (sched == 1) s = 0;
    while (s + 1 < nscan && D[s + 1].begin <= item) ++s;
    const BpBatchItem<T>& B = D[s];
    const int local = item - B.begin;
    const int zblk = local / B.colBlocks;
    bp_ref_body<UPDATE, ZG, T>(B.a, (local - zblk * B.colBlocks) * kWaves + wid, zblk);
  }
}


// ---------------------------------------------------------------------------
// Matched adjoint: the exact transpose of fp_kernel, in gather form.
// Input yp is the sinogram already multiplied by K * invdB (scale_matched_kernel).
// For each view the voxel's in-plane cell is located among the column footprints
// on its slice with the FP64 boundary lines fp_kernel evaluates, and its z cell
// among the row footprints (FP32, relative to the view's azi as in fp_kernel); the
// overlap weights are those of the forward projector.
// ---------------------------------------------------------------------------
template <bool UPDATE, int ZG>
__global__ __launch_bounds__(kBlock) void bp_matched_kernel(
    const float* __restrict__ yp, float* __restrict__ vol, const ViewP* __restrict__ views,
    const double2* __restrict__ bnd, const float4* __restrict__ cols,
    const float* __restrict__ Bz, const uint8_t* __restrict__ mask, Dims d, BpConsts c,
    int vb, int vs, int vc, const float* __restrict__ invCol, uint16_t* __restrict__ shadow) {
  const int lane = threadIdx.x & 63;
  const int col = blockIdx.x * kWaves + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (col >= d.XN * d.YN) return;
  const int zb = blockIdx.y * (64 * ZG) + lane;
  const int y = col / d.XN, x = col - y * d.XN;
  float* vcol = vol + (size_t)col * d.ZN;
  const float m = (float)mask[col];
  if (m == 0.f) {
    if constexpr (!UPDATE) {
#pragma unroll
      for (int g = 0; g < ZG; ++g)
        if (zb + 64 * g < d.ZN) vcol[zb + 64 * g] = 0.f;
    }
    return;
  }
  const float Px = ((float)x - d.ocx) * d.dx;
  const float Py = ((float)y - d.ocy) * d.dx;
  float acc[ZG];
  bool live[ZG];
#pragma unroll
  for (int g = 0; g < ZG; ++g) {
    acc[g] = 0.f;
    live[g] = zb + 64 * g < d.ZN;
  }
  const size_t frame = (size_t)d.DNU * d.DNV;
  const int DNU = d.DNU, DNV = d.DNV;
  for (int k = 0; k < vc; ++k) {
    const int p = vb + k * vs;
    const ViewP vp = views[p];
    const int ii = vp.xmarch ? x : y;
    const int j = vp.xmarch ? y : x;
    const double fi = (double)ii;
    const double2* bt = bnd + (size_t)p * (DNU + 1);
    const float4* ctab = cols + (size_t)p * DNU;
    const double dir = (double)vp.bdir;
    const double cl = (vp.bdir > 0) ? (double)j - 0.5 : -((double)j + 0.5);
    const double ch = cl + 1.0;
    // first guess from the fan angle of the voxel centre, then walk to the first
    // column whose footprint (the FP64 boundary lines of fp_kernel) reaches cl
    const float dX = Px - vp.sx, dY = Py - vp.sy;
    const float beta = asinf((vp.sy * dX - vp.sx * dY) * c.inv_sid * rsqrtf(dX * dX + dY * dY));
    int u = (int)fminf(fmaxf(floorf((beta - d.beta0) / d.dbeta_g), 0.f), (float)(DNU - 1));
    double su = dir * fma(fi, bt[u].y, bt[u].x);
    while (u > 0 && su > cl) {
      --u;
      su = dir * fma(fi, bt[u].y, bt[u].x);
    }
    double su1 = dir * fma(fi, bt[u + 1].y, bt[u + 1].x);
    while (u < DNU - 1 && su1 <= cl) {
      ++u;
      su = su1;
      su1 = dir * fma(fi, bt[u + 1].y, bt[u + 1].x);
    }
    const float* yk = yp + (size_t)k * frame;
    // z relative to azi, as fp_kernel
    const float az = vp.azf;
    for (; u < DNU && su < ch;) {
      const double wy = fmin(su1, ch) - fmax(su, cl);
      if (wy > 0.0) {
        const float4 ct = ctab[u];
        const float r = fmaf((float)ii, ct.y, ct.x);
        const float wyi = (float)wy * __builtin_amdgcn_rcpf((float)(su1 - su) * r);
        const float* yu = yk + (size_t)u * DNV;
        const float rinv = 1.0f / r;
        const float zlo0 = fmaf(r, Bz[0], az), zhiN = fmaf(r, Bz[DNV], az);
#pragma unroll
        for (int g = 0; g < ZG; ++g) {
          // rows whose z footprint [az + Bz[v] r, az + Bz[v+1] r] meets [zlo, zhi]
          const float zlo = (float)(zb + 64 * g - vp.azi) - 0.5f, zhi = zlo + 1.0f;
          const bool vis = live[g] && zhi > zlo0 && zlo < zhiN;
          if (!__any(vis)) continue;
          if (!vis) continue;
          int v = (int)fminf(fmaxf(floorf(((zlo - az) * rinv - d.B0) / d.dB), 0.f),
                             (float)(DNV - 1));
          float zl = fmaf(r, Bz[v], az);
          while (v > 0 && zl > zlo) {
            --v;
            zl = fmaf(r, Bz[v], az);
          }
          float zh = fmaf(r, Bz[v + 1], az);
          while (v < DNV - 1 && zh <= zlo) {
            ++v;
            zl = zh;
            zh = fmaf(r, Bz[v + 1], az);
          }
          float gsum = 0.f;
          for (; v < DNV && zl < zhi;) {
            const float wz = fminf(zh, zhi) - fmaxf(zl, zlo);
            if (wz > 0.f) gsum = fmaf(wz, yu[v], gsum);
            ++v;
            if (v < DNV) {
              zl = zh;
              zh = fmaf(r, Bz[v + 1], az);
            }
          }
          acc[g] = fmaf(wyi, gsum, acc[g]);
        }
      }
      ++u;
      if (u < DNU) {
        su = su1;
        su1 = dir * fma(fi, bt[u + 1].y, bt[u + 1].x);
      }
    }
  }
#pragma unroll
  for (int g = 0; g < ZG; ++g) {
    if (!live[g]) continue;
    const int z = zb + 64 * g;
    const float a = acc[g] * m;
    if constexpr (UPDATE) {
      const float nx = fmaf(a, invCol[(size_t)col * d.ZN + z], vcol[z]);
      vcol[z] = nx;
      if (shadow) shadow[(size_t)col * d.ZN + z] = to_bf16_dither(nx, (size_t)col * d.ZN + z);
    } else {
      vcol[z] = a;
    }
  }
}

// Rows of one detector column meeting the z cell [zlo, zlo + 1] of a voxel, integrated
// against the column's scaled sinogram yu with the forward projector's FP32 row
// boundaries az + r Bz[v] (Bz from LDS); the first row from the uniform-spacing guess,
// then corrected against the exact boundaries.
__device__ __forceinline__ float matched_rows(const float* __restrict__ yu,
                                              const float* __restrict__ sBz, int DNV, float r,
                                              float az, float zlo, float B0, float dB) {
  const float zhi = zlo + 1.0f;
  int v = (int)fminf(fmaxf(floorf(((zlo - az) * __builtin_amdgcn_rcpf(r) - B0) / dB), 0.f),
                     (float)(DNV - 1));
  float zl = fmaf(r, sBz[v], az);
  while (v > 0 && zl > zlo) {
    --v;
    zl = fmaf(r, sBz[v], az);
  }
  float zh = fmaf(r, sBz[v + 1], az);
  while (v < DNV - 1 && zh <= zlo) {
    ++v;
    zl = zh;
    zh = fmaf(r, sBz[v + 1], az);
  }
  float gsum = 0.f;
  for (; v < DNV && zl < zhi;) {
    const float wz = fminf(zh, zhi) - fmaxf(zl, zlo);
    if (wz > 0.f) gsum = fmaf(wz, yu[v], gsum);
    ++v;
    if (v < DNV) {
      zl = zh;
      zh = fmaf(r, sBz[v + 1], az);
    }
  }
  return gsum;
}

// The same sums as matched_rows for the (at most four) columns t < nu of one view, the
// rows taken as a fixed count NR (at least the number of rows of spacing r_t dBmin that
// can meet a cell of height 1): every column's first row is searched, then every
// sinogram value is loaded, then the rows are summed in order, rows with no overlap or
// past the detector adding nothing -- the sums and their order are those of matched_rows.
// ig[t] = 1 / (r_t dB), g0 = -B0 / dB give the first-row guess.
template <int NR>
__device__ __forceinline__ float matched_cols(const float* __restrict__ yk,
                                              const float* __restrict__ sBz, int DNV, int nu,
                                              const float (&w)[4], const float (&r)[4],
                                              const float (&ig)[4], float az, float g0,
                                              float zlo, float a) {
  const float zhi = zlo + 1.0f;
  int v[4];
  float zl[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    v[t] = 0;
    zl[t] = 0.f;
    if (t < nu) {
      int vv = (int)fminf(fmaxf(floorf(fmaf(zlo - az, ig[t], g0)), 0.f), (float)(DNV - 1));
      float l = fmaf(r[t], sBz[vv], az);
      while (vv > 0 && l > zlo) {
        --vv;
        l = fmaf(r[t], sBz[vv], az);
      }
      float h = fmaf(r[t], sBz[vv + 1], az);
      while (vv < DNV - 1 && h <= zlo) {
        ++vv;
        l = h;
        h = fmaf(r[t], sBz[vv + 1], az);
      }
      v[t] = vv;
      zl[t] = l;
    }
  }
  float yv[4][NR];
#pragma unroll
  for (int t = 0; t < 4; ++t) {
#pragma unroll
    for (int i = 0; i < NR; ++i)
      yv[t][i] = (t < nu) ? yk[(size_t)t * DNV + min(v[t] + i, DNV - 1)] : 0.f;
  }
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    if (t < nu && w[t] != 0.f) {
      float g = 0.f, lo = zl[t];
#pragma unroll
      for (int i = 0; i < NR; ++i) {
        const int vi = v[t] + i;
        const float hi = fmaf(r[t], sBz[min(vi + 1, DNV)], az);
        const float wz = fminf(hi, zhi) - fmaxf(lo, zlo);
        if (vi < DNV && wz > 0.f) g = fmaf(wz, yv[t][i], g);
        lo = hi;
      }
      a = fmaf(w[t], g, a);
    }
  }
  return a;
}

// Windowed matched adjoint: the transpose of fp_kernel as bp_matched_kernel computes it,
// with one wave per voxel column over all of its z.  Per view (64 views at a time, one
// per lane): the detector columns whose footprints on the voxel's slice meet its cell
// (first column u0, count nu; for nu <= 4 the in-plane weights w_t = overlap / ((tr - tl)
// r) and magnifications r_t), and the view's z-window of the column (the cells the
// detector's z range at those magnifications reaches, widened by one).  The lanes then
// take the window, each voxel summing w_t times its rows' integral over the columns in
// order (the same sequence of operations per voxel as bp_matched_kernel), into the
// column's LDS sums.  Dynamic LDS: Bz (DNV + 1 floats, 4-aligned), then kWaves * ZN.
template <bool UPDATE>
__global__ __launch_bounds__(kBlock) void bp_matched_win_kernel(
    const float* __restrict__ yp, float* __restrict__ vol, const ViewP* __restrict__ views,
    const double2* __restrict__ bnd, const float4* __restrict__ cols,
    const float* __restrict__ Bz, const uint8_t* __restrict__ mask, Dims d, BpConsts c,
    int vb, int vs, int vc, const float* __restrict__ invCol, uint16_t* __restrict__ shadow) {
  extern __shared__ float lds_m[];
  const int DNU = d.DNU, DNV = d.DNV;
  const int nbz = (DNV + 1 + 3) & ~3;
  float* sBz = lds_m;
  for (int i = threadIdx.x; i <= DNV; i += kBlock) sBz[i] = Bz[i];
  __syncthreads();
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = blockIdx.x * kWaves + wid;
  if (col >= d.XN * d.YN) return;
  float* lacc = lds_m + nbz + wid * d.ZN;
  const int y = col / d.XN, x = col - y * d.XN;
  float* vcol = vol + (size_t)col * d.ZN;
  const float m = (float)mask[col];
  if (m == 0.f) {
    if constexpr (!UPDATE) {
      for (int z = lane; z < d.ZN; z += 64) vcol[z] = 0.f;
    }
    return;
  }
  for (int z = lane; z < d.ZN; z += 64) lacc[z] = 0.f;
  const float Px = ((float)x - d.ocx) * d.dx;
  const float Py = ((float)y - d.ocy) * d.dx;
  const size_t frame = (size_t)DNU * DNV;
  const float ZNf = (float)d.ZN;
  for (int k0 = 0; k0 < vc; k0 += 64) {
    const int kl = k0 + lane;
    int q_u0 = 0, q_nu = 0, q_z0 = 0, q_z1 = -1;
    float q_w[4] = {0.f, 0.f, 0.f, 0.f}, q_r[4] = {1.f, 1.f, 1.f, 1.f};
    float q_ig[4] = {0.f, 0.f, 0.f, 0.f};
    float q_az = 0.f;
    int q_azi = 0;
    int q_nr = 0;
    if (kl < vc) {
      const int p = vb + kl * vs;
      const ViewP vp = views[p];
      const int ii = vp.xmarch ? x : y;
      const int j = vp.xmarch ? y : x;
      const double fi = (double)ii;
      const double2* bt = bnd + (size_t)p * (DNU + 1);
      const float4* ctab = cols + (size_t)p * DNU;
      const double dir = (double)vp.bdir;
      const double cl = (vp.bdir > 0) ? (double)j - 0.5 : -((double)j + 0.5);
      const double ch = cl + 1.0;
      // first guess from the fan angle of the voxel centre, then walk to the first
      // column whose footprint (the FP64 boundary lines of fp_kernel) reaches cl
      const float dX = Px - vp.sx, dY = Py - vp.sy;
      const float beta =
          asinf((vp.sy * dX - vp.sx * dY) * c.inv_sid * rsqrtf(dX * dX + dY * dY));
      int u = (int)fminf(fmaxf(floorf((beta - d.beta0) / d.dbeta_g), 0.f), (float)(DNU - 1));
      double su = dir * fma(fi, bt[u].y, bt[u].x);
      while (u > 0 && su > cl) {
        --u;
        su = dir * fma(fi, bt[u].y, bt[u].x);
      }
      double su1 = dir * fma(fi, bt[u + 1].y, bt[u + 1].x);
      while (u < DNU - 1 && su1 <= cl) {
        ++u;
        su = su1;
        su1 = dir * fma(fi, bt[u + 1].y, bt[u + 1].x);
      }
      // the columns u .. while su < ch (zero-overlap ones included: they add nothing)
      q_u0 = u;
      float rmin = 3.4e38f, rmax = -3.4e38f;
      int n = 0;
      for (; u < DNU && su < ch;) {
        const float4 ct = ctab[u];
        const float r = fmaf((float)ii, ct.y, ct.x);
        const double wy = fmin(su1, ch) - fmax(su, cl);
        if (n < 4) {
          q_w[n] = wy > 0.0 ? (float)wy * __builtin_amdgcn_rcpf((float)(su1 - su) * r) : 0.f;
          q_r[n] = r;
          q_ig[n] = __builtin_amdgcn_rcpf(r * d.dB);
        }
        rmin = fminf(rmin, r);
        rmax = fmaxf(rmax, r);
        ++n;
        ++u;
        if (u < DNU) {
          su = su1;
          su1 = dir * fma(fi, bt[u + 1].y, bt[u + 1].x);
        }
      }
      q_nu = n;
      // z relative to azi, as fp_kernel
      q_az = vp.azf;
      q_azi = vp.azi;
      if (n > 0) {
        // z cells [k - .5, k + .5] meeting [az + r Bz[0], az + r Bz[DNV]] for some r of
        // the columns (r > 0 beyond the source)
        const float lo = fminf(fmaf(rmin, Bz[0], vp.azf), fmaf(rmax, Bz[0], vp.azf));
        const float hi = fmaxf(fmaf(rmin, Bz[DNV], vp.azf), fmaf(rmax, Bz[DNV], vp.azf));
        const float fazi = (float)vp.azi;
        const float za = fminf(fmaxf(lo - 0.5f, -4.f - fazi), (ZNf + 4.f) - fazi);
        const float zb = fminf(fmaxf(hi + 0.5f, -4.f - fazi), (ZNf + 4.f) - fazi);
        q_z0 = max((int)floorf(za) - 1 + vp.azi, 0);
        q_z1 = min((int)ceilf(zb) + 1 + vp.azi, d.ZN - 1);
        // rows of spacing >= h meeting a cell of height 1: at most ceil(1 / h) + 1; h is
        // the smallest spacing rmin dBmin less the rounding of boundaries of size <= big
        const float big = fmaxf(fmaxf(fabsf(lo), fabsf(hi)), 1.f);
        const float h = rmin * d.dBmin * 0.99999f - 4.8e-7f * big;
        q_nr = h > 0.125f ? (int)ceilf(__builtin_amdgcn_rcpf(h) * 1.0001f) + 1 : 99;
      }
    }
    uint64_t live = __ballot(q_nu > 0 && q_z0 <= q_z1);
    while (live) {
      const int jl = __builtin_ctzll(live);
      live &= live - 1;
      const int k = k0 + jl;
      const int u0 = __builtin_amdgcn_readlane(q_u0, jl), nu = __builtin_amdgcn_readlane(q_nu, jl);
      const int z0 = __builtin_amdgcn_readlane(q_z0, jl), z1 = __builtin_amdgcn_readlane(q_z1, jl);
      const float az = rdl(q_az, jl);
      const int azi = __builtin_amdgcn_readlane(q_azi, jl);
      const int nr = __builtin_amdgcn_readlane(q_nr, jl);
      const float* yk = yp + (size_t)k * frame + (size_t)u0 * DNV;
      if (nu <= 4 && nr <= 5) {
        float w[4], r[4], ig[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          w[t] = rdl(q_w[t], jl);
          r[t] = rdl(q_r[t], jl);
          ig[t] = rdl(q_ig[t], jl);
        }
        const float g0 = -d.B0 / d.dB;
        for (int zz = z0; zz <= z1; zz += 64) {
          const int z = zz + lane;
          if (z > z1) continue;
          const float zlo = (float)(z - azi) - 0.5f;
          const float a0 = lacc[z];
          float a;
          switch (nr) {
            case 2: a = matched_cols<2>(yk, sBz, DNV, nu, w, r, ig, az, g0, zlo, a0); break;
            case 3: a = matched_cols<3>(yk, sBz, DNV, nu, w, r, ig, az, g0, zlo, a0); break;
            case 4: a = matched_cols<4>(yk, sBz, DNV, nu, w, r, ig, az, g0, zlo, a0); break;
            default: a = matched_cols<5>(yk, sBz, DNV, nu, w, r, ig, az, g0, zlo, a0); break;
          }
          lacc[z] = a;
        }
      } else if (nu <= 4) {
        float w[4], r[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          w[t] = rdl(q_w[t], jl);
          r[t] = rdl(q_r[t], jl);
        }
        for (int zz = z0; zz <= z1; zz += 64) {
          const int z = zz + lane;
          if (z > z1) continue;
          const float zlo = (float)(z - azi) - 0.5f;
          float a = lacc[z];
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            if (t < nu && w[t] != 0.f)
              a = fmaf(w[t], matched_rows(yk + t * DNV, sBz, DNV, r[t], az, zlo, d.B0, d.dB),
                       a);
          }
          lacc[z] = a;
        }
      } else {
        // more than four columns: their weights recomputed here, as in the lane stage
        const int p = vb + k * vs;
        const ViewP vp = views[p];
        const int ii = vp.xmarch ? x : y;
        const int j = vp.xmarch ? y : x;
        const double fi = (double)ii;
        const double2* bt = bnd + (size_t)p * (DNU + 1);
        const float4* ctab = cols + (size_t)p * DNU;
        const double dir = (double)vp.bdir;
        const double cl = (vp.bdir > 0) ? (double)j - 0.5 : -((double)j + 0.5);
        const double ch = cl + 1.0;
        for (int zz = z0; zz <= z1; zz += 64) {
          const int z = zz + lane;
          if (z > z1) continue;
          const float zlo = (float)(z - azi) - 0.5f;
          float a = lacc[z];
          for (int t = 0; t < nu; ++t) {
            const int u = u0 + t;
            const double su = dir * fma(fi, bt[u].y, bt[u].x);
            const double su1 = dir * fma(fi, bt[u + 1].y, bt[u + 1].x);
            const double wy = fmin(su1, ch) - fmax(su, cl);
            if (wy > 0.0) {
              const float4 ct = ctab[u];
              const float r = fmaf((float)ii, ct.y, ct.x);
              const float wyi = (float)wy * __builtin_amdgcn_rcpf((float)(su1 - su) * r);
              a = fmaf(wyi, matched_rows(yk + t * DNV, sBz, DNV, r, az, zlo, d.B0, d.dB), a);
            }
          }
          lacc[z] = a;
        }
      }
    }
  }
  for (int z = lane; z < d.ZN; z += 64) {
    const float a = lacc[z] * m;
    if constexpr (UPDATE) {
      const size_t i = (size_t)col * d.ZN + z;
      const float nx = fmaf(a, invCol[i], vcol[z]);
      vcol[z] = nx;
      if (shadow) shadow[i] = to_bf16_dither(nx, i);
    } else {
      vcol[z] = a;
    }
  }
}

// A view's detector columns meeting one voxel's cell on its slice: the boundary lines of
// fp_kernel in FP64, walked from the column that the voxel centre's fan angle suggests.
// next() steps to the next column while one meets the cell.
struct MatchedCols {
  const double2* bt;
  double fi, dir, cl, ch, su, su1;
  int u, DNU;
  __device__ __forceinline__ MatchedCols(const ViewP& vp, const double2* bnd, int p, int x, int y,
                                         float Px, float Py, const Dims& d, float inv_sid) {
    const int ii = vp.xmarch ? x : y, j = vp.xmarch ? y : x;
    DNU = d.DNU;
    fi = (double)ii;
    bt = bnd + (size_t)p * (DNU + 1);
    dir = (double)vp.bdir;
    cl = (vp.bdir > 0) ? (double)j - 0.5 : -((double)j + 0.5);
    ch = cl + 1.0;
    const float dX = Px - vp.sx, dY = Py - vp.sy;
    const float beta = asinf((vp.sy * dX - vp.sx * dY) * inv_sid * rsqrtf(dX * dX + dY * dY));
    u = (int)fminf(fmaxf(floorf((beta - d.beta0) / d.dbeta_g), 0.f), (float)(DNU - 1));
    su = at(u);
    while (u > 0 && su > cl) su = at(--u);
    su1 = at(u + 1);
    while (u < DNU - 1 && su1 <= cl) {
      ++u;
      su = su1;
      su1 = at(u + 1);
    }
  }
  __device__ __forceinline__ double at(int b) const {
    const double2 t = gload(bt, b);
    return dir * fma(fi, t.y, t.x);
  }
  __device__ __forceinline__ bool meets() const { return u < DNU && su < ch; }
  // overlap of the column with the cell (<= 0: none)
  __device__ __forceinline__ double overlap() const { return fmin(su1, ch) - fmax(su, cl); }
  __device__ __forceinline__ void next() {
    ++u;
    if (u < DNU) {
      su = su1;
      su1 = at(u + 1);
    }
  }
};

// Windowed matched adjoint with staged rows, for detectors of evenly spaced rows
// (d.even_rows; DNV <= 64 RC): bp_staged_body's scheme with one row set per detector column,
// since each column's rows have their own magnification r.  In units of the rows the cell
// of voxel z meets column t's rows over [T, T + s], T = T0 + (z - z0) s, s = 1 / (r dB), and
// its overlap with a row, times the column's in-plane overlap over its footprint's area, is
// the forward projector's weight: w_t = overlap dB / (tr - tl), r cancelling.  Lane l
// evaluates view k0 + l (columns, T0 and s in FP64); the row sets hold w_t y[u + t][v].
// Views of more than four columns take further records for the rest.
// Bound by VALU issue (0.75 of the chip's rate) and the texture unit's row loads.  256^2 x
// 128, 197 views of 888 x 64: 3.94 ms with a search and a gather of the rows per voxel
// (bp_matched_win_kernel), 0.91 ms; 512^2 x 256: 18.0 ms, 4.1 ms; 256^2 x 128 of 1.4 mm 5.7 ms,
// 2.2 ms.
//
// RC = kPacked: several views at a time, as bp_packed_body.
// 197 views of 888 columns, one view at a time and packed: 64^3, 16 rows 104 us, 60 us; 256^2 x
// 128, 16 rows 915 us, 584 us, 8 rows 911 us, 497 us.
template <int RC>
constexpr int kMatchedF = 4 * kRowsLds<RC> + 64 * 16;
template <>
constexpr int kMatchedF<kPacked> = 4 * kPackRowsLds + 64 * 16;
__host__ __device__ constexpr int bp_matched_floats(int RC, int sums) {
  return (RC == kPacked ? kMatchedF<kPacked>
          : RC == 1     ? kMatchedF<1>
          : RC == 2     ? kMatchedF<2>
                        : kMatchedF<4>) +
         ((sums + 3) & ~3);
}

// What the matched kernels read: the scaled sinogram and the plan's tables.
struct MatchedArgs {
  const float* yp;
  float* vol;
  const ViewP* views;
  const double2* bnd;
  const float4* cols;
  const float* Bz;
  const uint8_t* mask;
  Dims d;
  BpConsts c;
  int vb, vs, vc, lanes;
  const float* invCol;
  uint16_t* shadow;
};

// View kl's record of its columns c0 ... c0 + 3: (T0, s, w) of the n columns, their window, the
// offset of the first and the class as in BpRecord (1: shadows of more than two rows, or that
// leave the row set's zeros at an end of the window, or `exact`).
struct MatchedRecord {
  float4 t[4];
  int z0, z1, o, n, key;
  bool more;
};
__device__ __forceinline__ MatchedRecord matched_record(const MatchedArgs& A, int kl, int c0,
                                                        int x, int y, float Px, float Py,
                                                        int lanes, bool exact) {
  const Dims& d = A.d;
  const int DNU = d.DNU, DNV = d.DNV, p = A.vb + kl * A.vs;
  const float ZNf = (float)d.ZN;
  const double idB = 1.0 / d.dB_64;
  MatchedRecord v{};
  v.z1 = -1;
  const ViewP vp = A.views[p];
  const float4* ctab = A.cols + (size_t)p * DNU;
  const float fii = (float)(vp.xmarch ? x : y);
  MatchedCols mc(vp, A.bnd, p, x, y, Px, Py, d, A.c.inv_sid);
  v.o = (mc.u + c0) * DNV;
  float rt[4] = {1.f, 1.f, 1.f, 1.f}, wt[4] = {0.f, 0.f, 0.f, 0.f};
  float rmin = 3.4e38f, rmax = -3.4e38f;
  int n = -c0;
  for (; n < 4 && mc.meets(); mc.next(), ++n) {
    if (n < 0) continue;
    const float4 ct = ctab[mc.u];
    const float r = fmaf(fii, ct.y, ct.x);
    const double wy = mc.overlap();
    const float w = wy > 0.0 ? (float)(wy / (mc.su1 - mc.su) * d.dB_64) : 0.f;
#pragma unroll
    for (int t = 0; t < 4; ++t)
      if (n == t) {
        rt[t] = r;
        wt[t] = w;
      }
    rmin = fminf(rmin, r);
    rmax = fmaxf(rmax, r);
  }
  v.more = n == 4 && mc.meets();
  if (!(n > 0 && rmin > 0.f)) return v;
  // z cells [k - .5, k + .5] meeting [az + r Bz[0], az + r Bz[DNV]] for some column,
  // with a margin of 1e-2 (relative to azi, as fp_kernel)
  const float lo = fminf(fmaf(rmin, A.Bz[0], vp.azf), fmaf(rmax, A.Bz[0], vp.azf));
  const float hi = fmaxf(fmaf(rmin, A.Bz[DNV], vp.azf), fmaf(rmax, A.Bz[DNV], vp.azf));
  const float fazi = (float)vp.azi;
  const float za = fminf(fmaxf(lo - 0.51f, -4.f - fazi), (ZNf + 4.f) - fazi);
  const float zb = fminf(fmaxf(hi + 0.51f, -4.f - fazi), (ZNf + 4.f) - fazi);
  v.z0 = max((int)floorf(za) + 1 + vp.azi, 0);
  v.z1 = min((int)ceilf(zb) - 1 + vp.azi, d.ZN - 1);
  if (v.z0 > v.z1) return v;
  bool plain = !exact;
  const double e0 = (double)(v.z0 - vp.azi) - 0.5 - (double)vp.azf;
#pragma unroll
  for (int t = 0; t < 4; ++t)
    if (t < n) {
      const double s = idB / (double)rt[t];
      const float sf = (float)s, T0 = (float)(e0 * s - d.B0_64 * idB);
      // taps stay on the row set and its zeros over the whole window
      plain = plain && sf <= 2.f && T0 >= (float)-kPadRows &&
              fmaf((float)(v.z1 - v.z0), sf, T0) < (float)(DNV + kPadRows - 2);
      v.t[t] = make_float4(T0, sf, wt[t], 0.f);
    }
  v.n = n;
  v.key = plain ? 2 * n + (v.z1 - v.z0 >= lanes ? 1 : 0) : 1;
  return v;
}

// A voxel's share of a view of NU columns, TAPS as in bp_voxel (5 and 0: n of the NU columns):
// r[t] its records, R0 + t * set their first rows.
template <int NU, int TAPS>
__device__ __forceinline__ float matched_voxel(const float4 (&r)[NU], int n, float zi,
                                               const float* R0, int set, float DNVf) {
  float g = 0.f;
#pragma unroll
  for (int t = 0; t < NU; ++t) {
    const float T = fmaf(zi, r[t].y, r[t].x);
    if constexpr (TAPS == 5) {
      if (t < n) {
        const Overlap5 o = overlap5(T, r[t].y);
        const float* R = R0 + t * set + o.k;
#pragma unroll
        for (int i = 0; i < 5; ++i) g = fmaf(o.w[i], R[i], g);
      }
    } else if constexpr (TAPS == 0) {
      if (t < n && r[t].z != 0.f) g += tall_rows(R0 + t * set, T, r[t].y, DNVf);
    } else {
      const Overlap3 o = overlap3<3>(T, r[t].y);
      const float* R = R0 + t * set + o.k;
      g = t == 0 ? o.w0 * R[0] : fmaf(o.w0, R[0], g);
      g = fmaf(o.w1, R[1], g);
      g = fmaf(o.w2, R[2], g);
    }
  }
  return g;
}

template <bool UPDATE, int RC>
__global__ __launch_bounds__(kBlock, RC == 4 ? 4 : 6) void bp_matched_staged_kernel(MatchedArgs A,
                                                                                    int sums) {
  extern __shared__ float4 lds_win[];
  constexpr bool PACK = RC == kPacked;
  constexpr int SET = PACK ? kPackRowsLds : kRowsLds<PACK ? 1 : RC>;  // floats of a column's rows
  constexpr int NC = PACK ? 1 : RC;                                    // row chunks per lane
  const Dims& d = A.d;
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  float* rows = reinterpret_cast<float*>(lds_win) + wid * bp_matched_floats(RC, sums);
  float4* rec = reinterpret_cast<float4*>(rows + 4 * SET);  // [64][4]
  float* lacc = rows + kMatchedF<RC>;
  const int col = blockIdx.x * kWaves + wid;
  if (col >= d.XN * d.YN) return;
  const int y = col / d.XN, x = col - y * d.XN;
  float* vcol = A.vol + (size_t)col * d.ZN;
  const float mk = (float)A.mask[col];
  if (mk == 0.f) {
    if constexpr (!UPDATE) {
      for (int z = lane; z < d.ZN; z += 64) vcol[z] = 0.f;
    }
    return;
  }
  const int DNU = d.DNU, DNV = d.DNV, frame = DNU * DNV, ZN4 = (d.ZN + 3) & ~3;
  const Groups g(PACK ? A.lanes : 64, DNV, ZN4);  // (one group when not packed)
  for (int i = lane; i < sums; i += 64) lacc[i] = 0.f;
  int row[NC], slot[NC];
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    if constexpr (PACK) {
      g.zero_pads(rows + t * SET, DNV);
      row[0] = g.row;
      slot[0] = g.rows + g.slot;
    } else {
      stage_rows<NC>(rows + t * SET, DNV, lane, row, slot);
    }
  }
  const float Px = ((float)x - d.ocx) * d.dx, Py = ((float)y - d.ocy) * d.dx;
  const float lanef = (float)lane, glf = (float)g.gl;
  const float DNVf = (float)DNV;
  bool rest = false;
  // views' records, [64][4]; the free fourth entries: offset of the first column, z0, z1 - z0, n
  auto put = [&](MatchedRecord& v, int pos) {
    v.t[0].w = __int_as_float(lane * frame + v.o);
    v.t[1].w = __int_as_float(v.z0);
    v.t[2].w = __int_as_float(v.z1 - v.z0);
    v.t[3].w = __int_as_float(v.n);
#pragma unroll
    for (int t = 0; t < 4; ++t) rec[4 * pos + t] = v.t[t];
  };
  for (int k0 = 0; k0 < A.vc; k0 += 64) {
    const int kl = k0 + lane;
    MatchedRecord v{};
    if (kl < A.vc) v = matched_record(A, kl, 0, x, y, Px, Py, PACK ? g.L : 64, false);
    rest = rest || __any(v.key == 1 || v.more);
    if (!__any(v.key)) continue;
    const int q_o = lane * frame + v.o;
    int first[11], pos = lane;
    if constexpr (PACK) pos = sort_classes(v.key, first);
    if (v.key) put(v, pos);
    const Buf<float> P(A.yp + (size_t)k0 * frame, (uint32_t)min(64, A.vc - k0) * (uint32_t)frame);
    for_classes([&](auto NU_, auto MULTI_) {
      constexpr int NU = decltype(NU_)::value;
      constexpr bool MULTI = decltype(MULTI_)::value;
      constexpr int K = 2 * NU + (MULTI ? 1 : 0);
      struct Set {
        float y[NU][NC];
      };
      if constexpr (PACK) {
        const int n = first[K + 1] - first[K];
        if (!n) return;
        const float4* rc = rec + 4 * first[K];
        pipelined_n<Set>(
            g.rounds(n),
            [&](int i, Set& f) {
              const int o = __float_as_int(rc[4 * min(i * g.G + g.grp, n - 1)].w) + row[0];
#pragma unroll
              for (int t = 0; t < NU; ++t) f.y[t][0] = P.at(o, t * DNV);
            },
            [&](int i, const Set& f) {
              const int e = i * g.G + g.grp;
              const float4* re = rc + 4 * min(e, n - 1);
              float4 r[NU];
#pragma unroll
              for (int t = 0; t < NU; ++t) {
                r[t] = re[t];
                rows[t * SET + slot[0]] = r[t].z * f.y[t][0];
              }
              const int zf = __float_as_int(re[1].w);
              const int last = e < n && g.gl < g.L ? __float_as_int(re[2].w) : -1;
              const float* R0 = rows + g.rows + kPadRows;
              float* a = lacc + g.sums + zf + g.gl;
              if constexpr (MULTI) {
                float zi = glf;
                for (int zz = 0; __any(zz <= last); zz += g.L, zi += (float)g.L)
                  if (g.gl <= last - zz)
                    a[zz] += matched_voxel<NU, 3>(r, NU, zi, R0, SET, DNVf);
              } else {
                if (g.gl <= last) *a += matched_voxel<NU, 3>(r, NU, glf, R0, SET, DNVf);
              }
            });
      } else {
        const uint64_t m = __ballot(v.key == K);
        if (!m) return;
        pipelined<Set>(
            m,
            [&](int j, Set& f) {
              const int o = __builtin_amdgcn_readlane(q_o, j);
#pragma unroll
              for (int t = 0; t < NU; ++t)
#pragma unroll
                for (int h = 0; h < NC; ++h) f.y[t][h] = P.at(row[h], o + t * DNV);
            },
            [&](int j, const Set& f) {
              float4 r[NU];
#pragma unroll
              for (int t = 0; t < NU; ++t) {
                r[t] = rec[4 * j + t];
#pragma unroll
                for (int h = 0; h < NC; ++h) rows[t * SET + slot[h]] = r[t].z * f.y[t][h];
              }
              const int zf = __builtin_amdgcn_readlane(v.z0, j);
              const int n = __builtin_amdgcn_readlane(v.z1, j) - zf;
              auto pass = [&](float zi, int zz) {
                lacc[zf + zz + lane] +=
                    matched_voxel<NU, 3>(r, NU, zi, rows + kPadRows, SET, DNVf);
              };
              if constexpr (MULTI) {
                float zi = lanef;
                for (int zz = 0; zz <= n; zz += 64, zi += 64.f)
                  if (lane <= n - zz) pass(zi, zz);
              } else {
                if (lane <= n) pass(lanef, 0);
              }
            });
      }
    });
  }
  // records of key 1 and views' further columns; all where a sum is not finite
  const bool exact = reset_not_finite(lacc, sums);
  if (rest || exact)
    for (int k0 = 0, c0 = 0; k0 < A.vc;) {
      const int kl = k0 + lane;
      MatchedRecord v{};
      if (kl < A.vc) v = matched_record(A, kl, c0, x, y, Px, Py, 64, exact || c0 > 0);
      const uint64_t m = __ballot(v.key == 1);
      if (v.key == 1)
        put(v, PACK ? (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                                     __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0))
                    : lane);
      const Buf<float> P(A.yp + (size_t)k0 * frame,
                         (uint32_t)min(64, A.vc - k0) * (uint32_t)frame);
      struct Set {
        float y[4][NC];
      };
      // whether five taps stay on the row sets and their zeros over the whole window
      auto five = [&](const float4(&r)[4], int nc, int last) {
        bool ok = true;
#pragma unroll
        for (int t = 0; t < 4; ++t)
          ok = ok && (t >= nc || (r[t].y <= kTaps5 && r[t].x >= (float)-kPadRows &&
                                  fmaf((float)last, r[t].y, r[t].x) < (float)(DNV + 1)));
        return ok;
      };
      // the record at re, this lane's rows from offset o, voxels gl, gl + step, ...
      auto load = [&](const float4* re, Set& f) {
        const int o = __float_as_int(re[0].w), last = __float_as_int(re[3].w) - 1;
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
          for (int h = 0; h < NC; ++h) f.y[t][h] = P.at(o + row[h] + min(t, last) * DNV, 0);
      };
      auto use = [&](const float4* re, const Set& f, bool act, int gl, int step) {
        float4 r[4];
        bool own = exact;  // read the shadows' own rows only
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          r[t] = re[t];
#pragma unroll
          for (int h = 0; h < NC; ++h) {
            rows[t * SET + slot[h]] = r[t].z * f.y[t][h];
            own = own || not_finite(f.y[t][h]);
          }
        }
        const int zf = __float_as_int(re[1].w), nc = __float_as_int(re[3].w);
        const int last = act ? __float_as_int(re[2].w) : -1;
        const float* R0 = rows + (PACK ? g.rows : 0) + kPadRows;
        float* a = lacc + (PACK ? g.sums : 0) + zf;
        if (__any(own || (act && !five(r, nc, last)))) {
          for (int zz = gl; zz <= last; zz += step)
            a[zz] += matched_voxel<4, 0>(r, nc, (float)zz, R0, SET, DNVf);
        } else {
          for (int zz = gl; zz <= last; zz += step)
            a[zz] += matched_voxel<4, 5>(r, nc, (float)zz, R0, SET, DNVf);
        }
      };
      if (m) {
        if constexpr (PACK) {
          const int n = __builtin_popcountll(m);
          pipelined_n<Set>(
              g.rounds(n),
              [&](int i, Set& f) { load(rec + 4 * min(i * g.G + g.grp, n - 1), f); },
              [&](int i, const Set& f) {
                const int e = i * g.G + g.grp;
                use(rec + 4 * min(e, n - 1), f, e < n && g.gl < g.L, g.gl, g.L);
              });
        } else {
          pipelined<Set>(
              m, [&](int j, Set& f) { load(rec + 4 * j, f); },
              [&](int j, const Set& f) { use(rec + 4 * j, f, true, lane, 64); });
        }
      }
      const bool more = __any(v.more);
      c0 = more ? c0 + 4 : 0;
      k0 = more ? k0 : k0 + 64;
    }
  for (int z = lane; z < d.ZN; z += 64) {
    float a = lacc[z];
    if constexpr (PACK)
      for (int k = 1; k < g.G; ++k) a += lacc[k * ZN4 + z];
    a *= mk;
    if constexpr (UPDATE) {
      const size_t i = (size_t)col * d.ZN + z;
      const float nx = fmaf(a, A.invCol[i], vcol[z]);
      vcol[z] = nx;
      if (A.shadow) A.shadow[i] = to_bf16_dither(nx, i);
    } else {
      vcol[z] = a;
    }
  }
}

// yp[k][u][v] = y[k][u][v] * K(p,u,v) * invdB[v]: the per-ray factors of fp_kernel
// (y stored as float or BF16, yp FP32).
template <typename T>
__global__ __launch_bounds__(kBlock) void scale_matched_kernel(
    const T* __restrict__ in, float* __restrict__ out, const float4* __restrict__ cols,
    const float* __restrict__ h2, const float* __restrict__ invdB, Dims d, int vb, int vs) {
  const int k = blockIdx.y;
  const int p = vb + k * vs;
  const int ray = blockIdx.x * kBlock + threadIdx.x;
  if (ray >= d.DNU * d.DNV) return;
  const int u = ray / d.DNV, v = ray - u * d.DNV;
  const float4 ct = cols[(size_t)p * d.DNU + u];
  const float K = ct.w * sqrtf(ct.z + h2[v]) * invdB[v];
  const size_t o = (size_t)k * d.DNU * d.DNV + ray;
  out[o] = ld(in, o) * K;
}

__global__ void copy_kernel(float* __restrict__ dst, const float* __restrict__ src, size_t n) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x)
    dst[i] = src[i];
}

__global__ void fill_kernel(float* __restrict__ p, size_t n, float v) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x)
    p[i] = v;
}

__global__ void to_bf16_kernel(uint16_t* __restrict__ dst, const float* __restrict__ src,
                               size_t n) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x)
    dst[i] = to_bf16(src[i]);
}

__global__ void to_bf16_dither_kernel(uint16_t* __restrict__ dst, const float* __restrict__ src,
                                      size_t n) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x)
    dst[i] = to_bf16_dither(src[i], i);
}

// vol[col][z] *= mask[col] (the in-place masking of DD3_GPU.cu:1004-1011, on the device).
__global__ void mask_volume_kernel(float* __restrict__ vol, const float* __restrict__ maskf,
                                   int ZN, size_t n) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x)
    vol[i] *= maskf[i / ZN];
}

__global__ void from_bf16_kernel(float* __restrict__ dst, const uint16_t* __restrict__ src,
                                 size_t n) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x)
    dst[i] = ld(src, i);
}

// out = (in != 0) ? 1/in : 1  -- the guarded divisions of os_sart.m:30-31,38-39.
__global__ void inv_guard_kernel(const float* __restrict__ in, float* __restrict__ out,
                                 size_t n) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x) {
    const float a = in[i];
    out[i] = (a != 0.f) ? 1.0f / a : 1.0f;
  }
}

__global__ void axpy_kernel(float* __restrict__ y, const float* __restrict__ x, double a,
                            size_t n) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x)
    y[i] = (float)((double)y[i] + a * (double)x[i]);
}

__global__ void sub_kernel(float* __restrict__ out, const float* __restrict__ a,
                           const float* __restrict__ b, size_t n) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x)
    out[i] = a[i] - b[i];
}

// FP64 dot product: per-block partial sums (fixed order), then one block reduces.
__global__ __launch_bounds__(kBlock) void dot_partial_kernel(const float* __restrict__ a,
                                                             const float* __restrict__ b,
                                                             size_t n,
                                                             double* __restrict__ partials) {
  double s = 0.0;
  for (size_t i = blockIdx.x * (size_t)kBlock + threadIdx.x; i < n; i += (size_t)gridDim.x * kBlock)
    s += (double)a[i] * (double)b[i];
  block_sum2(s, 0.0, partials + 2 * blockIdx.x);
}

// The two vector steps of a CG iteration, with alpha = rr / pAp and beta = rr1 / rr taken from
// device memory, so that the host waits for no dot product: x += alpha p, r -= alpha t and the
// partial sums of r.r; then p = r + beta p.  64^3, 720 views of
// 256 x 16, three iterations: 1.41 ms with a copy and a wait per dot product, 1.26 ms.
__global__ __launch_bounds__(kBlock) void cg_step_kernel(float* __restrict__ x,
                                                         float* __restrict__ r,
                                                         const float* __restrict__ p,
                                                         const float* __restrict__ t,
                                                         const double* __restrict__ rr,
                                                         const double* __restrict__ pAp, size_t n,
                                                         double* __restrict__ partials) {
  const double a = *rr / *pAp;
  double s = 0.0;
  for (size_t i = blockIdx.x * (size_t)kBlock + threadIdx.x; i < n;
       i += (size_t)gridDim.x * kBlock) {
    x[i] = (float)((double)x[i] + a * (double)p[i]);
    const float ri = (float)((double)r[i] - a * (double)t[i]);
    r[i] = ri;
    s += (double)ri * (double)ri;
  }
  block_sum2(s, 0.0, partials + 2 * blockIdx.x);
}

__global__ void cg_direction_kernel(float* __restrict__ p, const float* __restrict__ r,
                                    const double* __restrict__ rr1,
                                    const double* __restrict__ rr, size_t n) {
  const double b = *rr1 / *rr;
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x)
    p[i] = (float)((double)r[i] + b * (double)p[i]);
}

// result[0..1] = the sums of nparts pairs.  One workgroup, bound by the latency of its loads: as
// many waves as it can have, eight pairs of each lane in flight.
// 64^3, 4608 pairs 5 us as before with 256 threads; 512^2 x 256, 43734 pairs: 45 us, 9.4 us.
constexpr int kReduceThreads = 1024;
__global__ __launch_bounds__(kReduceThreads) void reduce_pairs_kernel(
    const double2* __restrict__ partials, int nparts, double* __restrict__ result) {
  __shared__ double2 red[kReduceThreads / 64];
  double2 s = make_double2(0.0, 0.0);
  for (int i = threadIdx.x; i < nparts; i += 8 * kReduceThreads) {
    double2 q[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int j = i + k * kReduceThreads;
      q[k] = j < nparts ? partials[j] : make_double2(0.0, 0.0);
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      s.x += q[k].x;
      s.y += q[k].y;
    }
  }
  for (int off = 32; off > 0; off >>= 1) {
    s.x += __shfl_xor(s.x, off, 64);
    s.y += __shfl_xor(s.y, off, 64);
  }
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < kReduceThreads / 64; ++w) {
      s.x += red[w].x;
      s.y += red[w].y;
    }
    result[0] = s.x;
    result[1] = s.y;
  }
}

// One block per scan: items[blockIdx.x].out[0..1] = sums of its partial pairs.
__global__ __launch_bounds__(kBlock) void reduce_batch_kernel(const ReduceItem* __restrict__ items) {
  const ReduceItem it = items[blockIdx.x];
  double a = 0.0, b = 0.0;
  for (int i = threadIdx.x; i < it.n; i += kBlock) {
    a += it.partials[2 * i];
    b += it.partials[2 * i + 1];
  }
  block_sum2(a, b, it.out);
}

int grid_1d(size_t n) {
  size_t g = (n + 255) / 256;
  if (g > 65536) g = 65536;
  if (g < 1) g = 1;
  return (int)g;
}

int check_launch(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(CTR_ERR_HIP, std::string(what) + ": " + hipGetErrorString(e));
  return CTR_OK;
}

}  // namespace

// Lanes per item (log2) of the forward projector for a detector of DNV rows: the least
// lanes spent per column, each weighed by the instructions it issues per slice -- about 20
// with one column per wave, 25 in groups, and the FP64 evaluation of a slice (about 130)
// once per L slices.  16 rows: four columns per wave, 87 us against 212 us one thread per
// ray (64^3, 720 views); 40 rows: one column per wave (24 lanes idle), 0.94 ms against
// 2.19 ms (301^2 x 143, 234 views); 80 rows: groups of 16 without idle lanes.
int fp_lanes_log2(int DNV) {
  int best = 6;
  float cost = 1e30f;
  for (int lg = 6; lg >= 3; --lg) {
    const int L = 1 << lg;
    const float c = (float)((DNV + L - 1) / L * L) * ((lg == 6 ? 20.f : 25.f) + 130.f / L);
    if (c < cost) {
      cost = c;
      best = lg;
    }
  }
  return best;
}

static int fp_blocks_of(const Plan& P, int lg, int columns) {
  const int L = 1 << lg, per = kWaves << (6 - lg);  // items per workgroup
  const int items = columns * ((P.d.DNV + L - 1) / L);
  return (items + per - 1) / per;
}
static int fp_blocks_of(const Plan& P, int lg) { return fp_blocks_of(P, lg, P.d.DNU); }

int fp_column_blocks(const Plan& P, int columns) {
  return fp_blocks_of(P, fp_lanes_log2(P.d.DNV), columns);
}

int fp_columns_within(const Plan& P, long long blocks) {
  const int lg = fp_lanes_log2(P.d.DNV), L = 1 << lg;
  const long long items = blocks * (kWaves << (6 - lg));
  return (int)std::max(1ll, std::min<long long>(P.d.DNU, items / ((P.d.DNV + L - 1) / L)));
}

int fp_partial_blocks(const Plan& P, int vc) {
  if (P.method == CTR_METHOD_SAT) return fp_sat_blocks(P.d) * vc;
  return fp_blocks_of(P, fp_lanes_log2(P.d.DNV)) * vc;
}

int fp_partial_most(const Plan& P, int vc) {
  return std::max(fp_sat_blocks(P.d), fp_blocks_of(P, fp_lanes_log2(P.d.DNV))) * vc;
}

template <typename TV, typename TO>
FpArgs<TV, TO> fp_args(const Plan& P, const TV* vol, TO* out, int vb, int vs, const float* b,
                       const float* invRow, double* partials) {
  return FpArgs<TV, TO>{vol,  out,  P.views, P.bnd64, P.cols, P.Bz, P.h2,
                        P.invdB, P.maskf, P.mext, P.d, fp_lanes_log2(P.d.DNV), vb, vs,
                        b,    invRow, partials};
}

template <typename T>
BpArgs<T> bp_args(const Plan& P, const T* prj, float* vol, int vb, int vs, int vc,
                  const float* invCol, uint16_t* shadow) {
  return BpArgs<T>{prj, vol, P.views, P.src64, P.mask, P.d, P.bc, P.bc64, vb, vs, vc,
                   invCol, shadow, bp_pack_lanes(P, false)};
}

int fp_blocks_per_view(const Plan& P, bool colw) {
  return fp_blocks_of(P, colw ? 6 : fp_lanes_log2(P.d.DNV));
}

// f(one column per wave, FINE) with a launch's choices as integral constants.
template <typename F>
static void fp_variant(const Plan& P, F f) {
  using Y = std::true_type;
  using N = std::false_type;
  const bool colw = fp_lanes_log2(P.d.DNV) == 6;
  if (colw && P.d.fine) f(Y{}, Y{});
  else if (colw) f(Y{}, N{});
  else if (P.d.fine) f(N{}, Y{});
  else f(N{}, N{});
}

template <typename TV, typename TO>
int launch_fp(const Plan& P, const TV* vol, TO* out, int vb, int vs, int vc, hipStream_t st,
              const float* b, const float* invRow, double* partials) {
  if (vc <= 0) return CTR_OK;
  const FpArgs<TV, TO> A = fp_args<TV, TO>(P, vol, out, vb, vs, b, invRow, partials);
  const int bpv = fp_blocks_of(P, A.lg);
  const dim3 grid(xcd_chunked_grid((long long)bpv * vc));
  fp_variant(P, [&](auto C, auto F) {
    constexpr bool c = decltype(C)::value, f = decltype(F)::value;
    if (b)
      hipLaunchKernelGGL((fp_kernel<true, c, TV, TO, f>), grid, dim3(kBlock), 0, st, A, bpv, vc);
    else
      hipLaunchKernelGGL((fp_kernel<false, c, TV, TO, f>), grid, dim3(kBlock), 0, st, A, bpv, vc);
  });
  return check_launch("fp_kernel");
}

// The fused partial sums of columns u0 ... u0 + columns - 1 of view p alone (no output): the
// kernel on tables that begin there.
int launch_fp_columns(const Plan& P, const float* vol, int p, int u0, int columns, hipStream_t st,
                      const float* b, double* partials) {
  const size_t at = (size_t)p * P.d.DNU + u0;
  FpArgs<float, float> A = fp_args<float, float>(P, vol, nullptr, 0, 1, b + at * P.d.DNV, nullptr,
                                                 partials);
  A.views += p;
  A.bnd64 += at + p;
  A.cols += at;
  A.d.DNU = columns;
  const int bpv = fp_blocks_of(P, A.lg, columns);
  const dim3 grid(xcd_chunked_grid(bpv));
  fp_variant(P, [&](auto C, auto F) {
    hipLaunchKernelGGL((fp_kernel<true, decltype(C)::value, float, float, decltype(F)::value>),
                       grid, dim3(kBlock), 0, st, A, bpv, 1);
  });
  return check_launch("fp_kernel");
}

int launch_fp_ones(const Plan& P, float* out, int vb, int vs, int vc, hipStream_t st) {
  if (vc <= 0) return CTR_OK;
  const FpArgs<float, float> A =
      fp_args<float, float>(P, nullptr, out, vb, vs, nullptr, nullptr, nullptr);
  const int bpv = fp_blocks_of(P, A.lg);
  const dim3 grid(xcd_chunked_grid((long long)bpv * vc));
  fp_variant(P, [&](auto C, auto F) {
    hipLaunchKernelGGL((fp_ones_kernel<decltype(C)::value, decltype(F)::value>), grid,
                       dim3(kBlock), 0, st, A, bpv, vc);
  });
  return check_launch("fp_ones_kernel");
}

// Lanes of a packed wave's groups (bp_packed_body), 0 for one view at a time.  A group holds a
// view's rows and, where they fit half a wave, the voxels of a column that its cone covers at
// the grid's far edge, DNV l / (S dz) at distance l; a longer window takes a second pass.  The
// windows at the axis (matched: at the far edge) must fit two groups: 512^2 x 256, 32 rows on
// windows of 30 voxels, 38 at the far edge, one view at a time and packed: 2.13 ms, 1.92 ms
// (matched 3.48 ms, 3.65 ms).  The groups' column sums must fit kPackSums floats, a sixth of
// the LDS with four waves: at that limit (16 rows, 256^2 x 512) 578 us, 459 us (matched 938 us,
// 866 us).
int bp_pack_lanes(const Plan& P, bool matched) {
  const Dims& d = P.d;
  if (d.DNV > 32 || !bp_row_chunks(d.DNU, d.DNV)) return 0;
  const double perl = d.DNV / (std::fabs((double)P.bc.S) * d.dz);
  const double sid = 1.0 / P.bc64.inv_sid, R = 0.5 * std::max(d.XN, d.YN) * (double)d.dx;
  const double axis = perl * sid + 2.0, edge = perl * (sid + R) + 2.0;
  if (!((matched ? edge : axis) <= 32.0)) return 0;
  const int need = std::max({d.DNV, (int)std::min(edge, 32.0), 8});
  const int G = std::min(64 / need, kPackSums / ((d.ZN + 3) & ~3));
  return G >= 2 ? 64 / G : 0;
}

// Packed views need enough of them to pay for a group's own sums: 512^2 x 128, 16 rows, 8 views
// 223 us, 173 us one view at a time, 16 views 249 us, 255 us (64^3 7.9 us, 7.1 us; 8.4 us, 9.2 us);
// matched 330 us, 273 us; 381 us, 384 us.  One or two views do not pay for the classes' longer
// code: 512^2 x 128, 64 rows, one view 123 us, 114 us view by view (160 rows 158 us, 123 us;
// 64^3 6.7 us, 4.9 us), four views 150 us, 168 us.  Nor do the second loop's views where they are
// about half of all or more (Dims::coarse): 128^2 x 64, 100 views of 888 x 64, 2.8 mm voxels
// 323 us, 272 us; 1.4 mm 192 us, 159 us; 1 mm (not coarse) 93 us, 152 us; more rows gain nothing.
BpShape bp_shape(const Plan& P, bool matched, int vc) {
  const int ZN4 = (P.d.ZN + 3) & ~3, rc = bp_row_chunks(P.d.DNU, P.d.DNV);
  const BpShape staged{rc, ZN4};
  const int L = vc >= 16 ? bp_pack_lanes(P, matched) : 0;
  if (L) return {kPacked, 64 / L * ZN4};
  if (matched || !rc) return staged;
  if (vc <= 2 || (rc == 1 && P.d.coarse)) return {kPlain - rc / 2, ZN4};
  return staged;
}

// Row chunks (of 64) a staged wave holds for a detector, 0 for the unstaged form: over 256
// rows, or 64 frames past the staged loads' 32-bit byte offsets.
int bp_row_chunks(int DNU, int DNV) {
  if (DNV > 256 || (long long)DNU * DNV > (1ll << 23)) return 0;
  return DNV <= 64 ? 1 : DNV <= 128 ? 2 : 4;
}

int launch_bp_ones(const Plan& P, float* vol, int vb, int vs, int vc, hipStream_t st) {
  if (P.d.ZN > kWinMaxZ) return fail(CTR_ERR_ARG, "bp of ones: columns over the LDS limit");
  const BpArgs<float> A = bp_args<float>(P, nullptr, vol, vb, vs, vc, nullptr, nullptr);
  const dim3 wgrid((P.d.XN * P.d.YN + kWaves - 1) / kWaves);
  const BpShape sh = bp_shape(P, false, vc);
  const size_t lds = (size_t)kWaves * bp_win_floats(sh.rc, sh.sums) * sizeof(float);
#define CTR_BPO(RC) \
  hipLaunchKernelGGL(bp_win_ones_kernel<RC>, wgrid, dim3(kBlock), lds, st, A, sh.sums)
  switch (sh.rc) {
    case kPacked: CTR_BPO(kPacked); break;
    case kPlain: CTR_BPO(kPlain); break;
    case kPlain - 1: CTR_BPO(kPlain - 1); break;
    case kPlain - 2: CTR_BPO(kPlain - 2); break;
    case 1: CTR_BPO(1); break;
    case 2: CTR_BPO(2); break;
    case 4: CTR_BPO(4); break;
    default: CTR_BPO(0); break;
  }
#undef CTR_BPO
  return check_launch("bp_win_ones_kernel");
}

template <typename T>
int launch_bp(const Plan& P, const T* prj, float* vol, int vb, int vs, int vc, int kind,
              hipStream_t st, const float* invCol, int accumulate, uint16_t* shadow) {
  const int zg = std::min(4, (P.d.ZN + 63) / 64);
  dim3 rgrid((P.d.XN * P.d.YN + kWaves - 1) / kWaves, (P.d.ZN + 64 * zg - 1) / (64 * zg));
  if (kind == CTR_BP_MATCHED) {
    if constexpr (!std::is_same<T, float>::value) {
      return fail(CTR_ERR_ARG, "the matched back projector reads the FP32 scaled sinogram");
    } else {
      const BpShape sh = bp_shape(P, true, vc);
      const size_t slds = (size_t)kWaves * bp_matched_floats(sh.rc, sh.sums) * sizeof(float);
      if (P.d.even_rows && sh.rc != 0 && P.d.ZN <= kWinMaxZ && slds <= 65536) {
        const dim3 wgrid((P.d.XN * P.d.YN + kWaves - 1) / kWaves);
        const MatchedArgs M{prj, vol, P.views, P.bnd64, P.cols, P.Bz, P.mask, P.d, P.bc, vb, vs,
                            vc, bp_pack_lanes(P, true), accumulate ? invCol : nullptr,
                            accumulate ? shadow : nullptr};
#define CTR_BPMS(RC)                                                                           \
  do {                                                                                         \
    if (accumulate)                                                                            \
      hipLaunchKernelGGL((bp_matched_staged_kernel<true, RC>), wgrid, dim3(kBlock), slds, st,  \
                         M, sh.sums);                                                          \
    else                                                                                       \
      hipLaunchKernelGGL((bp_matched_staged_kernel<false, RC>), wgrid, dim3(kBlock), slds, st, \
                         M, sh.sums);                                                          \
  } while (0)
        switch (sh.rc) {
          case kPacked: CTR_BPMS(kPacked); break;
          case 1: CTR_BPMS(1); break;
          case 2: CTR_BPMS(2); break;
          default: CTR_BPMS(4); break;
        }
#undef CTR_BPMS
        return check_launch("bp_matched_staged_kernel");
      }
      // (unevenly spaced or over 256 rows) the searching windowed kernel while its row table
      // and column sums fit 64 KiB of LDS
      const size_t lds =
          ((size_t)((P.d.DNV + 1 + 3) & ~3) + (size_t)kWaves * P.d.ZN) * sizeof(float);
      if (P.d.ZN <= kWinMaxZ && lds <= 65536) {
        const dim3 wgrid((P.d.XN * P.d.YN + kWaves - 1) / kWaves);
        if (accumulate)
          hipLaunchKernelGGL((bp_matched_win_kernel<true>), wgrid, dim3(kBlock), lds, st, prj,
                             vol, P.views, P.bnd64, P.cols, P.Bz, P.mask, P.d, P.bc, vb, vs, vc,
                             invCol, shadow);
        else
          hipLaunchKernelGGL((bp_matched_win_kernel<false>), wgrid, dim3(kBlock), lds, st, prj,
                             vol, P.views, P.bnd64, P.cols, P.Bz, P.mask, P.d, P.bc, vb, vs, vc,
                             nullptr, nullptr);
        return check_launch("bp_matched_win_kernel");
      }
#define CTR_BPM(UPD, ZGV, IC, SH)                                                                \
  hipLaunchKernelGGL((bp_matched_kernel<UPD, ZGV>), rgrid, dim3(kBlock), 0, st, prj, vol, P.views, \
                     P.bnd64, P.cols, P.Bz, P.mask, P.d, P.bc, vb, vs, vc, IC, SH)
      if (accumulate) {
        switch (zg) {
          case 1: CTR_BPM(true, 1, invCol, shadow); break;
          case 2: CTR_BPM(true, 2, invCol, shadow); break;
          case 3: CTR_BPM(true, 3, invCol, shadow); break;
          default: CTR_BPM(true, 4, invCol, shadow); break;
        }
      } else {
        switch (zg) {
          case 1: CTR_BPM(false, 1, nullptr, nullptr); break;
          case 2: CTR_BPM(false, 2, nullptr, nullptr); break;
          case 3: CTR_BPM(false, 3, nullptr, nullptr); break;
          default: CTR_BPM(false, 4, nullptr, nullptr); break;
        }
      }
#undef CTR_BPM
      return check_launch("bp_matched_kernel");
    }
  }
  const BpArgs<T> A = bp_args<T>(P, prj, vol, vb, vs, vc, accumulate ? invCol : nullptr,
                                 accumulate ? shadow : nullptr);
  if (P.d.ZN <= kWinMaxZ) {
    const dim3 wgrid((P.d.XN * P.d.YN + kWaves - 1) / kWaves);
    const BpShape sh = bp_shape(P, false, vc);
    const size_t lds = (size_t)kWaves * bp_win_floats(sh.rc, sh.sums) * sizeof(float);
#define CTR_BPW(RC)                                                                           \
  do {                                                                                        \
    if (accumulate)                                                                           \
      hipLaunchKernelGGL((bp_win_kernel<true, T, RC>), wgrid, dim3(kBlock), lds, st, A,       \
                         sh.sums);                                                            \
    else                                                                                      \
      hipLaunchKernelGGL((bp_win_kernel<false, T, RC>), wgrid, dim3(kBlock), lds, st, A,      \
                         sh.sums);                                                            \
  } while (0)
    switch (sh.rc) {
      case kPacked: CTR_BPW(kPacked); break;
    case kPlain: CTR_BPW(kPlain); break;
    case kPlain - 1: CTR_BPW(kPlain - 1); break;
    case kPlain - 2: CTR_BPW(kPlain - 2); break;
      case 1: CTR_BPW(1); break;
      case 2: CTR_BPW(2); break;
      case 4: CTR_BPW(4); break;
      default: CTR_BPW(0); break;
    }
#undef CTR_BPW
    return check_launch("bp_win_kernel");
  }
#define CTR_BPREF(UPD, ZGV) \
  hipLaunchKernelGGL((bp_ref_kernel<UPD, ZGV, T>), rgrid, dim3(kBlock), 0, st, A)
  if (accumulate) {
    switch (zg) {
      case 1: CTR_BPREF(true, 1); break;
      case 2: CTR_BPREF(true, 2); break;
      case 3: CTR_BPREF(true, 3); break;
      default: CTR_BPREF(true, 4); break;
    }
  } else {
    switch (zg) {
      case 1: CTR_BPREF(false, 1); break;
      case 2: CTR_BPREF(false, 2); break;
      case 3: CTR_BPREF(false, 3); break;
      default: CTR_BPREF(false, 4); break;
    }
  }
#undef CTR_BPREF
  return check_launch("bp_ref_kernel");
}

// grid <= 0: one workgroup per item (hardware scheduling, per-scan XCD map)
template <typename T>
int launch_fp_batch(const FpBatchItem<T>* items, int nscan, int total, bool colw, bool fine,
                    int grid, int strided, hipStream_t st) {
  if (total <= 0) return CTR_OK;
  const int sched = grid <= 0 ? 2 : (strided ? 1 : 0);
  grid = grid <= 0 ? total : std::max(1, std::min(grid, total));
  auto launch = [&](auto C, auto F) {
    constexpr bool c = decltype(C)::value, f = decltype(F)::value;
    if (sched == 2)
      hipLaunchKernelGGL((fp_batch1_kernel<true, c, T, f>), dim3(grid), dim3(kBlock), 0, st,
                         items, nscan, total);
    else
      hipLaunchKernelGGL((fp_batch_kernel<true, c, T, f>), dim3(grid), dim3(kBlock), 0, st, items,
                         nscan, total, sched);
  };
  using Y = std::true_type;
  using N = std::false_type;
  if (colw && fine) launch(Y{}, Y{});
  else if (colw) launch(Y{}, N{});
  else if (fine) launch(N{}, Y{});
  else launch(N{}, N{});
  return check_launch("fp_batch_kernel");
}

template <typename T>
int launch_bp_batch(const BpBatchItem<T>* items, int nscan, int total, int zg, int grid,
                    int strided, hipStream_t st) {
  if (total <= 0) return CTR_OK;
  const int sched = grid <= 0 ? 2 : (strided ? 1 : 0);
  grid = grid <= 0 ? total : std::max(1, std::min(grid, total));
#define CTR_BPB(ZGV)                                                                       \
  hipLaunchKernelGGL((bp_batch_kernel<true, ZGV, T>), dim3(grid), dim3(kBlock), 0, st, items, \
                     nscan, total, sched)
  switch (zg) {
    case 1: CTR_BPB(1); break;
    case 2: CTR_BPB(2); break;
    case 3: CTR_BPB(3); break;
    case 4: CTR_BPB(4); break;
    default: return fail(CTR_ERR_ARG, "bp_batch: z groups must be 1..4");
  }
#undef CTR_BPB
  return check_launch("bp_batch_kernel");
}

template <typename T>
int launch_bp_batch_win(const BpBatchItem<T>* items, int nscan, int total, int sums, int rc,
                        int grid, int strided, hipStream_t st) {
  if (total <= 0) return CTR_OK;
  if (sums < 1 || sums > kWinMaxZ) return fail(CTR_ERR_ARG, "bp_batch_win: column height");
  const int sched = grid <= 0 ? 2 : (strided ? 1 : 0);
  grid = grid <= 0 ? total : std::max(1, std::min(grid, total));
  const size_t lds = (size_t)kWaves * bp_win_floats(rc, sums) * sizeof(float);
#define CTR_BPBW(RC)                                                                          \
  do {                                                                                        \
    if (sched == 2)                                                                           \
      hipLaunchKernelGGL((bp_batch_win1_kernel<T, RC>), dim3(grid), dim3(kBlock), lds, st,    \
                         items, nscan, total, sums);                                          \
    else                                                                                      \
      hipLaunchKernelGGL((bp_batch_win_kernel<T, RC>), dim3(grid), dim3(kBlock), lds, st,     \
                         items, nscan, total, sched, sums);                                   \
  } while (0)
  switch (rc) {
    case kPacked: CTR_BPBW(kPacked); break;
    case kPlain: CTR_BPBW(kPlain); break;
    case kPlain - 1: CTR_BPBW(kPlain - 1); break;
    case kPlain - 2: CTR_BPBW(kPlain - 2); break;
    case 1: CTR_BPBW(1); break;
    case 2: CTR_BPBW(2); break;
    case 4: CTR_BPBW(4); break;
    default: CTR_BPBW(0); break;
  }
#undef CTR_BPBW
  return check_launch("bp_batch_win_kernel");
}

int launch_reduce_batch(const ReduceItem* items, int nscan, hipStream_t st) {
  hipLaunchKernelGGL(reduce_batch_kernel, dim3(nscan), dim3(kBlock), 0, st, items);
  return check_launch("reduce_batch_kernel");
}

template <typename T>
int launch_scale_matched(const Plan& P, const T* in, float* out, int vb, int vs, int vc,
                         hipStream_t st) {
  if (vc <= 0) return CTR_OK;
  dim3 grid((P.d.DNU * P.d.DNV + kBlock - 1) / kBlock, vc);
  hipLaunchKernelGGL(scale_matched_kernel<T>, grid, dim3(kBlock), 0, st, in, out, P.cols, P.h2,
                     P.invdB, P.d, vb, vs);
  return check_launch("scale_matched_kernel");
}

template int launch_fp<float, float>(const Plan&, const float*, float*, int, int, int,
                                     hipStream_t, const float*, const float*, double*);
template int launch_fp<uint16_t, uint16_t>(const Plan&, const uint16_t*, uint16_t*, int, int,
                                           int, hipStream_t, const float*, const float*,
                                           double*);
template int launch_fp<float, uint16_t>(const Plan&, const float*, uint16_t*, int, int, int,
                                        hipStream_t, const float*, const float*, double*);
template int launch_bp<float>(const Plan&, const float*, float*, int, int, int, int, hipStream_t,
                              const float*, int, uint16_t*);
template int launch_bp<uint16_t>(const Plan&, const uint16_t*, float*, int, int, int, int,
                                 hipStream_t, const float*, int, uint16_t*);
template FpArgs<float> fp_args<float, float>(const Plan&, const float*, float*, int, int,
                                             const float*, const float*, double*);
template FpArgs<uint16_t> fp_args<uint16_t, uint16_t>(const Plan&, const uint16_t*, uint16_t*,
                                                      int, int, const float*, const float*,
                                                      double*);
template BpArgs<float> bp_args<float>(const Plan&, const float*, float*, int, int, int,
                                      const float*, uint16_t*);
template BpArgs<uint16_t> bp_args<uint16_t>(const Plan&, const uint16_t*, float*, int, int, int,
                                            const float*, uint16_t*);
template int launch_fp_batch<float>(const FpBatchItem<float>*, int, int, bool, bool, int, int,
                                    hipStream_t);
template int launch_fp_batch<uint16_t>(const FpBatchItem<uint16_t>*, int, int, bool, bool, int, int,
                                       hipStream_t);
template int launch_bp_batch<float>(const BpBatchItem<float>*, int, int, int, int, int,
                                    hipStream_t);
template int launch_bp_batch_win<float>(const BpBatchItem<float>*, int, int, int, int, int,
                                        int, hipStream_t);
template int launch_bp_batch_win<uint16_t>(const BpBatchItem<uint16_t>*, int, int, int, int,
                                           int, int, hipStream_t);
template int launch_bp_batch<uint16_t>(const BpBatchItem<uint16_t>*, int, int, int, int, int,
                                       hipStream_t);
template int launch_scale_matched<float>(const Plan&, const float*, float*, int, int, int,
                                         hipStream_t);
template int launch_scale_matched<uint16_t>(const Plan&, const uint16_t*, float*, int, int, int,
                                            hipStream_t);

int launch_to_bf16(uint16_t* dst, const float* src, size_t n, hipStream_t st) {
  hipLaunchKernelGGL(to_bf16_kernel, dim3(grid_1d(n)), dim3(256), 0, st, dst, src, n);
  return check_launch("to_bf16_kernel");
}

int launch_to_bf16_shadow(uint16_t* dst, const float* src, size_t n, hipStream_t st) {
  hipLaunchKernelGGL(to_bf16_dither_kernel, dim3(grid_1d(n)), dim3(256), 0, st, dst, src, n);
  return check_launch("to_bf16_dither_kernel");
}

int launch_mask_volume(const Plan& P, float* vol, hipStream_t st) {
  const size_t n = (size_t)P.d.XN * P.d.YN * P.d.ZN;
  hipLaunchKernelGGL(mask_volume_kernel, dim3(grid_1d(n)), dim3(256), 0, st, vol, P.maskf,
                     P.d.ZN, n);
  return check_launch("mask_volume_kernel");
}

int launch_from_bf16(float* dst, const uint16_t* src, size_t n, hipStream_t st) {
  hipLaunchKernelGGL(from_bf16_kernel, dim3(grid_1d(n)), dim3(256), 0, st, dst, src, n);
  return check_launch("from_bf16_kernel");
}

int launch_copy(float* dst, const float* src, size_t n, hipStream_t st) {
  hipLaunchKernelGGL(copy_kernel, dim3(grid_1d(n)), dim3(256), 0, st, dst, src, n);
  return check_launch("copy_kernel");
}

int launch_fill(float* p, size_t n, float v, hipStream_t st) {
  hipLaunchKernelGGL(fill_kernel, dim3(grid_1d(n)), dim3(256), 0, st, p, n, v);
  return check_launch("fill_kernel");
}

int launch_inv_guard(const float* in, float* out, size_t n, hipStream_t st) {
  hipLaunchKernelGGL(inv_guard_kernel, dim3(grid_1d(n)), dim3(256), 0, st, in, out, n);
  return check_launch("inv_guard_kernel");
}

int launch_axpy(float* y, const float* x, double a, size_t n, hipStream_t st) {
  hipLaunchKernelGGL(axpy_kernel, dim3(grid_1d(n)), dim3(256), 0, st, y, x, a, n);
  return check_launch("axpy_kernel");
}

int launch_sub(float* out, const float* a, const float* b, size_t n, hipStream_t st) {
  hipLaunchKernelGGL(sub_kernel, dim3(grid_1d(n)), dim3(256), 0, st, out, a, b, n);
  return check_launch("sub_kernel");
}

// result[0] = sum(a*b) in FP64; partials holds 2*nparts doubles.
int launch_dot(const float* a, const float* b, size_t n, double* partials, int nparts,
               double* result, hipStream_t st) {
  hipLaunchKernelGGL(dot_partial_kernel, dim3(nparts), dim3(kBlock), 0, st, a, b, n, partials);
  int rc = check_launch("dot_partial_kernel");
  if (rc) return rc;
  return launch_reduce_pairs(partials, nparts, result, st);
}

int launch_cg_update(float* x, float* r, float* p, const float* t, size_t n, const double* rr,
                     const double* pAp, double* rr1, double* partials, int nparts,
                     hipStream_t st) {
  hipLaunchKernelGGL(cg_step_kernel, dim3(nparts), dim3(kBlock), 0, st, x, r, p, t, rr, pAp, n,
                     partials);
  int rc = check_launch("cg_step_kernel");
  if (rc) return rc;
  if ((rc = launch_reduce_pairs(partials, nparts, rr1, st))) return rc;
  hipLaunchKernelGGL(cg_direction_kernel, dim3(grid_1d(n)), dim3(256), 0, st, p, r, rr1, rr, n);
  return check_launch("cg_direction_kernel");
}

int launch_reduce_pairs(const double* partials, int nparts, double* result, hipStream_t st) {
  hipLaunchKernelGGL(reduce_pairs_kernel, dim3(1), dim3(kReduceThreads), 0, st,
                     (const double2*)partials, nparts, result);
  return check_launch("reduce_pairs_kernel");
}

}  // namespace ctr

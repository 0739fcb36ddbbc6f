// k_distance.hip -- masked sliding distances (fastdistance, utils.jl:5-13)
// and valid cross-correlation (imfilter.jl:5-26) for gfx950.
//
// Two evaluations of the same map:
//   * exact:  D[c] = |(A2 - 2 AB) + B2| with A2, AB, B2 fused-multiply-add
//             chains in FP64 over the masked tile voxels in ascending
//             column-major order;
//   * scan:   AB in FP32 over disjoint boxes with the training image staged
//             through LDS, A2 from the exact per-mask map, and a rigorous
//             error bound, giving an interval [lo, hi] that contains the exact
//             FP64 value.  The scan feeds the tol-band superset; members of
//             the superset are recomputed exactly.
// The per-step kernels serve a batch of queries (independent tile steps of a
// wave, all realizations) per launch; blockIdx.z (or .y) selects the query.
#include "iq_internal.h"

// ---------------------------------------------------------------------------
// imfilter: out[c] = sum_j img[c+j] * krn[j]   (FP64, fma chain, column-major j)
// ---------------------------------------------------------------------------
extern "C" __global__ void __launch_bounds__(256)
k_imfilter(const double* __restrict__ img, int nx, int ny, int nz,
           const double* __restrict__ krn, int kx, int ky, int kz,
           double* __restrict__ out, int ox, int oy, int oz) {
  int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int64_t P = (int64_t)ox * oy * oz;
  if (c >= P) return;
  int cx = (int)(c % ox), cy = (int)((c / ox) % oy), cz = (int)(c / ((int64_t)ox * oy));
  const double* base = img + cx + (int64_t)nx * (cy + (int64_t)ny * cz);
  double acc = 0.0;
  int j = 0;
  for (int z = 0; z < kz; z++)
    for (int y = 0; y < ky; y++) {
      const double* row = base + (int64_t)nx * (y + (int64_t)ny * z);
      for (int x = 0; x < kx; x++, j++) acc = __builtin_fma(row[x], krn[j], acc);
    }
  out[c] = acc;
}

// ---------------------------------------------------------------------------
// Exact FP64 map of one query over all candidates (standalone fastdistance and
// the per-mask A2 maps).  MODE 0: D with the A2 and B2 chains; MODE 2: the A2
// chain alone.  toff: training-image offsets of the masked voxels in ascending
// column-major tile order; kv: query values.  Offsets and values are the same
// for every work-item and come through the scalar cache, 16 voxels ahead of
// their chains, so that 16 loads are in flight: 301,806 windows of 720 voxels
// take 62 us, 70 with 8 in flight, 156 with one (the vector instructions are
// ~25 us of it; a row of windows is not aligned, so a load touches 3 to 4
// cache lines).  OFF is the type of a work-item's byte offset: 32 bits go into
// the load as they are, 64 (images of 4 GiB and more) cost an addition each.
// B2 is chained by one wavefront of each workgroup (a launch of its own took
// 52 us).
// ---------------------------------------------------------------------------
template <typename T, int MODE, bool B2, typename OFF>
__device__ __forceinline__ void exact_chains(const T* __restrict__ img, OFF at, const int32_t* __restrict__ toff,
                                             const double* __restrict__ kv, int V, double& a2, double& ab, double& b2) {
  const auto ro = iq_const(toff);
  const auto kq = iq_const(kv);
  const auto rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)img, 0, -1, 0x00027000);
  const auto ld = [&](int o) {
    if constexpr (sizeof(OFF) == 8) {
      return (double)((const __attribute__((address_space(1))) T*)iq_glob(img))[at / sizeof(T) + (uint64_t)o];
    } else if constexpr (sizeof(T) == 4) {
      return (double)__builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, (int)at, (int)((uint32_t)o * 4u), 0));
    } else {
      return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(rsrc, (int)at, (int)((uint32_t)o * 8u), 0));
    }
  };
  int j = 0;
  for (; j + 16 <= V; j += 16) {
    double t[16], u[16];
#pragma unroll
    for (int i = 0; i < 16; i++) {
      t[i] = ld(ro[j + i]);
      if (MODE == 0) u[i] = kq[j + i];
    }
#pragma unroll
    for (int i = 0; i < 16; i++) {
      a2 = __builtin_fma(t[i], t[i], a2);
      if (MODE == 0) ab = __builtin_fma(t[i], u[i], ab);
      if (B2) b2 = __builtin_fma(u[i], u[i], b2);
    }
  }
  for (; j < V; j++) {
    const double t = ld(ro[j]);
    a2 = __builtin_fma(t, t, a2);
    if (MODE == 0) ab = __builtin_fma(t, kq[j], ab);
    if (B2) b2 = __builtin_fma(kq[j], kq[j], b2);
  }
}

template <typename T, int MODE, typename OFF>
__global__ void __launch_bounds__(256)
k_exact_map(const T* __restrict__ img, IqGeo g, const int32_t* __restrict__ toff,
            const double* __restrict__ kv, int V, double* __restrict__ out) {
  const int64_t c0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t c = c0 < g.P ? c0 : g.P - 1;
  const int cx = (int)(c % g.dist[0]), cy = (int)((c / g.dist[0]) % g.dist[1]);
  const int cz = (int)(c / ((int64_t)g.dist[0] * g.dist[1]));
  const OFF at = (OFF)((uint64_t)iq_lin3(g.ti, cx, cy, cz) * sizeof(T));
  double a2 = 0.0, ab = 0.0, b2 = 0.0;
  if (MODE == 2) {
    exact_chains<T, 2, false>(img, at, toff, kv, V, a2, ab, b2);
    if (c0 < g.P) out[c0] = a2;
    return;
  }
  __shared__ double b2s;
  // the chaining wavefront moves with the workgroup: each SIMD gets its share
  if (__builtin_amdgcn_readfirstlane(threadIdx.x >> 6) == (blockIdx.x & 3)) {
    exact_chains<T, MODE, MODE == 0>(img, at, toff, kv, V, a2, ab, b2);
    if ((threadIdx.x & 63) == 0) b2s = b2;
  } else {
    exact_chains<T, MODE, false>(img, at, toff, kv, V, a2, ab, b2);
  }
  __syncthreads();
  if (c0 < g.P) out[c0] = __builtin_fabs((a2 - 2.0 * ab) + b2s);
}

template <typename T, int MODE>
static void launch_exact_map(hipStream_t s, const T* img, const IqGeo& g, const int32_t* toff, const double* kv, int V, double* out) {
  const int64_t ni = (int64_t)g.ti[0] * g.ti[1] * g.ti[2];
  const dim3 gr((unsigned)((g.P + 255) / 256));
  if (ni * (int64_t)sizeof(T) < (1ll << 32))
    hipLaunchKernelGGL((k_exact_map<T, MODE, uint32_t>), gr, dim3(256), 0, s, img, g, toff, kv, V, out);
  else
    hipLaunchKernelGGL((k_exact_map<T, MODE, uint64_t>), gr, dim3(256), 0, s, img, g, toff, kv, V, out);
}

// ---------------------------------------------------------------------------
// Query staging, one workgroup per (query, source).  Source 0 is the overlap
// query (grid = the realization's simulation grid), 1 the hard-data query
// (grid = hard-data grid), 2+a the soft query of pair a (grid = aux[a]).
// Writes the query values at the masked voxels (ascending column-major), the
// box-ordered zero-padded FP32 copy for the scan, and the exact B2 chain; the
// overlap source also resets the query's reduction words.
// ---------------------------------------------------------------------------
#define PREP_LDS 8192

template <typename T>
__device__ __forceinline__ void query_prep_body(const IqDev* __restrict__ D, const IqQuery* __restrict__ qs, int qx,
                                                int src, double* kl) {
  const IqQuery q = qs[qx];
  const IqGeo& g = D->g;
  const IqStep& st = D->steps[q.step];
  const int64_t slot = q.slot;
  int V = 0;
  const int32_t* tv = nullptr;
  const IqMask* mask = nullptr;
  if (src == 0) {
    if (st.mask >= 0) {
      mask = &D->masks[st.mask];
      V = mask->V;
      tv = D->tvox + mask->off;
    }
    if (threadIdx.x == 0) {
      D->gmin_hi[slot] = 0x7f800000u;
      D->gmin64[slot] = 0x7ff0000000000000ull;
      D->nsup[slot] = 0;
      D->ncand[slot] = 0;
    }
  } else if (src == 1) {
    if (!q.multi || q.rep != q.slot || !st.hard) return;
    V = st.hcnt;
    tv = D->htvox + st.hoff;
  } else {
    if (!q.multi || q.rep != q.slot) return;
    V = g.tilevox;
    tv = D->tvox + D->full_off;
  }
  double* kv = D->kv + slot * D->kv_stride + (int64_t)src * g.tilevox;
  const int ox = st.origin[0], oy = st.origin[1], oz = st.origin[2];
  const IqReal& R = D->reals[q.real];
  const T* sim = (const T*)D->sims + R.sim_off;
  const double* dgrid = src == 1 ? R.hard : (src >= 2 ? R.aux[src - 2] : nullptr);
  // four voxels per pass: offsets, then grid values, all loads in flight
  const auto tvg = iq_glob(tv);
  const int t0 = g.tile[0], t1 = g.tile[1];
  for (int j0 = threadIdx.x; j0 < V; j0 += 4 * blockDim.x) {
    int t[4];
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const int j = j0 + u * (int)blockDim.x;
      t[u] = tvg[j < V ? j : 0];
    }
    int64_t gi[4];
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const int x = t[u] % t0, y = (t[u] / t0) % t1, z = t[u] / (t0 * t1);
      gi[u] = iq_lin3(R.pad, ox + x, oy + y, oz + z);
    }
    double v[4];
    if (src == 0) {  // uniform per group
#pragma unroll
      for (int u = 0; u < 4; u++) v[u] = (double)sim[gi[u]];
    } else {
#pragma unroll
      for (int u = 0; u < 4; u++) v[u] = dgrid[gi[u]];
    }
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const int j = j0 + u * (int)blockDim.x;
      if (j < V) {
        kv[j] = v[u];
        if (j < PREP_LDS) kl[j] = v[u];
      }
    }
  }
  if (src == 0 && mask && !q.multi && D->ti32 && D->kv32_on) {
    float* kv32 = D->kv32 + slot * D->kv32_stride;
    for (int b = 0; b < mask->nbox; b++) {
      const IqBox bx = mask->box[b];
      int n = bx.wxp * bx.wy * bx.wz;
      for (int i = threadIdx.x; i < n; i += blockDim.x) {
        int x = i % bx.wxp, y = (i / bx.wxp) % bx.wy, z = i / (bx.wxp * bx.wy);
        float v = 0.0f;
        if (x < bx.wx) v = (float)sim[iq_lin3(R.pad, ox + bx.x0 + x, oy + bx.y0 + y, oz + bx.z0 + z)];
        kv32[bx.kofs + i] = v;
      }
    }
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    // B2 chain in ascending voxel order; the next eight values are read from
    // LDS while the current eight run through the fmas
    double s = 0.0;
    int j = 0;
    const int vl = V < PREP_LDS ? V : PREP_LDS;
    double a[8];
    if (vl >= 8) {
#pragma unroll
      for (int i = 0; i < 8; i++) a[i] = kl[i];
    }
    for (; j + 8 <= vl; j += 8) {
      const int jn = j + 16 <= vl ? j + 8 : j;
      double an[8];
#pragma unroll
      for (int i = 0; i < 8; i++) an[i] = kl[jn + i];
#pragma unroll
      for (int i = 0; i < 8; i++) s = __builtin_fma(a[i], a[i], s);
#pragma unroll
      for (int i = 0; i < 8; i++) a[i] = an[i];
    }
    for (; j < vl; j++) s = __builtin_fma(kl[j], kl[j], s);
    for (; j < V; j++) s = __builtin_fma(kv[j], kv[j], s);  // beyond the LDS stage
    D->b2[slot * (2 + D->naux) + src] = s;
  }
}

template <typename T>
__global__ void __launch_bounds__(256)
k_query_prep(const IqDev* __restrict__ D, const IqQuery* __restrict__ qs) {
  __shared__ double kl[PREP_LDS];
  query_prep_body<T>(D, qs, blockIdx.x, blockIdx.y, kl);
}

template __global__ void k_query_prep<float>(const IqDev*, const IqQuery*);
template __global__ void k_query_prep<double>(const IqDev*, const IqQuery*);

// ---------------------------------------------------------------------------
// FP32 scan.  Work-item (lx, ly, lz) of the group owns R consecutive
// candidates along x.  Per box, the needed training-image block is staged in
// LDS with an R-interleaved row layout (element x of a row lives at
// (x % R) * S + x / R) so that lanes read consecutive words, conflict free,
// while each loaded word feeds R fused multiply-adds.
// Grid: x, y candidate blocks; z = candidate z-block + nbz * query.
// ---------------------------------------------------------------------------
template <int R, int LX, int LY, int LZ>
__global__ void __launch_bounds__(LX * LY * LZ)
k_scan_f32(const IqDev* __restrict__ D, const IqQuery* __restrict__ qs, int nbz) {
  extern __shared__ float lds[];
  const IqQuery q = qs[blockIdx.z / nbz];
  const IqStep& st = D->steps[q.step];
  if (q.multi || st.mask < 0) return;
  const IqGeo& g = D->g;
  const IqMask* mask = &D->masks[st.mask];
  const int64_t slot = q.slot;
  const float* __restrict__ ti = D->ti32;
  const float* __restrict__ kv32 = D->kv32 + slot * D->kv32_stride;
  const int tid = threadIdx.x;
  const int lx = tid % LX, ly = (tid / LX) % LY, lz = tid / (LX * LY);
  const int cx0 = blockIdx.x * (LX * R), cy0 = blockIdx.y * LY, cz0 = (blockIdx.z % nbz) * LZ;
  float acc[R];
#pragma unroll
  for (int i = 0; i < R; i++) acc[i] = 0.0f;
  const int nbox = mask->nbox;
  for (int b = 0; b < nbox; b++) {
    const IqBox bx = mask->box[b];
    const int wxp = bx.wxp;
    const int S = LX + wxp / R;              // interleave stride
    const int RXL = R * LX + wxp - 1;        // logical row length
    const int RY = LY + bx.wy - 1, RZ = LZ + bx.wz - 1;
    const int rowst = R * S;
    const int nst = RXL * RY * RZ;
    const int gx0 = cx0 + bx.x0, gy0 = cy0 + bx.y0, gz0 = cz0 + bx.z0;
    for (int i = tid; i < nst; i += LX * LY * LZ) {
      int x = i % RXL, y = (i / RXL) % RY, z = i / (RXL * RY);
      int gx = gx0 + x, gy = gy0 + y, gz = gz0 + z;
      float v = 0.0f;
      if (gx < g.ti[0] && gy < g.ti[1] && gz < g.ti[2]) v = ti[iq_lin3(g.ti, gx, gy, gz)];
      lds[(z * RY + y) * rowst + (x % R) * S + x / R] = v;
    }
    __syncthreads();
    const float* kb = kv32 + bx.kofs;
    for (int jz = 0; jz < bx.wz; jz++) {
      for (int jy = 0; jy < bx.wy; jy++) {
        const float* rowp = lds + ((lz + jz) * RY + (ly + jy)) * rowst + lx;
        const float* kp = kb + (jz * bx.wy + jy) * wxp;
        for (int jx = 0; jx < wxp; jx += 4) {
          const float* rp = rowp + jx / R;
          float v[R + 3];
#pragma unroll
          for (int m = 0; m < R + 3; m++) v[m] = rp[(m % R) * S + m / R];
          const float k0 = kp[jx], k1 = kp[jx + 1], k2 = kp[jx + 2], k3 = kp[jx + 3];
#pragma unroll
          for (int i = 0; i < R; i++) {
            acc[i] = __builtin_fmaf(v[i], k0, acc[i]);
            acc[i] = __builtin_fmaf(v[i + 1], k1, acc[i]);
            acc[i] = __builtin_fmaf(v[i + 2], k2, acc[i]);
            acc[i] = __builtin_fmaf(v[i + 3], k3, acc[i]);
          }
        }
      }
    }
    __syncthreads();
  }
  // bound and publish
  const double* a2map = D->a2maps[mask->a2];
  const double b2 = D->b2[slot * (2 + D->naux)];
  const double V = (double)mask->V;
  const double u32 = 0x1p-24, u64 = 0x1p-53;
  const double g32 = V * u32 / (1.0 - V * u32), g64 = V * u64 / (1.0 - V * u64);
  float* lo_out = D->lo32 + slot * g.P;
  float lmin = __builtin_inff();
  const int cy = cy0 + ly, cz = cz0 + lz;
#pragma unroll
  for (int i = 0; i < R; i++) {
    const int cx = cx0 + R * lx + i;
    if (cx < g.dist[0] && cy < g.dist[1] && cz < g.dist[2]) {
      int64_t c = iq_lin3(g.dist, cx, cy, cz);
      float lo = __builtin_inff(), hi = __builtin_inff();
      if (!D->disabled[c]) {
        double a2 = a2map[c];
        double s = __builtin_sqrt(a2 * b2) * (1.0 + 0x1p-30);
        double d = __builtin_fabs((a2 - 2.0 * (double)acc[i]) + b2);
        double e = (2.0 * (g32 + g64) * s + 4.0 * u64 * (a2 + b2 + 2.0 * s) + 2.0 * V * 0x1p-148) * (1.0 + 0x1p-30)
                   + 4.0 * u64 * d;
        lo = iq_f32_down(d - e > 0.0 ? d - e : 0.0);
        hi = iq_f32_up(d + e);
      }
      lo_out[c] = lo;
      lmin = fminf(lmin, hi);
    }
  }
  // workgroup min of the upper bounds -> one atomic per group
  __shared__ float red[LX * LY * LZ / 64];
  for (int o = 32; o > 0; o >>= 1) lmin = fminf(lmin, __shfl_xor(lmin, o));
  if ((tid & 63) == 0) red[tid >> 6] = lmin;
  __syncthreads();
  if (tid == 0) {
    float m = red[0];
    for (int w = 1; w < LX * LY * LZ / 64; w++) m = fminf(m, red[w]);
    atomicMin(&D->gmin_hi[slot], __float_as_uint(m));  // non-negative floats order like their bits
  }
}

// ---------------------------------------------------------------------------
// FP32 scan with a 2-D register block (3-D candidate grids): a work-item owns
// R x-candidates times RY y-candidates at one z; the lanes of a wavefront span
// x (LX) and z (LZ) and the four wavefronts span y, so every loop over
// training-image rows is uniform across the wavefront.  One LDS row segment
// (R + 3 words) feeds up to 4 * R * RY fused multiply-adds: the row at offset
// ty serves candidate row iy with query row jy = ty - iy.  LDS rows use the
// R-interleaved layout of k_scan_f32 (conflict-free lane reads); the z-plane
// stride is padded to 8 words modulo 64 banks.
// Grid: x, y candidate blocks; z = candidate z-block + nbz * query.
// ---------------------------------------------------------------------------
template <int R, int RY, int LX, int LZ>
__global__ void __launch_bounds__(256)
k_scan2_f32(const IqDev* __restrict__ D, const IqQuery* __restrict__ qs, int nbz, int perz) {
  constexpr int LY = 256 / (LX * LZ);
  extern __shared__ float lds[];
  const IqQuery q = qs[blockIdx.z / nbz];
  const IqStep& st = D->steps[q.step];
  if (q.multi || st.mask < 0) return;
  const IqGeo& g = D->g;
  const IqMask* mask = &D->masks[st.mask];
  const int64_t slot = q.slot;
  const float* __restrict__ ti = D->ti32;
  const float* __restrict__ kv32 = D->kv32 + slot * D->kv32_stride;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int lx = lane % LX, lz = lane / LX, ly = tid >> 6;
  const int cx0 = blockIdx.x * (LX * R), cy0 = blockIdx.y * (LY * RY), cz0 = (blockIdx.z % nbz) * LZ;
  float acc[RY][R];
#pragma unroll
  for (int a = 0; a < RY; a++)
#pragma unroll
    for (int i = 0; i < R; i++) acc[a][i] = 0.0f;
  const int nbox = mask->nbox;
  for (int b = 0; b < nbox; b++) {
    const IqBox bx = mask->box[b];
    const int wxp = bx.wxp, wy = bx.wy, wz = bx.wz;
    const int S = LX + wxp / R;
    const int RXL = R * LX + wxp - 1;
    const int RYT = LY * RY + wy - 1, RZ = LZ + wz - 1;
    const int rowst = R * S;
    const int plane = ((RYT * rowst + 55) / 64) * 64 + 8;  // = 8 (mod 64)
    const int gx0 = cx0 + bx.x0, gy0 = cy0 + bx.y0, gz0 = cz0 + bx.z0;
    // perz: stage the LZ planes of one jz at a time (large tiles), else all RZ planes once
    const int nplanes = perz ? LZ : RZ;
    const int nst = RXL * RYT * nplanes;
    const float* kb = kv32 + bx.kofs;
    const int nty = RY + wy - 1;
    for (int jz = 0; jz < wz; jz++) {
      if (jz == 0 || perz) {
        if (jz > 0) __syncthreads();
        const int zoff = perz ? jz : 0;
        for (int i = tid; i < nst; i += 256) {
          int x = i % RXL, y = (i / RXL) % RYT, z = i / (RXL * RYT);
          int gx = gx0 + x, gy = gy0 + y, gz = gz0 + zoff + z;
          float v = 0.0f;
          if (gx < g.ti[0] && gy < g.ti[1] && gz < g.ti[2]) v = ti[iq_lin3(g.ti, gx, gy, gz)];
          lds[z * plane + y * rowst + (x % R) * S + x / R] = v;
        }
        __syncthreads();
      }
      const float* zp = lds + (lz + (perz ? 0 : jz)) * plane + lx + (ly * RY) * rowst;
      const float* kz = kb + jz * wy * wxp;
      for (int ty = 0; ty < nty; ty++) {
        const float* rowp = zp + ty * rowst;
        for (int jx = 0; jx < wxp; jx += 4) {
          const float* rp = rowp + jx / R;
          float v[R + 3];
#pragma unroll
          for (int m = 0; m < R + 3; m++) v[m] = rp[(m % R) * S + m / R];
#pragma unroll
          for (int a = 0; a < RY; a++) {
            const int jy = ty - a;
            if (jy >= 0 && jy < wy) {
              const float* kp = kz + jy * wxp + jx;
              const float k0 = kp[0], k1 = kp[1], k2 = kp[2], k3 = kp[3];
#pragma unroll
              for (int i = 0; i < R; i++) {
                acc[a][i] = __builtin_fmaf(v[i], k0, acc[a][i]);
                acc[a][i] = __builtin_fmaf(v[i + 1], k1, acc[a][i]);
                acc[a][i] = __builtin_fmaf(v[i + 2], k2, acc[a][i]);
                acc[a][i] = __builtin_fmaf(v[i + 3], k3, acc[a][i]);
              }
            }
          }
        }
      }
    }
    __syncthreads();
  }
  const double* a2map = D->a2maps[mask->a2];
  const double b2 = D->b2[slot * (2 + D->naux)];
  const double V = (double)mask->V;
  const double u32 = 0x1p-24, u64 = 0x1p-53;
  const double g32 = V * u32 / (1.0 - V * u32), g64 = V * u64 / (1.0 - V * u64);
  float* lo_out = D->lo32 + slot * g.P;
  float lmin = __builtin_inff();
  const int cz = cz0 + lz;
#pragma unroll
  for (int a = 0; a < RY; a++) {
    const int cy = cy0 + ly * RY + a;
#pragma unroll
    for (int i = 0; i < R; i++) {
      const int cx = cx0 + R * lx + i;
      if (cx < g.dist[0] && cy < g.dist[1] && cz < g.dist[2]) {
        int64_t c = iq_lin3(g.dist, cx, cy, cz);
        float lo = __builtin_inff(), hi = __builtin_inff();
        if (!D->disabled[c]) {
          double a2 = a2map[c];
          double sq = __builtin_sqrt(a2 * b2) * (1.0 + 0x1p-30);
          double d = __builtin_fabs((a2 - 2.0 * (double)acc[a][i]) + b2);
          double e = (2.0 * (g32 + g64) * sq + 4.0 * u64 * (a2 + b2 + 2.0 * sq) + 2.0 * V * 0x1p-148) * (1.0 + 0x1p-30)
                     + 4.0 * u64 * d;
          lo = iq_f32_down(d - e > 0.0 ? d - e : 0.0);
          hi = iq_f32_up(d + e);
        }
        lo_out[c] = lo;
        lmin = fminf(lmin, hi);
      }
    }
  }
  __shared__ float red[4];
  for (int o = 32; o > 0; o >>= 1) lmin = fminf(lmin, __shfl_xor(lmin, o));
  if (lane == 0) red[ly] = lmin;
  __syncthreads();
  if (tid == 0) {
    float m = fminf(fminf(red[0], red[1]), fminf(red[2], red[3]));
    atomicMin(&D->gmin_hi[slot], __float_as_uint(m));
  }
}

template __global__ void k_scan2_f32<4, 4, 8, 8>(const IqDev*, const IqQuery*, int, int);
template __global__ void k_scan2_f32<4, 4, 16, 4>(const IqDev*, const IqQuery*, int, int);

// ---------------------------------------------------------------------------
// MFMA scan (multi-query GEMM): AB[c, q] = sum_k A[c, k] * B[k, q] with
// A[c, k] = TI[c + voxel(k)] and B[k, q] = query q's value at voxel(k) (zero
// outside q's mask), on v_mfma_f32_32x32x16_bf16: 32 candidates (consecutive
// x) by 32 queries by 16 voxels per instruction, FP32 accumulation.  FP32
// data is split t = hi + lo (two bf16) and three products are accumulated
// (hi*hi, hi*lo, lo*hi); bf16-exact data (small integer codes) needs one.
// Each wavefront owns four 32-candidate rows (consecutive y) of one z, the
// group (two to four wavefronts, chosen per plan so that the groups of a
// launch pack the compute units evenly) 8 to 16 rows; the block of each box is
// staged in LDS from a packed copy of the image, y fastest, and A fragments
// are read from it column by column (scan_frags).
// What bounds it: split data the matrix cores at the card's power (70 % of the
// cycles at 1.7 GHz for 2.9M candidates, 1.2 PFLOP/s issued, the rate of a large
// library product), so LDS and permute work saved buys clock; bf16-exact data
// the instructions around its four MFMAs a k-step.  Per launch, a region in the
// image's order with eight words a row read, and this form: 2.9M candidates 65
// queries 6,185 and 5,844 us; 302k candidates 26 queries 108 and 98 us; 403k
// candidates, facies, 604 and 502 us.  Tried: two query tiles a group (bf16,
// 180 registers: 21 % slower), four wavefronts per SIMD (equal).
// Grid: x blocks (32), y blocks (4 x wavefronts), z = candidate z + dist_z * query tile.
// ---------------------------------------------------------------------------
typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 iq_bf16x8;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float iq_f32x16;
typedef unsigned int iq_u32x4 __attribute__((ext_vector_type(4)));

__device__ inline uint32_t iq_bf16_rne(float f) {  // round-to-nearest-even bf16 bits of a finite float
  uint32_t u = __float_as_uint(f);
  return (u + 0x7fffu + ((u >> 16) & 1u)) >> 16;
}

__device__ inline uint32_t iq_split_word(float t) {  // hi | lo << 16
  uint32_t h = iq_bf16_rne(t);
  float r = t - __uint_as_float(h << 16);
  return h | (iq_bf16_rne(r) << 16);
}

// B fragments of a batch: lane l of (tile, step) holds the eight values of
// chunk 2*step + l/32 for query tile*32 + l%32, as bf16 hi and lo.
__device__ __forceinline__ void mfma_bprep_body(const IqDev* __restrict__ D, const IqQuery* __restrict__ qs, int nq,
                                                int step, int tile, int lane) {
  const int nstep = D->ktab.nstep;
  const int qi = tile * 32 + (lane & 31);
  uint32_t h[4] = {0u, 0u, 0u, 0u}, l[4] = {0u, 0u, 0u, 0u};
  if (qi < nq) {
    const IqQuery q = qs[qi];
    const IqStep& st = D->steps[q.step];
    if (!q.multi && st.mask >= 0) {
      const IqGeo& g = D->g;
      const IqChunk ch = D->chunks[2 * step + (lane >> 5)];
      const uint8_t* mb = D->maskbits + (int64_t)st.mask * g.tilevox;
      const IqReal& R = D->reals[q.real];
      if (ch.nx > 0) {
        // mask bytes, then grid values of the chunk's (up to) eight voxels,
        // each batch of loads in flight together; positions past the box
        // repeat its first voxel and are dropped
        int64_t gi[8];
        uint8_t on[8];
#pragma unroll
        for (int e = 0; e < 8; e++) {
          const int ey = e & (ch.cy - 1), ex = e / ch.cy;
          const bool in = ey < ch.ny && ex < ch.nx;
          const int x = ch.jx + (in ? ex : 0), y = ch.jy + (in ? ey : 0), z = ch.jz;
          on[e] = in ? mb[x + g.tile[0] * (y + g.tile[1] * z)] : 0;
          gi[e] = iq_lin3(R.pad, st.origin[0] + x, st.origin[1] + y, st.origin[2] + z);
        }
        float v[8];
        if (D->ti_f32) {
          const float* sim32 = (const float*)D->sims + R.sim_off;
#pragma unroll
          for (int e = 0; e < 8; e++) v[e] = sim32[gi[e]];
        } else {
          const double* sim64 = (const double*)D->sims + R.sim_off;
#pragma unroll
          for (int e = 0; e < 8; e++) v[e] = (float)(sim64[gi[e]] * D->scan_s);
        }
#pragma unroll
        for (int e = 0; e < 8; e++) {
          if (!on[e]) continue;
          const uint32_t wv = iq_split_word(v[e]);
          h[e >> 1] |= (wv & 0xffffu) << (16 * (e & 1));
          l[e >> 1] |= (wv >> 16) << (16 * (e & 1));
        }
      }
    }
  }
  const int64_t o = ((int64_t)tile * nstep + step) * 64 + lane;
  D->bh[o] = make_uint4(h[0], h[1], h[2], h[3]);
  D->bl[o] = make_uint4(l[0], l[1], l[2], l[3]);
}

__global__ void __launch_bounds__(64)
k_mfma_bprep(const IqDev* __restrict__ D, const IqQuery* __restrict__ qs, int nq) {
  mfma_bprep_body(D, qs, nq, blockIdx.x, blockIdx.y, threadIdx.x);
}

// Query preparation and B fragments in one launch (both read the grid, neither
// reads what the other writes): blocks [0, nq) prepare one query each (the
// overlap source), the others hold four (k-step, query tile) items, one per
// wavefront.
template <typename T>
__global__ void __launch_bounds__(256)
k_prep_bprep(const IqDev* __restrict__ D, const IqQuery* __restrict__ qs, int nq, int nitems) {
  __shared__ double kl[PREP_LDS];
  if ((int)blockIdx.x < nq) {
    query_prep_body<T>(D, qs, blockIdx.x, 0, kl);
    return;
  }
  const int item = ((int)blockIdx.x - nq) * 4 + (int)(threadIdx.x >> 6);
  if (item >= nitems) return;
  const int nstep = D->ktab.nstep;
  mfma_bprep_body(D, qs, nq, item % nstep, item / nstep, threadIdx.x & 63);
}
template __global__ void k_prep_bprep<float>(const IqDev*, const IqQuery*, int, int);
template __global__ void k_prep_bprep<double>(const IqDev*, const IqQuery*, int, int);

// FP32 copy of an A2 map, times s2 (scan_s2), for the scan's interval bound;
// NaN marks a disabled window (an A2 that overflows FP32 becomes +inf and
// stays a candidate)
__global__ void __launch_bounds__(256)
k_a2_f32(const double* __restrict__ a2, const uint8_t* __restrict__ disabled, int64_t P, double s2, float* __restrict__ out) {
  for (int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x; c < P; c += (int64_t)gridDim.x * 256)
    out[c] = disabled[c] ? __builtin_nanf("") : (float)(a2[c] * s2);
}

// The image in the words the scan stages, y fastest: word (y, x, z) holds the
// bf16 split (hi | lo << 16) of its voxel (SPLIT), or its voxel and the next
// along y as a bf16 pair (bf16-exact data).  Written once per plan; `n` words,
// those past the image zero (a staged region may run past it).
template <bool SPLIT>
__global__ void __launch_bounds__(256)
k_scan_pack(const float* __restrict__ ti, int t0, int t1, int t2, uint32_t* __restrict__ out, int64_t n) {
  const int64_t nv = (int64_t)t0 * t1 * t2;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
    uint32_t v = 0;
    if (i < nv) {
      const int y = (int)(i % t1), x = (int)((i / t1) % t0), z = (int)(i / ((int64_t)t0 * t1));
      const float* p = ti + x + (int64_t)t0 * (y + (int64_t)t1 * z);
      if (SPLIT) v = iq_split_word(*p);
      else v = iq_bf16_rne(*p) | (y + 1 < t1 ? iq_bf16_rne(p[t0]) << 16 : 0u);
    }
    out[i] = v;
  }
}
template __global__ void k_scan_pack<true>(const float*, int, int, int, uint32_t*, int64_t);
template __global__ void k_scan_pack<false>(const float*, int, int, int, uint32_t*, int64_t);

// A fragments of four candidate rows (consecutive y) for one chunk, taken as
// four pairs of voxels along y, off[c] words from the lane's first: whatever
// the chunk's shape the code is the same, without a branch between the reads
// and the MFMAs (one by shape cost a fifth of the kernel's time).  The rows'
// pairs overlap, so a pair takes five words for the four rows together, 20 a
// chunk; a chunk along x takes 8 words a row, 32.  at and off are even: 8-byte
// reads.
typedef unsigned int iq_u32x2 __attribute__((ext_vector_type(2)));
template <bool SPLIT>
__device__ __forceinline__ void scan_frags(const uint32_t* lw, int at, const int (&off)[4], uint4 (&h)[4], uint4 (&l)[4]) {
  uint32_t w[4][6];
#pragma unroll
  for (int c = 0; c < 4; c++) {
    const uint32_t* p = lw + at + off[c];
    const iq_u32x2 v0 = ((const iq_u32x2*)p)[0], v1 = ((const iq_u32x2*)p)[1];
    w[c][0] = v0.x; w[c][1] = v0.y; w[c][2] = v1.x; w[c][3] = v1.y;
    if (SPLIT) w[c][4] = p[4];
  }
#pragma unroll
  for (int i = 0; i < 4; i++) {
    uint32_t a[4], b[4];
#pragma unroll
    for (int c = 0; c < 4; c++) {
      a[c] = SPLIT ? __builtin_amdgcn_perm(w[c][i + 1], w[c][i], 0x05040100u) : w[c][i];
      b[c] = SPLIT ? __builtin_amdgcn_perm(w[c][i + 1], w[c][i], 0x07060302u) : 0u;
    }
    h[i] = make_uint4(a[0], a[1], a[2], a[3]);
    if (SPLIT) l[i] = make_uint4(b[0], b[1], b[2], b[3]);
  }
}

// LIST: candidates within the band of the least upper bound known so far are
// listed (lo32: bounds, band: candidates, ncand: how many; every member of the
// final superset is among them) in place of a store of every bound, which no
// line is whole in (the lanes hold a candidate of 32 queries each) and the
// selection reads again.  The bound returned by the atomic is waited for: read
// ahead of the k-steps it is too old (facies scans took a tenth longer).  Scan
// and selection over 402,075 windows of 24x24x6 codes, 512 queries: 1,306 us
// with the store, 864 with the list; 64 queries 184 and 136, 32 queries 89 and
// 87.  In a launch of a few groups no group knows another's bound and the wait
// is not covered: one query tile in 4 groups 22 and 25 (scan_lists draws the
// line).
template <bool SPLIT, bool LIST>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3)))
k_scan_mfma(const IqDev* __restrict__ D, const IqQuery* __restrict__ qs, int nq, double gerr,
            const int32_t* __restrict__ kofs_tab, int exact) {
  extern __shared__ __align__(16) uint32_t lw[];
  __shared__ float red[4][32], thr[32];
  __shared__ int sslot[32];
  const IqGeo& g = D->g;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int row = lane & 31, kb = lane >> 5;
  const int tile = blockIdx.z / g.dist[2];
  const int cz = blockIdx.z % g.dist[2];
  const int nw = (int)(blockDim.x >> 6), NT = (int)blockDim.x;  // 2 to 4 wavefronts, 4 rows each
  const int cx0 = blockIdx.x * 32, cy0 = blockIdx.y * 4 * nw;
  const bool wlive = cy0 + 4 * w < g.dist[1];  // uniform per wavefront
  const int nstep = D->ktab.nstep;
  const int t0 = g.ti[0], t1 = g.ti[1];
  const int d0 = g.dist[0], d1 = g.dist[1];
  const auto tiw = iq_glob(D->tiw);
  const auto kofs = iq_glob(kofs_tab);
  const auto bhp = iq_glob((const iq_u32x4*)(D->bh + (int64_t)tile * nstep * 64 + lane));
  const auto blp = iq_glob((const iq_u32x4*)(D->bl + (int64_t)tile * nstep * 64 + lane));
  iq_f32x16 acc[4];
#pragma unroll
  for (int i = 0; i < 4; i++)
#pragma unroll
    for (int v = 0; v < 16; v++) acc[i][v] = 0.0f;
  for (int b = 0; b < D->ktab.nbox; b++) {
    const IqKBox kbx = D->ktab.box[b];
    const int ry = iq_scan_ry(kbx.wyr, nw), rx = iq_scan_rx(kbx.wxr);
    // The box's region goes straight to LDS, a word a lane, all loads in
    // flight (no registers, no tests: the packed image has room past its end,
    // and what a candidate outside the grid reads does not matter).
    {
      const int n = ry * rx * kbx.wz;
      int y = (int)threadIdx.x % ry, x = (int)threadIdx.x / ry % rx, z = (int)threadIdx.x / (ry * rx);
      const int sy = NT % ry, sx = NT / ry % rx, sz = NT / (ry * rx);
      int gi = cy0 + kbx.y0 + y + t1 * (cx0 + kbx.x0 + x + t0 * (cz + kbx.z0 + z));
      const int sg = sy + t1 * (sx + t0 * sz);
      if (b) __syncthreads();  // the previous box's region is no longer read
      for (int i0 = 64 * w; i0 < n; i0 += NT) {
        if (i0 + lane < n)
          __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(tiw + gi),
                                           (__attribute__((address_space(3))) void*)(lw + i0), 4, 0, 0);
        y += sy;
        x += sx;
        gi += sg;
        if (y >= ry) { y -= ry; x++; gi += t1 - ry; }
        if (x >= rx) { x -= rx; gi += t1 * (t0 - rx); }
      }
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
    }
    if (!wlive) continue;  // every candidate row of this wavefront is past the grid
    const int lane_off = 4 * w + ry * row;
    int off[4];  // the chunk's pairs of voxels: cy / 2 a column
#pragma unroll
    for (int c = 0; c < 4; c++) off[c] = 2 * c % kbx.cy + ry * (2 * c / kbx.cy);
    // k-steps: B fragments and chunk offsets are loaded ahead, one step for
    // split data (a step's twelve MFMAs cover the load; two ahead are no
    // faster), AHEAD for the four MFMAs of bf16-exact data.  There the loads
    // past the box's end repeat its last step's: with a test the wait of the
    // loop's head is for every load in flight.  Scans of codes with the list,
    // 126 launches on average: 522 us two ahead with the test, 479 four ahead
    // without, 457 eight (with the store, one round: 93, 88, 96);
    // consecutive MFMAs use different accumulators
    constexpr int AHEAD = SPLIT ? 2 : (LIST ? 8 : 4);
    iq_u32x4 bh[AHEAD], bl[AHEAD];
    int ko[AHEAD];
    auto fetch = [&](int u, int step) {
      bh[u] = bhp[(int64_t)step * 64];
      if (SPLIT) bl[u] = blp[(int64_t)step * 64];
      ko[u] = kofs[2 * step + kb];
    };
    auto mfmas = [&](int u) {
      uint4 h[4], l[4];
      scan_frags<SPLIT>(lw, ko[u] + lane_off, off, h, l);
      const iq_bf16x8 qh = __builtin_bit_cast(iq_bf16x8, bh[u]);
#pragma unroll
      for (int i = 0; i < 4; i++)
        acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(iq_bf16x8, h[i]), qh, acc[i], 0, 0, 0);
      if (SPLIT) {
        const iq_bf16x8 ql = __builtin_bit_cast(iq_bf16x8, bl[u]);
#pragma unroll
        for (int i = 0; i < 4; i++)
          acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(iq_bf16x8, h[i]), ql, acc[i], 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; i++)
          acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(iq_bf16x8, l[i]), qh, acc[i], 0, 0, 0);
      }
    };
    const int s0 = kbx.s0, s1 = kbx.s1;
    if constexpr (SPLIT) {
      if (s0 < s1) fetch(1, s0);
      for (int step = s0; step < s1; step++) {
        bh[0] = bh[1];
        bl[0] = bl[1];
        ko[0] = ko[1];
        if (step + 1 < s1) fetch(1, step + 1);
        mfmas(0);
      }
    } else {
#pragma unroll
      for (int u = 0; u < AHEAD; u++) fetch(u, s0 + u < s1 ? s0 + u : s1 - 1);
      int step = s0;
      for (; step + AHEAD <= s1; step += AHEAD) {
#pragma unroll
        for (int u = 0; u < AHEAD; u++) {
          mfmas(u);
          fetch(u, step + AHEAD + u < s1 ? step + AHEAD + u : s1 - 1);
        }
      }
#pragma unroll
      for (int u = 0; u + 1 < AHEAD; u++)
        if (step + u < s1) mfmas(u);
    }
  }
  // epilogue: lane holds C[row'][col] for col = lane % 32 (its query)
  const int qi = tile * 32 + row;
  float lmin = __builtin_inff();
  bool live = false;
  int64_t slot = 0;
  float B = 0.0f, sB = 0.0f, k1 = 0.0f, k2 = 0.0f, tiny2 = 0.0f;
  const float* a2p = nullptr;
  if (qi < nq) {
    const IqQuery q = qs[qi];
    const IqStep& st = D->steps[q.step];
    live = !q.multi && st.mask >= 0;
    slot = q.slot;
    if (live) {
      // Interval around the oracle's FP64 distance, evaluated in FP32:
      // |AB32 - AB| <= gerr sum|a||b| and sum|a||b| <= S = sqrt(A2) sqrt(B2)
      // (square roots of operands clamped up to 2^-100, rounded up by
      // 2^-19); 8 u32 (A2 + B2 + 2S) covers the FP32 conversions and the
      // evaluation of d as well as the oracle's own FP64 rounding.  The main
      // term carries a 2^-10 margin for its own FP32 evaluation, the small
      // terms are doubled to cover the rounding of d -/+ e, and lo / hi are
      // pushed outward by 2^-20.  A2 = NaN marks a disabled window.  All of it
      // is in units of scan_s2: the operands are a power of two times the
      // image's values, so its distances are that power squared times these.
      const IqMask& m = D->masks[st.mask];
      a2p = D->a2f[m.a2];
      B = (float)(D->b2[slot * (2 + D->naux)] * D->scan_s2);
      sB = __builtin_amdgcn_sqrtf(fmaxf(B, 0x1p-100f)) * (1.0f + 0x1p-19f);
      const double V = (double)m.V;
      const double g64 = V * 0x1p-53 / (1.0 - V * 0x1p-53);
      const float gs2 = (float)((gerr + g64) * (1.0 + 0x1p-10)) * 2.0f * (1.0f + 0x1p-10f);
      const float u32 = 0x1p-24f;
      tiny2 = 2.0f * (float)(1e3 * V * 0x1p-125);
      // e = gs2 S + 2 (8 u32 ((A + B) + 2 S)) + tiny2, regrouped as
      // S (gs2 + 32 u32) + 16 u32 (A + B) + tiny2 and evaluated by two fmas:
      // fewer roundings than the plain sum, each within the margins above
      k1 = gs2 + 32.0f * u32;
      k2 = 16.0f * u32;
    }
  }
  // (integer codes: every operand and result is an integer below 2^24)
  const auto bound = [&](auto codes, float a, float ab, float& hi) {
    const float d = __builtin_fabsf(__builtin_fmaf(-2.0f, ab, a) + B);  // 2 ab is exact
    float lo = d;
    hi = d;
    if constexpr (!codes.value) {
      const float S = __builtin_amdgcn_sqrtf(fmaxf(a, 0x1p-100f)) * sB;
      const float e = __builtin_fmaf(S, k1, __builtin_fmaf(a + B, k2, tiny2));
      lo = fmaxf(d - e, 0.0f) * (1.0f - 0x1p-20f);
      hi = (d + e) * (1.0f + 0x1p-20f);
    }
    if (a != a) lo = hi = __builtin_inff();
    return lo;
  };
  const auto bounds = [&](auto codes) {
    const auto a2f = iq_glob(a2p);
    const auto lo_out = iq_globw(D->lo32 + slot * g.P);
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int cy = cy0 + 4 * w + i;
      if (cy >= d1) break;  // uniform per wavefront
      const int64_t rb = (int64_t)d0 * (cy + (int64_t)d1 * cz) + cx0 + 4 * kb;
      const int xl = d0 - cx0 - 4 * kb;  // candidates of this row left to the lane
      float A[16];
#pragma unroll
      for (int v = 0; v < 16; v++) {
        const int ox = 8 * (v >> 2) + (v & 3);
        A[v] = a2f[ox < xl ? rb + ox : rb - 4 * kb];
      }
#pragma unroll
      for (int v = 0; v < 16; v++) {
        const int ox = 8 * (v >> 2) + (v & 3);
        float hi;
        const float lo = bound(codes, A[v], acc[i][v], hi);
        if (LIST) acc[i][v] = ox < xl ? lo : __builtin_inff();
        if (ox < xl) {
          if (!LIST) lo_out[rb + ox] = lo;
          lmin = fminf(lmin, hi);
        }
      }
    }
  };
  if (live) {
    if (exact) bounds(std::true_type());
    else bounds(std::false_type());
  }
  if constexpr (!LIST) {
    lmin = fminf(lmin, __shfl_xor(lmin, 32));
    if (kb == 0) red[w][row] = lmin;
    __syncthreads();
    if (w == 0 && kb == 0 && live) {
      float m = red[0][row];
      for (int i = 1; i < nw; i++) m = fminf(m, red[i][row]);
      atomicMin(&D->gmin_hi[slot], __float_as_uint(m));
    }
    return;
  }
  lmin = fminf(lmin, __shfl_xor(lmin, 32));
  if (kb == 0) {
    red[w][row] = lmin;
    if (w == 0) sslot[row] = live ? (int)slot : -1;
  }
  __syncthreads();
  // this group's share of the queries' bitmaps is cleared for the selection
  {
    const int nwg = (int)(gridDim.x * gridDim.y) * g.dist[2];
    const int fb = (int)blockIdx.x + (int)gridDim.x * ((int)blockIdx.y + (int)gridDim.y * cz);
    const int per = (int)((D->nw64 + nwg - 1) / nwg);
    for (int i = threadIdx.x; i < 32 * per; i += NT) {
      const int64_t wd = (int64_t)fb * per + i % per;
      const int sl = sslot[i / per];
      if (sl >= 0 && wd < D->nw64) D->bitmap[sl * D->nw64 + wd] = 0ull;
    }
  }
  if (w == 0 && kb == 0) {
    float T = -1.0f;
    if (live) {
      float m = red[0][row];
      for (int i = 1; i < nw; i++) m = fminf(m, red[i][row]);
      const float U = fminf(m, __uint_as_float(atomicMin(&D->gmin_hi[slot], __float_as_uint(m))));
      T = fminf(iq_f32_up((1.0 + D->tol) * (double)U), __FLT_MAX__);
    }
    thr[row] = T;
  }
  __syncthreads();
  const float T = thr[row];
  const int rows = d1 - cy0 - 4 * w;  // uniform per wavefront
  int n = 0;
#pragma unroll
  for (int i = 0; i < 4; i++)
    if (i < rows)
#pragma unroll
      for (int v = 0; v < 16; v++) n += acc[i][v] <= T;
  if (__ballot(live && n > 0) == 0ull) return;  // uniform per wavefront
  if (!live) n = 0;
  const int other = __shfl_xor(n, 32);
  int base = 0;
  if (kb == 0 && n + other > 0) base = atomicAdd(&D->ncand[slot], n + other);
  base = __shfl(base, row) + (kb ? other : 0);
  if (n == 0) return;
  const auto lo_out = iq_globw(D->lo32 + slot * g.P);
  const auto id_out = iq_globw(D->band + slot * g.P);
#pragma unroll
  for (int i = 0; i < 4; i++) {
    if (i >= rows) break;
    const int64_t r0 = (int64_t)d0 * (cy0 + 4 * w + i + (int64_t)d1 * cz) + cx0 + 4 * kb;
#pragma unroll
    for (int v = 0; v < 16; v++)
      if (acc[i][v] <= T && base < g.P) {
        lo_out[base] = acc[i][v];
        id_out[base] = (int32_t)(r0 + 8 * (v >> 2) + (v & 3));
        base++;
      }
  }
}

template __global__ void k_scan_mfma<true, false>(const IqDev*, const IqQuery*, int, double, const int32_t*, int);
template __global__ void k_scan_mfma<true, true>(const IqDev*, const IqQuery*, int, double, const int32_t*, int);
template __global__ void k_scan_mfma<false, false>(const IqDev*, const IqQuery*, int, double, const int32_t*, int);
template __global__ void k_scan_mfma<false, true>(const IqDev*, const IqQuery*, int, double, const int32_t*, int);

// What a listing scan of the slots [0, n) starts from, as k_query_prep leaves it.
__global__ void __launch_bounds__(64) k_scan_reset(const IqDev* __restrict__ D, int n) {
  for (int i = threadIdx.x; i < n; i += 64) {
    D->gmin_hi[i] = 0x7f800000u;
    D->ncand[i] = 0;
  }
}

#define IQ_SCAN_INST(R, LX, LY, LZ) \
  template __global__ void k_scan_f32<R, LX, LY, LZ>(const IqDev*, const IqQuery*, int);
IQ_SCAN_INST(4, 8, 8, 4)
IQ_SCAN_INST(4, 16, 4, 4)
IQ_SCAN_INST(2, 16, 8, 2)
IQ_SCAN_INST(4, 8, 16, 2)

// ---------------------------------------------------------------------------
// Band superset: lo <= T where T = round_up(fl(fl(1+tol) * U)) and U is the
// least upper bound of the scan, so every exact band member is selected.
// One bitmap bit per candidate (ballot words of 64 candidates) and an
// unordered list of the members, one reservation a wavefront.  `exact`: the
// scan's values are the exact distances (integer codes), so members get theirs
// here, with the exact minimum, and no recheck follows.
// Grid: (candidate blocks, query).
// ---------------------------------------------------------------------------
#define SEL_PT 8
__global__ void __launch_bounds__(256)
k_band_select(const IqDev* __restrict__ D, const IqQuery* __restrict__ qs, int exact) {
  const IqQuery q = qs[blockIdx.y];
  const IqStep& st = D->steps[q.step];
  if (q.multi || st.mask < 0) return;
  const int64_t P = D->g.P;
  const int64_t slot = q.slot;
  const double U = (double)__uint_as_float(D->gmin_hi[slot]);
  const float Tf = iq_f32_up((1.0 + D->tol) * U);
  const auto lo = iq_glob(D->lo32 + slot * P);
  const int lane = threadIdx.x & 63;
  if (exact && blockIdx.x == 0 && threadIdx.x == 0)
    D->gmin64[slot] = (unsigned long long)__double_as_longlong(U);
  // a wavefront covers SEL_PT words of 64 consecutive candidates
  const int64_t c0 = ((int64_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * 64 * SEL_PT + lane;
  float v[SEL_PT];
#pragma unroll
  for (int j = 0; j < SEL_PT; j++) {
    const int64_t c = c0 + 64 * j;
    v[j] = lo[c < P ? c : 0];
  }
  unsigned long long bal[SEL_PT];
  int total = 0;
#pragma unroll
  for (int j = 0; j < SEL_PT; j++) {
    const int64_t c = c0 + 64 * j;
    bal[j] = __ballot(c < P && v[j] <= Tf);
    total += __popcll(bal[j]);
    if (lane == 0 && (c >> 6) < D->nw64) D->bitmap[slot * D->nw64 + (c >> 6)] = bal[j];
  }
  if (!total) return;  // uniform
  int base = 0;
  if (lane == 0) base = atomicAdd(&D->nsup[slot], total);
  base = __builtin_amdgcn_readfirstlane(base);
#pragma unroll
  for (int j = 0; j < SEL_PT; j++) {
    const int64_t c = c0 + 64 * j;
    if ((bal[j] >> lane) & 1ull) {
      D->sup[slot * P + base + __popcll(bal[j] & ((1ull << lane) - 1ull))] = (int32_t)c;
      if (exact) D->dexact[slot * P + c] = (double)v[j];
    }
    base += __popcll(bal[j]);
  }
}

// The same superset from the list of the MFMA scan, whose bitmap is cleared.
// Grid: (list blocks, query).
__global__ void __launch_bounds__(256)
k_list_select(const IqDev* __restrict__ D, const IqQuery* __restrict__ qs, int exact) {
  const IqQuery q = qs[blockIdx.y];
  const IqStep& st = D->steps[q.step];
  if (q.multi || st.mask < 0) return;
  const int64_t P = D->g.P;
  const int64_t slot = q.slot;
  const double U = (double)__uint_as_float(D->gmin_hi[slot]);
  const float Tf = iq_f32_up((1.0 + D->tol) * U);
  if (exact && blockIdx.x == 0 && threadIdx.x == 0)
    D->gmin64[slot] = (unsigned long long)__double_as_longlong(U);
  const int64_t cnt = D->ncand[slot], n = cnt < P ? cnt : P;
  const auto lo = iq_glob(D->lo32 + slot * P);
  const auto id = iq_glob(D->band + slot * P);
  const int lane = threadIdx.x & 63;
  for (int64_t i0 = (int64_t)blockIdx.x * 256 + (threadIdx.x & ~63); i0 < n; i0 += (int64_t)gridDim.x * 256) {
    const int64_t i = i0 + lane;
    const float v = i < n ? lo[i] : __builtin_inff();
    const int32_t c = i < n ? id[i] : 0;
    const bool in = i < n && v <= Tf;
    const unsigned long long bal = __ballot(in);
    if (!bal) continue;  // uniform per wavefront
    int base = 0;
    if (lane == 0) base = atomicAdd(&D->nsup[slot], __popcll(bal));
    base = __builtin_amdgcn_readfirstlane(base);
    if (in) {
      D->sup[slot * P + base + __popcll(bal & ((1ull << lane) - 1ull))] = c;
      atomicOr(&D->bitmap[slot * D->nw64 + (c >> 6)], 1ull << (c & 63));
      if (exact) D->dexact[slot * P + c] = (double)v;
    }
  }
}

// ---------------------------------------------------------------------------
// Exact recheck of the superset: the FMA chain over the masked voxels in
// ascending column-major order, so the FP64 value is the oracle's bit for
// bit.  Large supersets: one work-item per member, the query values and
// window offsets staged in LDS RC_CHUNK at a time for the whole workgroup.
// At most RC_SMALL members: one wavefront per member, window and query
// values staged by the wavefront, every lane running the same chain (short
// latency when the superset is small).  The exact minimum is reduced with an
// integer atomic on the non-negative double bits.
// Grid: (query, groups per query), 256 work-items per group.
// ---------------------------------------------------------------------------
#define RC_CHUNK 1024
#define RC_SMALL 512  // default of IqDev::rc_small
#define RC_WCH 512
#define RC_GROUPS 128  // member groups per query: 512 members in one pass, more loop
__global__ void __launch_bounds__(256)
k_band_recheck(const IqDev* __restrict__ D, const IqQuery* __restrict__ qs) {
  __shared__ double kl[RC_CHUNK];
  __shared__ int32_t ol[RC_CHUNK];
  __shared__ double wl[4 * 2 * RC_WCH];
  __shared__ unsigned long long wbest[4];
  // grid (query, member group): the groups holding members of every query
  // are dispatched first, and groups past a query's superset leave at once
  const IqQuery q = qs[blockIdx.x];
  const int grp = blockIdx.y, ngrp = gridDim.y;
  const int n = D->nsup[q.slot];
  const int rcs = D->rc_small;
  if (grp * (n <= rcs ? 4 : 256) >= n) return;
  const IqStep& st = D->steps[q.step];
  if (q.multi || st.mask < 0) return;
  const IqGeo& g = D->g;
  const int64_t slot = q.slot;
  const IqMask& m = D->masks[st.mask];
  const int V = m.V;
  const int32_t* toff = D->toff + m.off;
  const double* kv = D->kv + slot * D->kv_stride;
  const double* a2map = D->a2maps[m.a2];
  const double b2 = D->b2[slot * (2 + D->naux)];
  double* dex = D->dexact + slot * g.P;
  unsigned long long best = 0x7ff0000000000000ull;
  if (n <= rcs) {  // few members: a wavefront per member, its chain fed from LDS
    // the wavefront stages RC_WCH window and query values per chunk and loads
    // the next chunk into registers while the chain runs over the current one
    double* tl = wl + (threadIdx.x >> 6) * (2 * RC_WCH);
    double* ql = tl + RC_WCH;
    const int lane = threadIdx.x & 63;
    const auto toffg = iq_glob(toff);
    const auto kvg = iq_glob(kv);
    const bool f32 = D->ti_f32;
    const auto ti32 = iq_glob((const float*)D->ti);
    const auto ti64 = iq_glob((const double*)D->ti);
    const int d0 = g.dist[0], d1 = g.dist[1];
    for (int e = grp * 4 + (int)(threadIdx.x >> 6); e < n; e += ngrp * 4) {
      const int32_t c = D->sup[slot * g.P + e];  // candidate indices fit 31 bits
      const int cx = c % d0, cy = (c / d0) % d1, cz = c / (d0 * d1);
      const int64_t base = iq_lin3(g.ti, cx, cy, cz);
      double rt[RC_WCH / 64], rq[RC_WCH / 64];
      // all offsets of a chunk first, then all window values (two latencies)
      auto fetch = [&](int j0) {
        int32_t o[RC_WCH / 64];
#pragma unroll
        for (int i = 0; i < RC_WCH / 64; i++) {
          const int k = j0 + lane + 64 * i;
          const int kc = k < V ? k : 0;
          o[i] = toffg[kc];
          rq[i] = kvg[kc];
        }
        if (f32) {  // uniform: the training image is read in its own element type
#pragma unroll
          for (int i = 0; i < RC_WCH / 64; i++) rt[i] = (double)ti32[base + o[i]];
        } else {
#pragma unroll
          for (int i = 0; i < RC_WCH / 64; i++) rt[i] = ti64[base + o[i]];
        }
#pragma unroll
        for (int i = 0; i < RC_WCH / 64; i++) {
          const bool ok = j0 + lane + 64 * i < V;
          rt[i] = ok ? rt[i] : 0.0;
          rq[i] = ok ? rq[i] : 0.0;
        }
      };
      fetch(0);
      double ab = 0.0;
      for (int j0 = 0; j0 < V; j0 += RC_WCH) {
        const int nj = V - j0 < RC_WCH ? V - j0 : RC_WCH;
#pragma unroll
        for (int i = 0; i < RC_WCH / 64; i++) {
          tl[lane + 64 * i] = rt[i];
          ql[lane + 64 * i] = rq[i];
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        if (j0 + RC_WCH < V) fetch(j0 + RC_WCH);  // next chunk in flight during the chain
        // the ordered chain runs on lane 0 alone (the other lanes' LDS reads
        // would only repeat its values and take LDS bandwidth from other
        // wavefronts); eight LDS pairs of the next group in flight while the
        // fmas of the current group run
        if (lane == 0) {
          int k = 0;
          double t[8], u[8];
          if (nj >= 8) {
#pragma unroll
            for (int i = 0; i < 8; i++) { t[i] = tl[i]; u[i] = ql[i]; }
          }
          for (; k + 8 <= nj; k += 8) {
            double tn[8], un[8];
            const int kn = k + 16 <= nj ? k + 8 : k;
#pragma unroll
            for (int i = 0; i < 8; i++) { tn[i] = tl[kn + i]; un[i] = ql[kn + i]; }
#pragma unroll
            for (int i = 0; i < 8; i++) ab = __builtin_fma(t[i], u[i], ab);
#pragma unroll
            for (int i = 0; i < 8; i++) { t[i] = tn[i]; u[i] = un[i]; }
          }
          for (; k < nj; k++) ab = __builtin_fma(tl[k], ql[k], ab);
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      }
      if (lane == 0) {
        const double d = __builtin_fabs((a2map[c] - 2.0 * ab) + b2);
        dex[c] = d;
        const unsigned long long bits = (unsigned long long)__double_as_longlong(d);
        best = bits < best ? bits : best;
      }
    }
  }
  for (int e0 = grp * 256; n > rcs && e0 < n; e0 += ngrp * 256) {  // uniform over the group
    const int e = e0 + (int)threadIdx.x;
    const bool live = e < n;
    int64_t c = 0, base = 0;
    if (live) {
      c = D->sup[slot * g.P + e];
      const int cx = (int)(c % g.dist[0]), cy = (int)((c / g.dist[0]) % g.dist[1]);
      const int cz = (int)(c / ((int64_t)g.dist[0] * g.dist[1]));
      base = iq_lin3(g.ti, cx, cy, cz);
    }
    double ab = 0.0;
    for (int j0 = 0; j0 < V; j0 += RC_CHUNK) {
      const int nj = V - j0 < RC_CHUNK ? V - j0 : RC_CHUNK;
      __syncthreads();
      for (int k = threadIdx.x; k < nj; k += 256) {
        kl[k] = kv[j0 + k];
        ol[k] = toff[j0 + k];
      }
      __syncthreads();
      if (live) {  // 16 window loads in flight, then the ordered fmas
        int k = 0;
        if (D->ti_f32) {
          const float* ti = (const float*)D->ti + base;
          for (; k + 16 <= nj; k += 16) {
            float t[16];
#pragma unroll
            for (int i = 0; i < 16; i++) t[i] = ti[ol[k + i]];
#pragma unroll
            for (int i = 0; i < 16; i++) ab = __builtin_fma((double)t[i], kl[k + i], ab);
          }
          for (; k < nj; k++) ab = __builtin_fma((double)ti[ol[k]], kl[k], ab);
        } else {
          const double* ti = (const double*)D->ti + base;
          for (; k + 16 <= nj; k += 16) {
            double t[16];
#pragma unroll
            for (int i = 0; i < 16; i++) t[i] = ti[ol[k + i]];
#pragma unroll
            for (int i = 0; i < 16; i++) ab = __builtin_fma(t[i], kl[k + i], ab);
          }
          for (; k < nj; k++) ab = __builtin_fma(ti[ol[k]], kl[k], ab);
        }
      }
    }
    if (live) {
      const double d = __builtin_fabs((a2map[c] - 2.0 * ab) + b2);
      dex[c] = d;
      const unsigned long long bits = (unsigned long long)__double_as_longlong(d);
      best = bits < best ? bits : best;
    }
  }
  for (int o = 32; o > 0; o >>= 1) {
    const unsigned long long other = __shfl_xor(best, o);
    best = other < best ? other : best;
  }
  if ((threadIdx.x & 63) == 0) wbest[threadIdx.x >> 6] = best;
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long b = wbest[0];
    for (int i = 1; i < 4; i++) b = wbest[i] < b ? wbest[i] : b;
    if (b != 0x7ff0000000000000ull) atomicMin(&D->gmin64[slot], b);
  }
}

// Exact recheck with a lane per member: the same ordered FMA chain (so the
// same FP64 value), each member's chain run by one lane.  A wavefront serves
// RCL_MPW members; for every block of 64 masked voxels it loads the members'
// window values one member at a time (lane l: voxel l of that window, so
// each load is a few contiguous runs of the window), transposes them through
// LDS with the block's 64 query values (lane l loads value l), and lanes
// 0..RCL_MPW-1 then chain over their member's row, reading the query values
// from LDS (one address for all lanes).  The next block's loads are issued
// before the current block's chains run.  (Query values read by scalar
// loads inside the chain: 280 us per launch at the 2.9M-candidate workload;
// the scalar cache does not hold a query's 38 KB, and every 16 chain steps
// waited on a scalar load.)  Few members per wavefront keep
// one round of loads per block and many wavefronts per query.
// Grid: (query, RCL_GROUPS wavefronts or more), members beyond loop.
#define RCL_GROUPS 32
#define RCL_WIDE 8192  // most wavefronts of a launch over a rounded image
#define RCL_MPW 16
template <typename E>
__device__ __forceinline__ double rcl_chain(const IqDev* __restrict__ D, int64_t base, const int32_t* __restrict__ toff,
                                            const double* kvp, int V, E (*tile)[65], double* kt) {
  const int lane = threadIdx.x;
  const auto ti = iq_glob((const E*)D->ti);
  const auto kv = iq_glob(kvp);
  int64_t bj[RCL_MPW];
#pragma unroll
  for (int u = 0; u < RCL_MPW; u++)
    bj[u] = (int64_t)(uint32_t)__builtin_amdgcn_readlane((int)base, u) |
            ((int64_t)__builtin_amdgcn_readlane((int)(base >> 32), u) << 32);
  E t[RCL_MPW];
  double kq;
  {
    const int i = lane < V ? lane : 0;
    const int32_t o = toff[i];
#pragma unroll
    for (int u = 0; u < RCL_MPW; u++) t[u] = ti[bj[u] + o];
    kq = kv[i];
  }
  double ab = 0.0;
  for (int v0 = 0; v0 < V; v0 += 64) {
    const int nv = V - v0 < 64 ? V - v0 : 64;
#pragma unroll
    for (int u = 0; u < RCL_MPW; u++) tile[u][lane] = t[u];
    kt[lane] = kq;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const int v1 = v0 + 64;
    if (v1 < V) {  // the next block's window and query values, in flight during the chains
      const int i = v1 + (v1 + lane < V ? lane : 0);
      const int32_t o = toff[i];
#pragma unroll
      for (int u = 0; u < RCL_MPW; u++) t[u] = ti[bj[u] + o];
      kq = kv[i];
    }
    if (lane < RCL_MPW) {
      const E* row = tile[lane];
      if (nv == 64) {
#pragma unroll 16
        for (int i = 0; i < 64; i++) ab = __builtin_fma((double)row[i], kt[i], ab);
      } else {
        for (int i = 0; i < nv; i++) ab = __builtin_fma((double)row[i], kt[i], ab);
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
  return ab;
}

__global__ void __launch_bounds__(64)
k_band_recheck_lanes(const IqDev* __restrict__ D, const IqQuery* __restrict__ qs) {
  __shared__ double tile_mem[RCL_MPW * 65];  // the transposed block (doubles, or floats in its first half)
  __shared__ double kt[64];                  // the block's query values
  const IqQuery q = qs[blockIdx.x];
  const int n = D->nsup[q.slot];
  if ((int)blockIdx.y * RCL_MPW >= n) return;
  const IqStep& st = D->steps[q.step];
  if (q.multi || st.mask < 0) return;
  const IqGeo& g = D->g;
  const int64_t slot = q.slot;
  const IqMask& m = D->masks[st.mask];
  const int V = m.V;
  const int32_t* toff = D->toff + m.off;
  const double* kvp = D->kv + slot * D->kv_stride;
  const double* a2map = D->a2maps[m.a2];
  const double b2 = D->b2[slot * (2 + D->naux)];
  double* dex = D->dexact + slot * g.P;
  const int lane = threadIdx.x;
  unsigned long long best = 0x7ff0000000000000ull;
  for (int e0 = blockIdx.y * RCL_MPW; e0 < n; e0 += gridDim.y * RCL_MPW) {  // uniform over the wavefront
    const int e = e0 + lane;
    const bool live = lane < RCL_MPW && e < n;
    int64_t c = 0, base = 0;
    if (live) {
      c = D->sup[slot * g.P + e];
      const int cx = (int)(c % g.dist[0]), cy = (int)((c / g.dist[0]) % g.dist[1]);
      const int cz = (int)(c / ((int64_t)g.dist[0] * g.dist[1]));
      base = iq_lin3(g.ti, cx, cy, cz);
    }
    const double ab = D->ti_f32 ? rcl_chain<float>(D, base, toff, kvp, V, (float(*)[65])tile_mem, kt)
                                : rcl_chain<double>(D, base, toff, kvp, V, (double(*)[65])tile_mem, kt);
    if (live) {
      const double d = __builtin_fabs((a2map[c] - 2.0 * ab) + b2);
      dex[c] = d;
      const unsigned long long bits = (unsigned long long)__double_as_longlong(d);
      best = bits < best ? bits : best;
    }
  }
  for (int o = 32; o > 0; o >>= 1) {
    const unsigned long long other = __shfl_xor(best, o);
    best = other < best ? other : best;
  }
  if (lane == 0 && best != 0x7ff0000000000000ull) atomicMin(&D->gmin64[slot], best);
}

// ---------------------------------------------------------------------------
// Exact maps of the hard-data source (relaxation): one work-item per
// candidate, grid (candidate blocks, query).  Every tile has its own list of
// hard voxels, and A2 is chained along with AB.  The map depends on the step
// alone, so the batch's first query of a step makes it for all realizations.
// Disabled candidates are +inf (iqsim.jl:207,217,226).  This form gathers the
// windows from the image: a tile usually holds a handful of points, for which
// staging its windows' region (k_hard_maps_tiled) costs more than it saves.
// ---------------------------------------------------------------------------
// A tile takes the tiled form from this many hard points for every voxel that
// form stages per candidate.  Gathered and tiled, us a launch by points of a
// tile: 225 x 225 candidates, tile 32 x 32 (5.8 voxels): 8: 10, 14; 24: 15, 14;
// 32: 19, 15; 128: 55, 22; 71 x 71 x 36 candidates, tile 20 x 20 x 5 (17.4): 8: 21, 110;
// 48: 70, 120; 96: 132, 133; 128: 172, 142.
#define HARD_TILED 5
__global__ void __launch_bounds__(256)
k_hard_maps(const IqDev* __restrict__ D, const IqQuery* __restrict__ qs) {
  const IqQuery q = qs[blockIdx.y];
  const IqStep& st = D->steps[q.step];
  if (!q.multi || q.rep != q.slot || !st.hard || st.hcnt >= D->hard_min) return;
  const IqGeo& g = D->g;
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= g.P) return;
  const int64_t slot = q.slot;
  double* out = D->maps + (slot * D->nmap + 1) * g.P;
  if (D->disabled[c]) { out[c] = __builtin_inf(); return; }
  const int V = st.hcnt;
  const int32_t* toff = D->htoff + st.hoff;
  const double* kv = D->kv + slot * D->kv_stride + (int64_t)g.tilevox;
  const double b2 = D->b2[slot * (2 + D->naux) + 1];
  int cx = (int)(c % g.dist[0]), cy = (int)((c / g.dist[0]) % g.dist[1]);
  int cz = (int)(c / ((int64_t)g.dist[0] * g.dist[1]));
  const int64_t base = iq_lin3(g.ti, cx, cy, cz);
  double a2 = 0.0, ab = 0.0;
  if (D->ti_f32) {
    const float* ti = (const float*)D->ti;
    for (int j = 0; j < V; j++) {
      double t = (double)ti[base + toff[j]];
      a2 = __builtin_fma(t, t, a2);
      ab = __builtin_fma(t, kv[j], ab);
    }
  } else {
    const double* ti = (const double*)D->ti;
    for (int j = 0; j < V; j++) {
      double t = ti[base + toff[j]];
      a2 = __builtin_fma(t, t, a2);
      ab = __builtin_fma(t, kv[j], ab);
    }
  }
  out[c] = __builtin_fabs((a2 - 2.0 * ab) + b2);
}

// Tiled form for tiles with many hard points: a workgroup of MX x MY
// work-items owns MX x MY candidates at one z (32 x 16 where the region fits,
// else 16 x 16: rows of 32 consecutive candidates keep a half-wavefront's
// 8-byte reads on distinct LDS banks, and 512-wide groups hold more wavefronts
// per compute unit); the training-image region their windows cover is staged
// in LDS as FP64.  The query values and the voxels' region offsets (prepared
// per plan) are the same for every work-item and come through scalar loads.
// Grid: (x blocks * y blocks * dist z, query); LDS = the region (the host
// checks it fits).
template <int MT_X, int MT_Y>
__global__ void __launch_bounds__(MT_X * MT_Y)
k_hard_maps_tiled(const IqDev* __restrict__ D, const IqQuery* __restrict__ qs) {
  extern __shared__ double mreg[];
  const IqQuery q = qs[blockIdx.y];
  const IqStep& st = D->steps[q.step];
  if (!q.multi || q.rep != q.slot || !st.hard || st.hcnt < D->hard_min) return;
  const IqGeo& g = D->g;
  const int nbx = (g.dist[0] + MT_X - 1) / MT_X, nby = (g.dist[1] + MT_Y - 1) / MT_Y;
  const int bx = blockIdx.x % nbx, by = (blockIdx.x / nbx) % nby, cz = blockIdx.x / (nbx * nby);
  const int64_t slot = q.slot;
  double* out = D->maps + (slot * D->nmap + 1) * g.P;
  const int V = st.hcnt;
  const int RX = MT_X + g.tile[0] - 1, RY = MT_Y + g.tile[1] - 1, RZ = g.tile[2];
  const int nreg = RX * RY * RZ;
  double* reg = mreg;
  const int gx0 = bx * MT_X, gy0 = by * MT_Y;
  for (int i = threadIdx.x; i < nreg; i += blockDim.x) {
    const int x = i % RX, y = (i / RX) % RY, z = i / (RX * RY);
    const int gx = gx0 + x, gy = gy0 + y, gz = cz + z;
    double v = 0.0;
    if (gx < g.ti[0] && gy < g.ti[1]) {
      const int64_t o = iq_lin3(g.ti, gx, gy, gz);
      v = D->ti_f32 ? (double)((const float*)D->ti)[o] : ((const double*)D->ti)[o];
    }
    reg[i] = v;
  }
  // query values and region offsets are the same for every work-item:
  // constant-address loads (scalar unit, no LDS traffic)
  const auto kq = iq_const(D->kv + slot * D->kv_stride + (int64_t)g.tilevox);
  const auto ro = iq_const(D->rhtvox + st.hoff);
  __syncthreads();
  const int lx = threadIdx.x % MT_X, ly = threadIdx.x / MT_X;
  const int cx = gx0 + lx, cy = gy0 + ly;
  if (cx >= g.dist[0] || cy >= g.dist[1]) return;
  const int64_t c = iq_lin3(g.dist, cx, cy, cz);
  if (D->disabled[c]) { out[c] = __builtin_inf(); return; }
  const double b2 = D->b2[slot * (2 + D->naux) + 1];
  const double* r0 = reg + lx + RX * ly;
  double a2 = 0.0, ab = 0.0;
  int j = 0;
  for (; j + 8 <= V; j += 8) {
    double t[8], u[8];
#pragma unroll
    for (int i = 0; i < 8; i++) { t[i] = r0[ro[j + i]]; u[i] = kq[j + i]; }
#pragma unroll
    for (int i = 0; i < 8; i++) { a2 = __builtin_fma(t[i], t[i], a2); ab = __builtin_fma(t[i], u[i], ab); }
  }
  for (; j < V; j++) { const double t = r0[ro[j]]; a2 = __builtin_fma(t, t, a2); ab = __builtin_fma(t, kq[j], ab); }
  out[c] = __builtin_fabs((a2 - 2.0 * ab) + b2);
}

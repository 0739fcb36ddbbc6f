// k_maps.hip -- exact FP64 distance maps of many queries on the matrix cores
// (fastdistance, utils.jl:5-13, for every candidate: the maps the relaxation
// works on, and the overlap maps of images the FP32 scans do not take).
//
// D[c] = |(A2[c] - 2 AB[c]) + B2| with AB an FP64 fused-multiply-add chain
// over the listed tile voxels in ascending column-major order.
// v_mfma_f64_4x4x4_4b evaluates exactly that chain: each output is
// fma(a3, b3, fma(a2, b2, fma(a1, b1, fma(a0, b0, c)))), rounded at every
// step (checked against the scalar chain on 10^6 outputs, with cancellation,
// subnormals, infinities and NaN), so a loop of them over the voxels, four at
// a time, is the chain bit for bit.  One query a work-item on the vector units
// reads one 8-byte LDS word per fma and stops at the LDS rate (15 TFLOP/s
// measured); here a word feeds four to sixteen queries.  Of the two FP64
// shapes the 16x16x4 one runs at 47 TFLOP/s on this chip and the 4x4x4 one,
// four blocks side by side, at 75.
#include "iq_internal.h"

#define MM_BX 32            // candidates of a group along x
#define MM_BY 16            // and along y
#define MM_Q 16             // queries of a tile (four groups of four)
#define MM_STEP 16          // voxels of a step (four MFMAs deep)
#define MM_LDS (80 * 1024)  // staged region: two groups of 512 work-items a compute unit

typedef double iq_f64x2 __attribute__((ext_vector_type(2)));

// Query values of the tiles in fragment order: entry
// ((((tile * stride + step) * 2 + h) * 4 + g) * 16 + k * 4 + i) * 2 + e holds
// query 4 g + i at voxel 16 step + 4 (2 h + e) + k of the list (zero past the
// list and past the tile's queries).  Grid: (steps, tiles).
__global__ void __launch_bounds__(256)
k_maps_pack(const IqDev* __restrict__ D, const IqQuery* __restrict__ qs, const IqMapTile* __restrict__ tiles,
            double* __restrict__ pack, int stride) {
  const IqMapTile& T = tiles[blockIdx.y];
  if (T.list < 0) return;
  const IqMapList L = D->mlists[T.list];
  const int step = blockIdx.x;
  if (step >= L.ns) return;
  const int t = threadIdx.x;
  const int e = t & 1, i = (t >> 1) & 3, k = (t >> 3) & 3, g = (t >> 5) & 3, h = t >> 7;
  const int qi = 4 * g + i;
  const int j = D->mvox[(int64_t)(L.s0 + step) * MM_STEP + 4 * (2 * h + e) + k];
  double v = 0.0;
  if (qi < T.n && j >= 0) {
    const int64_t slot = qs[T.q[qi]].slot;
    v = D->kv[slot * D->kv_stride + (int64_t)(T.src < 0 ? 0 : T.src) * D->g.tilevox + j];
  }
  pack[((int64_t)blockIdx.y * stride + step) * 256 + t] = v;
}

// The chains of one wavefront over steps [s0, s1): four blocks of sixteen
// candidates (lane % 16 each; base[t] is the lane's first window voxel in the
// staged region), NQ groups of four queries.  An MFMA takes the candidates as
// B (candidate lane % 16, voxel lane / 16) and the queries as A (query
// lane % 4, voxel lane / 16, the same for the four blocks) and leaves
// (candidate lane % 16, query lane / 16).  The last step of a list's chunk may
// hold pad voxels (offset -1): their window values are replaced by zero, which
// leaves a chain as it is whatever the image holds.
template <int NQ>
__device__ __forceinline__ void map_chains(const double* reg, const int (&base)[4], const int4* ofs_, const iq_f64x2* pk_,
                                           int s0, int s1, double (&acc)[NQ][4]) {
  const auto ofs = iq_glob((const iq_u32x4*)ofs_);
  const auto pk = iq_glob(pk_);
  iq_u32x4 o = ofs[s0 * 4];
  iq_f64x2 a[2][NQ];
#pragma unroll
  for (int h = 0; h < 2; h++)
#pragma unroll
    for (int g = 0; g < NQ; g++) a[h][g] = pk[((int64_t)s0 * 2 + h) * 64 + g * 16];
  for (int s = s0; s < s1; s++) {
    const int sn = s + 1 < s1 ? s + 1 : s;
    const iq_u32x4 on = ofs[sn * 4];
    const bool last = s + 1 == s1;
#pragma unroll
    for (int h = 0; h < 2; h++) {
#pragma unroll
      for (int e = 0; e < 2; e++) {
        const int oo = (int)o[2 * h + e];
        double b[4];
#pragma unroll
        for (int t = 0; t < 4; t++) b[t] = reg[base[t] + (last ? (oo < 0 ? 0 : oo) : oo)];
        if (last) {
#pragma unroll
          for (int t = 0; t < 4; t++) b[t] = oo < 0 ? 0.0 : b[t];
        }
#pragma unroll
        for (int g = 0; g < NQ; g++)
#pragma unroll
          for (int t = 0; t < 4; t++) acc[g][t] = __builtin_amdgcn_mfma_f64_4x4x4f64(a[h][g][e], b[t], acc[g][t], 0, 0, 0);
      }
      // this half's query values of the next step, in flight during the other half
#pragma unroll
      for (int g = 0; g < NQ; g++) a[h][g] = pk[((int64_t)sn * 2 + h) * 64 + g * 16];
    }
    o = on;
  }
}

template <int NQ>
__device__ __forceinline__ void map_tile(const IqDev* __restrict__ D, const IqQuery* __restrict__ qs, const IqMapTile& T,
                                         const double* pack, int stride, double* reg) {
  const IqGeo& g = D->g;
  const int nbx = (g.dist[0] + MM_BX - 1) / MM_BX, nby = (g.dist[1] + MM_BY - 1) / MM_BY;
  const int bx = blockIdx.x % nbx, by = (blockIdx.x / nbx) % nby, cz = blockIdx.x / (nbx * nby);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int c = lane & 15, k = lane >> 4;
  const int gx0 = bx * MM_BX, gy0 = by * MM_BY;
  const int RX = D->map_rx;
  const bool wlive = gy0 + 2 * w < g.dist[1];  // uniform per wavefront
  double acc[NQ][4];
#pragma unroll
  for (int i = 0; i < NQ; i++)
#pragma unroll
    for (int t = 0; t < 4; t++) acc[i][t] = 0.0;
  int base[4];
#pragma unroll
  for (int t = 0; t < 4; t++) base[t] = 16 * (t & 1) + c + RX * (2 * w + (t >> 1));
  const IqMask* mask = nullptr;
  const double* img64 = nullptr;
  const double* a2map = nullptr;
  if (T.src >= 2) {
    img64 = D->auxti[T.src - 2];
    a2map = D->a2soft[T.src - 2];
  } else if (T.list >= 0) {
    mask = &D->masks[T.list];
    a2map = D->a2maps[mask->a2];
    if (!D->ti_f32) img64 = (const double*)D->ti;
  }
  if (T.list >= 0) {
    const IqMapList L = D->mlists[T.list];
    const int4* ofs = D->mofs + (int64_t)L.s0 * 4 + k;
    const iq_f64x2* pk = (const iq_f64x2*)pack + (int64_t)blockIdx.y * stride * 128 + k * 4 + (lane & 3);
    const auto f32 = iq_glob((const float*)D->ti);
    const auto f64 = iq_glob(img64);
    for (int ch = 0; ch < L.nc; ch++) {
      const IqMapChunk C = D->mchunks[L.c0 + ch];
      const int RY = MM_BY + C.ny - 1;
      const int n = RX * RY * C.nz;
      if (ch) __syncthreads();  // the previous chunk's region is no longer read
      for (int i0 = threadIdx.x; i0 < n; i0 += 4 * 512) {  // four loads in flight
        double v[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
          const int i = i0 + 512 * u;
          const int x = i % RX, y = (i / RX) % RY, z = i / (RX * RY);
          const int gx = gx0 + C.x0 + x, gy = gy0 + C.y0 + y, gz = cz + C.z0 + z;
          const bool in = i < n && gx < g.ti[0] && gy < g.ti[1];
          const int64_t o = in ? iq_lin3(g.ti, gx, gy, gz) : 0;
          v[u] = img64 ? f64[o] : (double)f32[o];
          if (!in) v[u] = 0.0;
        }
#pragma unroll
        for (int u = 0; u < 4; u++)
          if (i0 + 512 * u < n) reg[i0 + 512 * u] = v[u];
      }
      __syncthreads();
      if (wlive) map_chains<NQ>(reg, base, ofs, pk, C.s0, C.s1, acc);
    }
  }
  if (!wlive) return;
#pragma unroll
  for (int t = 0; t < 4; t++) {
    const int cx = gx0 + 16 * (t & 1) + c, cy = gy0 + 2 * w + (t >> 1);
    if (cx >= g.dist[0] || cy >= g.dist[1]) continue;
    const int64_t ci = iq_lin3(g.dist, cx, cy, cz);
    const bool dis = D->disabled[ci] != 0;
    const double a2 = a2map ? a2map[ci] : 0.0;
#pragma unroll
    for (int i = 0; i < NQ; i++) {
      const int qi = 4 * i + k;
      if (qi >= T.n) continue;
      const int64_t slot = qs[T.q[qi]].slot;
      const double b2 = D->b2[slot * (2 + D->naux) + (T.src < 0 ? 0 : T.src)];
      double* out = T.src < 0 ? D->dexact + slot * g.P : D->maps + (slot * D->nmap + T.src) * g.P;
      out[ci] = dis ? __builtin_inf() : __builtin_fabs((a2 - 2.0 * acc[i][t]) + b2);
    }
  }
}

// Maps of the tiles: up to sixteen queries that share a voxel list (an overlap
// mask, or the whole tile for a soft pair) and the image it is read from.  A
// group of eight wavefronts owns 32 x 16 candidates at one z; the region their
// windows cover is staged in LDS as FP64, whole where it fits MM_LDS, else in
// chunks of planes or rows in the list's order.  Grid: (x blocks * y blocks *
// dist z, tiles).
// Measured (512x512 image, tile 48x48, 216,225 candidates, soft and hard data,
// four realizations): 1,322 us a wave, 43 TFLOP/s of the distinct maps' work;
// a map per query and source on the vector units, soft maps repeated for every
// realization, took 7,962 us.
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(4)))
k_maps_mfma(const IqDev* __restrict__ D, const IqQuery* __restrict__ qs, const IqMapTile* __restrict__ tiles,
            const double* __restrict__ pack, int stride) {
  extern __shared__ double mm_reg[];
  const IqMapTile& T = tiles[blockIdx.y];
  switch ((T.n + 3) / 4) {  // uniform
    case 1: map_tile<1>(D, qs, T, pack, stride, mm_reg); break;
    case 2: map_tile<2>(D, qs, T, pack, stride, mm_reg); break;
    case 3: map_tile<3>(D, qs, T, pack, stride, mm_reg); break;
    default: map_tile<4>(D, qs, T, pack, stride, mm_reg); break;
  }
}

// The chain of one candidate over V listed voxels: offsets and query values
// come through LDS, MG_DEEP window values are in flight at once.  `img` is the
// image at the candidate's first voxel.
#define MG_DEEP 64
#define MG_CHUNK 1024
template <typename T>
__device__ __forceinline__ double gather_chain(const T* img_, const int32_t* toff, const double* kv, int V, int32_t* ol, double* kl) {
  const auto img = iq_glob(img_);
  double ab = 0.0;
  for (int j0 = 0; j0 < V; j0 += MG_CHUNK) {
    const int n = V - j0 < MG_CHUNK ? V - j0 : MG_CHUNK;
    if (j0) __syncthreads();  // the previous chunk is no longer read
    for (int k = threadIdx.x; k < (n + MG_DEEP - 1) / MG_DEEP * MG_DEEP; k += (int)blockDim.x) {
      ol[k] = k < n ? toff[j0 + k] : 0;
      kl[k] = k < n ? kv[j0 + k] : 0.0;
    }
    __syncthreads();
    for (int k0 = 0; k0 < n; k0 += MG_DEEP) {
      T t[MG_DEEP];
#pragma unroll
      for (int i = 0; i < MG_DEEP; i++) t[i] = img[ol[k0 + i]];
      if (k0 + MG_DEEP <= n) {
#pragma unroll
        for (int i = 0; i < MG_DEEP; i++) ab = __builtin_fma((double)t[i], kl[k0 + i], ab);
      } else {  // past the list: zero times zero, whatever the image holds
#pragma unroll
        for (int i = 0; i < MG_DEEP; i++) ab = __builtin_fma(k0 + i < n ? (double)t[i] : 0.0, kl[k0 + i], ab);
      }
    }
  }
  return ab;
}

// The same maps, of little work: a work-item per candidate gathers its window
// from the image, a query at a time, in one launch.  What bounds it is the
// latency of the loads of the few wavefronts there are, so groups are of one,
// over as many compute units as they reach (4,232 candidates, 192 voxels: 13.8
// us in groups of four, 10.2 of one; k_maps_pack and k_maps_mfma 15.6).  Grid:
// (candidate blocks, tiles, queries of a tile).
__global__ void __launch_bounds__(64)
k_maps_gather(const IqDev* __restrict__ D, const IqQuery* __restrict__ qs, const IqMapTile* __restrict__ tiles) {
  __shared__ int32_t ol[MG_CHUNK];
  __shared__ double kl[MG_CHUNK];
  const IqMapTile& T = tiles[blockIdx.y];
  if ((int)blockIdx.z >= T.n) return;
  const IqGeo& g = D->g;
  const int64_t slot = qs[T.q[blockIdx.z]].slot;
  const int src = T.src < 0 ? 0 : T.src;
  const int64_t c0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t c = c0 < g.P ? c0 : g.P - 1;
  const int cx = (int)(c % g.dist[0]), cy = (int)((c / g.dist[0]) % g.dist[1]);
  const int cz = (int)(c / ((int64_t)g.dist[0] * g.dist[1]));
  const int64_t at = iq_lin3(g.ti, cx, cy, cz);
  const double* kv = D->kv + slot * D->kv_stride + (int64_t)src * g.tilevox;
  double a2 = 0.0, ab = 0.0;
  if (T.src >= 2) {
    a2 = D->a2soft[T.src - 2][c];
    ab = gather_chain(D->auxti[T.src - 2] + at, D->toff + D->full_off, kv, g.tilevox, ol, kl);
  } else if (T.list >= 0) {
    const IqMask& m = D->masks[T.list];
    a2 = D->a2maps[m.a2][c];
    if (D->ti_f32) ab = gather_chain((const float*)D->ti + at, D->toff + m.off, kv, m.V, ol, kl);
    else ab = gather_chain((const double*)D->ti + at, D->toff + m.off, kv, m.V, ol, kl);
  }
  if (c0 >= g.P) return;
  const double b2 = D->b2[slot * (2 + D->naux) + src];
  double* out = T.src < 0 ? D->dexact + slot * g.P : D->maps + (slot * D->nmap + src) * g.P;
  out[c] = D->disabled[c] ? __builtin_inf() : __builtin_fabs((a2 - 2.0 * ab) + b2);
}

// Plain queries whose training image the FP32 scans do not take (values out
// of range, or Float64 values dominated by a common offset): their overlap
// maps are exact for every candidate (k_maps_mfma), all enabled candidates
// form the superset.  Grid: (candidate blocks, query).
__global__ void __launch_bounds__(256)
k_band_all(const IqDev* __restrict__ D, const IqQuery* __restrict__ qs) {
  const IqQuery q = qs[blockIdx.y];
  const IqStep& st = D->steps[q.step];
  if (q.multi || st.mask < 0) return;
  const IqGeo& g = D->g;
  const int64_t slot = q.slot;
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const bool in = c < g.P && !D->disabled[c];
  const unsigned long long bal = __ballot(in);
  if ((threadIdx.x & 63) == 0 && (c >> 6) < D->nw64) D->bitmap[slot * D->nw64 + (c >> 6)] = bal;
  unsigned long long bits = in ? (unsigned long long)__double_as_longlong(D->dexact[slot * g.P + c]) : 0x7ff0000000000000ull;
  for (int o = 32; o > 0; o >>= 1) {
    unsigned long long other = __shfl_xor(bits, o);
    bits = other < bits ? other : bits;
  }
  if ((threadIdx.x & 63) == 0 && bal) atomicMin(&D->gmin64[slot], bits);
}

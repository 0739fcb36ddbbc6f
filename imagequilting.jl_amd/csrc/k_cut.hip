// k_cut.hip -- boundary cut (graphcut.jl:5-84) and paste (iqsim.jl:252-281).
//
// One workgroup per overlap slab.  The first slice along the cut
// axis is tied to the source and the last to the sink with infinite capacity
// (graphcut.jl:56-70), so both are contracted into the terminals and a
// preflow push-relabel runs on the interior slices, its state in registers and
// LDS (global scratch beyond CUT_REG_MAX interior nodes).  The schedule is
// synchronous: a relabel phase, a push phase (only the higher endpoint of an
// edge can push on it, so every residual pair has one writer) and a gather
// phase that adds incoming flow in a fixed neighbour order; a global relabel
// (exact residual BFS distance to the sink) runs every iq_gr_freq(n) rounds
// (8, or 24 above 1,024 interior nodes) and decides termination.  The result is deterministic and matches the oracle's
// restatement bit for bit.  Cut mask = voxels that cannot reach the sink in
// the residual graph (graphcut.jl:79-81).
#include "iq_internal.h"

template <typename T>
__device__ inline double cut_cap(const T* A, const T* B, int64_t u, int64_t v, int64_t w, bool wok);

template <>
__device__ inline double cut_cap<float>(const float* A, const float* B, int64_t u, int64_t v, int64_t w, bool wok) {
  float Au = A[u], Av = A[v], Bu = B[u], Bv = B[v];
  float Du = __builtin_fabsf(Au - Bu), Dv = __builtin_fabsf(Av - Bv);
  float gAu = __builtin_fabsf(Av - Au), gBu = __builtin_fabsf(Bv - Bu);
  float gAv = wok ? __builtin_fabsf(A[w] - Av) : gAu;
  float gBv = wok ? __builtin_fabsf(B[w] - Bv) : gBu;
  float num = Du + Dv;
  float g = ((gAu + gAv) + gBu) + gBv;
  return (double)num / ((double)g + 0x1p-52);
}

template <>
__device__ inline double cut_cap<double>(const double* A, const double* B, int64_t u, int64_t v, int64_t w, bool wok) {
  double Du = __builtin_fabs(A[u] - B[u]), Dv = __builtin_fabs(A[v] - B[v]);
  double gAu = __builtin_fabs(A[v] - A[u]), gBu = __builtin_fabs(B[v] - B[u]);
  double gAv = wok ? __builtin_fabs(A[w] - A[v]) : gAu;
  double gBv = wok ? __builtin_fabs(B[w] - B[v]) : gBu;
  return (Du + Dv) / ((((gAu + gAv) + gBu) + gBv) + 0x1p-52);
}

// Slab view: element (x,y,z) of the slab lives at base + x*sx + y*sy + z*sz.
template <typename T>
struct SlabView {
  const T* base;
  int64_t st[3];
  __device__ int64_t at(int x, int y, int z) const { return x * st[0] + y * st[1] + z * st[2]; }
};

template <typename T>
__device__ double slab_cap(const SlabView<T>& A, const SlabView<T>& B, const int s[3], int c0, int c1, int c2, int d) {
  int c[3] = {c0, c1, c2};
  int cv[3] = {c0, c1, c2};
  cv[d] += 1;
  int cw[3] = {c0, c1, c2};
  cw[d] += 2;
  bool wok = cw[d] < s[d];
  int64_t u = A.at(c[0], c[1], c[2]), v = A.at(cv[0], cv[1], cv[2]);
  int64_t w = wok ? A.at(cw[0], cw[1], cw[2]) : 0;
  // A and B share strides only when both live in the same array; use per-view offsets
  int64_t ub = B.at(c[0], c[1], c[2]), vb = B.at(cv[0], cv[1], cv[2]);
  int64_t wb = wok ? B.at(cw[0], cw[1], cw[2]) : 0;
  // evaluate with the element order of graphcut.jl:37-52
  T Au = A.base[u], Av = A.base[v], Bu = B.base[ub], Bv = B.base[vb];
  T Aw = wok ? A.base[w] : (T)0, Bw = wok ? B.base[wb] : (T)0;
  T a3[3] = {Au, Av, Aw}, b3[3] = {Bu, Bv, Bw};
  return cut_cap<T>(a3, b3, 0, 1, 2, wok);
}

struct CutState {
  double *e, *rt, *rf, *rb, *pr;
  int32_t *h, *hn, *fl;
};

__device__ inline void cut_bind(CutState& S, char* mem, int n) {
  S.e = (double*)mem;
  S.rt = S.e + n;
  S.rf = S.rt + n;
  S.rb = S.rf + 3 * n;
  S.pr = S.rb + 3 * n;
  S.h = (int32_t*)(S.pr + 3 * n);
  S.hn = S.h + n;
  S.fl = S.hn + n;
}

// bytes of state per interior node
#define CUT_NODE_BYTES (8 * 11 + 4 * 3)

// Minimum cut of one slab (graphcut.jl:5-84) by the whole workgroup: writes
// keep = mask XOR side for every slab voxel into out (slab column-major).
// A and B are strided views (the simulation grid and the chosen training-image
// window); S points at global scratch sized for the interior nodes.
template <typename T>
__device__ void cut_slab(const SlabView<T>& A, const SlabView<T>& B, const int s[3], int dim, uint8_t side,
                         uint8_t* out, char* mem, int32_t* err, int64_t* rounds) {
  const int TEAM = (int)blockDim.x;
  const int L = s[dim];
  const int nvox = s[0] * s[1] * s[2];
  // terminal slices
  for (int p = threadIdx.x; p < nvox; p += TEAM) {
    int c[3] = {p % s[0], (p / s[0]) % s[1], p / (s[0] * s[1])};
    uint8_t m = (c[dim] == L - 1) ? 0 : 1;
    out[p] = m ^ side;
  }
  if (L <= 2) return;
  int si[3] = {s[0], s[1], s[2]};
  si[dim] = L - 2;
  const int n = si[0] * si[1] * si[2];
  const int HMAX = n + 1;
  const int GR = iq_gr_freq(n);
  const int ist[3] = {1, si[0], si[0] * si[1]};
  CutState S;
  cut_bind(S, mem, n);

  // build: capacities of graphcut.jl:22-54 on interior edges; saturated source edges
  for (int u = threadIdx.x; u < n; u += TEAM) {
    int ic[3] = {u % si[0], (u / si[0]) % si[1], u / (si[0] * si[1])};
    int pc[3] = {ic[0], ic[1], ic[2]};
    pc[dim] += 1;
    int f = 0;
    double e = 0.0, rt = 0.0;
    for (int d = 0; d < 3; d++) {
      double c = 0.0;
      if (ic[d] + 1 < si[d]) { f |= 1 << d; c = slab_cap<T>(A, B, s, pc[0], pc[1], pc[2], d); }
      S.rf[3 * u + d] = c;
      S.rb[3 * u + d] = c;
      S.pr[3 * u + d] = 0.0;
    }
    if (pc[dim] == 1) {
      int q[3] = {pc[0], pc[1], pc[2]};
      q[dim] -= 1;
      e = e + slab_cap<T>(A, B, s, q[0], q[1], q[2], dim);
    }
    if (pc[dim] == L - 2) { f |= 8; rt = slab_cap<T>(A, B, s, pc[0], pc[1], pc[2], dim); }
    S.e[u] = e;
    S.rt[u] = rt;
    S.fl[u] = f;
  }
  __syncthreads();

  int64_t total = 0;
  for (;;) {
    // global relabel
    for (int u = threadIdx.x; u < n; u += TEAM) S.h[u] = ((S.fl[u] & 8) && S.rt[u] > 0.0) ? 1 : HMAX;
    __syncthreads();
    for (int lev = 1;; lev++) {
      int ch = 0;
      for (int u = threadIdx.x; u < n; u += TEAM) {
        if (S.h[u] != HMAX) continue;
        int ic[3] = {u % si[0], (u / si[0]) % si[1], u / (si[0] * si[1])};
        bool hit = false;
        for (int d = 0; d < 3 && !hit; d++) {
          if (ic[d] > 0) {
            int v = u - ist[d];
            if (S.rb[3 * v + d] > 0.0 && S.h[v] == lev) hit = true;
          }
          if (!hit && (S.fl[u] & (1 << d))) {
            int v = u + ist[d];
            if (S.rf[3 * u + d] > 0.0 && S.h[v] == lev) hit = true;
          }
        }
        if (hit) { S.h[u] = lev + 1; ch = 1; }
      }
      if (!__syncthreads_or(ch)) break;
    }
    int act = 0;
    for (int u = threadIdx.x; u < n; u += TEAM) act |= (S.e[u] > 0.0 && S.h[u] < HMAX);
    if (!__syncthreads_or(act)) break;
    if (total > IQ_PR_LIMIT) {
      if (threadIdx.x == 0) atomicCAS(err, 0, IQ_KERR_ITER);
      break;
    }
    for (int it = 0; it < GR; it++) {
      // relabel phase (also clears the push records of the previous round)
      for (int u = threadIdx.x; u < n; u += TEAM) {
        S.pr[3 * u] = 0.0; S.pr[3 * u + 1] = 0.0; S.pr[3 * u + 2] = 0.0;
        int hu = S.h[u];
        int nh = hu;
        if (S.e[u] > 0.0 && hu < HMAX) {
          int ic[3] = {u % si[0], (u / si[0]) % si[1], u / (si[0] * si[1])};
          bool adm = false;
          int mh = HMAX;
          if ((S.fl[u] & 8) && S.rt[u] > 0.0) { if (hu == 1) adm = true; mh = 0; }
          for (int d = 0; d < 3; d++) {
            if (ic[d] > 0) {
              int v = u - ist[d];
              if (S.rb[3 * v + d] > 0.0) { int hv = S.h[v]; if (hu == hv + 1) adm = true; if (hv < mh) mh = hv; }
            }
            if (S.fl[u] & (1 << d)) {
              int v = u + ist[d];
              if (S.rf[3 * u + d] > 0.0) { int hv = S.h[v]; if (hu == hv + 1) adm = true; if (hv < mh) mh = hv; }
            }
          }
          if (!adm) nh = (mh + 1 < HMAX) ? mh + 1 : HMAX;
        }
        S.hn[u] = nh;
      }
      __syncthreads();
      for (int u = threadIdx.x; u < n; u += TEAM) S.h[u] = S.hn[u];
      __syncthreads();
      // push phase
      for (int u = threadIdx.x; u < n; u += TEAM) {
        double ex = S.e[u];
        int hu = S.h[u];
        if (!(ex > 0.0 && hu < HMAX)) continue;
        int ic[3] = {u % si[0], (u / si[0]) % si[1], u / (si[0] * si[1])};
        if ((S.fl[u] & 8) && hu == 1 && S.rt[u] > 0.0) {
          double r = S.rt[u];
          double dl = ex < r ? ex : r;
          ex -= dl;
          S.rt[u] = r - dl;
        }
        for (int d = 0; d < 3 && ex > 0.0; d++) {
          if (ic[d] > 0) {
            int v = u - ist[d];
            if (hu == S.h[v] + 1) {
              double r = S.rb[3 * v + d];
              if (r > 0.0) {
                double dl = ex < r ? ex : r;
                ex -= dl;
                S.rb[3 * v + d] = r - dl;
                S.rf[3 * v + d] += dl;
                S.pr[3 * v + d] = -dl;
              }
            }
          }
          if (ex > 0.0 && (S.fl[u] & (1 << d))) {
            int v = u + ist[d];
            if (hu == S.h[v] + 1) {
              double r = S.rf[3 * u + d];
              if (r > 0.0) {
                double dl = ex < r ? ex : r;
                ex -= dl;
                S.rf[3 * u + d] = r - dl;
                S.rb[3 * u + d] += dl;
                S.pr[3 * u + d] = dl;
              }
            }
          }
        }
        S.e[u] = ex;
      }
      __syncthreads();
      // gather phase
      int a2 = 0;
      for (int u = threadIdx.x; u < n; u += TEAM) {
        int ic[3] = {u % si[0], (u / si[0]) % si[1], u / (si[0] * si[1])};
        double ex = S.e[u];
        for (int d = 0; d < 3; d++) {
          if (ic[d] > 0) {
            double q = S.pr[3 * (u - ist[d]) + d];
            if (q > 0.0) ex += q;
          }
          if (S.fl[u] & (1 << d)) {
            double q = S.pr[3 * u + d];
            if (q < 0.0) ex += -q;
          }
        }
        S.e[u] = ex;
        a2 |= (ex > 0.0 && S.h[u] < HMAX);
      }
      total++;
      if (!__syncthreads_or(a2)) break;
    }
  }
  for (int u = threadIdx.x; u < n; u += TEAM) {
    int ic[3] = {u % si[0], (u / si[0]) % si[1], u / (si[0] * si[1])};
    int pc[3] = {ic[0], ic[1], ic[2]};
    pc[dim] += 1;
    uint8_t m = (S.h[u] < HMAX) ? 0 : 1;
    out[pc[0] + s[0] * (pc[1] + s[1] * pc[2])] = m ^ side;
  }
  if (threadIdx.x == 0 && rounds) {
    atomicAdd((unsigned long long*)rounds, (unsigned long long)total);
    atomicAdd((unsigned long long*)rounds + 2, 1ull);
  }
}

// Register-resident form of cut_slab: same schedule, same arithmetic,
// bit-identical result.  A work-item owns nodes u = tid + k * TEAM, k < NPT;
// their excess, sink residual, height and the residuals of their six outgoing
// edges (towards the minus and the plus neighbour per axis; zero where the
// edge is absent) stay in registers: only the owner reads them.  A push from u
// to w lowers u's outgoing residual at once and leaves the amount in w's inbox
// (LDS, one slot per direction a push can come from, so each slot has one
// writer); w adds it to its excess and to its own outgoing residual on that
// edge at the start of the next round, in the same fixed order as the
// reference schedule's gather.  LDS holds only the inboxes (6 doubles per
// node) and the heights (double buffered, 16-bit): 52 bytes per node.
//
// A round is two barriers around straight-line code: with one node a lane its
// time is the length of that instruction stream (one wavefront per SIMD), with
// six node-wavefronts per SIMD (1,536 nodes) its issue slots, so what the
// schedule allows is done without branches, tests and clears:
//   * a wavefront with excess rewrites all six outgoing amounts of its nodes,
//     zeros included, so a received amount needs no test (adding zero changes
//     nothing) and no clearing; it writes zeros once more in the first round
//     without excess, then skips the push altogether.  The slot of an absent
//     edge is the node's own inbox slot that no neighbour writes;
//   * heights are valid labels (h(u) <= h(v) + 1 on every residual edge u->v:
//     relabels take a minimum over neighbours that only rise, and a push opens
//     an edge from the lower to the higher end), so an active node's relabel,
//     with or without an admissible edge, is min over residual edges of
//     h(v) + 1;
//   * neighbour indices and inbox addresses are formed once per slab.
// 96 slabs side by side, with tests, branches and clears and now: 200 nodes on
// 256 lanes 129 and 87 us, 576 nodes on 256 lanes with three each 455 us and on
// 576 lanes 152 us, 1,536 nodes 741 and 489 us.  The node state must start on a
// 16-byte boundary: 8-byte LDS accesses that straddle one run ten times slower.
//
// OR of a predicate over the team: wavefront votes into one of three LDS words
// behind a single barrier; the word used next is cleared before the barrier
// (its last readers passed an earlier one).
template <bool WAVE>
__device__ __forceinline__ void team_sync() {
  if constexpr (WAVE) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  } else {
    __syncthreads();
  }
}

template <bool WAVE>
__device__ __forceinline__ bool team_or(bool p, int* tflag, int& ph) {
  const bool w = __any(p);
  if constexpr (WAVE) {
    team_sync<true>();
    return w;
  } else {
    const int nx = ph == 2 ? 0 : ph + 1;
    if (w && (threadIdx.x & 63) == 0) tflag[ph] = 1;
    if (threadIdx.x == 0) tflag[nx] = 0;
    __syncthreads();
    const int r = __builtin_amdgcn_readfirstlane(tflag[ph]);
    ph = nx;
    return r != 0;
  }
}

// The same in two parts: the vote and its barrier, returning the word to read;
// the word itself, to be tested (readfirstlane) before the next barrier.
template <bool WAVE>
__device__ __forceinline__ int team_vote(bool p, int* tflag, int& ph) {
  if constexpr (WAVE) {
    team_sync<true>();
    return 0;
  } else {
    const int cur = ph, nx = ph == 2 ? 0 : ph + 1;
    if (p) tflag[cur] = 1;
    if (threadIdx.x == 0) tflag[nx] = 0;
    __syncthreads();
    ph = nx;
    return cur;
  }
}
template <bool WAVE>
__device__ __forceinline__ int team_votes(bool p, const int* tflag, int cur) {
  if constexpr (WAVE) return __any(p);
  else return tflag[cur];
}

// max(x, 0) with zero for NaN (infinite less infinite), and the lesser of two
// numbers: one instruction each (the compiler's own forms quiet their operands
// first, which no value here needs).
__device__ __forceinline__ double cut_pos(double x) {
  double y;
  asm("v_max_f64 %0, %1, 0" : "=v"(y) : "v"(x));
  return y;
}
__device__ __forceinline__ double cut_min(double x, double z) {
  double y;
  asm("v_min_f64 %0, %1, %2" : "=v"(y) : "v"(x), "v"(z));
  return y;
}

#define CUT_FAST_NODE_BYTES (8 * 6 + 2 * 2)
#define CUT_TEAM_MAX 1024
#define CUT_REG_MAX (3 * CUT_TEAM_MAX)  // nodes of the register-resident form (159,744 bytes of LDS)

// mem: CUT_FAST_NODE_BYTES for every node, the count rounded up to a multiple
// of 64; TEAM = 64 (WAVE) or the workgroup's size, a multiple of 64.
template <typename T, int NPT, bool WAVE, bool SKIP = (NPT > 1)>
__device__ __forceinline__ void cut_slab_fast(const SlabView<T>& A, const SlabView<T>& B, const int s[3], int dim, uint8_t side,
                                              uint8_t* out, char* mem, int32_t* err, int64_t* rounds) {
  const int TEAM = WAVE ? 64 : (int)blockDim.x;
  const int L = s[dim];
  const int nvox = s[0] * s[1] * s[2];
  for (int p = threadIdx.x; p < nvox; p += TEAM) {
    int c[3] = {p % s[0], (p / s[0]) % s[1], p / (s[0] * s[1])};
    uint8_t m = (c[dim] == L - 1) ? 0 : 1;
    out[p] = m ^ side;
  }
  if (L <= 2) return;
  int si[3] = {s[0], s[1], s[2]};
  si[dim] = L - 2;
  const int n = si[0] * si[1] * si[2];
  const int np = (n + 63) & ~63;
  const int HMAX = n + 1;
  const int GR = iq_gr_freq(n);
  const int ist[3] = {1, si[0], si[0] * si[1]};
  __shared__ int tflag[3];
  int ph = 0;
  // inbox of node w: [d np + w] the amount its minus neighbour along d pushed
  // up to it, [(3 + d) np + w] what its plus neighbour pushed down
  double* inb = (double*)mem;
  int16_t* h = (int16_t*)(inb + 6 * np);  // committed heights
  int16_t* hn = h + np;                   // next heights
  // per owned node: excess, sink residual, outgoing residuals towards the
  // minus (om) and plus (op) neighbours, height; neighbour indices (the node
  // itself where the edge is absent) and the inbox slots its pushes go to
  bool live[NPT];  // uniform per wavefront: it holds nodes (its lanes past n hold isolated ones)
  double e[NPT], rt[NPT], om[NPT][3], op[NPT][3];
  int hr[NPT], vm[NPT][3], vp[NPT][3], qm[NPT][3], qp[NPT][3];
  bool dirty[NPT];  // uniform per wavefront: it wrote a nonzero amount last round
#pragma unroll
  for (int k = 0; k < NPT; k++) {
    const int u = threadIdx.x + k * TEAM;
    live[k] = (int)(threadIdx.x & ~63u) + k * TEAM < n;
    dirty[k] = false;
    e[k] = 0.0;
    rt[k] = 0.0;
    hr[k] = HMAX;
    int ic[3] = {u % si[0], (u / si[0]) % si[1], u / (si[0] * si[1])};
    int pc[3] = {ic[0], ic[1], ic[2]};
    pc[dim] += 1;
    for (int d = 0; d < 3; d++) {
      om[k][d] = 0.0;
      op[k][d] = 0.0;
      vm[k][d] = u;
      vp[k][d] = u;
      qm[k][d] = d * np + u;
      qp[k][d] = (3 + d) * np + u;
      if (u >= n) continue;
      // an edge's capacity is the same both ways; each end evaluates it
      if (ic[d] + 1 < si[d]) {
        op[k][d] = slab_cap<T>(A, B, s, pc[0], pc[1], pc[2], d);
        vp[k][d] = u + ist[d];
        qp[k][d] = d * np + u + ist[d];
      }
      if (ic[d] > 0) {
        int q[3] = {pc[0], pc[1], pc[2]};
        q[d] -= 1;
        om[k][d] = slab_cap<T>(A, B, s, q[0], q[1], q[2], d);
        vm[k][d] = u - ist[d];
        qm[k][d] = (3 + d) * np + u - ist[d];
      }
    }
    if (u < n) {
      if (pc[dim] == 1) {
        int q[3] = {pc[0], pc[1], pc[2]};
        q[dim] -= 1;
        e[k] = e[k] + slab_cap<T>(A, B, s, q[0], q[1], q[2], dim);
      }
      if (pc[dim] == L - 2) rt[k] = slab_cap<T>(A, B, s, pc[0], pc[1], pc[2], dim);
    }
    if (live[k]) {
#pragma unroll
      for (int d = 0; d < 6; d++) inb[d * np + u] = 0.0;
    }
  }
  if (threadIdx.x < 3) tflag[threadIdx.x] = 0;
  team_sync<WAVE>();

  int64_t total = 0, levels = 0;
  for (;;) {
    // global relabel (exact residual distance to the sink): the least fixed
    // point of h(u) = min over residual edges u->v of h(v) + 1 from these
    // starting values, which relaxing in any order reaches as well as a
    // level-by-level BFS does (every label written is the length of a real
    // path, and labels only decrease).
#pragma unroll
    for (int k = 0; k < NPT; k++)
      if (live[k]) {
        hr[k] = rt[k] > 0.0 ? 1 : HMAX;
        h[threadIdx.x + k * TEAM] = (int16_t)hr[k];
      }
    team_sync<WAVE>();
    int rm[NPT][3], rp[NPT][3];  // the neighbour, or the node itself where the edge is saturated
#pragma unroll
    for (int k = 0; k < NPT; k++)
#pragma unroll
      for (int d = 0; d < 3; d++) {
        const int u = threadIdx.x + k * TEAM;
        rm[k][d] = om[k][d] > 0.0 ? vm[k][d] : u;
        rp[k][d] = op[k][d] > 0.0 ? vp[k][d] : u;
      }
    for (;;) {
      // Each wavefront relaxes its own nodes until they hold still (no
      // barrier; labels of other wavefronts' nodes read meanwhile are valid
      // upper bounds), then one team OR asks whether any wavefront lowered a
      // label; a pass in which none did ends the relabel.  Labels strictly
      // decrease, so both loops end.
      bool ch = false;
      for (;;) {
        bool lc = false;
#pragma unroll
        for (int r = 0; r < 2; r++) {
#pragma unroll
          for (int k = 0; k < NPT; k++) {
            if (!live[k]) continue;
            const int u = threadIdx.x + k * TEAM;
            const int hu = hr[k];
            const int a0 = h[rm[k][0]], a1 = h[rm[k][1]], a2 = h[rm[k][2]];
            const int b0 = h[rp[k][0]], b1 = h[rp[k][1]], b2 = h[rp[k][2]];
            const int best = min(min(min(a0, a1), min(a2, b0)), min(b1, b2)) + 1;
            hr[k] = min(best, hu);
            h[u] = (int16_t)hr[k];
            lc |= best < hu;
          }
          __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
          __builtin_amdgcn_wave_barrier();
          __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        }
        if (!__any(lc)) break;
        ch = true;
      }
      levels++;
      if (!team_or<WAVE>(ch, tflag, ph)) break;
    }
    bool act = false;
#pragma unroll
    for (int k = 0; k < NPT; k++)
      if (live[k]) act |= e[k] > 0.0 && hr[k] < HMAX;
    if (!team_or<WAVE>(act, tflag, ph)) break;
    if (total > IQ_PR_LIMIT) {
      if (threadIdx.x == 0) atomicCAS(err, 0, IQ_KERR_ITER);
      break;
    }
    for (int it = 0; it <= GR; it++) {
      // phase A: take in the previous round's pushes, then relabel
      int hu[NPT];  // the height a push goes to, or -2
      bool any[NPT];
      bool a2 = false;
#pragma unroll
      for (int k = 0; k < NPT; k++) {
        const int u = threadIdx.x + k * TEAM;
        any[k] = false;
        hu[k] = -2;
        if (!live[k]) continue;
        int hm[3], hp[3];
#pragma unroll
        for (int d = 0; d < 3; d++) {
          hm[d] = h[vm[k][d]];
          hp[d] = h[vp[k][d]];
        }
        if (it > 0) {
          double im[3], ip[3];
#pragma unroll
          for (int d = 0; d < 3; d++) {
            im[d] = inb[d * np + u];
            ip[d] = inb[(3 + d) * np + u];
          }
          double ex = e[k];
#pragma unroll
          for (int d = 0; d < 3; d++) {
            ex += im[d];
            om[k][d] = om[k][d] + im[d];
            ex += ip[d];
            op[k][d] = op[k][d] + ip[d];
          }
          e[k] = ex;
        }
        const bool active = e[k] > 0.0 && hr[k] < HMAX;
        a2 |= active;
        any[k] = !SKIP || __any(active);
        if (any[k]) {
          int mh = HMAX;
#pragma unroll
          for (int d = 0; d < 3; d++) {
            mh = min(mh, om[k][d] > 0.0 ? hm[d] : HMAX);
            mh = min(mh, op[k][d] > 0.0 ? hp[d] : HMAX);
          }
          mh = rt[k] > 0.0 ? 0 : mh;
          // past the last round (it == GR) the heights are not used again
          hr[k] = active ? min(mh + 1, HMAX) : hr[k];
          hu[k] = active && mh + 1 < HMAX ? mh : -2;
        }
        hn[u] = (int16_t)hr[k];
      }
      total += it > 0;
      const int cur = team_vote<WAVE>(a2, tflag, ph);
      if (it == GR) break;
      const int more = team_votes<WAVE>(a2, tflag, cur);  // read below, past the push
      { int16_t* t = h; h = hn; hn = t; }
      // phase B: push with the new heights (an edge has one pusher per
      // round, its higher end: the residuals it reads are its own)
#pragma unroll
      for (int k = 0; k < NPT; k++) {
        if (!live[k]) continue;
        if (any[k]) {
          int hm[3], hp[3];
#pragma unroll
          for (int d = 0; d < 3; d++) {
            hm[d] = h[vm[k][d]];
            hp[d] = h[vp[k][d]];
          }
          // what each admissible edge can take
          double cm[3], cp[3];
          const double ct = cut_pos(hu[k] == 0 ? rt[k] : 0.0);
#pragma unroll
          for (int d = 0; d < 3; d++) {
            cm[d] = cut_pos(hu[k] == hm[d] ? om[k][d] : 0.0);
            cp[d] = cut_pos(hu[k] == hp[d] ? op[k][d] : 0.0);
          }
          double ex = e[k];
          const double dt = cut_min(cut_pos(ex), ct);
          ex -= dt;
          rt[k] -= dt;
#pragma unroll
          for (int d = 0; d < 3; d++) {
            const double d0 = cut_min(cut_pos(ex), cm[d]);
            ex -= d0;
            om[k][d] -= d0;
            inb[qm[k][d]] = d0;
            const double d1 = cut_min(cut_pos(ex), cp[d]);
            ex -= d1;
            op[k][d] -= d1;
            inb[qp[k][d]] = d1;
          }
          e[k] = ex;
          dirty[k] = true;
        } else if (dirty[k]) {
#pragma unroll
          for (int d = 0; d < 3; d++) {
            inb[qm[k][d]] = 0.0;
            inb[qp[k][d]] = 0.0;
          }
          dirty[k] = false;
        }
      }
      team_sync<WAVE>();
      // no node was active: the push above changed nothing
      if (it > 0 && !__builtin_amdgcn_readfirstlane(more)) break;
    }
  }
#pragma unroll
  for (int k = 0; k < NPT; k++) {
    const int u = threadIdx.x + k * TEAM;
    if (u >= n) continue;
    int ic[3] = {u % si[0], (u / si[0]) % si[1], u / (si[0] * si[1])};
    int pc[3] = {ic[0], ic[1], ic[2]};
    pc[dim] += 1;
    uint8_t m = (h[u] < HMAX) ? 0 : 1;
    out[pc[0] + s[0] * (pc[1] + s[1] * pc[2])] = m ^ side;
  }
  if (threadIdx.x == 0 && rounds) {
    atomicAdd((unsigned long long*)rounds, (unsigned long long)total);
    atomicAdd((unsigned long long*)rounds + 1, (unsigned long long)levels);
    atomicAdd((unsigned long long*)rounds + 2, 1ull);
  }
}

// One slab by the whole workgroup (a multiple of 64 work-items): up to NPT
// register-resident nodes a lane; NPT = 0: up to three on CUT_TEAM_MAX lanes,
// node state in global scratch beyond CUT_REG_MAX nodes.
template <typename T, int NPT>
__device__ __forceinline__ void cut_dispatch(const SlabView<T>& A, const SlabView<T>& B, const int s[3], int dim, uint8_t side,
                                             uint8_t* out, char* lds, char* gmem, int32_t* err, int64_t* rounds) {
  const int n = s[0] * s[1] * s[2] / s[dim] * (s[dim] > 2 ? s[dim] - 2 : 0);
  const int team = (int)blockDim.x;
  constexpr int MOST = NPT == 0 ? 3 : NPT;
  if (NPT == 0 && n > CUT_REG_MAX) cut_slab<T>(A, B, s, dim, side, out, gmem, err, rounds);
  else if (MOST >= 3 && n > 2 * team) cut_slab_fast<T, 3, false>(A, B, s, dim, side, out, lds, err, rounds);
  else if (MOST >= 2 && n > team) cut_slab_fast<T, 2, false>(A, B, s, dim, side, out, lds, err, rounds);
  else cut_slab_fast<T, 1, false>(A, B, s, dim, side, out, lds, err, rounds);
}

// The slab blockIdx.x of query blockIdx.y: A = the realization's grid over the
// tile, B = the picked training-image window (iqsim.jl:244-273).  False when
// there is none.
template <typename T>
__device__ __forceinline__ bool cut_views(const IqDev* __restrict__ D, const IqQuery* __restrict__ qs, SlabView<T>& A,
                                          SlabView<T>& B, int s[3], int& dim, int& side, uint8_t*& out, char*& gmem) {
  const IqQuery q = qs[blockIdx.y];
  const IqStep& st = D->steps[q.step];
  if ((int)blockIdx.x >= st.ncut) return false;
  const int64_t slot = q.slot;
  const int64_t pk = D->pick[slot];
  if (pk < 0) return false;
  const IqGeo& g = D->g;
  const IqSlab sl = st.slab[blockIdx.x];
  for (int d = 0; d < 3; d++) s[d] = sl.sz[d];
  dim = sl.dim;
  side = sl.side;
  const int rc[3] = {(int)(pk % g.dist[0]), (int)((pk / g.dist[0]) % g.dist[1]),
                     (int)(pk / ((int64_t)g.dist[0] * g.dist[1]))};
  const IqReal& R = D->reals[q.real];
  A.base = (const T*)D->sims + R.sim_off +
           iq_lin3(R.pad, st.origin[0] + sl.lo[0], st.origin[1] + sl.lo[1], st.origin[2] + sl.lo[2]);
  A.st[0] = 1; A.st[1] = R.pad[0]; A.st[2] = (int64_t)R.pad[0] * R.pad[1];
  B.base = (const T*)D->ti + iq_lin3(g.ti, rc[0] + sl.lo[0], rc[1] + sl.lo[1], rc[2] + sl.lo[2]);
  B.st[0] = 1; B.st[1] = g.ti[0]; B.st[2] = (int64_t)g.ti[0] * g.ti[1];
  out = D->keep + (slot * IQ_MAX_SLAB + blockIdx.x) * g.tilevox;
  gmem = D->cutscratch ? D->cutscratch + (slot * IQ_MAX_SLAB + blockIdx.x) * D->cutscratch_per : nullptr;
  return true;
}

// Batched cut: grid (slab, query).  The workgroup has a lane for every node of
// the plan's largest slab, up to CUT_TEAM_MAX, then two or three nodes a lane.
// In a plan with slabs beyond CUT_REG_MAX nodes (NPT = 0) each slab takes the
// form of its own size.
template <typename T, int NPT>
__global__ void __launch_bounds__(CUT_TEAM_MAX)
k_graphcut(const IqDev* __restrict__ D, const IqQuery* __restrict__ qs) {
  extern __shared__ __align__(16) char cut_lds[];
  SlabView<T> A, B;
  int s[3], dim, side;
  uint8_t* out;
  char* gmem;
  if (!cut_views<T>(D, qs, A, B, s, dim, side, out, gmem)) return;
  cut_dispatch<T, NPT>(A, B, s, dim, (uint8_t)side, out, cut_lds, gmem, D->err, D->rounds);
}

#define CUT_INST(T)                                                       \
  template __global__ void k_graphcut<T, 0>(const IqDev*, const IqQuery*); \
  template __global__ void k_graphcut<T, 1>(const IqDev*, const IqQuery*); \
  template __global__ void k_graphcut<T, 2>(const IqDev*, const IqQuery*); \
  template __global__ void k_graphcut<T, 3>(const IqDev*, const IqQuery*);
CUT_INST(float)
CUT_INST(double)

// Plans whose slabs all have at most CUT_WAVE_MAX interior nodes: one
// wavefront per slab, one node a lane, no workgroup barriers in the
// push-relabel rounds.  (Two nodes a lane cost more than the barriers of twice
// the lanes: 90-node slabs take 49 us on one wavefront and 34 us on two.)
#define CUT_WAVE_MAX 64
template <typename T>
__global__ void __launch_bounds__(64)
k_graphcut_wave(const IqDev* __restrict__ D, const IqQuery* __restrict__ qs) {
  extern __shared__ __align__(16) char cut_lds[];
  SlabView<T> A, B;
  int s[3], dim, side;
  uint8_t* out;
  char* gmem;
  if (!cut_views<T>(D, qs, A, B, s, dim, side, out, gmem)) return;
  cut_slab_fast<T, 1, true>(A, B, s, dim, (uint8_t)side, out, cut_lds, D->err, D->rounds);
}

template __global__ void k_graphcut_wave<float>(const IqDev*, const IqQuery*);
template __global__ void k_graphcut_wave<double>(const IqDev*, const IqQuery*);

// Standalone cut of one slab pair (iq_graphcut): A and B both column-major of extents s.
template <typename T, int NPT>
__global__ void __launch_bounds__(CUT_TEAM_MAX)
k_graphcut_host(const T* __restrict__ a, const T* __restrict__ b, int s0, int s1, int s2, int dim,
                uint8_t* __restrict__ out, char* __restrict__ gmem, int32_t* __restrict__ err) {
  extern __shared__ __align__(16) char cut_lds[];
  const int s[3] = {s0, s1, s2};
  SlabView<T> A, B;
  A.base = a; A.st[0] = 1; A.st[1] = s0; A.st[2] = (int64_t)s0 * s1;
  B.base = b; B.st[0] = 1; B.st[1] = s0; B.st[2] = (int64_t)s0 * s1;
  if constexpr (NPT == 0) cut_slab<T>(A, B, s, dim, (uint8_t)0, out, gmem, err, nullptr);  // launched for such a slab alone
  else cut_dispatch<T, NPT>(A, B, s, dim, (uint8_t)0, out, cut_lds, gmem, err, nullptr);
}

#define CUT_HOST_INST(T)                                                                                         \
  template __global__ void k_graphcut_host<T, 0>(const T*, const T*, int, int, int, int, uint8_t*, char*, int32_t*); \
  template __global__ void k_graphcut_host<T, 1>(const T*, const T*, int, int, int, int, uint8_t*, char*, int32_t*); \
  template __global__ void k_graphcut_host<T, 2>(const T*, const T*, int, int, int, int, uint8_t*, char*, int32_t*); \
  template __global__ void k_graphcut_host<T, 3>(const T*, const T*, int, int, int, int, uint8_t*, char*, int32_t*);
CUT_HOST_INST(float)
CUT_HOST_INST(double)

template <typename T>
__global__ void __launch_bounds__(64)
k_graphcut_host_wave(const T* __restrict__ a, const T* __restrict__ b, int s0, int s1, int s2, int dim,
                     uint8_t* __restrict__ out, int32_t* __restrict__ err) {
  extern __shared__ __align__(16) char cut_lds[];
  const int s[3] = {s0, s1, s2};
  SlabView<T> A, B;
  A.base = a; A.st[0] = 1; A.st[1] = s0; A.st[2] = (int64_t)s0 * s1;
  B.base = b; B.st[0] = 1; B.st[1] = s0; B.st[2] = (int64_t)s0 * s1;
  cut_slab_fast<T, 1, true>(A, B, s, dim, (uint8_t)0, out, cut_lds, err, nullptr);
}

template __global__ void k_graphcut_host_wave<float>(const float*, const float*, int, int, int, int, uint8_t*, int32_t*);
template __global__ void k_graphcut_host_wave<double>(const double*, const double*, int, int, int, int, uint8_t*, int32_t*);

// Paste (iqsim.jl:278): voxels whose OR-ed keep flag is 0 take the picked
// training-image window; the keep flags are the debug cut grid (iqsim.jl:281).
// Grid: (tile blocks, query).
template <typename T>
__global__ void __launch_bounds__(256)
k_paste(const IqDev* __restrict__ D, const IqQuery* __restrict__ qs) {
  const IqQuery q = qs[blockIdx.y];
  const int64_t slot = q.slot;
  const int64_t pk = D->pick[slot];
  if (pk < 0) return;
  const IqGeo& g = D->g;
  const IqStep& st = D->steps[q.step];
  const int rc[3] = {(int)(pk % g.dist[0]), (int)((pk / g.dist[0]) % g.dist[1]),
                     (int)(pk / ((int64_t)g.dist[0] * g.dist[1]))};
  const int ns = st.nslab;
  const IqReal& R = D->reals[q.real];
  T* sim = (T*)D->sims + R.sim_off;
  uint8_t* cut = D->cuts + R.sim_off;
  const T* ti = (const T*)D->ti;
  const uint8_t* keep = D->keep + slot * IQ_MAX_SLAB * g.tilevox;
  for (int j = blockIdx.x * blockDim.x + threadIdx.x; j < g.tilevox; j += gridDim.x * blockDim.x) {
    int x = j % g.tile[0], y = (j / g.tile[0]) % g.tile[1], z = j / (g.tile[0] * g.tile[1]);
    uint8_t k = 0;
    for (int s = 0; s < ns; s++) {
      const IqSlab& sl = st.slab[s];
      int a = x - sl.lo[0], b = y - sl.lo[1], c = z - sl.lo[2];
      if (a >= 0 && b >= 0 && c >= 0 && a < sl.sz[0] && b < sl.sz[1] && c < sl.sz[2]) {
        if (s < st.ncut) {
          k |= keep[(int64_t)s * g.tilevox + a + sl.sz[0] * (b + sl.sz[1] * c)];
        } else {
          // two slices, no interior: the slice next to the source keeps the
          // grid, the other takes the window (negated for a next slab), as
          // the cut kernels write for such a slab
          const int cd = sl.dim == 0 ? a : (sl.dim == 1 ? b : c);
          k |= (uint8_t)((cd == sl.sz[sl.dim] - 1 ? 0 : 1) ^ sl.side);
        }
      }
    }
    int64_t gi = iq_lin3(R.pad, st.origin[0] + x, st.origin[1] + y, st.origin[2] + z);
    if (!k) sim[gi] = ti[iq_lin3(g.ti, rc[0] + x, rc[1] + y, rc[2] + z)];
    cut[gi] = k;
  }
}

template __global__ void k_paste<float>(const IqDev*, const IqQuery*);
template __global__ void k_paste<double>(const IqDev*, const IqQuery*);

// Fill helpers (no memset nodes: the run may be captured in a graph)
template <typename T>
__global__ void k_fill(T* __restrict__ p, int64_t n, T v) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) p[i] = v;
}
template __global__ void k_fill<float>(float*, int64_t, float);
template __global__ void k_fill<double>(double*, int64_t, double);
template __global__ void k_fill<uint8_t>(uint8_t*, int64_t, uint8_t);
template __global__ void k_fill<int64_t>(int64_t*, int64_t, int64_t);
template __global__ void k_fill<int32_t>(int32_t*, int64_t, int32_t);

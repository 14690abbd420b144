// (T) correction of the converged closed-shell amplitudes, FP64.
//
// For every occupied triple i >= j >= k of a molecule (the work item):
//   w_ijk^abc = sum_d (bd|ai) t_kj^cd - sum_l (ck|jl) t_il^ab,
//   W_ijk^abc = sum of w over the six simultaneous permutations of (ia),(jb),(kc),
//   V_ijk^abc = t_i^a (bj|ck) + t_j^b (ai|ck) + t_k^c (ai|bj),
//   R3(W)_abc = 4 W_abc + W_bca + W_cab - 2 (W_acb + W_bac + W_cba),
//   E[T]_ijk  = sum_abc W R3(W) / (3 D),  E[ST]_ijk = sum_abc V R3(W) / (3 D),
// D = e_i + e_j + e_k - e_a - e_b - e_c.  R3's coefficients are constant on
// the conjugacy classes of S3, so the per-triple sums are invariant under
// permutations of (i,j,k): ordered triples are covered by i >= j >= k with
// weights 6, 3 or 1.  The reference's spin-orbital loop
// (src/methods/coupledCluster/mod_cc.f90:2028-2111) evaluates -E[T] (c1) and
// -E[ST] (c2) of the same amplitudes.
//
// The kernels are persistent: a fixed grid of workgroups walks the work items
// of the molecules of one size class (v <= 16, v <= 24, v <= 32); each workgroup
// builds W of its item in LDS with FP64 matrix-core products (six
// permutations, each a v^2 x v x (v + o) product), then reduces the energy.
// Per-item partials are summed per molecule in a fixed order, so results are
// bitwise reproducible.
#include <hip/hip_runtime.h>

#include "hcc_triples.h"

namespace hcc {

constexpr int kTripThreads = 256;

// Loads through buffer resources: a padding element takes an offset past the
// resource's range and reads 0 in hardware, with no branch and no select, and
// unlike a load through a descriptor's (generic) pointer it does not count
// against the LDS counter.  Every array of a molecule stays far below 2 GiB.
constexpr int kTripPad = 0x7ffffff8;
__device__ __forceinline__ __amdgpu_buffer_rsrc_t trip_rsrc(const double* p) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, 0x7ffffff0, 0x00020000);
}
__device__ __forceinline__ double trip_load(__amdgpu_buffer_rsrc_t r, bool in, int element) {
  return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, in ? element * 8 : kTripPad, 0, 0));
}

// Orders the wave's LDS accesses before this point with those after it, of all
// its lanes.  LDS serves a wave in program order, so this costs no instruction;
// it keeps the compiler from moving an access across.
__device__ __forceinline__ void wave_lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
}

// permutation s of three positions: position k of the permuted triple takes entry kPerm[s][k]
__constant__ int kPerm[6][3] = {{0, 1, 2}, {0, 2, 1}, {1, 0, 2}, {1, 2, 0}, {2, 0, 1}, {2, 1, 0}};

__device__ double trip_block_sum(double v, double* red) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  double r = red[0];
  for (int k = 1; k < kTripThreads / 64; ++k) r += red[k];
  __syncthreads();
  return r;
}

// Items of molecules with v <= VM (16 or 24) on the matrix cores, W resident in
// LDS.  For permutation s the product Y[(x,y)][z] = sum_d A[p][x][y][d]
// t2[r][q][z][d] - sum_l t2[p][l][x][y] (ql|rz) is a (v^2 x v) x (v + o)
// FP64 MFMA product: A fragments stream from memory (rows (x,y), K = d
// contiguous; the t2 rows are contiguous along (x,y)), the B operands
// (t2[r][q][z][d] as [d][z], (ql|rz) as [l][z], zero-padded to 32 x 32) sit in
// LDS; each 16 x 16 tile is added into W at the permuted positions.
// V_MFMA_F64_16X16X4F64: lane t holds A[t % 16][t / 16] and B[t / 16][t % 16];
// D[row][col] is element row / 4 of lane col + 16 (row % 4).
//
// Bound by the matrix cores and, at the smaller sizes, by the latency of an
// item's few phases.  A wave owns whole x values of a permutation pair: both
// permutations of a pair add to the slab of W of their common x, so a wave
// orders its own read-modify-writes and the workgroup meets only between
// pairs.  (With row tiles dealt out to all waves, each tile needed a barrier
// between the two permutations, 30 an item at v = 24, and the matrix cores
// were busy 23 % of the cycles: 512 ragged molecules of 10 to 48 sites took
// 116 ms.  Now they take 90, the matrix cores busy 34 % at v <= 24 and 28 % at
// v <= 16.)  v <= 16 has its own instance of 4 waves whose 51 KB of LDS let three
// items share a CU; a single one leaves the CU idle while it stages.
typedef double trip_d4 __attribute__((ext_vector_type(4)));
constexpr int kTripKL = kTripMaxOV / 4;        // K steps over l
// W[a][b][c] at a S2 + b S1 + c with S1 = v + 1 and S2 = v S1 + 1 (both odd):
// accesses along any one index are free of LDS bank conflicts.
// The two permutations of a pair share the A operand, so their B operands sit
// side by side as one operand of 2v columns (the first permutation's at
// columns z, the second's at v + z): ceil(2v / 16) column tiles per product
// instead of 2 ceil(v / 16), no padding columns for v = 24 (48 = 3 x 16).
template <int VM>
struct TripLds {
  static constexpr int kThreads = VM <= 16 ? 256 : 512;
  static constexpr int kBC = 2 * VM;                          // combined B columns
  static constexpr int kKD = VM / 4;                          // K steps over d
  // doubles: W[v^3], B operands 2 x 32 x kBC (reused for the L slices of the
  // energy pass), orbital energies and t1 rows, reduction
  static constexpr int kW = VM * (VM * (VM + 1) + 1);
  static constexpr int kE = 4 * VM;
  static constexpr size_t kBytes = sizeof(double) * (kW + 2 * 32 * kBC + kE + 2 * (kThreads / 64));
  static_assert(VM % 8 == 0 && kBC % 16 == 0, "whole K steps and column tiles");
};

template <int VM>
__global__ __launch_bounds__(TripLds<VM>::kThreads) __attribute__((amdgpu_waves_per_eu(VM <= 16 ? 3 : 2))) void
k_triples_mfma(const TripMol* __restrict__ mols, const int2* __restrict__ items, int total, double* __restrict__ part) {
  constexpr int kTripMfmaThreads = TripLds<VM>::kThreads, kTripBC = TripLds<VM>::kBC, kTripKD = TripLds<VM>::kKD;
  constexpr int kTripLdsW = TripLds<VM>::kW, kTripLdsE = TripLds<VM>::kE;
  extern __shared__ double lds[];
  double* W = lds;
  double* Tb = W + kTripLdsW;                 // [d][c], 32 x kTripBC: t_rq^{z d} | t_qr^{z d}
  double* Qb = Tb + 32 * kTripBC;             // [l][c], 32 x kTripBC: (ql|rz) | (rl|qz)
  double* E = Qb + 32 * kTripBC;              // e_vir (v), t1 rows of i, j, k
  double* red = E + kTripLdsE;                // kTripMfmaThreads / 64
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, l16 = lane & 15, kq = lane >> 4;
  constexpr int nwave = kTripMfmaThreads / 64;
  int2 next = (int)blockIdx.x < total ? items[blockIdx.x] : int2{0, 0};
  for (int item = blockIdx.x; item < total; item += gridDim.x) {
    const int2 info = next;   // molecule, packed triple; the next item's is loaded now
    if (item + (int)gridDim.x < total) next = items[item + gridDim.x];
    const TripMol& M = mols[info.x];
    const int o = M.o, v = M.v, n = M.n;
    const int packed = info.y;
    const int occ[3] = {packed & 0xff, (packed >> 8) & 0xff, (packed >> 16) & 0xff};
    const int vv = v * v, ct_n = (2 * v + 15) >> 4;
    const int S1 = v + 1, S2 = v * S1 + 1;
    // the wave's x values and its rows (x, y) of every product
    const int x0 = wave * v / nwave, x1 = (wave + 1) * v / nwave, row0 = x0 * v, row1 = x1 * v;
    for (int e = x0 * S2 + lane; e < x1 * S2; e += 64) W[e] = 0.0;   // the first pair's x is a: the wave's own slab
    const int i = occ[0], j = occ[1], k = occ[2];
    const __amdgpu_buffer_rsrc_t rA = trip_rsrc(M.A), rB = trip_rsrc(M.B), rL = trip_rsrc(M.L), rt2 = trip_rsrc(M.t2);
    // operands of the next phase, loaded into registers while the current
    // phase runs: the B operands of pair h (kStg elements of each 32 x kTripBC
    // array per thread), then the L slices, virtual orbital energies and t1 rows
    constexpr int kStg = 32 * kTripBC / kTripMfmaThreads;   // elements per B array and thread
    constexpr int kStgL = (3 * VM * VM + kTripMfmaThreads - 1) / kTripMfmaThreads;
    static_assert(kStg * kTripMfmaThreads == 32 * kTripBC, "staging covers each B array exactly");
    static_assert(kStgL + 1 <= 2 * kStg, "the staging registers hold the energy-pass data");
    static_assert(3 * VM * VM <= 2 * 32 * kTripBC, "the B region holds the L slices");
    static_assert(kTripMfmaThreads >= 4 * VM, "one energy-pass vector element per thread");
    double stg[2 * kStg];
    auto fetch_b = [&](int h) {
      const int q = occ[kPerm[2 * h][1]], r = occ[kPerm[2 * h][2]];
#pragma unroll
      for (int u = 0; u < kStg; ++u) {
        const int e = threadIdx.x + u * kTripMfmaThreads, row = e / kTripBC, c = e - row * kTripBC;
        const bool first = c < v, second = !first && c < 2 * v;
        const int z = first ? c : c - v;
        const bool dz = row < v && (first || second), lz = row < o && (first || second);
        // first: t_rq^{z d} and (ql|rz); second: t_qr^{z d} and (rl|qz); d, l = row
        const int tt = first ? ((r * o + q) * v + z) * v + row : ((q * o + r) * v + z) * v + row;
        const int bb = first ? ((q * o + row) * o + r) * v + z : ((r * o + row) * o + q) * v + z;
        stg[u] = trip_load(rt2, dz, tt);
        stg[kStg + u] = trip_load(rB, lz, bb);
      }
    };
    // energy-pass data: element e of [Ljk | Lik | Lij] (3 v^2 <= kStgL x threads)
    // and of [e_vir | t1_i | t1_j | t1_k] (4 v <= threads)
    auto fetch_e = [&]() {
#pragma unroll
      for (int u = 0; u < kStgL; ++u) {
        const int e = threadIdx.x + u * kTripMfmaThreads, w = e / vv, f = e - w * vv;
        const int pair = w == 0 ? j * o + k : (w == 1 ? i * o + k : i * o + j);
        stg[u] = trip_load(rL, w < 3, pair * vv + f);
      }
      const int w = threadIdx.x / v, f = threadIdx.x - w * v;
      const int row = w == 1 ? i : (w == 2 ? j : k);
      stg[kStgL] = w == 0 ? M.F[(long)(o + f) * n + o + f] : (w < 4 ? M.t1[(long)row * v + f] : 0.0);
    };
    fetch_b(0);
    // permutations 2h and 2h + 1 share p (hence the A fragments) and swap q, r;
    // the second one's output for (x, y, z) lands where the first one's lands
    // for (x, z, y): both stay within the wave's x values, each tile adds the
    // first, then the second
    for (int h = 0; h < 3; ++h) {
      const int s = 2 * h;
      const int p = occ[kPerm[s][0]];
      const int stride3[3] = {S2, S1, 1};
      const int sx = stride3[kPerm[s][0]], sy = stride3[kPerm[s][1]], sz = stride3[kPerm[s][2]];
      __syncthreads();
#pragma unroll
      for (int u = 0; u < kStg; ++u) {
        const int e = threadIdx.x + u * kTripMfmaThreads;
        Tb[e] = stg[u];
        Qb[e] = stg[kStg + u];
      }
      __syncthreads();
      if (h < 2) fetch_b(h + 1);
      else fetch_e();
      const int Ap = p * vv * v;     // [(x,y)][d] of A
      const int Up = p * o * vv;     // [l][(x,y)] of t2
      // A fragments of the next tile are prefetched; the t2 rows (contiguous
      // along (x, y)) are loaded at the tile (prefetching them too measured
      // slower)
      double fa[kTripKD], fu[kTripKL], na[kTripKD];
      auto fetch = [&](int row) {
        const bool rin = row < row1;
#pragma unroll
        for (int k = 0; k < kTripKD; ++k) {
          const int d = 4 * k + kq;
          na[k] = trip_load(rA, rin && d < v, Ap + row * v + d);
        }
      };
      fetch(row0 + l16);
      for (int rb = row0; rb < row1; rb += 16) {
        // column tiles of the combined B operand: columns c < v belong to
        // permutation 2h (z = c), v <= c < 2v to permutation 2h + 1 (z = c - v)
        constexpr int kCt = kTripBC / 16;
        trip_d4 acc[kCt];
#pragma unroll
        for (int ct = 0; ct < kCt; ++ct) acc[ct] = trip_d4{0.0, 0.0, 0.0, 0.0};
        // (x, y) of the lane's four output rows rb + kq + 4 e, from one division
        // and carries; nr of them are the wave's
        int rx[4], ry[4];
        const int nr = (row1 - rb - kq + 3) >> 2;
        {
          const int base = rb + kq;
          int x = base / v, y = base - x * v;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            rx[e] = x;
            ry[e] = y;
            y += 4;
            while (y >= v) {
              y -= v;
              ++x;
            }
          }
        }
#pragma unroll
        for (int k = 0; k < kTripKD; ++k) fa[k] = na[k];
#pragma unroll
        for (int k = 0; k < kTripKL; ++k) {
          const int l = 4 * k + kq, row = rb + l16;
          fu[k] = -trip_load(rt2, row < row1 && l < o, Up + l * vv + row);
        }
        if (rb + 16 < row1) fetch(rb + 16 + l16);
#pragma unroll
        for (int k = 0; k < kTripKD; ++k) {
          if (4 * k >= v) break;
          const int d = 4 * k + kq;
#pragma unroll
          for (int ct = 0; ct < kCt; ++ct) {
            if (ct >= ct_n) break;
            acc[ct] = __builtin_amdgcn_mfma_f64_16x16x4f64(fa[k], Tb[d * kTripBC + 16 * ct + l16], acc[ct], 0, 0, 0);
          }
        }
#pragma unroll
        for (int k = 0; k < kTripKL; ++k) {
          if (4 * k >= o) break;
          const int l = 4 * k + kq;
#pragma unroll
          for (int ct = 0; ct < kCt; ++ct) {
            if (ct >= ct_n) break;
            acc[ct] = __builtin_amdgcn_mfma_f64_16x16x4f64(fu[k], Qb[l * kTripBC + 16 * ct + l16], acc[ct], 0, 0, 0);
          }
        }
        // permutation 2h: rows (x, y), columns z < v at x sx + y sy + z sz
#pragma unroll
        for (int ct = 0; ct < kCt; ++ct) {
          const int z = 16 * ct + l16;
          if (ct >= ct_n || z >= v) continue;
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (e < nr) W[rx[e] * sx + ry[e] * sy + z * sz] += acc[ct][e];
        }
        wave_lds_order();   // other lanes' elements are updated next
        // permutation 2h + 1: columns v + z of the same tiles at x sx + y sz + z sy
#pragma unroll
        for (int ct = 0; ct < kCt; ++ct) {
          const int z = 16 * ct + l16 - v;
          if (ct >= ct_n || z < 0 || z >= v) continue;
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (e < nr) W[rx[e] * sx + ry[e] * sz + z * sy] += acc[ct][e];
        }
        wave_lds_order();   // and the next tile's rows share x with this one's
      }
    }
    // energy of the item: L slices (jb|kc), (ia|kc), (ia|jb) (in the B-operand
    // region), virtual orbital energies and t1 rows of i, j, k in LDS
    __syncthreads();
    double* Ljk = Tb;
    double* Lik = Tb + vv;
    double* Lij = Tb + 2 * vv;
    double* ev = E;
    double* t1i = E + v;
    double* t1j = t1i + v;
    double* t1k = t1j + v;
#pragma unroll
    for (int u = 0; u < kStgL; ++u) {
      const int e = threadIdx.x + u * kTripMfmaThreads;
      if (e < 3 * vv) Tb[e] = stg[u];
    }
    if ((int)threadIdx.x < 4 * v) E[threadIdx.x] = stg[kStgL];
    __syncthreads();
    const double eijk = M.F[(long)i * n + i] + M.F[(long)j * n + j] + M.F[(long)k * n + k];
    double eT = 0.0, eST = 0.0;
    // element e = (a v + b) v + c; the thread's elements step by the block
    // size, whose (a, b, c) step is added with carries instead of dividing
    const int st_a = kTripMfmaThreads / vv, st_r = kTripMfmaThreads - st_a * vv, st_b = st_r / v,
              st_c = st_r - st_b * v;
    int a = (int)threadIdx.x / vv, b, c;
    {
      const int r = (int)threadIdx.x - a * vv;
      b = r / v;
      c = r - b * v;
    }
    for (int e = threadIdx.x; e < vv * v; e += kTripMfmaThreads) {
      const double Wabc = W[a * S2 + b * S1 + c];
      const double r3 = 4.0 * Wabc + W[b * S2 + c * S1 + a] + W[c * S2 + a * S1 + b] -
                        2.0 * (W[a * S2 + c * S1 + b] + W[b * S2 + a * S1 + c] + W[c * S2 + b * S1 + a]);
      const double g = r3 / (3.0 * (eijk - ev[a] - ev[b] - ev[c]));
      const double V = t1i[a] * Ljk[b * v + c] + t1j[b] * Lik[a * v + c] + t1k[c] * Lij[a * v + b];
      eT += Wabc * g;
      eST += V * g;
      c += st_c;
      b += st_b;
      a += st_a;
      if (c >= v) {
        c -= v;
        ++b;
      }
      if (b >= v) {
        b -= v;
        ++a;
      }
    }
    // block sums (fixed order)
    for (int off = 32; off > 0; off >>= 1) {
      eT += __shfl_xor(eT, off);
      eST += __shfl_xor(eST, off);
    }
    if (lane == 0) {
      red[wave] = eT;
      red[nwave + wave] = eST;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      double t = 0.0, st = 0.0;
      for (int w = 0; w < nwave; ++w) {
        t += red[w];
        st += red[nwave + w];
      }
      const double m = (i > j && j > k) ? 6.0 : ((i == j && j == k) ? 1.0 : 3.0);
      part[2 * item] = m * t;
      part[2 * item + 1] = m * st;
    }
  }
}

// Items of molecules with 24 < v <= 32, whose W (up to 262 KB) does not fit in
// LDS.  The virtual index splits into two blocks (16, and v - 16 padded to 16
// in the products).  R3 mixes only elements whose indices are permutations of
// each other, so the 16^3 blocks of W fall into four classes closed under
// permutation -- indices all in block 0, one in block 1, one in block 0, all in
// block 1 -- of one or three blocks: a class is built in LDS (up to 105 KB),
// reduced to its energy and dropped; every block is built once.
//
// For a block and a permutation pair (p; q, r) a wave takes whole x (two of
// 16): each permutation is one 16 x 16 tile over K = d and l, whose A operand
// streams from the caches straight into registers (the next x's are loaded
// meanwhile), B operands sit in LDS.  Bound by the matrix cores in principle
// (3072 instructions per wave and item at v = o = 32) and by those operand
// loads: one 512-byte read per matrix instruction (matrix cores busy 36 % of the
// cycles, the return path of the loads 77 %).  Six molecules of 54 to 64 sites
// take 19.9 ms (18 TF/s); a kernel of vector FMAs with W in global memory took
// 275 ms.
constexpr int kTbThreads = 512;
constexpr int kTbS1 = 17, kTbS2 = 16 * kTbS1 + 1, kTbBlk = 16 * kTbS2;   // strides and size of a 16^3 block (odd strides)
constexpr int kTbP = 33;                                                   // pitch of the 32 x 32 operand matrices
constexpr int kTbMat = 32 * kTbP;
constexpr size_t kTbBytes = sizeof(double) * (3 * kTbBlk + 6 * kTbMat + 4 * 32 + 2 * (kTbThreads / 64));

__global__ __launch_bounds__(kTbThreads) __attribute__((amdgpu_waves_per_eu(2))) void k_triples_blocked(
    const TripMol* __restrict__ mols, const int2* __restrict__ items, int total, double* __restrict__ part) {
  extern __shared__ double lds[];
  double* const W = lds;                    // up to three blocks: the odd index first, second, third
  double* const Tm = W + 3 * kTbBlk;        // t_rq^{z d} at [z][d] (= t_qr^{d z})
  double* const Bq = Tm + kTbMat;           // (ql|rz) at [l][z]
  double* const Br = Bq + kTbMat;           // (rl|qz) at [l][z]
  double* const Ls = Br + kTbMat;           // (jb|kc), (ia|kc), (ia|jb)
  double* const ev = Ls + 3 * kTbMat;       // virtual orbital energies, t1 rows of i, j, k (32 each)
  double* const red = ev + 4 * 32;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, l16 = lane & 15, kq = lane >> 4;
  constexpr int nwave = kTbThreads / 64;
  constexpr int kStg = 1024 / kTbThreads;   // elements of a 32 x 32 matrix per thread
  for (int item = blockIdx.x; item < total; item += gridDim.x) {
    const int2 info = items[item];
    const TripMol& M = mols[info.x];
    const int o = M.o, v = M.v, n = M.n, vv = v * v;
    const int occ[3] = {info.y & 0xff, (info.y >> 8) & 0xff, (info.y >> 16) & 0xff};
    const int i = occ[0], j = occ[1], k = occ[2];
    const int b1 = v - 16;   // size of block 1 (block 0 has 16)
    const __amdgpu_buffer_rsrc_t rA = trip_rsrc(M.A), rB = trip_rsrc(M.B), rL = trip_rsrc(M.L), rt2 = trip_rsrc(M.t2);
    double stg[3 * kStg];
    auto fetch_b = [&](int h) {
      const int q = occ[kPerm[2 * h][1]], r = occ[kPerm[2 * h][2]];
#pragma unroll
      for (int u = 0; u < kStg; ++u) {
        const int e = t + u * kTbThreads, row = e >> 5, c = e & 31;
        stg[3 * u] = trip_load(rt2, row < v && c < v, ((r * o + q) * v + row) * v + c);
        stg[3 * u + 1] = trip_load(rB, row < o && c < v, ((q * o + row) * o + r) * v + c);
        stg[3 * u + 2] = trip_load(rB, row < o && c < v, ((r * o + row) * o + q) * v + c);
      }
    };
    fetch_b(0);
    __syncthreads();   // the previous item's energy pass has read Ls and ev
#pragma unroll
    for (int u = 0; u < 3 * kStg; ++u) {
      const int e = t + u * kTbThreads, w = e >> 10, row = (e >> 5) & 31, c = e & 31;
      const int pair = w == 0 ? j * o + k : (w == 1 ? i * o + k : i * o + j);
      Ls[w * kTbMat + row * kTbP + c] = trip_load(rL, row < v && c < v, pair * vv + row * v + c);
    }
    if (t < 128) {
      const int w = t >> 5, f = t & 31, row = w == 1 ? i : (w == 2 ? j : k);
      ev[t] = f < v ? (w == 0 ? M.F[(long)(o + f) * n + o + f] : M.t1[(long)row * v + f]) : 0.0;
    }
    const double eijk = M.F[(long)i * n + i] + M.F[(long)j * n + j] + M.F[(long)k * n + k];
    double eT = 0.0, eST = 0.0;
#pragma unroll 1
    for (int cls = 0; cls < 4; ++cls) {
      // class: the common block E and, in the mixed classes, the odd block O
      const int E = cls >> 1, O = cls == 1 ? 1 : (cls == 2 ? 0 : E), nslot = E == O ? 1 : 3;
#pragma unroll 1
      for (int h = 0; h < 3; ++h) {
        const int pp = kPerm[2 * h][0], pq = kPerm[2 * h][1], pr = kPerm[2 * h][2];
        const int p = occ[pp];
        const int stride3[3] = {kTbS2, kTbS1, 1};
        const int sx = stride3[pp], sy = stride3[pq], sz = stride3[pr];
        __syncthreads();   // the previous pair's products and the previous class's energy pass are done
#pragma unroll
        for (int u = 0; u < kStg; ++u) {
          const int e = t + u * kTbThreads, at = (e >> 5) * kTbP + (e & 31);
          Tm[at] = stg[3 * u];
          Bq[at] = stg[3 * u + 1];
          Br[at] = stg[3 * u + 2];
        }
        __syncthreads();
        fetch_b(h < 2 ? h + 1 : 0);
        const int Ap = p * vv * v, Up = p * o * vv;   // [(x, y)][d] of A, [l][(x, y)] of t2
        // A operands of (slot, x): rows y of q's block and y' of r's block.  The
        // next (slot, x)'s take their registers as soon as the products have
        // read them.
        double aq[8], ar[8], uq[8], ur[8];
        auto base = [&](int slot, int x, int& xg, bool& inq, bool& inr) {
          const int bx = pp == slot ? O : E, yq = 16 * (pq == slot ? O : E) + l16, yr = 16 * (pr == slot ? O : E) + l16;
          const bool in = slot < nslot && x < (bx ? b1 : 16);
          xg = (16 * bx + x) * v + yq;
          inq = in && yq < v;
          inr = in && yr < v;
          return yr - yq;
        };
        auto fetch_a = [&](int slot, int x) {
          int xg;
          bool inq, inr;
          const int dr = base(slot, x, xg, inq, inr);
          const int eq = Ap + xg * v + kq, er = eq + dr * v;
#pragma unroll
          for (int s = 0; s < 8; ++s) {
            aq[s] = trip_load(rA, inq && 4 * s + kq < v, eq + 4 * s);
            ar[s] = trip_load(rA, inr && 4 * s + kq < v, er + 4 * s);
          }
        };
        auto fetch_u = [&](int slot, int x) {
          int xg;
          bool inq, inr;
          const int dr = base(slot, x, xg, inq, inr);
          const int eq = Up + xg + kq * vv, er = eq + dr;
#pragma unroll
          for (int s = 0; s < 8; ++s) {
            uq[s] = trip_load(rt2, inq && 4 * s + kq < o, eq + 4 * s * vv);
            ur[s] = trip_load(rt2, inr && 4 * s + kq < o, er + 4 * s * vv);
          }
        };
        fetch_a(0, wave);
        fetch_u(0, wave);
#pragma unroll 1
        for (int u = 0; u < 2 * nslot; ++u) {   // x = wave, wave + 8 of every block
          const int slot = u >> 1, x = wave + nwave * (u & 1);
          const int bx = pp == slot ? O : E, by = pq == slot ? O : E, bz = pr == slot ? O : E;
          double* const Wb = W + slot * kTbBlk;
          const int ny = by ? b1 : 16, nz = bz ? b1 : 16;
          const double* const Tz = Tm + (16 * bz + l16) * kTbP;   // column z: t_rq^{z d}, d along the row
          const double* const Ty = Tm + 16 * by + l16;            // column z' (of q): t_qr^{z' d} = t_rq^{d z'}
          const double* const Qz = Bq + 16 * bz + l16;
          const double* const Ry = Br + 16 * by + l16;
          trip_d4 a0 = {0.0, 0.0, 0.0, 0.0}, a1 = {0.0, 0.0, 0.0, 0.0};
          if (x < (bx ? b1 : 16)) {
#pragma unroll
            for (int s = 0; s < 8; ++s) {
              const int d = 4 * s + kq;
              a0 = __builtin_amdgcn_mfma_f64_16x16x4f64(aq[s], Tz[d], a0, 0, 0, 0);
              a1 = __builtin_amdgcn_mfma_f64_16x16x4f64(ar[s], Ty[d * kTbP], a1, 0, 0, 0);
            }
          }
          fetch_a((u + 1) >> 1, wave + nwave * ((u + 1) & 1));
          if (x < (bx ? b1 : 16)) {
#pragma unroll
            for (int s = 0; s < 8; ++s) {
              const int l = 4 * s + kq;
              a0 = __builtin_amdgcn_mfma_f64_16x16x4f64(-uq[s], Qz[l * kTbP], a0, 0, 0, 0);
              a1 = __builtin_amdgcn_mfma_f64_16x16x4f64(-ur[s], Ry[l * kTbP], a1, 0, 0, 0);
            }
          }
          fetch_u((u + 1) >> 1, wave + nwave * ((u + 1) & 1));
          if (x >= (bx ? b1 : 16)) continue;
          // the block's first contribution stores (it covers the x slab)
          double* const Wx = Wb + x * sx;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int y = kq + 4 * e;
            if (y < ny && l16 < nz) {
              double* const w = Wx + y * sy + l16 * sz;
              *w = h == 0 ? a0[e] : *w + a0[e];
            }
          }
          wave_lds_order();   // other lanes' elements of the x slab are updated next
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int y = kq + 4 * e;
            if (y < nz && l16 < ny) Wx[y * sz + l16 * sy] += a1[e];
          }
        }
      }
      __syncthreads();
      // energy of the class.  Mixed: a runs over the odd block and (b, c) over
      // the common one; the three cyclic elements abc, bca, cab of every ordered
      // (b, c) are taken together, with P their sum and Q that of the other three:
      // R3(abc) = 3 W_abc + P - 2 Q, likewise the others.  Uniform: every element
      // alone by the same formula.
      const int na = O ? b1 : 16, nb = E ? b1 : 16, oa = 16 * O, ob = 16 * E;
      const int c = t & 15, b = (t >> 4) & 15, bg = ob + b, cg = ob + c;
      const double* const Ljk = Ls;
      const double* const Lik = Ls + kTbMat;
      const double* const Lij = Ls + 2 * kTbMat;
      const double* const t1i = ev + 32;
      const double* const t1j = ev + 64;
      const double* const t1k = ev + 96;
      const double* const W1 = nslot == 3 ? W + kTbBlk : W;
      const double* const W2 = nslot == 3 ? W + 2 * kTbBlk : W;
      if (b < nb && c < nb)
        for (int a = t >> 8; a < na; a += kTbThreads >> 8) {
          const int ag = oa + a;
          const double wabc = W[a * kTbS2 + b * kTbS1 + c], wbca = W2[b * kTbS2 + c * kTbS1 + a],
                       wcab = W1[c * kTbS2 + a * kTbS1 + b];
          const double wacb = W[a * kTbS2 + c * kTbS1 + b], wbac = W1[b * kTbS2 + a * kTbS1 + c],
                       wcba = W2[c * kTbS2 + b * kTbS1 + a];
          const double g = 1.0 / (3.0 * (eijk - ev[ag] - ev[bg] - ev[cg]));
          const double m = (wabc + wbca + wcab) - 2.0 * (wacb + wbac + wcba);
          const double r0 = (3.0 * wabc + m) * g;
          eT += wabc * r0;
          eST += (t1i[ag] * Ljk[bg * kTbP + cg] + t1j[bg] * Lik[ag * kTbP + cg] + t1k[cg] * Lij[ag * kTbP + bg]) * r0;
          if (nslot == 3) {
            const double r1 = (3.0 * wbca + m) * g, r2 = (3.0 * wcab + m) * g;
            eT += wbca * r1 + wcab * r2;
            // (i, j, k) with (b, c, a), then with (c, a, b)
            eST += (t1i[bg] * Ljk[cg * kTbP + ag] + t1j[cg] * Lik[bg * kTbP + ag] + t1k[ag] * Lij[bg * kTbP + cg]) * r1;
            eST += (t1i[cg] * Ljk[ag * kTbP + bg] + t1j[ag] * Lik[cg * kTbP + bg] + t1k[bg] * Lij[cg * kTbP + ag]) * r2;
          }
        }
    }
    // block sums (fixed order)
    for (int off = 32; off > 0; off >>= 1) {
      eT += __shfl_xor(eT, off);
      eST += __shfl_xor(eST, off);
    }
    if (lane == 0) {
      red[wave] = eT;
      red[nwave + wave] = eST;
    }
    __syncthreads();
    if (t == 0) {
      double sT = 0.0, sST = 0.0;
      for (int w = 0; w < nwave; ++w) {
        sT += red[w];
        sST += red[nwave + w];
      }
      const double m = (i > j && j > k) ? 6.0 : ((i == j && j == k) ? 1.0 : 3.0);
      part[2 * item] = m * sT;
      part[2 * item + 1] = m * sST;
    }
  }
}

// out[2 m] = E[T], out[2 m + 1] = E[ST]: one workgroup per molecule, the sums
// of its threads' strided items combined in a fixed order (one lane per
// molecule took 1 ms over up to 2600 items)
__global__ __launch_bounds__(kTripThreads) void k_triples_final(const int2* __restrict__ range,
                                                                const double* __restrict__ part,
                                                                double* __restrict__ out) {
  __shared__ double red[kTripThreads / 64];
  const int mol = blockIdx.x;
  double t = 0.0, st = 0.0;
#pragma unroll 4
  for (int it = range[mol].x + threadIdx.x; it < range[mol].y; it += kTripThreads) {
    t += part[2 * (long)it];
    st += part[2 * (long)it + 1];
  }
  t = trip_block_sum(t, red);
  st = trip_block_sum(st, red);
  if (threadIdx.x == 0) {
    out[2 * mol] = t;
    out[2 * mol + 1] = st;
  }
}

// one class's kernel over its items, on `per_cu` workgroups a CU
template <class K>
static hipError_t launch_class(K kernel, int threads, size_t bytes, int per_cu, int cus, const TripMol* mols,
                               const int2* items, int first, int count, double* part, hipStream_t s) {
  if (count <= 0) return hipSuccess;
  const hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
  if (e != hipSuccess) return e;
  const int grid = count < per_cu * cus ? count : per_cu * cus;
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(threads), bytes, s, mols, items + first, count, part + 2 * (long)first);
  return hipGetLastError();
}

int trip_class(int v) { return v <= 16 ? 0 : (v <= 24 ? 1 : 2); }

hipError_t launch_triples(const TripMol* mols, int nm, const int2* range, const int2* items, const int* count, int cus,
                          double* part, double* out, hipStream_t s) {
  hipError_t e = launch_class(k_triples_blocked, kTbThreads, kTbBytes, 1, cus, mols, items, count[0] + count[1],
                              count[2], part, s);
  if (e == hipSuccess)
    e = launch_class(k_triples_mfma<24>, TripLds<24>::kThreads, TripLds<24>::kBytes, 1, cus, mols, items, count[0],
                     count[1], part, s);
  if (e == hipSuccess)
    e = launch_class(k_triples_mfma<16>, TripLds<16>::kThreads, TripLds<16>::kBytes, 3, cus, mols, items, 0, count[0],
                     part, s);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_triples_final, dim3(nm), dim3(kTripThreads), 0, s, range, part, out);
  return hipGetLastError();
}

}  // namespace hcc

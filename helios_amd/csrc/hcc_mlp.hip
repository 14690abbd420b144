// Learned T2 guess: a 3-layer MLP (16 -> 64 -> 64 -> 1, exact-erf GELU) that
// corrects the MP2 amplitudes, t2 = t_mp2 + y / Dp, Dp = e_a + e_b - e_i - e_j.
// The network sees 16 features of each amplitude (MP2 amplitude, the two
// integrals (ia|jb) and (ib|ja), denominator, orbital energies about the
// midgap, site-localisation overlaps of the four orbitals, size) and predicts
// y = Dp (t_ccsd - t_mp2), the residual-scaled correction.
//
// Matrix-core layout.  One wave evaluates 16 amplitudes with
// V_MFMA_F32_16X16X32_BF16 in the transposed form Z^T = W X^T, so that a
// lane (sample n = lane & 15, group g = lane >> 4) holds hidden units
// 16 mb + 4 g + r (mb = 0..3, r = 0..3) of its sample after each layer.  The
// next layer's B operand must hold, per lane, 8 consecutive k-slots 8g..8g+7
// of its sample: k-slot q of step s is mapped to hidden unit
// 16 (2 s + q / 4) + 4 g + q % 4, which is exactly what the lane already
// holds, and the A operand (W2) is loaded in the same permuted k order.  No
// LDS round trip is needed between layers.  Weights and layer inputs are
// BF16, accumulation FP32; biases, GELU and the output layer are FP32.
//
// Training (GPU, deterministic): one kernel per mini-batch takes every wave's
// samples forward (same device function), backward and into weight-gradient
// sums on the matrix cores, 16 samples at a time; a second kernel reduces the
// workgroups' sums in a fixed order and applies Adam.  No atomics anywhere:
// results are bitwise reproducible.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <numeric>
#include <string>
#include <vector>

#include "../../include/helios_ccsd.h"
#include "hcc_mlp.h"

namespace hcc {

typedef float f4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ float bfr(float x) { return (float)(__bf16)x; }
__device__ __forceinline__ float gelu(float z) { return 0.5f * z * (1.f + erff(z * 0.70710678118654752f)); }
// gelu(z) and its derivative, which share the error function
__device__ __forceinline__ float gelu_both(float z, float& prime) {
  const float e = 1.f + erff(z * 0.70710678118654752f);
  prime = 0.5f * e + z * expf(-0.5f * z * z) * 0.39894228040143268f;
  return 0.5f * z * e;
}

// ---------------------------------------------------------------------------
// features
// ---------------------------------------------------------------------------
// The 16 features of an amplitude from the quantities of its pair
// representative: orbital energies e_i, e_j, e_a, e_b, the midgap mu, the
// integrals K = (ia|jb) and X = (ib|ja), the site-localisation overlaps
// O_ij, O_ab, O_ia, O_jb, O_ib, O_ja and the site count.  Returns the MP2
// amplitude t and Dp.  (One formula for the guess, the training rows and
// every kernel that evaluates the network, so their features agree bitwise.)
__device__ __forceinline__ void features_of(double ei, double ej, double ea, double eb, double mu, double K, double X,
                                            double oij, double oab, double oia, double ojb, double oib, double oja,
                                            int N, float* f, double& t, double& Dp) {
  Dp = (ea + eb) - (ei + ej);
  t = -K / Dp;
  f[0] = (float)(10.0 * t);
  f[1] = (float)(K / 2.0);
  f[2] = (float)(X / 2.0);
  f[3] = (float)(Dp / 10.0);
  f[4] = (float)(2.0 / Dp);
  f[5] = (float)(((ei + ej) - 2.0 * mu) / 10.0);
  f[6] = (float)(((ea + eb) - 2.0 * mu) / 10.0);
  f[7] = (float)(fabs(ei - ej) / 10.0);
  f[8] = (float)(fabs(ea - eb) / 10.0);
  f[9] = (float)oij;
  f[10] = (float)oab;
  f[11] = (float)((oia + ojb) / 2.0);
  f[12] = (float)(fabs(oia - ojb) / 2.0);
  f[13] = (float)((oib + oja) / 2.0);
  f[14] = (float)(fabs(oib - oja) / 2.0);
  f[15] = (float)(10.0 / N);
}

// Features of amplitude (i, j, a, b) (virtual indices from 0), computed from
// the pair's representative (i a) <= (j b) so that t2 stays exactly
// pair-symmetric.  Returns the MP2 amplitude and Dp.
__device__ void amp_features(const Mol& M, int i, int j, int a, int b, float* f, double& t, double& Dp) {
  const int N = M.n, o = M.o, v = M.v;
  if (i * v + a > j * v + b) {
    int x = i; i = j; j = x;
    x = a; a = b; b = x;
  }
  const double* F = M.F;
  const double ei = F[(long)i * N + i], ej = F[(long)j * N + j];
  const double ea = F[(long)(o + a) * N + o + a], eb = F[(long)(o + b) * N + o + b];
  const double mu = 0.5 * (F[(long)(o - 1) * N + o - 1] + F[(long)o * N + o]);
  const double K = M.Gklcd[(((long)i * o + j) * v + a) * v + b];   // (ia|jb)
  const double X = M.Gklcd[(((long)i * o + j) * v + b) * v + a];   // (ib|ja)
  const double* O = M.Ov;
  features_of(ei, ej, ea, eb, mu, K, X, O[(long)i * N + j], O[(long)(o + a) * N + o + b], O[(long)i * N + o + a],
              O[(long)j * N + o + b], O[(long)i * N + o + b], O[(long)j * N + o + a], N, f, t, Dp);
}

__device__ __forceinline__ void decode(long e, int o, int v, int& i, int& j, int& a, int& b) {
  b = (int)(e % v);
  a = (int)((e / v) % v);
  j = (int)((e / ((long)v * v)) % o);
  i = (int)(e / ((long)o * v * v));
}

// ---------------------------------------------------------------------------
// network in matrix-core operand order
// ---------------------------------------------------------------------------
struct Net {
  bf8 w1[4];        // layer 1, A operand of hidden block mb: W1[16 mb + row][8 g + q] (g < 2)
  bf8 w2[4][2];     // layer 2, A operand of block mb, k-step s: W2[16 mb + row][unit(s, g, q)]
  float b1[16], b2[16], w3[16];   // this lane's units 16 mb + 4 g + r at index 4 mb + r
  float b3;
};

__device__ __forceinline__ int unit(int s, int g, int q) { return 16 * (2 * s + (q >> 2)) + 4 * g + (q & 3); }

__device__ void net_load(Net& N, const float* __restrict__ w, int lane) {
  const int row = lane & 15, g = lane >> 4;
#pragma unroll
  for (int mb = 0; mb < 4; ++mb) {
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      N.w1[mb][q] = (__bf16)(g < 2 ? w[kOffW1 + (16 * mb + row) * kMlpF + 8 * g + q] : 0.f);
#pragma unroll
      for (int s = 0; s < 2; ++s) N.w2[mb][s][q] = (__bf16)w[kOffW2 + (16 * mb + row) * kMlpH + unit(s, g, q)];
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int u = 16 * mb + 4 * g + r;
      N.b1[4 * mb + r] = w[kOffB1 + u];
      N.b2[4 * mb + r] = w[kOffB2 + u];
      N.w3[4 * mb + r] = bfr(w[kOffW3 + u]);
    }
  }
  N.b3 = w[kOffB3];
}

// what the backward pass needs of this lane's units: gelu' at z1 and z2, the
// rounded first hidden layer and the second
struct Acts {
  float d1[16], h1r[16], d2[16], h2[16];
};

// Forward pass of the wave's 16 samples; x holds features 8g..8g+7 of sample
// lane & 15 (zeros for g >= 2).  Every lane returns its sample's output.
template <bool STORE>
__device__ float net_forward(const Net& N, const bf8 x, Acts& A) {
  f4 c1[4];
#pragma unroll
  for (int mb = 0; mb < 4; ++mb)
    c1[mb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(N.w1[mb], x, f4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
  bf8 hb[2];
#pragma unroll
  for (int mb = 0; mb < 4; ++mb)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float z = c1[mb][r] + N.b1[4 * mb + r];
      const float h = STORE ? gelu_both(z, A.d1[4 * mb + r]) : gelu(z);
      hb[mb >> 1][4 * (mb & 1) + r] = (__bf16)h;
      if (STORE) A.h1r[4 * mb + r] = bfr(h);
    }
  f4 c2[4];
#pragma unroll
  for (int mb = 0; mb < 4; ++mb) {
    c2[mb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(N.w2[mb][0], hb[0], f4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    c2[mb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(N.w2[mb][1], hb[1], c2[mb], 0, 0, 0);
  }
  float p = 0.f;
#pragma unroll
  for (int mb = 0; mb < 4; ++mb)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float z = c2[mb][r] + N.b2[4 * mb + r];
      const float h = STORE ? gelu_both(z, A.d2[4 * mb + r]) : gelu(z);
      p += N.w3[4 * mb + r] * h;
      if (STORE) A.h2[4 * mb + r] = h;
    }
  p += __shfl_xor(p, 16);
  p += __shfl_xor(p, 32);
  return p + N.b3;
}

__device__ __forceinline__ bf8 pack_x(const float* f, int g) {
  bf8 x;
#pragma unroll
  for (int q = 0; q < 8; ++q) x[q] = (__bf16)(g == 0 ? f[q] : (g == 1 ? f[8 + q] : 0.f));
  return x;
}

// ---------------------------------------------------------------------------
// solver-side kernels
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_mlp_overlap(const Mol* __restrict__ mols, Ragged rg, int nm) {
  const int mol = rg.bmol[blockIdx.x];
  const Mol& M = mols[mol];
  const long e = (long)(blockIdx.x - rg.prefix[mol]) * 256 + threadIdx.x;
  const int N = M.n;
  if (e >= (long)N * N) return;
  const int p = (int)(e / N), q = (int)(e % N);
  double s = 0.0;
  for (int mu = 0; mu < N; ++mu) {
    const double cp = M.C[(long)mu * N + p], cq = M.C[(long)mu * N + q];
    s += (cp * cp) * (cq * cq);
  }
  M.Ov[e] = N * s;
}

// The learned guess over the occupied block pairs i <= j of a molecule
// (o(o+1)/2 pairs; each workgroup takes guess_pairs_per_workgroup(v)
// consecutive ones, about 1024 amplitudes, so the network is loaded once per
// workgroup).
// Every (a, b) of block (i, j) with i < j is a pair representative
// ((i a) <= (j b)); for i = j those with a <= b are.  The block's integrals
// (kc|ld) at [i][j][:][:], the virtual-virtual overlaps and the overlap rows
// of i and j are read once, coalesced, into LDS; the network runs once per
// representative; t2[i][j][a][b] is written directly (consecutive b per wave)
// and the mirror block t2[j][i][b][a] through an LDS transpose, so t2 stays
// exactly pair-symmetric and every global access is coalesced.
constexpr int kGuessV = 32;   // v <= 32 (larger molecules: k_mlp_guess_pairs)
// Three waves per SIMD (168 VGPRs and a few spilled registers) hide the GELU
// chain's latency better than the two that the full register set allows:
// 38 -> 30 ms for the 4096-molecule batch (four waves spill 280 bytes a lane).
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3, 8))) void k_mlp_guess_blocks(const Mol* __restrict__ mols, Ragged rg, int nm,
                                                          const float* __restrict__ w) {
  __shared__ double sK[kGuessV * kGuessV], sOvv[kGuessV * kGuessV], sT[kGuessV * (kGuessV + 1)];
  __shared__ double sOi[kGuessV], sOj[kGuessV], sEv[kGuessV];
  const int mol = rg.bmol[blockIdx.x];
  const Mol& M = mols[mol];
  const int N = M.n, o = M.o, v = M.v, vv = v * v;
  if (v > kGuessV) return;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, n = lane & 15, g = lane >> 4;
  Net net;
  net_load(net, w, lane);
  Acts unused;
  const double* F = M.F;
  const double* O = M.Ov;
  const double mu = 0.5 * (F[(long)(o - 1) * N + o - 1] + F[(long)o * N + o]);
  for (int e = threadIdx.x; e < vv; e += 256) sOvv[e] = O[(long)(o + e / v) * N + o + e % v];
  for (int e = threadIdx.x; e < v; e += 256) sEv[e] = F[(long)(o + e) * N + o + e];
  const int npb = o * (o + 1) / 2, bpw = guess_pairs_per_workgroup(v);
  const int pb0 = (blockIdx.x - rg.prefix[mol]) * bpw, pb1 = min(npb, pb0 + bpw);
  for (int pb = pb0; pb < pb1; ++pb) {
    int j = (int)((sqrt(8.0 * pb + 1.0) - 1.0) * 0.5);
    while (j * (j + 1) / 2 > pb) --j;
    while ((j + 1) * (j + 2) / 2 <= pb) ++j;
    const int i = pb - j * (j + 1) / 2;   // i <= j < o
    const long blk = ((long)i * o + j) * vv;
    __syncthreads();   // the previous pair's LDS reads and mirror writes are done
    for (int e = threadIdx.x; e < vv; e += 256) sK[e] = M.Gklcd[blk + e];
    for (int e = threadIdx.x; e < v; e += 256) {
      sOi[e] = O[(long)i * N + o + e];
      sOj[e] = O[(long)j * N + o + e];
    }
    __syncthreads();
    const double ei = F[(long)i * N + i], ej = F[(long)j * N + j];
    const double oij = O[(long)i * N + j];
    // representatives in order: (a, b) row-major over the block (i < j), or
    // the upper triangle a <= b row by row (i = j)
    const int nrep = i < j ? vv : v * (v + 1) / 2;
    for (int base = wave * 16; base < nrep; base += 64) {
      const int q = base + n;
      const bool ok = q < nrep;
      int a = 0, b = 0;
      if (ok) {
        if (i < j) {
          a = q / v;
          b = q - a * v;
        } else {
          // row a of the upper triangle starts at a v - a (a - 1) / 2
          a = (int)(((2.0 * v + 1.0) - sqrt((2.0 * v + 1.0) * (2.0 * v + 1.0) - 8.0 * q)) * 0.5);
          while (a > 0 && a * v - a * (a - 1) / 2 > q) --a;
          while ((a + 1) * v - (a + 1) * a / 2 <= q) ++a;
          b = a + (q - (a * v - a * (a - 1) / 2));
        }
      }
      float f[kMlpF];
#pragma unroll
      for (int r = 0; r < kMlpF; ++r) f[r] = 0.f;
      double t = 0.0, Dp = 1.0;
      if (ok && g < 2)
        features_of(ei, ej, sEv[a], sEv[b], mu, sK[a * v + b], sK[b * v + a], oij, sOvv[a * v + b], sOi[a], sOj[b],
                    sOi[b], sOj[a], N, f, t, Dp);
      const float y = net_forward<false>(net, pack_x(f, g), unused);
      if (ok && g == 0) {
        const double val = t + (double)y / Dp;
        M.t2[blk + a * v + b] = val;
        if (i < j) sT[b * (kGuessV + 1) + a] = val;   // t2[j][i][b][a]
        else M.t2[blk + b * v + a] = val;
      }
    }
    if (i < j) {
      __syncthreads();
      const long mblk = ((long)j * o + i) * vv;
      for (int e = threadIdx.x; e < vv; e += 256) M.t2[mblk + e] = sT[(e / v) * (kGuessV + 1) + e % v];
    }
  }
}

// Molecules with v > 32: one network evaluation per amplitude pair; work item
// p enumerates the pairs (mm, nn) = ((i a), (j b)) with mm <= nn
// (p = nn (nn + 1) / 2 + mm), and the value is written to t2[i][j][a][b] and
// its mirror t2[j][i][b][a].  4 waves x 16 groups x 16 amplitudes per workgroup.
__global__ __launch_bounds__(256) void k_mlp_guess_pairs(const Mol* __restrict__ mols, Ragged rg, int nm,
                                                         const float* __restrict__ w) {
  const int mol = rg.bmol[blockIdx.x];
  const Mol& M = mols[mol];
  const int o = M.o, v = M.v;
  if (v <= kGuessV) return;
  const long ne = (long)o * v, npair = ne * (ne + 1) / 2;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, n = lane & 15, g = lane >> 4;
  const long base = (long)(blockIdx.x - rg.prefix[mol]) * 1024 + wave * 256;
  Net net;
  net_load(net, w, lane);
  Acts unused;
  for (int grp = 0; grp < 16; ++grp) {
    const long p = base + grp * 16 + n;
    const bool ok = p < npair;
    float f[kMlpF];
#pragma unroll
    for (int q = 0; q < kMlpF; ++q) f[q] = 0.f;
    double t = 0.0, Dp = 1.0;
    long e = 0, em = 0;
    if (ok) {
      long nn = (long)((sqrt(8.0 * (double)p + 1.0) - 1.0) * 0.5);
      while (nn * (nn + 1) / 2 > p) --nn;
      while ((nn + 1) * (nn + 2) / 2 <= p) ++nn;
      const long mm = p - nn * (nn + 1) / 2;
      const int i = (int)(mm / v), a = (int)(mm % v), j = (int)(nn / v), b = (int)(nn % v);
      e = (((long)i * o + j) * v + a) * v + b;
      em = (((long)j * o + i) * v + b) * v + a;
      if (g < 2) amp_features(M, i, j, a, b, f, t, Dp);
    }
    const float y = net_forward<false>(net, pack_x(f, g), unused);
    if (ok && g == 0) {
      const double val = t + (double)y / Dp;
      M.t2[e] = val;
      M.t2[em] = val;
    }
  }
}

void mlp_overlaps(const Mol* mols, Ragged rgNN, int nm, hipStream_t s) {
  if (rgNN.nblocks > 0) hipLaunchKernelGGL(k_mlp_overlap, dim3(rgNN.nblocks), dim3(256), 0, s, mols, rgNN, nm);
}
void mlp_guess(const Mol* mols, Ragged rgPairBlk, Ragged rgPairL, int nm, bool any_large, const float* params,
               hipStream_t s) {
  if (rgPairBlk.nblocks > 0)
    hipLaunchKernelGGL(k_mlp_guess_blocks, dim3(rgPairBlk.nblocks), dim3(256), 0, s, mols, rgPairBlk, nm, params);
  if (any_large && rgPairL.nblocks > 0)
    hipLaunchKernelGGL(k_mlp_guess_pairs, dim3(rgPairL.nblocks), dim3(256), 0, s, mols, rgPairL, nm, params);
}

// ---------------------------------------------------------------------------
// training kernels
// ---------------------------------------------------------------------------
__device__ __forceinline__ unsigned mix32(unsigned h) {
  h ^= h >> 16;
  h *= 0x7feb352du;
  h ^= h >> 15;
  h *= 0x846ca68bu;
  h ^= h >> 16;
  return h;
}

// training rows of the converged molecules: per_mol hashed amplitudes each
__global__ __launch_bounds__(256) void k_mlp_collect(const Mol* __restrict__ mols, const State* __restrict__ st, int nm,
                                                     int per_mol, unsigned seed, float* __restrict__ rows,
                                                     int* __restrict__ where) {
  const long gid = (long)blockIdx.x * 256 + threadIdx.x;
  if (gid >= (long)nm * per_mol) return;
  const int mol = (int)(gid / per_mol), s = (int)(gid % per_mol);
  const Mol& M = mols[mol];
  const long n2 = (long)M.o * M.o * M.v * M.v;
  const unsigned h = mix32(seed ^ mix32(0x9e3779b9u * (unsigned)(mol + 1) + 0x85ebca6bu * (unsigned)s));
  const long e = (long)(h % (unsigned long)n2);
  float* r = rows + gid * kMlpRow;
  where[2 * gid] = mol;
  where[2 * gid + 1] = (int)e;
  if (st[mol].status != 1) {
    for (int q = 0; q < kMlpRow; ++q) r[q] = 0.f;
    return;
  }
  int i, j, a, b;
  decode(e, M.o, M.v, i, j, a, b);
  float f[kMlpF];
  double t, Dp;
  amp_features(M, i, j, a, b, f, t, Dp);
  for (int q = 0; q < kMlpF; ++q) r[q] = f[q];
  r[kMlpF] = (float)(Dp * (M.t2[e] - t));
  r[kMlpF + 1] = 1.f;
}

// Forward over rows base .. base + nb - 1: per-workgroup loss sums (fixed
// order) to lossp[blockIdx.x], outputs to yout unless null.
__global__ __launch_bounds__(256) void k_mlp_forward(const float* __restrict__ w, const float* __restrict__ rows,
                                                     long base, int nb, double* __restrict__ lossp,
                                                     float* __restrict__ yout) {
  __shared__ double sl[256];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, n = lane & 15, g = lane >> 4;
  Net net;
  net_load(net, w, lane);
  for (int grp = 0; grp < 4; ++grp) {
    const int loc = wave * 64 + grp * 16 + n;
    const int sb = blockIdx.x * 256 + loc;
    const bool ok = sb < nb;
    const float* R = rows + (ok ? base + sb : 0) * kMlpRow;
    float f[kMlpF];
#pragma unroll
    for (int q = 0; q < kMlpF; ++q) f[q] = ok ? R[q] : 0.f;
    Acts A;
    const float y = net_forward<false>(net, pack_x(f, g), A);
    const float tg = ok ? R[kMlpF] : 0.f, wt = ok ? R[kMlpF + 1] : 0.f;
    const float d = y - tg;
    if (g == 0) sl[loc] = ok ? (double)(wt * d * d) : 0.0;
    if (yout != nullptr && ok && g == 0) yout[sb] = y;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    double s = 0.0;
    for (int k = 0; k < 256; ++k) s += sl[k];
    lossp[blockIdx.x] = s;
  }
}

// Loss and weight gradient of a mini-batch: sample sb is row
// ((base + sb) pa + pc) mod ns (a permutation of the rows for gcd(pa, ns) = 1).
// A workgroup takes `per_block` samples (64 or 256) and writes their loss and
// its gradient sums, part[blockIdx.x][kMlpParams]; samples past nb add zero.
//
// Everything between the rows and the sums stays in registers and LDS, 16
// samples of a wave at a time:
//  * forward as in the guess (BF16 operands, FP32 accumulation);
//  * dz2 = dy w3 gelu'(z2) on the lane that holds the unit, dz1 = (W2^T dz2)
//    gelu'(z1) with V_MFMA_F32_16X16X4F32: the K step (mb, r) takes units
//    16 mb + 4 g + r of the four lane groups, which is what they hold, so dz2
//    is the B operand as it stands;
//  * dW2 += dz2 h1^T and dW1 += dz1 x^T with the samples along K (FP32
//    products and sums, 80 accumulators a lane), from an LDS transpose with a
//    row pitch of 80 floats (reads and 16-byte writes without bank conflicts);
//    the biases and dW3 are summed per lane.
// Bound by the GELU arithmetic and this chain's latency: one wave per SIMD,
// for the accumulators and the network's operands take over 256 registers.
// The separate forward, backward and per-parameter gradient kernels, with 400
// activations a sample through memory, took 420 us for 65000 rows; this one
// takes 59 (477 -> 97 us for the whole call, 195 -> 63 us for a few thousand rows).
constexpr int kGradThreads = 256;
constexpr int kGradLd = 80;
constexpr int kGradW2Ld = 68;
constexpr int kGradWave = 16 * (3 * kGradLd + 16);   // floats of a wave: dz2, h1, dz1 [n][80], x [n][16]
constexpr int kGradLds = 4 * kGradWave + kMlpH * kGradW2Ld > 4 * kOffB3 ? 4 * kGradWave + kMlpH * kGradW2Ld : 4 * kOffB3;
__global__ __launch_bounds__(kGradThreads) __attribute__((amdgpu_waves_per_eu(1, 1))) void k_mlp_gradient(
    const float* __restrict__ w, const float* __restrict__ rows, long ns, long pa, long pc, long base, int nb,
    int per_block, double* __restrict__ lossp, float* __restrict__ part) {
  __shared__ __attribute__((aligned(16))) float lds[kGradLds];
  __shared__ double sl[kGradThreads];
  __shared__ float sb3[4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, n = lane & 15, g = lane >> 4;
  float* const D2 = lds + wave * kGradWave;
  float* const H1 = D2 + 16 * kGradLd;
  float* const D1 = H1 + 16 * kGradLd;
  float* const Xs = D1 + 16 * kGradLd;
  float* const W2s = lds + 4 * kGradWave;   // W2[k][j], rounded
  for (int q = threadIdx.x; q < kMlpH * kMlpH; q += kGradThreads) W2s[(q >> 6) * kGradW2Ld + (q & 63)] = bfr(w[kOffW2 + q]);
  Net net;
  net_load(net, w, lane);
  f4 gw2[4][4], gw1[4];
  float gb1[16], gb2[16], gw3[16], gb3 = 0.f;
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    gw1[a] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int b = 0; b < 4; ++b) gw2[a][b] = f4{0.f, 0.f, 0.f, 0.f};
  }
#pragma unroll
  for (int u = 0; u < 16; ++u) gb1[u] = gb2[u] = gw3[u] = 0.f;
  double loss = 0.0;
  const int passes = per_block / 64;
  for (int pass = 0; pass < passes; ++pass) {
    const int sb = blockIdx.x * per_block + (wave * passes + pass) * 16 + n;
    const bool ok = sb < nb;
    const float* R = rows + (ok ? ((base + sb) * pa + pc) % ns : 0) * kMlpRow;
    float f[kMlpF];
#pragma unroll
    for (int q = 0; q < kMlpF; ++q) f[q] = ok ? R[q] : 0.f;
    const float tg = ok ? R[kMlpF] : 0.f, wt = ok ? R[kMlpF + 1] : 0.f;
    Acts A;
    const float y = net_forward<true>(net, pack_x(f, g), A);
    const float d = y - tg, dy = ok ? 2.f * wt * d / (float)nb : 0.f;
    if (g == 0) loss += ok ? (double)(wt * d * d) : 0.0;
    float dz2[16];
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      dz2[u] = dy * net.w3[u] * A.d2[u];
      gb2[u] += dz2[u];
      gw3[u] += dy * A.h2[u];
    }
    gb3 += dy;
    __syncthreads();   // the previous pass has read the tiles (first pass: W2s is written)
#pragma unroll
    for (int mb = 0; mb < 4; ++mb) {
      *reinterpret_cast<f4*>(&D2[n * kGradLd + 16 * mb + 4 * g]) = f4{dz2[4 * mb], dz2[4 * mb + 1], dz2[4 * mb + 2], dz2[4 * mb + 3]};
      *reinterpret_cast<f4*>(&H1[n * kGradLd + 16 * mb + 4 * g]) = f4{A.h1r[4 * mb], A.h1r[4 * mb + 1], A.h1r[4 * mb + 2], A.h1r[4 * mb + 3]};
    }
    if (g < 2)
#pragma unroll
      for (int q = 0; q < 8; ++q) Xs[n * 16 + 8 * g + q] = bfr(g == 0 ? f[q] : f[8 + q]);
    f4 c[4];
#pragma unroll
    for (int jb = 0; jb < 4; ++jb) c[jb] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int mb = 0; mb < 4; ++mb)
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int jb = 0; jb < 4; ++jb)
          c[jb] = __builtin_amdgcn_mfma_f32_16x16x4f32(W2s[(16 * mb + 4 * g + r) * kGradW2Ld + 16 * jb + n],
                                                       dz2[4 * mb + r], c[jb], 0, 0, 0);
#pragma unroll
    for (int jb = 0; jb < 4; ++jb) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        c[jb][r] *= A.d1[4 * jb + r];
        gb1[4 * jb + r] += c[jb][r];
      }
      *reinterpret_cast<f4*>(&D1[n * kGradLd + 16 * jb + 4 * g]) = c[jb];
    }
    __syncthreads();
    // samples 4 s + g along K: rows are the units of a block, columns those of the layer below
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const float* const d2 = D2 + (4 * s + g) * kGradLd + n;
      const float* const h1 = H1 + (4 * s + g) * kGradLd + n;
      const float* const d1 = D1 + (4 * s + g) * kGradLd + n;
      const float x = Xs[(4 * s + g) * 16 + n];
      float hk[4];
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) hk[kb] = h1[16 * kb];
#pragma unroll
      for (int mb = 0; mb < 4; ++mb) {
        const float a = d2[16 * mb];
#pragma unroll
        for (int kb = 0; kb < 4; ++kb) gw2[mb][kb] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, hk[kb], gw2[mb][kb], 0, 0, 0);
        gw1[mb] = __builtin_amdgcn_mfma_f32_16x16x4f32(d1[16 * mb], x, gw1[mb], 0, 0, 0);
      }
    }
  }
  // the lanes of a group hold the same units: sums over their samples
#pragma unroll
  for (int off = 1; off < 16; off <<= 1) {
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      gb1[u] += __shfl_xor(gb1[u], off);
      gb2[u] += __shfl_xor(gb2[u], off);
      gw3[u] += __shfl_xor(gw3[u], off);
    }
    gb3 += __shfl_xor(gb3, off);
  }
  sl[threadIdx.x] = loss;
  __syncthreads();
  float* const S = lds + wave * kOffB3;   // this wave's sums in parameter order
#pragma unroll
  for (int mb = 0; mb < 4; ++mb)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int m = 16 * mb + 4 * g + r;
      S[kOffW1 + m * kMlpF + n] = gw1[mb][r];
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) S[kOffW2 + m * kMlpH + 16 * kb + n] = gw2[mb][kb][r];
      if (n == 0) {
        S[kOffB1 + m] = gb1[4 * mb + r];
        S[kOffB2 + m] = gb2[4 * mb + r];
        S[kOffW3 + m] = gw3[4 * mb + r];
      }
    }
  if (lane == 0) sb3[wave] = gb3;
  __syncthreads();
  float* const P = part + (long)blockIdx.x * kMlpParams;
  for (int q = threadIdx.x; q < kOffB3; q += kGradThreads)
    P[q] = lds[q] + lds[kOffB3 + q] + lds[2 * kOffB3 + q] + lds[3 * kOffB3 + q];
  if (threadIdx.x == 0) {
    P[kOffB3] = sb3[0] + sb3[1] + sb3[2] + sb3[3];
    double s = 0.0;
    for (int k = 0; k < 4; ++k)
      for (int q = 0; q < 16; ++q) s += sl[64 * k + q];
    lossp[blockIdx.x] = s;
  }
}

// fixed-order reduction of the workgroups' sums (8 threads per parameter, 32
// consecutive parameters of a sum row per load), then (update) one Adam step
__global__ __launch_bounds__(256) void k_mlp_adam(float* __restrict__ w, float* __restrict__ m1, float* __restrict__ m2,
                                                  float* __restrict__ grad, const float* __restrict__ part, int nchunk,
                                                  float lr, float bc1, float bc2, int update) {
  __shared__ float red[8][32];
  const int p = blockIdx.x * 32 + (threadIdx.x & 31), grp = threadIdx.x >> 5;
  float g = 0.f;
  if (p < kMlpParams)
#pragma unroll 8
    for (int c = grp; c < nchunk; c += 8) g += part[(long)c * kMlpParams + p];
  red[grp][threadIdx.x & 31] = g;
  __syncthreads();
  if (grp != 0 || p >= kMlpParams) return;
  for (int c = 1; c < 8; ++c) g += red[c][threadIdx.x];
  grad[p] = g;
  if (!update) return;
  const float a = 0.9f * m1[p] + 0.1f * g;
  const float b = 0.999f * m2[p] + 0.001f * g * g;
  m1[p] = a;
  m2[p] = b;
  w[p] -= lr * (a / bc1) / (sqrtf(b / bc2) + 1e-8f);
}

}  // namespace hcc

// ---------------------------------------------------------------------------
// trainer object and its C ABI
// ---------------------------------------------------------------------------
using namespace hcc;

struct hcc_mlp {
  int device = 0;
  hipStream_t stream = nullptr;
  float *w = nullptr, *m1 = nullptr, *m2 = nullptr, *grad = nullptr;
  float* rows = nullptr;
  int* where = nullptr;
  long cap = 0, count = 0;
  // mini-batch buffers (grown on demand): gradient sums per workgroup, loss sums
  int pcap = 0;
  float* part = nullptr;
  double* lossp = nullptr;
  long lcap = 0;
  long step = 0;
  std::string err;
};

namespace {

template <class T>
void dalloc(T** p, size_t count) {
  if (*p) HCHECK(hipFree(*p));
  *p = nullptr;
  HCHECK(hipMalloc((void**)p, std::max<size_t>(1, count) * sizeof(T)));
}

// Samples per workgroup of the gradient kernel: 64 (16 per wave) keep up to
// 256 CUs busy on mini-batches; beyond 16384 samples 256 bound the number of
// gradient sums to reduce (65000 samples: 1016 sums of 21 KB instead of 254).
int samples_per_block(long nb) { return nb <= 16384 ? 64 : 256; }

// a buffer of `count` times `each` elements; a failed growth leaves none (capacity 0)
template <class T, class N>
void grow(T** p, N* cap, N count, size_t each) {
  if (count <= *cap) return;
  *cap = 0;
  dalloc(p, (size_t)count * each);
  *cap = count;
}

void ensure_part(hcc_mlp* net, int blocks) { grow(&net->part, &net->pcap, blocks, kMlpParams); }

void ensure_loss(hcc_mlp* net, long blocks) { grow(&net->lossp, &net->lcap, blocks, 1); }

// one mini-batch of nb samples on `blocks` workgroups (those past nb add
// zero): loss and gradient; update = Adam step
void batch_step(hcc_mlp* net, long ns, long pa, long pc, long base, int nb, int blocks, int per_block, double* lossp,
                bool update, float lr) {
  hipStream_t s = net->stream;
  hipLaunchKernelGGL(k_mlp_gradient, dim3(blocks), dim3(kGradThreads), 0, s, net->w, net->rows, ns, pa, pc, base, nb,
                     per_block, lossp, net->part);
  float bc1 = 1.f, bc2 = 1.f;
  if (update) {
    net->step += 1;
    bc1 = (float)(1.0 - std::pow(0.9, (double)net->step));
    bc2 = (float)(1.0 - std::pow(0.999, (double)net->step));
  }
  hipLaunchKernelGGL(k_mlp_adam, dim3((kMlpParams + 31) / 32), dim3(256), 0, s, net->w, net->m1, net->m2,
                     net->grad, net->part, blocks, lr, bc1, bc2, update ? 1 : 0);
  HCHECK(hipGetLastError());
}

long gcd_l(long a, long b) {
  while (b) {
    long t = a % b;
    a = b;
    b = t;
  }
  return a;
}

}  // namespace

#define MLP_BEGIN                   \
  if (net == nullptr) return HCC_E_ARG; \
  try {                             \
    HCHECK(hipSetDevice(net->device));
#define MLP_END                                                          \
  }                                                                      \
  catch (const HipError& he) {                                           \
    net->err = std::string(he.what) + ": " + hipGetErrorString(he.e);   \
    return HCC_E_HIP;                                                    \
  }                                                                      \
  catch (const std::string& se) {                                        \
    net->err = se;                                                       \
    return HCC_E_ARG;                                                    \
  }                                                                      \
  catch (const std::bad_alloc&) {                                        \
    net->err = "host allocation failed";                                 \
    return HCC_E_MEMORY;                                                 \
  }                                                                      \
  return HCC_OK;

extern "C" {

int hcc_mlp_create(hcc_mlp** out, int device, long capacity) {
  if (out == nullptr || capacity < 0) return HCC_E_ARG;
  *out = nullptr;
  hcc_mlp* net = new hcc_mlp();
  net->device = device;
  int rc = [&]() -> int {
    MLP_BEGIN
    HCHECK(hipStreamCreateWithFlags(&net->stream, hipStreamNonBlocking));
    dalloc(&net->w, kMlpParams);
    dalloc(&net->m1, kMlpParams);
    dalloc(&net->m2, kMlpParams);
    dalloc(&net->grad, kMlpParams);
    HCHECK(hipMemset(net->w, 0, kMlpParams * sizeof(float)));
    HCHECK(hipMemset(net->m1, 0, kMlpParams * sizeof(float)));
    HCHECK(hipMemset(net->m2, 0, kMlpParams * sizeof(float)));
    dalloc(&net->rows, (size_t)capacity * kMlpRow);
    dalloc(&net->where, (size_t)capacity * 2);
    // 256 workgroups' gradient sums, with the trainer's other arrays: enough for
    // 16384 samples at 64 a workgroup and for 65536 at 256.  Allocated by the first
    // gradient call, the 5 MB cost it 0.35 ms (larger calls grow them)
    const int blocks = (int)std::min<long>(256, (capacity + 63) / 64);
    ensure_part(net, blocks);
    ensure_loss(net, blocks);
    net->cap = capacity;
    MLP_END
  }();
  if (rc != HCC_OK) {
    hcc_mlp_destroy(net);
    return rc;
  }
  *out = net;
  return HCC_OK;
}

void hcc_mlp_destroy(hcc_mlp* net) {
  if (net == nullptr) return;
  (void)hipSetDevice(net->device);
  for (void* p : {(void*)net->w, (void*)net->m1, (void*)net->m2, (void*)net->grad, (void*)net->rows,
                  (void*)net->where, (void*)net->part, (void*)net->lossp})
    if (p) (void)hipFree(p);
  if (net->stream) (void)hipStreamDestroy(net->stream);
  delete net;
}

const char* hcc_mlp_last_error(const hcc_mlp* net) { return net ? net->err.c_str() : "null trainer"; }

int hcc_mlp_set_params(hcc_mlp* net, const float* params, int count) {
  if (net == nullptr || params == nullptr) return HCC_E_ARG;
  if (count != kMlpParams) {
    net->err = "parameter count must be HCC_MLP_PARAMS";
    return HCC_E_ARG;
  }
  MLP_BEGIN
  HCHECK(hipMemcpy(net->w, params, kMlpParams * sizeof(float), hipMemcpyHostToDevice));
  HCHECK(hipMemset(net->m1, 0, kMlpParams * sizeof(float)));
  HCHECK(hipMemset(net->m2, 0, kMlpParams * sizeof(float)));
  net->step = 0;
  MLP_END
}

int hcc_mlp_get_params(hcc_mlp* net, float* params, int count) {
  if (net == nullptr || params == nullptr) return HCC_E_ARG;
  if (count != kMlpParams) {
    net->err = "parameter count must be HCC_MLP_PARAMS";
    return HCC_E_ARG;
  }
  MLP_BEGIN
  HCHECK(hipMemcpy(params, net->w, kMlpParams * sizeof(float), hipMemcpyDeviceToHost));
  MLP_END
}

int hcc_mlp_collect(hcc_mlp* net, hcc_ctx* ctx, int per_molecule, unsigned seed, long* added) {
  if (net == nullptr || ctx == nullptr || per_molecule < 1) return HCC_E_ARG;
  BatchView bv;
  if (!batch_view(ctx, &bv)) {
    net->err = "the context holds no solved molecules";
    return HCC_E_STATE;
  }
  if (bv.device != net->device) {
    net->err = "trainer and context are on different devices";
    return HCC_E_ARG;
  }
  const long nrow = (long)bv.nm * per_molecule;
  if (net->count + nrow > net->cap) {
    net->err = "sample capacity exceeded";
    return HCC_E_ARG;
  }
  MLP_BEGIN
  HCHECK(hipStreamSynchronize(bv.stream));
  mlp_overlaps(bv.dm, bv.rgNN, bv.nm, net->stream);
  const long blocks = (nrow + 255) / 256;
  hipLaunchKernelGGL(k_mlp_collect, dim3((unsigned)blocks), dim3(256), 0, net->stream, bv.dm, bv.dst, bv.nm,
                     per_molecule, seed, net->rows + net->count * kMlpRow, net->where + net->count * 2);
  HCHECK(hipGetLastError());
  HCHECK(hipStreamSynchronize(net->stream));
  net->count += nrow;
  if (added) *added = nrow;
  MLP_END
}

int hcc_mlp_samples(hcc_mlp* net, long* count) {
  if (net == nullptr || count == nullptr) return HCC_E_ARG;
  *count = net->count;
  return HCC_OK;
}

int hcc_mlp_read_samples(hcc_mlp* net, long first, long count, float* rows, int* where) {
  if (net == nullptr || first < 0 || count < 0 || first + count > net->count) return HCC_E_ARG;
  MLP_BEGIN
  if (rows && count)
    HCHECK(hipMemcpy(rows, net->rows + first * kMlpRow, count * kMlpRow * sizeof(float), hipMemcpyDeviceToHost));
  if (where && count)
    HCHECK(hipMemcpy(where, net->where + first * 2, count * 2 * sizeof(int), hipMemcpyDeviceToHost));
  MLP_END
}

int hcc_mlp_write_samples(hcc_mlp* net, const float* rows, long count) {
  if (net == nullptr || rows == nullptr || count < 0) return HCC_E_ARG;
  if (count > net->cap) {
    net->err = "sample capacity exceeded";
    return HCC_E_ARG;
  }
  MLP_BEGIN
  if (count) HCHECK(hipMemcpy(net->rows, rows, count * kMlpRow * sizeof(float), hipMemcpyHostToDevice));
  std::vector<int> wh((size_t)count * 2, -1);
  if (count) HCHECK(hipMemcpy(net->where, wh.data(), wh.size() * sizeof(int), hipMemcpyHostToDevice));
  net->count = count;
  MLP_END
}

int hcc_mlp_gradient(hcc_mlp* net, long first, int count, double* loss, float* grad) {
  if (net == nullptr || first < 0 || count < 1 || first + count > net->count) return HCC_E_ARG;
  MLP_BEGIN
  const int per = samples_per_block(count), blocks = (count + per - 1) / per;
  ensure_part(net, blocks);
  ensure_loss(net, blocks);
  batch_step(net, net->count, 1, 0, first, count, blocks, per, net->lossp, false, 0.f);
  std::vector<double> lp(blocks);
  HCHECK(hipMemcpyAsync(lp.data(), net->lossp, blocks * sizeof(double), hipMemcpyDeviceToHost, net->stream));
  if (grad) HCHECK(hipMemcpyAsync(grad, net->grad, kMlpParams * sizeof(float), hipMemcpyDeviceToHost, net->stream));
  HCHECK(hipStreamSynchronize(net->stream));
  if (loss) *loss = std::accumulate(lp.begin(), lp.end(), 0.0) / count;
  MLP_END
}

int hcc_mlp_train(hcc_mlp* net, int epochs, int batch, float lr, float lr_final, unsigned seed, double* epoch_loss) {
  if (net == nullptr || epochs < 1 || batch < 1 || !(lr > 0.f) || lr_final < 0.f) return HCC_E_ARG;
  if (net->count < 1) {
    net->err = "no training samples";
    return HCC_E_STATE;
  }
  MLP_BEGIN
  const long ns = net->count;
  const int nb = (int)std::min<long>(batch, ns);
  const long steps = (ns + nb - 1) / nb;
  const int per = samples_per_block(nb), bpb = (nb + per - 1) / per;
  ensure_part(net, bpb);
  ensure_loss(net, steps * bpb);
  const long total = steps * (long)epochs;
  std::vector<double> lp((size_t)steps * bpb);
  unsigned h = seed * 2654435761u + 12345u;
  for (int ep = 0; ep < epochs; ++ep) {
    // row permutation (q * pa + pc) mod ns with gcd(pa, ns) = 1
    h = h * 1664525u + 1013904223u;
    long pa = ns > 1 ? 1 + ((long)(0.6180339887 * ns) + (long)(h % 997u)) % (ns - 1) : 1;
    while (gcd_l(pa, ns) != 1) pa = pa + 1 < ns ? pa + 1 : 1;
    h = h * 1664525u + 1013904223u;
    const long pc = (long)(h % (unsigned long)ns);
    for (long k = 0; k < steps; ++k) {
      const long base = k * nb;
      const int cnt = (int)std::min<long>(nb, ns - base);
      const double frac = (double)(ep * steps + k) / (double)std::max<long>(1, total - 1);
      const float lrk = (float)(lr_final + 0.5 * (lr - lr_final) * (1.0 + std::cos(3.14159265358979 * frac)));
      batch_step(net, ns, pa, pc, base, cnt, bpb, per, net->lossp + k * bpb, true, lrk);
    }
    HCHECK(hipMemcpyAsync(lp.data(), net->lossp, lp.size() * sizeof(double), hipMemcpyDeviceToHost, net->stream));
    HCHECK(hipStreamSynchronize(net->stream));
    if (epoch_loss) epoch_loss[ep] = std::accumulate(lp.begin(), lp.end(), 0.0) / (double)ns;
  }
  MLP_END
}

int hcc_mlp_evaluate(hcc_mlp* net, double* loss) {
  if (net == nullptr || loss == nullptr) return HCC_E_ARG;
  if (net->count < 1) {
    net->err = "no samples";
    return HCC_E_STATE;
  }
  MLP_BEGIN
  const long ns = net->count;
  const long blocks = (ns + 255) / 256;
  ensure_loss(net, blocks);
  hipLaunchKernelGGL(k_mlp_forward, dim3((unsigned)blocks), dim3(256), 0, net->stream, net->w, net->rows, 0L, (int)ns,
                     net->lossp, (float*)nullptr);
  HCHECK(hipGetLastError());
  std::vector<double> lp(blocks);
  HCHECK(hipMemcpyAsync(lp.data(), net->lossp, blocks * sizeof(double), hipMemcpyDeviceToHost, net->stream));
  HCHECK(hipStreamSynchronize(net->stream));
  *loss = std::accumulate(lp.begin(), lp.end(), 0.0) / (double)ns;
  MLP_END
}

int hcc_mlp_predict(hcc_mlp* net, const float* features, long count, float* y) {
  if (net == nullptr || features == nullptr || y == nullptr || count < 1 || count > (1L << 30)) return HCC_E_ARG;
  MLP_BEGIN
  float* rows = nullptr;
  float* yd = nullptr;
  dalloc(&rows, (size_t)count * kMlpRow);
  dalloc(&yd, (size_t)count);
  std::vector<float> h((size_t)count * kMlpRow, 0.f);
  for (long r = 0; r < count; ++r)
    for (int q = 0; q < kMlpF; ++q) h[(size_t)r * kMlpRow + q] = features[(size_t)r * kMlpF + q];
  HCHECK(hipMemcpy(rows, h.data(), h.size() * sizeof(float), hipMemcpyHostToDevice));
  const long blocks = (count + 255) / 256;
  double* lp = nullptr;
  dalloc(&lp, (size_t)blocks);
  hipLaunchKernelGGL(k_mlp_forward, dim3((unsigned)blocks), dim3(256), 0, net->stream, net->w, rows, 0L, (int)count,
                     lp, yd);
  HCHECK(hipGetLastError());
  HCHECK(hipStreamSynchronize(net->stream));
  HCHECK(hipMemcpy(y, yd, count * sizeof(float), hipMemcpyDeviceToHost));
  HCHECK(hipFree(rows));
  HCHECK(hipFree(yd));
  HCHECK(hipFree(lp));
  MLP_END
}

}  // extern "C"

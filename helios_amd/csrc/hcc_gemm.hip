// Grouped composite-strided GEMM on CDNA4 matrix cores.
//
// One launch runs every problem of a table (one problem per molecule, or a
// single problem): C = alpha * A B + beta * C.  Work items are 64x64 output
// tiles; 256 threads (4 waves of 64) per tile, each wave owning a 32x32
// quadrant computed with 2x2 V_MFMA_F64_16X16X4_F64 blocks.  Operand tiles
// are staged through LDS (k-major), with the next k-slab prefetched into
// registers while the current one feeds the matrix cores.
//
// Tile -> workgroup mapping is XCD-aware: consecutive workgroups are spread
// round-robin over the 8 XCDs by the dispatcher, so workgroup b takes tile
// b / 8 of XCD b % 8's contiguous run (XcdMap), which keeps a molecule's tiles
// (which share operands) in one L2.
#include <type_traits>

#include "hcc_internal.h"

namespace hcc {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef double d2 __attribute__((ext_vector_type(2)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));

// Operand pointers arrive as generic pointers inside GemmProb; loads through
// them compile to FLAT instructions, which also count against the LDS
// counter, so waiting for the LDS fragment reads would wait for the next
// slab's prefetch as well.  Global-address-space views give GLOBAL loads that
// stay in flight across the matrix-core work of the current slab.
typedef __attribute__((address_space(1))) double gdouble;
__device__ __forceinline__ const gdouble* gptr(const double* p) { return (const gdouble*)p; }
__device__ __forceinline__ gdouble* gptr(double* p) { return (gdouble*)p; }

// Operand loads through buffer resources: a masked (padding) element uses a
// byte offset beyond the resource's range and reads 0 in hardware, so no
// select follows the load and nothing has to wait for it before the next
// slab's store to LDS.  Valid offsets stay below 2 GiB (the largest operand is
// far smaller).
constexpr int kRsrcBytes = 0x7ffffff0;
constexpr unsigned kPadByte = 0x80000000u;
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const double* p) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, kRsrcBytes, 0x00020000);
}
__device__ __forceinline__ double bload(__amdgpu_buffer_rsrc_t r, int byte_off) {
  return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, byte_off, 0, 0));
}
// 16 bytes at an 8-byte aligned offset
__device__ __forceinline__ d2 bload2(__amdgpu_buffer_rsrc_t r, int byte_off) {
  return __builtin_bit_cast(d2, __builtin_amdgcn_raw_buffer_load_b128(r, byte_off, 0, 0));
}
// r / radix for 0 <= r < kMaxIndex, 1 <= radix < kMaxRadix (exact, see Operand)
__device__ __forceinline__ int quot(int r, double inv) { return (int)(((double)r + 0.5) * inv); }
__device__ __forceinline__ int row_off(const Operand& o, int r) {
  const int q = quot(r, o.ir);
  return q * o.srh + (r - q * o.rr) * o.srl;
}
__device__ __forceinline__ int col_off(const Operand& o, int c) {
  const int q = quot(c, o.ic);
  return q * o.sch + (c - q * o.rc) * o.scl;
}
// the same for output rows and columns, which may run over pairs
__device__ __forceinline__ int out_row(const Operand& o, int r) {
  if (o.rr > 0) return row_off(o, r);
  int i, j;
  pair_of(r, -o.rr, i, j);
  return i * o.srh + j * o.srl;
}
__device__ __forceinline__ int out_col(const Operand& o, int c) {
  if (o.rc > 0) return col_off(o, c);
  int i, j;
  pair_of(c, -o.rc, i, j);
  return i * o.sch + j * o.scl;
}

// Problem owning global tile `tile`: one load from the table's tile map
// (a binary search over problems would be a chain of dependent loads).
__device__ __forceinline__ int find_problem(const int* __restrict__ tile_prob, int tile) {
  return tile_prob[tile];
}

// Position of tile lt of a problem of tiles_m x tiles_n tiles: bands of H tile
// rows, column by column within a band.  An XCD runs a contiguous range of lt,
// so the tiles it has in flight cover a block of about H x (in flight / H)
// and share that block's operand panels in its L2; row by row they would cover
// one or two full rows and stream all of B once per row.  Solves with rows
// and with bands: 100 sites (40 x 40 tiles of 64) 223 and 207 ms; 120 sites in
// mixed precision (29 x 29 tiles of 128 in the correction forms, where B's
// panels came from memory at 2.5 TB/s) 544 and 446 ms, correction levels included.
template <int H>
__device__ __forceinline__ void tile_pos(int lt, int tiles_m, int tiles_n, int& tm, int& tn) {
  const int band = lt / (H * tiles_n), r = lt - band * H * tiles_n, h = min(H, tiles_m - band * H);
  tn = r / h;
  tm = band * H + r - tn * h;
}
// band heights: the square root of the tiles an XCD's 32 CUs hold
constexpr int kBand64 = 12, kBand128 = 8;

// ---------------------------------------------------------------------------
// FP64 kernel: output tile BM x BN, 32x32 per wave (4 waves or 1), 16-deep K
// slabs staged through LDS.
//
// What bounds it: the matrix cores, and next to them the return path of the
// vector loads -- a 64-lane 8-byte load occupies it for 16 cycles, as long as
// a 16-byte one (31 and 62 bytes a cycle).  In a 100-site solve the matrix cores
// are busy 72 % of the kernel's cycles and the return path 64 % (with 8-byte
// loads and one launch per contraction 44 to 53 % and 41 to 62 %), over 512 ragged
// molecules 64 and 78 %.  So an operand is staged in 16-byte pairs along its
// unit-stride dimension wherever pairs exist (GemmProb::modes):
//   mode 0  pairs along K, staged [row][k];
//   mode 1  pairs along the rows (columns of B), staged [k][row];
//   mode 2  single elements, staged [k][row]: any strides.
// Pairs along K never straddle a run of an odd composite radix: K is
// enumerated with one padding element behind each such run (GemmProb::krun),
// and a pair whose second element is padding (bit 0 of its K-table entry)
// drops it.  Measured with single loads and with pairs, TF/s of 2 M N K: one
// 100-site molecule's 2500^3 contractions 42-50 and 45-53, its solve 313 and
// 287 ms; 512 ragged molecules of 10 to 48 sites 37-41 and 38-43, 316 and
// 305 ms (64 at 4096^3, where the last wave of tiles weighs little).  The
// register bound keeps the accumulators in VGPRs: with a larger budget the
// compiler moves them to AGPRs and back every slab.
//
// A wave in its matrix work has priority over those staging (100 sites: 4.04 and
// 3.96 ms for an iteration's contractions).
//
// Fragments are read from LDS 16 bytes at a time too: mode 0 gives a lane two
// consecutive K, used by the two halves of an 8-deep step (the K order within
// a step is free), modes 1 and 2 two consecutive rows, one for each of the
// wave's two 16-row blocks (bank conflicts 5 to 7 % of the cycles).
// ---------------------------------------------------------------------------
constexpr int kPk = kBK + 2;   // pitch of the [row][k] staging layout (16-byte aligned rows)

template <int BM, int BN>
struct F64Tile {
  static constexpr int kT = 64 * (BM / 32) * (BN / 32);
  // pitch of the [k][row] layout: == 16 (mod 32) doubles, so that the
  // fragment reads of neighbouring K fall in disjoint bank halves
  static constexpr int kPa = BM + 16;
  static constexpr int kPb = BN + 16;
  static constexpr int kLdsA = BM * kPk > kBK * kPa ? BM * kPk : kBK * kPa;
  static constexpr int kLdsB = BN * kPk > kBK * kPb ? BN * kPk : kBK * kPb;
  // K-offset table length (LDS) per chunk: small enough that the table does
  // not limit the workgroups per CU
  static constexpr int kKT = BM >= 64 ? 1024 : 512;
};

#define HCC_F64_THREADS(BM_, BN_) (64 * ((BM_) / 32) * ((BN_) / 32))

// staged pieces of thread t (of T) in an R-row x 16 slab: piece i is the pair
// or element at (row(t, i), k(t, i))
template <int MODE, int R, int T>
struct F64Stage {
  static constexpr int kN = (MODE == 2 ? R * kBK : R * kBK / 2) / T;   // pieces per thread
  static constexpr int kNK = MODE == 0 ? 1 : kN;                        // distinct K per thread
  static_assert(kN * T == (MODE == 2 ? R * kBK : R * kBK / 2) && T % 8 == 0, "staging covers the slab");
  static __device__ __forceinline__ int row(int t, int i) {
    return MODE == 0 ? t / 8 + (T / 8) * i : (MODE == 1 ? 2 * (t % (R / 2)) : t % R);
  }
  static __device__ __forceinline__ int k(int t, int i) {
    return MODE == 0 ? 2 * (t % 8) : (MODE == 1 ? t / (R / 2) + (2 * T / R) * i : t / R + (T / R) * i);
  }
};

// one tile of problem P: staging modes MA of A, MB of B
template <int BM, int BN, int MA, int MB>
__device__ __forceinline__ void gemm_f64_tile(const GemmProb& P, int lt, double* As, double* Bs, unsigned* koffA,
                                              unsigned* koffB) {
  using TL = F64Tile<BM, BN>;
  constexpr int T = TL::kT;
  using SA = F64Stage<MA, BM, T>;
  using SB = F64Stage<MB, BN, T>;
  const int tiles_n = (P.N + BN - 1) / BN, tiles_m = (P.M + BM - 1) / BM;
  const int ks = lt / (tiles_m * tiles_n);
  lt -= ks * tiles_m * tiles_n;
  int tm, tn;
  tile_pos<kBand64>(lt, tiles_m, tiles_n, tm, tn);
  const int m0 = tm * BM, n0 = tn * BN;
  const int kbeg = ks * P.kchunk;
  const int kend = min(P.kpad, kbeg + P.kchunk);
  const int t = threadIdx.x;
  const int lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int wm = (wave / (BN / 32)) * 32, wn = (wave % (BN / 32)) * 32;

  // fixed (non-K) byte offsets of this thread's staged pieces; kPadByte
  // marks padding, as it does in the K tables: every sum with one sentinel
  // lies past the resources (reads 0), a sum of two wraps to the operand's
  // first elements, whose products only reach padding rows or columns.  The
  // second element of a pair at an odd problem's last row is the next one in
  // memory (the arenas end in padding) and reaches a padding row only.
  unsigned fa[SA::kN], fb[SB::kN];
#pragma unroll
  for (int i = 0; i < SA::kN; ++i) {
    const int m = m0 + SA::row(t, i);
    fa[i] = m < P.M ? 8u * (unsigned)out_row(P.A, m) : kPadByte;
  }
#pragma unroll
  for (int i = 0; i < SB::kN; ++i) {
    const int n = n0 + SB::row(t, i);
    fb[i] = n < P.N ? 8u * (unsigned)out_col(P.B, n) : kPadByte;
  }
  const __amdgpu_buffer_rsrc_t rA = rsrc(P.A.p), rB = rsrc(P.B.p);
  d2 ra[SA::kN], rb[SB::kN];   // mode 2 uses the first element
  unsigned ca = 0, cb = 0;     // mode 0: bit 0 = the pair's second element is padding

  d4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = d4{0.0, 0.0, 0.0, 0.0};

  for (int c0 = kbeg; c0 < kend; c0 += TL::kKT) {
    const int clen = min(kend - c0, TL::kKT);
    __syncthreads();
    // K offsets of the chunk, with a slab of padding behind it for the last,
    // partial slab and the final prefetch
    for (int q = t; q < clen + 2 * kBK; q += T) {
      const int kp = c0 + q;
      const int hi = P.krun > 0 ? quot(kp, P.irun) : 0, lo = kp - hi * (P.krun + 1);
      const int k = kp - hi, run = P.krun > 0 ? P.krun : P.K;   // krun = 0: one run of K
      const bool in = q < clen && lo < run && k < P.K;
      const unsigned last = lo + 1 >= run ? 1u : 0u;
      koffA[q] = in ? 8u * (unsigned)col_off(P.A, k) | last : kPadByte;
      koffB[q] = in ? 8u * (unsigned)row_off(P.B, k) | last : kPadByte;
    }
    __syncthreads();
    auto load = [&](int kl0) {
      unsigned ka[SA::kNK], kb[SB::kNK];
#pragma unroll
      for (int i = 0; i < SA::kNK; ++i) ka[i] = koffA[kl0 + SA::k(t, i)];
#pragma unroll
      for (int i = 0; i < SB::kNK; ++i) kb[i] = koffB[kl0 + SB::k(t, i)];
      if (MA == 0) ca = ka[0];
      if (MB == 0) cb = kb[0];
#pragma unroll
      for (int i = 0; i < SA::kN; ++i) {
        const int off = (int)(fa[i] + (ka[MA == 0 ? 0 : i] & ~1u));
        if (MA == 2) ra[i][0] = bload(rA, off);
        else ra[i] = bload2(rA, off);
      }
#pragma unroll
      for (int i = 0; i < SB::kN; ++i) {
        const int off = (int)(fb[i] + (kb[MB == 0 ? 0 : i] & ~1u));
        if (MB == 2) rb[i][0] = bload(rB, off);
        else rb[i] = bload2(rB, off);
      }
    };
    load(0);
    for (int k0 = 0; k0 < clen; k0 += kBK) {
#pragma unroll
      for (int i = 0; i < SA::kN; ++i) {
        if (MA == 0) {
          if (ca & 1u) ra[i][1] = 0.0;
          *(d2*)&As[SA::row(t, i) * kPk + SA::k(t, i)] = ra[i];
        } else if (MA == 1) {
          *(d2*)&As[SA::k(t, i) * TL::kPa + SA::row(t, i)] = ra[i];
        } else {
          As[SA::k(t, i) * TL::kPa + SA::row(t, i)] = ra[i][0];
        }
      }
#pragma unroll
      for (int i = 0; i < SB::kN; ++i) {
        if (MB == 0) {
          if (cb & 1u) rb[i][1] = 0.0;
          *(d2*)&Bs[SB::row(t, i) * kPk + SB::k(t, i)] = rb[i];
        } else if (MB == 1) {
          *(d2*)&Bs[SB::k(t, i) * TL::kPb + SB::row(t, i)] = rb[i];
        } else {
          Bs[SB::k(t, i) * TL::kPb + SB::row(t, i)] = rb[i][0];
        }
      }
      __syncthreads();
      load(k0 + kBK);   // the last prefetch reads only padding
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int kk = 0; kk < kBK; kk += 8) {
        const int kg = kk + 2 * (lane >> 4), l = lane & 15;
        d2 a[2], b[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          a[i] = MA == 0 ? *(const d2*)&As[(wm + 16 * i + l) * kPk + kg] : *(const d2*)&As[(kg + i) * TL::kPa + wm + 2 * l];
          b[i] = MB == 0 ? *(const d2*)&Bs[(wn + 16 * i + l) * kPk + kg] : *(const d2*)&Bs[(kg + i) * TL::kPb + wn + 2 * l];
        }
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
              acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(MA == 0 ? a[i][h] : a[h][i], MB == 0 ? b[j][h] : b[h][j],
                                                               acc[i][j], 0, 0, 0);
      }
      __builtin_amdgcn_s_setprio(0);
      __syncthreads();
    }
  }

  // epilogue: for the FP64 MFMA, D[row][col] of a 16x16 block sits in lane
  // (col + 16*(row%4)), element row/4; modes 1 and 2 interleave the rows
  // (columns) of the two blocks
  gdouble* __restrict__ W = gptr(P.ksplit > 1 ? P.ws + (long)ks * P.M * P.N : P.C.p);
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int col = n0 + wn + (MB == 0 ? 16 * j + (lane & 15) : 2 * (lane & 15) + j);
    if (col >= P.N) continue;
    const int co = P.ksplit > 1 ? col : out_col(P.C, col);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int br = (lane >> 4) + 4 * r, row = m0 + wm + (MA == 0 ? 16 * i + br : 2 * br + i);
        if (row >= P.M) continue;
        if (P.ksplit > 1) {
          W[(long)row * P.N + co] = acc[i][j][r];
          continue;
        }
        const int o = out_row(P.C, row) + co;
        double v = P.alpha * acc[i][j][r];
        if (P.beta != 0.0) v += P.beta * W[o];
        W[o] = v;
      }
    }
  }
}

template <int BM, int BN>
__global__ __launch_bounds__(HCC_F64_THREADS(BM, BN)) __attribute__((amdgpu_waves_per_eu(BM == 64 ? 5 : 3))) void gemm_f64_kernel(const GemmProb* __restrict__ probs,
                                                                           const int* __restrict__ tile_prob,
                                                                           XcdMap xcd,
                                                                           const int* __restrict__ active) {
  using TL = F64Tile<BM, BN>;
  __shared__ __attribute__((aligned(16))) double As[TL::kLdsA];
  __shared__ __attribute__((aligned(16))) double Bs[TL::kLdsB];
  __shared__ unsigned koffA[TL::kKT + 2 * kBK];
  __shared__ unsigned koffB[TL::kKT + 2 * kBK];
  const int x = blockIdx.x & 7, tile = xcd.begin[x] + (int)(blockIdx.x >> 3);
  if (tile >= xcd.begin[x + 1]) return;
  const GemmProb P = probs[find_problem(tile_prob, tile)];
  if (active != nullptr && active[P.mol] == 0) return;
  const int lt = tile - P.tile_begin + P.lt0;
#define HCC_F64_TILE(MA, MB) \
  case 3 * MA + MB: gemm_f64_tile<BM, BN, MA, MB>(P, lt, As, Bs, koffA, koffB); break;
  switch (P.modes) {   // uniform over the workgroup
    HCC_F64_TILE(0, 0)
    HCC_F64_TILE(0, 1)
    HCC_F64_TILE(0, 2)
    HCC_F64_TILE(1, 0)
    HCC_F64_TILE(1, 1)
    HCC_F64_TILE(1, 2)
    HCC_F64_TILE(2, 0)
    HCC_F64_TILE(2, 1)
    HCC_F64_TILE(2, 2)
  }
#undef HCC_F64_TILE
}

// ---------------------------------------------------------------------------
// Correction-form ("dual") GEMM of the mixed-precision inner iterations:
//   C = alpha * (A0 dB + dA (B0 + dB)) + beta * C
// which is the change of A B between the outer point (A0, B0) and the current
// point (A0 + dA, B0 + dB), so with BF16 operands the rounding error is
// proportional to the size of the correction, not of A B.  FP64 form: 64x64
// tiles, 16-deep slabs; BF16 form below.
// ---------------------------------------------------------------------------
constexpr int kDualLds64 = 64 * kPk;   // [row][k] staging; [k][row] takes less
template <bool AKF, bool BNF>
__device__ __forceinline__ void gemm_dual_f64_tile(const GemmProb& P, int lt, double* A0s, double* dAs, double* dBs,
                                                   double* Bfs) {
  constexpr int BM = 64, BN = 64, T = 256, BK = 16, NE = 4;
  constexpr int kPa = BM + 2, kPb = BN + 2;
  static_assert(BK * kPa <= kDualLds64 && BK * kPb <= kDualLds64, "staging fits");
  const int tiles_n = (P.N + BN - 1) / BN, tiles_m = (P.M + BM - 1) / BM;
  const int ks = lt / (tiles_m * tiles_n);
  lt -= ks * tiles_m * tiles_n;
  int tm, tn;
  tile_pos<kBand64>(lt, tiles_m, tiles_n, tm, tn);
  const int m0 = tm * BM, n0 = tn * BN;
  const int kbeg = ks * P.kchunk, kend = min(P.K, kbeg + P.kchunk);
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
  const bool hasA = P.dA != nullptr, hasB = P.dB != nullptr;
  int fa[NE], fb[NE], kqa[NE], kqb[NE];
#pragma unroll
  for (int i = 0; i < NE; ++i) {
    const int q = t + i * T;
    const int m = m0 + (AKF ? q / BK : q % BM);
    kqa[i] = AKF ? q % BK : q / BM;
    fa[i] = m < P.M ? out_row(P.A, m) : -1;
    const int n = n0 + (BNF ? q % BN : q / BK);
    kqb[i] = BNF ? q / BN : q % BK;
    fb[i] = n < P.N ? out_col(P.B, n) : -1;
  }
  const gdouble* __restrict__ A0 = gptr(P.A.p);
  const float* __restrict__ dA = P.dA;
  const gdouble* __restrict__ B0 = gptr(P.B.p);
  const float* __restrict__ dB = P.dB;
  double ra0[NE], rda[NE], rdb[NE], rbf[NE];
  auto load = [&](int k0) {
#pragma unroll
    for (int i = 0; i < NE; ++i) {
      int k = k0 + kqa[i];
      bool ok = fa[i] >= 0 && k < kend;
      int o = ok ? fa[i] + col_off(P.A, k) : 0;
      const double a0 = A0[o], da = hasA ? (double)dA[o] : 0.0;
      ra0[i] = ok ? a0 : 0.0;
      rda[i] = (ok && hasA) ? da : 0.0;
      k = k0 + kqb[i];
      ok = fb[i] >= 0 && k < kend;
      o = ok ? fb[i] + row_off(P.B, k) : 0;
      const double b0 = B0[o], db = hasB ? (double)dB[o] : 0.0;
      rdb[i] = (ok && hasB) ? db : 0.0;
      rbf[i] = ok ? b0 + rdb[i] : 0.0;
    }
  };
  d4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = d4{0.0, 0.0, 0.0, 0.0};
  load(kbeg);
  for (int k0 = kbeg; k0 < kend; k0 += BK) {
#pragma unroll
    for (int i = 0; i < NE; ++i) {
      const int q = t + i * T;
      const int ia = AKF ? (q / BK) * kPk + q % BK : (q / BM) * kPa + q % BM;
      const int ib = BNF ? (q / BN) * kPb + q % BN : (q / BK) * kPk + q % BK;
      A0s[ia] = ra0[i];
      dAs[ia] = rda[i];
      dBs[ib] = rdb[i];
      Bfs[ib] = rbf[i];
    }
    __syncthreads();
    load(min(k0 + BK, kend));
#pragma unroll
    for (int kk = 0; kk < BK; kk += 4) {
      const int kr = kk + (lane >> 4);
      const int ma = wm + (lane & 15), nb = wn + (lane & 15);
      const int ia0 = AKF ? ma * kPk + kr : kr * kPa + ma;
      const int ia1 = AKF ? (ma + 16) * kPk + kr : kr * kPa + ma + 16;
      const int ib0 = BNF ? kr * kPb + nb : nb * kPk + kr;
      const int ib1 = BNF ? kr * kPb + nb + 16 : (nb + 16) * kPk + kr;
      const double a0 = A0s[ia0], a1 = A0s[ia1], e0 = dAs[ia0], e1 = dAs[ia1];
      const double b0 = dBs[ib0], b1 = dBs[ib1], f0 = Bfs[ib0], f1 = Bfs[ib1];
      acc[0][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b0, acc[0][0], 0, 0, 0);
      acc[0][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b1, acc[0][1], 0, 0, 0);
      acc[1][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b0, acc[1][0], 0, 0, 0);
      acc[1][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b1, acc[1][1], 0, 0, 0);
      acc[0][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(e0, f0, acc[0][0], 0, 0, 0);
      acc[0][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(e0, f1, acc[0][1], 0, 0, 0);
      acc[1][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(e1, f0, acc[1][0], 0, 0, 0);
      acc[1][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(e1, f1, acc[1][1], 0, 0, 0);
    }
    __syncthreads();
  }
  if (P.ksplit > 1) {
    gdouble* __restrict__ W = gptr(P.ws + (long)ks * P.M * P.N);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int col = n0 + wn + 16 * j + (lane & 15);
      if (col >= P.N) continue;
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int row = m0 + wm + 16 * i + (lane >> 4) + 4 * r;
          if (row < P.M) W[(long)row * P.N + col] = acc[i][j][r];
        }
    }
    return;
  }
  float* __restrict__ Cp = P.Cd;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int col = n0 + wn + 16 * j + (lane & 15);
    if (col >= P.N) continue;
    const int co = out_col(P.C, col);
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = m0 + wm + 16 * i + (lane >> 4) + 4 * r;
        if (row >= P.M) continue;
        const int o = out_row(P.C, row) + co;
        double v = P.alpha * acc[i][j][r];
        if (P.beta != 0.0) v += P.beta * Cp[o];
        Cp[o] = v;
      }
  }
}

__global__ __launch_bounds__(256) void gemm_dual_f64(const GemmProb* __restrict__ probs,
                                                     const int* __restrict__ tile_prob, XcdMap xcd,
                                                     const int* __restrict__ active) {
  __shared__ double A0s[kDualLds64], dAs[kDualLds64], dBs[kDualLds64], Bfs[kDualLds64];
  const int x = blockIdx.x & 7, tile = xcd.begin[x] + (int)(blockIdx.x >> 3);
  if (tile >= xcd.begin[x + 1]) return;
  const GemmProb P = probs[find_problem(tile_prob, tile)];
  if (active != nullptr && active[P.mol] == 0) return;
  const int lt = tile - P.tile_begin + P.lt0;
  switch (P.modes & 3) {   // uniform over the workgroup
    case 0: gemm_dual_f64_tile<false, false>(P, lt, A0s, dAs, dBs, Bfs); break;
    case 1: gemm_dual_f64_tile<true, false>(P, lt, A0s, dAs, dBs, Bfs); break;
    case 2: gemm_dual_f64_tile<false, true>(P, lt, A0s, dAs, dBs, Bfs); break;
    default: gemm_dual_f64_tile<true, true>(P, lt, A0s, dAs, dBs, Bfs); break;
  }
}

// HA / HB: the operand has a correction (dA / dB non-null for every problem
// of the table).  A constant A needs only A0 dB, a constant B only dA B0.
//
// Output tiles of 128, 64 or 32 square, 32-deep K slabs.  Staging bounds this
// kernel (the matrix cores need 16 instructions per slab and wave): LDS stores
// and fragment reads first, then the return path of the loads, so elements
// move four at a time:
//  * an operand that is contiguous along K is loaded in quads of K, 16 bytes
//    of the FP32 correction and the 12 bytes around 4 BF16 values (which start
//    at any even byte), lanes along K (KC);
//  * any other operand is loaded one element per lane, the lanes along its
//    rows, four consecutive K per thread;
//  * both store four consecutive K of a row to LDS as 8 bytes.
// A quad never straddles a run of an operand's composite K: K is enumerated
// with every run padded to a multiple of four (GemmProb::krun), and the K
// table's low two bits hold how many of a quad's elements are padding.
// Offsets are row + K-table entry with no compare or select: a padding row or K
// carries the sentinel kPad, and any sum that includes it lies past the end of
// the resources (which read 0).  Measured with single elements (16-bit LDS
// stores along K) and with quads: a 3600^3 correction with both operands
// contiguous along K 346 and 285 us for one product, 558 and 520 us for two;
// 512 ragged molecules' 406 and 336, 439 and 362 us; solves of 2048 ragged
// molecules 796 and 761 ms, of 120 sites 326 and 318 ms.  What remains is the
// latency of a slab (two barriers, 12 to 16 waves a CU): of the 128 x 128 tiles'
// cycles in a 120-site solve, matrix cores 15 %, load return 80 %, LDS conflicts
// 18 %; a conflict-free permuted LDS layout measured equal.
constexpr unsigned kPad = 1u << 29;   // 4 x (element index) of a padding row or K
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc_h(const void* p, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, bytes, 0x00020000);
}
// staged group i of thread t (of T) in an R-row slab: four consecutive K from
// k(t, i) of row(t, i)
template <bool KC, int R, int T>
struct DualStage {
  static constexpr int kN = R * 8 / T;
  static __device__ __forceinline__ int row(int t, int i) { return KC ? t / 8 + (T / 8) * i : t % R; }
  static __device__ __forceinline__ int k(int t, int i) { return KC ? 4 * (t % 8) : 4 * (t / R) + (4 * T / R) * i; }
};
constexpr int kDualBK = 32;   // 64-deep slabs measured slower (K padding of the short contractions, fewer waves)
constexpr int kDualLD = kDualBK + 8;   // LDS pitch of a staged row
constexpr int kDualKT = 512;           // K-table chunk
typedef unsigned u2v __attribute__((ext_vector_type(2)));
typedef unsigned u3v __attribute__((ext_vector_type(3)));
typedef unsigned u4v __attribute__((ext_vector_type(4)));
typedef __bf16 bf4 __attribute__((ext_vector_type(4)));

// One operand's staging: X0 (BF16 copy of the outer point, loaded with LX0)
// and the correction dX (FP32, loaded with LDX)
template <bool KC, bool LX0, bool LDX, int R, int T>
struct DualOperand {
  using S = DualStage<KC, R, T>;
  static constexpr int N = S::kN;
  __amdgpu_buffer_rsrc_t r0, rd;
  unsigned f[KC ? N : 1];   // 4 x row offsets
  unsigned q0[N][KC ? 3 : 4];
  f4 qd[N];
  unsigned pad, sh[KC ? N : 1];   // KC: padding elements of the quad, byte shift of its BF16 values
  unsigned odd;                   // KC: byte distance of the BF16 block from the dword before it
  __device__ __forceinline__ void bind(const __bf16* x0, const float* dx) {
    odd = KC ? (unsigned)(reinterpret_cast<unsigned long>(x0) & 2u) : 0u;
    r0 = rsrc_h(reinterpret_cast<const char*>(x0) - odd, 1 << 28);
    rd = rsrc_h(dx, 1 << 29);
  }
  __device__ __forceinline__ void load(const unsigned* koff, int kl0, int t) {
    if (KC) {
      const unsigned e = koff[kl0 + S::k(t, 0)];
      pad = e & 3u;
#pragma unroll
      for (int i = 0; i < N; ++i) {
        const unsigned o = f[i] + (e & ~3u);
        if (LX0) {
          const unsigned h = (o >> 1) + odd;
          const u3v w = __builtin_amdgcn_raw_buffer_load_b96(r0, (int)(h & ~3u), 0, 0);
          q0[i][0] = w[0], q0[i][1] = w[1], q0[i][2] = w[2];
          sh[i] = h & 2u;
        }
        if (LDX) qd[i] = __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(rd, (int)o, 0, 0));
      }
    } else {
#pragma unroll
      for (int i = 0; i < N; ++i) {
        const u4v e = *reinterpret_cast<const u4v*>(&koff[kl0 + S::k(t, i)]);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const unsigned o = f[0] + e[j];
          if (LX0) q0[i][j] = (unsigned short)__builtin_amdgcn_raw_buffer_load_b16(r0, (int)(o >> 1), 0, 0);
          if (LDX) qd[i][j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rd, (int)o, 0, 0));
        }
      }
    }
  }
  // 4 BF16 values of X0
  __device__ __forceinline__ u2v x0(int i) const {
    if (KC)
      return u2v{__builtin_amdgcn_alignbyte(q0[i][1], q0[i][0], sh[i]), __builtin_amdgcn_alignbyte(q0[i][2], q0[i][1], sh[i])};
    return u2v{q0[i][0] | (q0[i][1] << 16), q0[i][2] | (q0[i][3] << 16)};
  }
  static __device__ __forceinline__ u2v round(f4 x) { return __builtin_bit_cast(u2v, __builtin_convertvector(x, bf4)); }
  // X0 + dX (X0 alone for a constant operand), rounded once
  __device__ __forceinline__ u2v sum(int i) const {
    const u2v b = x0(i);
    if (!LDX) return b;
    f4 x;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const unsigned u = KC ? (j & 1 ? b[j / 2] & 0xffff0000u : b[j / 2] << 16) : q0[i][j] << 16;
      x[j] = __builtin_bit_cast(float, u) + qd[i][j];
    }
    return round(x);
  }
  __device__ __forceinline__ void store(__bf16* lds, int t, int i, u2v v) const {
    if (KC) {
      v[0] &= pad == 3 ? 0xffffu : ~0u;
      v[1] &= pad == 0 ? ~0u : (pad == 1 ? 0xffffu : 0u);
    }
    *reinterpret_cast<u2v*>(&lds[S::row(t, i) * kDualLD + S::k(t, i)]) = v;
  }
};

// TS: output tile edge, 32 (2 waves of 32x16), 64 (4 waves of 32x32) or 128
// (8 waves of 32x64).  SK (short K, at most two slabs): the next slab is loaded
// after the current one's matrix-core work instead of during it; the staging
// registers are then dead during that work, which lets more waves share a SIMD
// (a one- or two-slab tile is mostly fixed latency, hidden by more tiles per CU)
template <bool KA, bool KB, bool HA, bool HB, int TS, bool SK>
__device__ __forceinline__ void gemm_dual_tile(const GemmProb& P, int lt, __bf16* A0s, __bf16* dAs, __bf16* dBs,
                                               __bf16* Bfs, unsigned* koffA, unsigned* koffB) {
  constexpr int BK = kDualBK, BM = TS, BN = TS, T = TS * 4, LD = kDualLD;
  constexpr int FM = 2, FN = TS / 32;   // 16x16 blocks per wave along M and N
  constexpr int KT = kDualKT;
  const int tiles_n = (P.N + BN - 1) / BN, tiles_m = (P.M + BM - 1) / BM;
  const int ks = lt / (tiles_m * tiles_n);
  lt -= ks * tiles_m * tiles_n;
  int tm, tn;
  tile_pos<TS == 128 ? kBand128 : kBand64>(lt, tiles_m, tiles_n, tm, tn);
  const int m0 = tm * BM, n0 = tn * BN;
  const int kbeg = ks * P.kchunk, kend = min(P.kpad, kbeg + P.kchunk);
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  // waves: 2 along N (32 FN columns each), T / 128 along M (32 rows each)
  const int wm = (wave >> 1) * 32, wn = (wave & 1) * (16 * FN);
  // A0 dB needs A0 and dB (HB), dA (B0 + dB) needs dA and B0 (HA); BF16
  // resources of 2^28 bytes, FP32 of 2^29 (valid element indices stay below
  // 2^27, checked by the host)
  using OA = DualOperand<KA, HB, HA, BM, T>;
  using OB = DualOperand<KB, HA, HB, BN, T>;
  OA A;
  OB B;
  A.bind(P.hA, HA ? P.dA : nullptr);
  B.bind(P.hB, HB ? P.dB : nullptr);
#pragma unroll
  for (int i = 0; i < (KA ? OA::N : 1); ++i) {
    const int m = m0 + OA::S::row(t, i);
    A.f[i] = m < P.M ? 4u * (unsigned)out_row(P.A, m) : kPad;
  }
#pragma unroll
  for (int i = 0; i < (KB ? OB::N : 1); ++i) {
    const int n = n0 + OB::S::row(t, i);
    B.f[i] = n < P.N ? 4u * (unsigned)out_col(P.B, n) : kPad;
  }
  f4 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = f4{0.f, 0.f, 0.f, 0.f};
  const int run = P.krun > 0 ? P.krun : P.K, runp = (P.krun + 3) & ~3;   // krun = 0: one run of K
  for (int c0 = kbeg; c0 < kend; c0 += KT) {
    const int clen = min(kend - c0, KT);
    __syncthreads();
    // 4 x K offsets of the chunk; entries past its end (read by the last,
    // partial slab and the final prefetch) carry kPad
    for (int q = t; q < KT + BK; q += T) {
      const int kp = c0 + q, hi = P.krun > 0 ? quot(kp, P.irun) : 0, lo = kp - hi * runp, k = hi * P.krun + lo;
      const bool in = q < clen && lo < run && k < P.K;
      const unsigned pad = (unsigned)max(0, 4 - (run - lo));
      koffA[q] = in ? 4u * (unsigned)col_off(P.A, k) | (KA ? pad : 0u) : kPad;
      koffB[q] = in ? 4u * (unsigned)row_off(P.B, k) | (KB ? pad : 0u) : kPad;
    }
    __syncthreads();
    auto load = [&](int kl0) {
      A.load(koffA, kl0, t);
      B.load(koffB, kl0, t);
    };
    load(0);
    for (int kl = 0; kl < clen; kl += BK) {
#pragma unroll
      for (int i = 0; i < OA::N; ++i) {
        if (HB) A.store(A0s, t, i, A.x0(i));
        if (HA) A.store(dAs, t, i, OA::round(A.qd[i]));
      }
#pragma unroll
      for (int i = 0; i < OB::N; ++i) {
        if (HB) B.store(dBs, t, i, OB::round(B.qd[i]));
        if (HA) B.store(Bfs, t, i, B.sum(i));
      }
      __syncthreads();
      if (!SK) load(kl + BK);   // the last prefetch reads only padding
      const int kq = 8 * (lane >> 4);
      // product with A from Xa, B from Xb (LDS [row][k])
      auto product = [&](const __bf16* Xa, const __bf16* Xb) {
        bf8 a[FM], b[FN];
#pragma unroll
        for (int f = 0; f < FM; ++f) a[f] = *reinterpret_cast<const bf8*>(&Xa[(wm + 16 * f + (lane & 15)) * LD + kq]);
#pragma unroll
        for (int f = 0; f < FN; ++f) b[f] = *reinterpret_cast<const bf8*>(&Xb[(wn + 16 * f + (lane & 15)) * LD + kq]);
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int j = 0; j < FN; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
      };
      if (HB) product(A0s, dBs);
      if (HA) product(dAs, Bfs);
      __syncthreads();
      if (SK && kl + BK < clen) load(kl + BK);
    }
  }
  // epilogue: V_MFMA_F32_16X16X32_BF16 leaves D[row][col] of a 16x16 block in
  // lane col + 16 (row / 4), element row % 4
  if (P.ksplit > 1) {
    double* __restrict__ W = P.ws + (long)ks * P.M * P.N;
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      const int col = n0 + wn + 16 * j + (lane & 15);
      if (col >= P.N) continue;
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int row = m0 + wm + 16 * i + 4 * (lane >> 4) + r;
          if (row < P.M) W[(long)row * P.N + col] = (double)acc[i][j][r];
        }
    }
    return;
  }
  float* __restrict__ Cp = P.Cd;
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    const int col = n0 + wn + 16 * j + (lane & 15);
    if (col >= P.N) continue;
    const int co = out_col(P.C, col);
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = m0 + wm + 16 * i + 4 * (lane >> 4) + r;
        if (row >= P.M) continue;
        const int o = out_row(P.C, row) + co;
        double v = P.alpha * (double)acc[i][j][r];
        if (P.beta != 0.0) v += P.beta * Cp[o];
        Cp[o] = v;
      }
  }
}

// One launch per tile kind runs problems of every layout and operand kind
// (GemmProb::modes, uniform over a workgroup).
template <int TS, bool SK>
__global__ __launch_bounds__(TS * 4) __attribute__((amdgpu_waves_per_eu(SK ? 6 : 4, 8))) void gemm_dual_bf16(
    const GemmProb* __restrict__ probs, const int* __restrict__ tile_prob, XcdMap xcd,
    const int* __restrict__ active) {
  __shared__ __attribute__((aligned(16))) __bf16 A0s[TS * kDualLD];
  __shared__ __attribute__((aligned(16))) __bf16 dAs[TS * kDualLD];
  __shared__ __attribute__((aligned(16))) __bf16 dBs[TS * kDualLD];
  __shared__ __attribute__((aligned(16))) __bf16 Bfs[TS * kDualLD];
  __shared__ __attribute__((aligned(16))) unsigned koffA[kDualKT + kDualBK];
  __shared__ __attribute__((aligned(16))) unsigned koffB[kDualKT + kDualBK];
  const int x = blockIdx.x & 7, tile = xcd.begin[x] + (int)(blockIdx.x >> 3);
  if (tile >= xcd.begin[x + 1]) return;
  const GemmProb P = probs[find_problem(tile_prob, tile)];
  if (active != nullptr && active[P.mol] == 0) return;
  const int lt = tile - P.tile_begin + P.lt0;
#define HCC_DUAL_TILE(AK, BN, HA, HB) \
  case AK + 2 * BN + 4 * HA + 8 * HB: gemm_dual_tile<AK, !BN, HA, HB, TS, SK>(P, lt, A0s, dAs, dBs, Bfs, koffA, koffB); break;
#define HCC_DUAL_LAYOUTS(HA, HB) \
  HCC_DUAL_TILE(0, 0, HA, HB) HCC_DUAL_TILE(1, 0, HA, HB) HCC_DUAL_TILE(0, 1, HA, HB) HCC_DUAL_TILE(1, 1, HA, HB)
  switch (P.modes) {
    HCC_DUAL_LAYOUTS(1, 0)
    HCC_DUAL_LAYOUTS(0, 1)
    HCC_DUAL_LAYOUTS(1, 1)
  }
#undef HCC_DUAL_LAYOUTS
#undef HCC_DUAL_TILE
}

static int longest_run(const XcdMap& xcd) {
  int longest = 0;
  for (int x = 0; x < 8; ++x) longest = longest > xcd.begin[x + 1] - xcd.begin[x] ? longest : xcd.begin[x + 1] - xcd.begin[x];
  return longest;
}

template <int TS, bool SK>
static void launch_dual(const GemmProb* probs, const int* tp, const XcdMap& xcd, const int* active, hipStream_t s) {
  hipLaunchKernelGGL((gemm_dual_bf16<TS, SK>), dim3(8 * longest_run(xcd)), dim3(4 * TS), 0, s, probs, tp, xcd, active);
}

hipError_t launch_gemm_dual(const GemmProb* probs, const int* tp, const XcdMap& xcd, const int* active, hipStream_t s,
                            bool bf16, int tile, bool short_k) {
  if (longest_run(xcd) <= 0) return hipSuccess;
  if (!bf16) {
    if (tile != 64) return hipErrorInvalidValue;
    hipLaunchKernelGGL(gemm_dual_f64, dim3(8 * longest_run(xcd)), dim3(256), 0, s, probs, tp, xcd, active);
  } else if (tile == 64) {
    if (short_k) launch_dual<64, true>(probs, tp, xcd, active, s);
    else launch_dual<64, false>(probs, tp, xcd, active, s);
  } else if (tile == 32) {
    if (short_k) launch_dual<32, true>(probs, tp, xcd, active, s);
    else launch_dual<32, false>(probs, tp, xcd, active, s);
  } else if (tile == 256) {
    launch_dual<128, false>(probs, tp, xcd, active, s);
  } else {
    return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

// fixed-order sum of the split-K partials into C
__global__ __launch_bounds__(256) void splitk_reduce_kernel(const GemmProb* __restrict__ probs,
                                                            const int* __restrict__ prefix,
                                                            const int* __restrict__ block_prob,
                                                            const int* __restrict__ active) {
  const int b = blockIdx.x;
  const int lo = block_prob[b];
  const GemmProb& P = probs[lo];
  if (P.ksplit <= 1) return;
  if (active != nullptr && active[P.mol] == 0) return;
  const long e = (long)(b - prefix[lo]) * 256 + threadIdx.x;
  const long mn = (long)P.M * P.N;
  if (e >= mn) return;
  const int row = e / P.N, col = e % P.N;
  // the adds are a chain; the loads of 16 partials are in flight together (one
  // load at a time: 53 us for the 211 partials of a 120-site molecule's thin
  // contractions, 13 us so)
  const gdouble* __restrict__ W = gptr((const double*)P.ws) + e;
  constexpr int kBatch = 16;
  double s = 0.0;
  for (int k0 = 0; k0 < P.ksplit; k0 += kBatch) {
    double part[kBatch];
#pragma unroll
    for (int k = 0; k < kBatch; ++k) part[k] = k0 + k < P.ksplit ? W[(k0 + k) * mn] : 0.0;
#pragma unroll
    for (int k = 0; k < kBatch; ++k) s += part[k];
  }
  const int o = out_row(P.C, row) + out_col(P.C, col);
  double v = P.alpha * s;
  if (P.Cd != nullptr) {   // FP32 correction output
    if (P.beta != 0.0) v += P.beta * P.Cd[o];
    P.Cd[o] = (float)v;
    return;
  }
  if (P.beta != 0.0) v += P.beta * P.C.p[o];
  P.C.p[o] = v;
}

hipError_t launch_splitk_reduce(const GemmProb* probs, const int* prefix, const int* block_prob, int nblocks,
                                const int* active, hipStream_t s) {
  if (nblocks <= 0) return hipSuccess;
  hipLaunchKernelGGL(splitk_reduce_kernel, dim3(nblocks), dim3(256), 0, s, probs, prefix, block_prob, active);
  return hipGetLastError();
}

// Compacted table: dst[i] = src[idx[i]] with tile_begin = tbeg[i] (the live
// problems of a table, their tiles renumbered consecutively)
__global__ __launch_bounds__(256) void k_compact_probs(const GemmProb* __restrict__ src, const int* __restrict__ idx,
                                                       const int* __restrict__ tbeg, int n, GemmProb* __restrict__ dst) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  GemmProb p = src[idx[i]];
  p.tile_begin = tbeg[i];
  dst[i] = p;
}

// out[x] = i with prefix[i] <= x < prefix[i + 1] (prefix: n + 1 ascending entries)
__global__ __launch_bounds__(256) void k_expand_prefix(const int* __restrict__ prefix, int n, int* __restrict__ out,
                                                       int total) {
  const int x = blockIdx.x * blockDim.x + threadIdx.x;
  if (x >= total) return;
  int lo = 0, hi = n - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (prefix[mid] <= x) lo = mid; else hi = mid - 1;
  }
  out[x] = lo;
}

hipError_t launch_expand_prefix(const int* prefix, int n, int* out, int total, hipStream_t s) {
  if (total > 0) hipLaunchKernelGGL(k_expand_prefix, dim3((total + 255) / 256), dim3(256), 0, s, prefix, n, out, total);
  return hipGetLastError();
}

hipError_t launch_compact_table(const GemmProb* src, const int* idx, const int* tbeg, const int* rpre, int n,
                                int tiles, int red, GemmProb* dst, int* tile_prob, int* red_bprob, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_compact_probs, dim3((n + 255) / 256), dim3(256), 0, s, src, idx, tbeg, n, dst);
  if (tiles > 0) hipLaunchKernelGGL(k_expand_prefix, dim3((tiles + 255) / 256), dim3(256), 0, s, tbeg, n, tile_prob, tiles);
  if (red > 0) hipLaunchKernelGGL(k_expand_prefix, dim3((red + 255) / 256), dim3(256), 0, s, rpre, n, red_bprob, red);
  return hipGetLastError();
}

void set_f64_modes(GemmProb& p) {
  const int ra = one_run_cols(p.A) ? 0 : p.A.rc, rb = one_run_rows(p.B) ? 0 : p.B.rr;   // runs along K
  int ma = unit_cols(p.A) ? 0 : (unit_rows(p.A) && (one_run_rows(p.A) || (p.A.rr > 0 && p.A.rr % 2 == 0)) ? 1 : 2);
  int mb = unit_cols(p.B) ? (one_run_cols(p.B) || (p.B.rc > 0 && p.B.rc % 2 == 0) ? 1 : 2) : (unit_rows(p.B) ? 0 : 2);
  // a padded enumeration for one operand's odd runs shifts the other's pairs
  // against its own runs unless they are the same
  p.krun = 0;
  if (ma == 0 && ra % 2 == 1) p.krun = ra;
  if (mb == 0 && rb > 0 && p.krun > 0 && rb != p.krun) mb = 2;
  if (mb == 0 && rb % 2 == 1 && p.krun == 0) {
    p.krun = rb;
    if (ma == 0 && ra > 0) ma = 2;
  }
  p.modes = 3 * ma + mb;
  p.kpad = p.krun > 0 ? p.K + p.K / p.krun : p.K;
  p.irun = 1.0 / (p.krun + 1);
}

void set_dual_modes(GemmProb& p, bool bf16) {
  const bool ka = unit_cols(p.A) || !unit_rows(p.A), kb = !unit_cols(p.B) && unit_rows(p.B);
  p.krun = 0;
  p.kpad = p.K;
  int qa = ka, qb = kb;
  if (bf16) {
    // quads along K need unit stride; runs along K (0: one run)
    const int ra = one_run_cols(p.A) ? 0 : p.A.rc, rb = one_run_rows(p.B) ? 0 : p.B.rr;
    qa = qa && unit_cols(p.A);
    // padding one operand's runs shifts the other's quads against its own runs
    // unless they are the same
    if (qa && ra % 4 != 0) p.krun = ra;
    if (qb && rb > 0 && p.krun > 0 && rb != p.krun) qb = 0;
    if (qb && rb % 4 != 0 && p.krun == 0) {
      p.krun = rb;
      if (ra > 0) qa = 0;
    }
    const int runp = (p.krun + 3) / 4 * 4;
    if (p.krun > 0) p.kpad = p.K / p.krun * runp + p.K % p.krun;
    p.irun = p.krun > 0 ? 1.0 / runp : 0.0;
  }
  p.modes = qa | (!qb << 1) | ((p.dA != nullptr) << 2) | ((p.dB != nullptr) << 3);
}

template <int BM, int BN>
static void launch_f64(const GemmProb* probs, const int* tp, const XcdMap& xcd, const int* active, hipStream_t s) {
  hipLaunchKernelGGL((gemm_f64_kernel<BM, BN>), dim3(8 * longest_run(xcd)), dim3(HCC_F64_THREADS(BM, BN)), 0, s, probs, tp, xcd,
                     active);
}

hipError_t launch_gemm_f64(const GemmProb* probs, const int* tile_prob, const XcdMap& xcd, const int* active,
                           hipStream_t s, int tile) {
  if (longest_run(xcd) <= 0) return hipSuccess;
  if (tile == 32) launch_f64<32, 32>(probs, tile_prob, xcd, active, s);
  else if (tile == 128) launch_f64<128, 32>(probs, tile_prob, xcd, active, s);
  else launch_f64<64, 64>(probs, tile_prob, xcd, active, s);
  return hipGetLastError();
}

}  // namespace hcc

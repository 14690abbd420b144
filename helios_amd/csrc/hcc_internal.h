// Internal declarations of libhelios_ccsd (not part of the C ABI).
//
// Layout conventions (all device arrays row-major, one molecule after another
// in per-buffer arenas):
//   C[mu][p]        MO coefficients, column p = MO p (occupied first)
//   t1[i][a]        o x v
//   t2[i][j][a][b]  o*o*v*v, pair-symmetric: t2[i][j][a][b] == t2[j][i][b][a]
//
// A GEMM operand is addressed through "composite" indices: a row (or column)
// index r is split as r = hi * radix + lo and the element offset is
// hi * s_hi + lo * s_lo.  With one composite index per dimension every
// permuted tensor contraction of the T1-dressed CCSD residual becomes a plain
// GEMM with no transposition pass.
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>

namespace hcc {

// HIP failure inside the library; the C ABI turns it into HCC_E_HIP
struct HipError {
  hipError_t e;
  const char* what;
};

#define HCHECK(x)                                        \
  do {                                                   \
    hipError_t e_ = (x);                                 \
    if (e_ != hipSuccess) throw HipError{e_, #x};        \
  } while (0)

struct Operand {
  double* p;        // base of this molecule's block
  int rr, rc;       // radices of the row and column composite indices (1 .. kMaxRadix)
  int srh, srl;     // row offset = (r / rr) * srh + (r % rr) * srl
  int sch, scl;     // col offset = (c / rc) * sch + (c % rc) * scl
  double ir, ic;    // 1 / rr and 1 / rc (FP64, round to nearest)
};
// Composite indices stay below kMaxIndex and radices below kMaxRadix, so the
// kernels' quotient floor((r + 1/2) * (1 / radix)) is exact: (r + 1/2) / radix
// lies at least 2^-17 from an integer, the FP64 rounding error is below 2^-25.
constexpr int kMaxRadix = 1 << 16;
constexpr int kMaxIndex = 1 << 27;
// A negative rr (rc) = -o enumerates rows (columns) over the pairs (i, j),
// i <= j < o, in row-major order instead: offset = i * srh + j * srl.
__device__ __forceinline__ void pair_of(int r, int o, int& i, int& j) {
  const int s = o * (o + 1) / 2 - 1 - r;   // counted from the last pair: h full rows of 1 .. h pairs behind it
  int h = (int)((sqrtf(8.f * (float)s + 1.f) - 1.f) * 0.5f);   // off by at most one (s < 2^27)
  if (h * (h + 1) / 2 > s) --h;
  if ((h + 1) * (h + 2) / 2 <= s) ++h;
  i = o - 1 - h;
  j = o - 1 - (s - h * (h + 1) / 2);
}
inline Operand make_operand(double* p, int rr, int rc, int srh, int srl, int sch, int scl) {
  return Operand{p, rr, rc, srh, srl, sch, scl, 1.0 / rr, 1.0 / rc};
}

// the unit stride of an operand's columns or rows, and whether that dimension
// is one contiguous run (else it comes in runs of its radix)
inline bool unit_cols(const Operand& o) { return (o.rc == 1 ? o.sch : o.scl) == 1; }
inline bool unit_rows(const Operand& o) { return (o.rr == 1 ? o.srh : o.srl) == 1; }
inline bool one_run_cols(const Operand& o) { return o.rc == 1 || o.sch == o.rc; }
inline bool one_run_rows(const Operand& o) { return o.rr == 1 || o.srh == o.rr; }

struct GemmProb {
  Operand A, B, C;  // A: M x K, B: K x N, C: M x N
  int M, N, K;
  double alpha, beta;
  int tile_begin;   // first global tile of this problem (of this part of it)
  int lt0;          // a problem spread over the XCDs: first tile of this part
  int mol;          // molecule index (for the active mask)
  int ksplit;       // number of K chunks (1: no split)
  int kchunk;       // K range of one chunk (multiple of the K tile), in kpad's enumeration
  // staging modes: FP64 kernel, 3 MA + MB (see gemm_f64_kernel); correction
  // kernels, A along K | B along its columns << 1 | (dA != 0) << 2 | (dB != 0) << 3.
  // K is enumerated with padding behind every run of krun (0: no such runs): one
  // element in the FP64 kernel, up to a multiple of 4 in the BF16 one; kpad
  // elements long, irun = 1 / (padded run)
  int modes;
  int krun, kpad;
  double irun;
  double* ws;       // split-K partials: ksplit x M x N, row-major (ksplit > 1)
  // correction ("delta") form, used by the mixed-precision inner iterations:
  // Cd += alpha * (A0 dB + dA (B0 + dB)) with A0 = A.p, B0 = B.p and the FP32
  // corrections dA, dB, Cd (Cd at C's offsets); a null dA or dB marks an
  // operand that does not change with the amplitudes
  const float* dA;
  const float* dB;
  float* Cd;
  // BF16 copies of A0 and B0 (same element offsets), refreshed at every outer
  // point; the BF16 correction kernel reads A0 and B0 from them
  const __bf16* hA;
  const __bf16* hB;
};

// Tile shape of the FP64 MFMA GEMM.
constexpr int kBM = 64, kBN = 64, kBK = 16, kThreads = 256;

// tiles [begin[x], begin[x + 1]) of a table run on XCD x
struct XcdMap {
  int begin[9];
};

// launches one grouped GEMM over all problems of a table (device memory)
// tile: 64 (64x64 tiles, 256 threads), 32 (32x32 tiles, 64 threads) or 128
// (128x32 tiles, 256 threads, for outputs at most 32 columns wide);
// tile_prob: problem index of every global tile of the table
hipError_t launch_gemm_f64(const GemmProb* probs, const int* tile_prob, const XcdMap& xcd,
                           const int* active, hipStream_t s, int tile = 64);
// staging modes and K enumeration of a problem for the FP64 kernel
void set_f64_modes(GemmProb& p);
// the same for a correction-form problem on the BF16 (or the FP64) kernel
void set_dual_modes(GemmProb& p, bool bf16);
// correction-form GEMM (see GemmProb::dA/dB); bf16 = 1 rounds the operands to
// BF16 for V_MFMA_F32_16X16X32_BF16 (FP32 accumulation; tile kinds 32, 64 and
// 256 = 128x128 output tiles), 0 keeps FP64 (tile kind 64 only)
// short_k: no problem has K above 64 (a variant with more waves in flight)
hipError_t launch_gemm_dual(const GemmProb* probs, const int* tile_prob, const XcdMap& xcd, const int* active,
                            hipStream_t s, bool bf16, int tile, bool short_k);
// C = alpha * sum_k ws_k + beta * C for the split problems of a table;
// prefix: block prefix over the table's problems (256 elements per block),
// block_prob: problem index of every reduction block
hipError_t launch_splitk_reduce(const GemmProb* probs, const int* prefix, const int* block_prob, int nblocks,
                                const int* active, hipStream_t s);

// out[x] = i with prefix[i] <= x < prefix[i + 1] for x < total (prefix: n + 1
// ascending entries; zero-length ranges are never chosen for a valid x)
hipError_t launch_expand_prefix(const int* prefix, int n, int* out, int total, hipStream_t s);
// Compacts a table to its live problems: dst[i] = src[idx[i]] with
// tile_begin = tbeg[i], tile_prob over the renumbered tiles (tbeg: n + 1
// entries, tiles = tbeg[n]) and red_bprob over the split-K reduction blocks
// (rpre: n + 1 entries, red = rpre[n])
hipError_t launch_compact_table(const GemmProb* src, const int* idx, const int* tbeg, const int* rpre, int n,
                                int tiles, int red, GemmProb* dst, int* tile_prob, int* red_bprob, hipStream_t s);

}  // namespace hcc

// izh_field.hip -- charge deposition, open-boundary Poisson solve and E field.
//
// Deposition: CIC weights as deposit_BeamBunch forms them, accumulated as
// fixed-point integers (scale 2^e from the total |charge|), so the sum is
// exact and independent of the order atomics land in: bitwise
// deterministic.
//
// Poisson: the Hockney doubled-grid convolution of openBC3D
// (src/Appl/Field.f90:239-331), factored into batched 1D FFTs over lines:
//   fwd-x (real, half zero) -> fwd-y (half zero) -> z: FFT * G^ * IFFT fused
//   in LDS, keeping only the first half -> inv-y (keep half) -> inv-x (C2R).
// Only the first octant of the result is ever stored.  G^ of the even
// extended integrated Green function is real and even, so it is built and
// stored on the (nx+1)(ny+1)(nz+1) half-grid and folded on use.
// Each block transforms B lines of length L (B*L = 2048 points, 4096 in the
// fused z pass) in LDS with in-place radix-2 stages: decimation in
// frequency for forward transforms (natural in, bit-reversed out) and
// decimation in time for the inverse of the fused z pass (bit-reversed in,
// natural out), so no reorder pass is needed between them.
#include <algorithm>
#include <array>
#include <atomic>
#include <cmath>
#include <cstring>
#include <map>
#include <vector>

#include "izh_device.hpp"

namespace izh {
namespace {

template <typename T>
struct cx {
  T re, im;
};

template <typename T>
__device__ inline cx<T> cmul(cx<T> a, cx<T> b) {
  return {a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re};
}

// Threads per line-kernel block: 512 puts four waves per SIMD on a CU that
// holds two 4096-point z-pass blocks in LDS (256 left two, and the solve
// 8% slower).
constexpr int kFftThreads = 512;
constexpr int kFftPoints = 2048;  // points per block in LDS
constexpr int kFftPointsZ = 4096; // the fused z pass: 8 lines of 512 at 128x128x256
constexpr int kFftMinLine = 8;    // shortest line (a mesh of 4 nodes doubled)

// kLoadFx: the deposit's fixed-point charge, converted to the grid type as it
// is read; the pass also leaves the converted grid in Lines::rho and the
// accumulator cleared for the next deposit.  kLoadIgf: an even line of the
// integrated Green function, the 8-corner difference of its antiderivative.
enum Load { kLoadReal = 0, kLoadCplx = 1, kLoadEven = 2, kLoadHerm = 3, kLoadFx = 4,
            kLoadIgf = 5 };
enum Store { kStoreCplx = 0, kStoreReal = 1 };

struct Lines {
  const void *src;
  void *dst;
  int64_t nf, ns;          // lines = nf * ns, f fastest
  int64_t nfv;             // lines with f >= nfv are padding: not read or written
  int64_t sf, ss, se;      // source strides (elements)
  int64_t df, ds, de;      // destination strides
  int L, log2L, B, log2B, Lin, Lout;
  uint64_t nf_mul;         // ceil(2^40 / nf): line / nf by a multiply
  double out_scale;
  // fused z pass: multiply by the half-grid G^ folded in the line's y index
  const void *green;
  int64_t gkx, gky;        // G^ strides of ky and kz: ldx*(nz+1), ldx
  int my;                  // doubled y length, for folding the line's y index
  void *rho;               // kLoadFx: the converted grid
  double fx_inv;           // kLoadFx: grid value of one fixed-point unit
  int tx, ty;              // kLoadIgf: corners per row, rows per plane
  const void *far;         // kLoadIgf: G away from the origin (T)
  const IgfBox *box;       // kLoadIgf: where the corners hold
};

// 8-corner difference of the antiderivative at the cells' corners
// (src/Appl/Field.f90:420-428), node (i, j, k) at c of a grid of tx x ty
// corners per plane.
__device__ inline double igf_diff(const double *__restrict__ t, int64_t c, int64_t tx,
                                  int64_t txy) {
  return t[c + 1 + tx + txy] - t[c + tx + txy] - t[c + 1 + txy] + t[c + txy] -
         t[c + 1 + tx] + t[c + tx] + t[c + 1] - t[c];
}

// The integrated Green function far from the origin: the mean of 1/r over a
// cell, as the Taylor series of 1/r averaged over the cell up to eighth order.
// With a = x^2/r^4 (b, c for y, z) it is a polynomial over r,
//   g = (1/r) sum of C_ijk a^i b^j c^k, i + j + k <= 4, C_000 = 1,
// whose coefficients hold the mesh sizes (igf_block, igf_table).  The 8-corner
// difference of the antiderivative costs three arctangents and three
// logarithms per corner and cancels: its relative error grows with r^3, 1e-12
// at kIgfFar cell half diagonals and 1e-9 at 64 of cells 1:1:4.  The truncated
// series is off by at most rho^-10 / 11 at rho half diagonals, 1.5e-12 at
// kIgfFar and less than rounding from 30 on, whatever the cell (the bound is a
// needle's; 1.1e-13 at kIgfFar for cells up to 1:1:4, 5.3e-13 for 1:4:16; at
// ten half diagonals series and corners meet for cubes).  So only the box
// within kIgfFar of the origin keeps the corners.  The deposit's launch, which
// forms G beside the deposit, fell from 60 to 40 us on 128^3 (150k particles,
// FP64; 2.2M corners, 27 us of the deposit's own) and from 245 to 199 us on
// 128x128x256 (10M, mixed).
constexpr int kIgfOrder = 4;                    // pairs of derivatives
constexpr int kIgfTerms = 35;
constexpr double kIgfFar = 12.0;
// Nodes from which the series is used: below, its preparation takes as long as
// the corners it saves (deposit's launch and x pass of 64^3: 24.3 us either
// way; of 64x64x128 42.4 against 45.9).
constexpr int64_t kIgfSeriesNodes = 400000;

// Place of C_ijk: i outermost, then j, then k.
__host__ __device__ constexpr int igf_term(int i, int j, int k) {
  // terms of the i's before: T(4) + T(3) + ..., T(n) = (n+1)(n+2)/2
  return (i > 0 ? 15 : 0) + (i > 1 ? 10 : 0) + (i > 2 ? 6 : 0) + (i > 3 ? 3 : 0) +
         j * (kIgfOrder + 1 - i) - j * (j - 1) / 2 + k;
}
static_assert(igf_term(kIgfOrder, 0, 0) == kIgfTerms - 1 && igf_term(1, 0, 0) == 15 &&
              igf_term(0, 0, 4) == 4 && igf_term(0, 1, 0) == 5, "igf_term");

// C: the coefficients, uniform over the wavefront.
__device__ inline double igf_far(const double (&C)[kIgfTerms], double x2, double y2, double z2) {
  const double ir = rsqrt(x2 + y2 + z2), ir2 = ir * ir, ir4 = ir2 * ir2;
  const double a = x2 * ir4, b = y2 * ir4, c = z2 * ir4;
  double s = 0.0;
#pragma unroll
  for (int i = kIgfOrder; i >= 0; i--) {
    double p = 0.0;
#pragma unroll
    for (int j = kIgfOrder - i; j >= 0; j--) {
      double q = 0.0;
#pragma unroll
      for (int k = kIgfOrder - i - j; k >= 0; k--) q = fma(q, c, C[igf_term(i, j, k)]);
      p = fma(p, b, q);
    }
    s = fma(s, a, p);
  }
  return s * ir;
}

// G at node (i, j, k): the corners' difference in the box near the origin,
// elsewhere the grid the series left (igf_block).
template <typename T>
__device__ inline T igf_value(const Lines &p, int i, int j, int k, const int near[3]) {
  if (i < near[0] && j < near[1] && k < near[2]) {
    const int64_t txy = (int64_t)p.tx * p.ty;
    return (T)igf_diff((const double *)p.src, i + j * (int64_t)p.tx + k * txy, p.tx, txy);
  }
  return ((const T *)p.far)[i + (p.tx - 1) * (j + (p.ty - 1) * (int64_t)k)];
}

// Logical block of physical block p of n: the hardware deals blocks to the
// 8 XCDs in turn (block p to XCD p mod 8), each XCD with its own L2.  XCD x
// takes the x-th contiguous run of logical blocks, one after another, so
// blocks whose lines share 128-byte lines of a spectrum or of G^ (FP32 rows,
// G^'s runs of 8 values) read them through one L2.  A bijection of [0, n)
// for any n (the first n mod 8 XCDs take one block more).
__device__ inline int xcd_block(int p, int n) {
  const int x = p & 7, base = n >> 3, extra = n & 7;
  return x * base + min(x, extra) + (p >> 3);
}

__device__ inline int bitrev(int v, int bits) {
  return (int)(__brev((unsigned)v) >> (32 - bits));
}

// In-place radix-2 decimation in frequency (natural in, bit-reversed out) and
// decimation in time (bit-reversed in, natural out) over the B lines of a
// block.  Up to three consecutive radix-2 stages run in registers on groups
// of 8 elements: the elements a run of stages combines form closed groups
// (stride = the run's smallest half), so each group is read from LDS once per
// three stages.  Every element sees the same butterflies with the same
// twiddles, in the same order, as the stage-by-stage transform.  tw: L/2
// twiddles exp(-2 pi i k / L) in LDS.
// Position of point m in its line's LDS row.  Without it the radix-8 groups
// of the later runs put the lanes of a wavefront on a few banks (group
// stride 1: 16-byte points 128 bytes apart); XOR-ing the low 4 bits with
// m >> 3 spreads every access pattern of the kernel over all banks.  mask
// is 15 for lines of 64 points or more, else 0 (short lines do no better).
__device__ inline int lds_pos(int m, int mask) { return m ^ ((m >> 3) & mask); }

// The K stages of one run on a group held in registers: v[j] is position
// m0 + j * 2^ls of its line, r = m0 mod 2^ls.
template <typename T, bool DIT, int K>
__device__ __attribute__((always_inline)) inline void run_regs(cx<T> (&v)[1 << K], int ls,
                                                               int r, int log2L,
                                                               const cx<T> *tw, bool inverse) {
  constexpr int span = 1 << K;
#pragma unroll
  for (int st = 0; st < K; st++) {
    const int e = DIT ? st : K - 1 - st;  // pair distance 2^e in the group
    const int lt = log2L - 1 - ls - e;    // log2 of the twiddle stride
#pragma unroll
    for (int j = 0; j < span; j++) {
      if ((j >> e) & 1) continue;
      const int k = r + ((j & ((1 << e) - 1)) << ls);
      cx<T> w = tw[k << lt];
      if (inverse) w.im = -w.im;
      const cx<T> u = v[j], x = v[j + (1 << e)];
      if (DIT) {
        const cx<T> y = cmul<T>(x, w);
        v[j] = {u.re + y.re, u.im + y.im};
        v[j + (1 << e)] = {u.re - y.re, u.im - y.im};
      } else {
        v[j] = {u.re + x.re, u.im + x.im};
        v[j + (1 << e)] = cmul<T>({u.re - x.re, u.im - x.im}, w);
      }
    }
  }
}

template <typename T, bool DIT, int K>
__device__ inline void fft_run(cx<T> *buf, int log2L, int LP, int lines, const cx<T> *tw,
                               bool inverse, int done, int mask) {
  constexpr int span = 1 << K;
  // DIF runs halves L/2 .. 1 downwards, DIT 1 .. L/2 upwards; every size
  // here is a power of two, so the group index splits with shifts and masks
  const int ls = DIT ? done : log2L - done - K;  // log2 of the group stride
  const int s = 1 << ls;
  const int lpl = log2L - K;                     // log2 of the groups per line
  const int ngroups = lines << lpl;
  for (int g = threadIdx.x; g < ngroups; g += kFftThreads) {
    const int lb = g >> lpl, q = g & ((1 << lpl) - 1);
    const int blk = q >> ls, r = q & (s - 1);
    const int row = lb * LP, m0 = (blk << (ls + K)) + r;
    cx<T> v[span];
#pragma unroll
    for (int j = 0; j < span; j++) v[j] = buf[row + lds_pos(m0 + j * s, mask)];
    run_regs<T, DIT, K>(v, ls, r, log2L, tw, inverse);
#pragma unroll
    for (int j = 0; j < span; j++) buf[row + lds_pos(m0 + j * s, mask)] = v[j];
  }
  __syncthreads();
}

// The fused z pass's middle: the forward transform's last run (stages
// log2L-3 .. log2L-1, groups of 8 neighbouring positions) and the inverse
// transform's first run (stages 0 .. 2, the same groups) with the multiply by
// G^ between them, in registers: two LDS round trips and two barriers fewer
// than running them apart.  Thread t takes the group of positions 8q .. 8q+7
// of line lb, lb = t mod B and q = t / B (lanes walk across the block's lines,
// so their G^ values, gv[j] for position 8q + j, were read in runs of
// neighbouring x lines); one group per thread (PTS / 8 == kFftThreads).
template <typename T>
__device__ __attribute__((always_inline)) inline void fft_conv_middle(
    cx<T> *buf, int LP, int log2L, int log2B, const cx<T> *tw, bool inverse,
    const T (&gv)[8], int mask) {
  const int lb = threadIdx.x & ((1 << log2B) - 1), q = threadIdx.x >> log2B;
  const int row = lb * LP, m0 = q << 3;
  cx<T> v[8];
#pragma unroll
  for (int j = 0; j < 8; j++) v[j] = buf[row + lds_pos(m0 + j, mask)];
  run_regs<T, false, 3>(v, 0, 0, log2L, tw, inverse);
#pragma unroll
  for (int j = 0; j < 8; j++) v[j] = {v[j].re * gv[j], v[j].im * gv[j]};
  run_regs<T, true, 3>(v, 0, 0, log2L, tw, true);
#pragma unroll
  for (int j = 0; j < 8; j++) buf[row + lds_pos(m0 + j, mask)] = v[j];
  __syncthreads();
}

// Stages [from, to) of the transform (all of them by default), in runs of
// up to three.
template <typename T, bool DIT>
__device__ __attribute__((always_inline)) inline void fft_stages(
    cx<T> *buf, int LP, int log2L, int lines, const cx<T> *tw, bool inverse, int mask,
    int from = 0, int to = -1) {
  if (to < 0) to = log2L;
  int done = from;
  while (done < to) {
    const int k = min(3, to - done);
    if (k == 3)
      fft_run<T, DIT, 3>(buf, log2L, LP, lines, tw, inverse, done, mask);
    else if (k == 2)
      fft_run<T, DIT, 2>(buf, log2L, LP, lines, tw, inverse, done, mask);
    else
      fft_run<T, DIT, 1>(buf, log2L, LP, lines, tw, inverse, done, mask);
    done += k;
  }
}

// line = f + nf * s for f < nf: s by a multiply with nf_mul = ceil(2^40 / nf),
// exact for line < 2^24 and nf < 2^16 (run_lines checks both).
__device__ inline void line_fs(int line, const Lines &p, int &f, int &s) {
  s = (int)(((uint64_t)(uint32_t)line * p.nf_mul) >> 40);
  f = line - s * (int)p.nf;
}

// Thread t of a block -> (line in block, element) with coalesced addresses:
// unit element stride -> consecutive threads walk one line; otherwise they
// walk across neighbouring lines (unit line stride).
__device__ inline void map_thread(int t, int64_t estride, int log2L, int log2B, int &lb,
                                  int &m) {
  if (estride == 1) {
    lb = t >> log2L;
    m = t & ((1 << log2L) - 1);
  } else {
    m = t >> log2B;
    lb = t & ((1 << log2B) - 1);
  }
}

// PAIR: two real lines share one complex transform (line 2j in the real
// part, line 2j+1 in the imaginary part).  Real even input (kLoadEven) gives
// a real even spectrum each, so the parts separate directly; real input
// (kLoadReal) is separated from Z(k) and conj Z(L-k) when stored; two
// Hermitian spectra (kLoadHerm) are combined as X + iY, whose inverse has
// the two real outputs as its parts.
// PTS points of B = PTS/L lines per block; each line is held in LDS at a
// pitch of L+1 points, so lanes that walk across lines (a line stride
// other than 1, or the fused z pass's multiply) do not all hit one bank.
// LL: log2 of the line length when it is fixed at compile time (the common
// lengths, so every index split and LDS position folds), 0 to take it from p.
// buf: kFftLds<PTS> points of LDS, tw: L/2 twiddles of it; block bid of nb.
template <int PTS>
constexpr int kFftLds = PTS + PTS / kFftMinLine;

template <typename T, int LOAD, int STORE, bool CONV, bool PAIR, int PTS, int LL>
__device__ __attribute__((always_inline)) inline void fft_lines_block(
    const Lines &p, const cx<T> *__restrict__ twg, int inverse, int bid, int nb, cx<T> *buf,
    cx<T> *tw) {
  static_assert(PTS == 2048 || PTS == 4096, "points per block");
  constexpr int kLog2Pts = PTS == 4096 ? 12 : 11;
  const int log2L = LL ? LL : p.log2L;
  const int L = 1 << log2L;
  const int log2B = kLog2Pts - log2L;
  const int B = 1 << log2B;
  const int LP = L + 1;
  const int mask = L >= 64 ? 15 : 0;
  // twiddles are written to LDS together with the line data below
  constexpr int kTwPer = PTS / 2 / kFftThreads;  // L/2 <= PTS/2
  cx<T> twv[kTwPer];
#pragma unroll
  for (int it = 0; it < kTwPer; it++) {
    const int t = threadIdx.x + it * kFftThreads;
    T re = (T)0, im = (T)0;
    if (t < (L >> 1)) {
      const cx<T> v = twg[t];
      re = v.re; im = v.im;
    }
    twv[it] = {re, im};
  }
  const int nf = (int)p.nf;
  const int nlines = nf * (int)p.ns;
  const int line0 = xcd_block(bid, nb) * B;
  // fused z pass: fetch the G^ values of the thread's group of the fused
  // middle run first, so their latency hides behind the forward transform.
  // Lanes walk across the block's lines first (neighbouring x indices,
  // neighbouring addresses of G^); the forward spectrum is bit-reversed, so
  // position m of a line holds natural frequency kz = bitrev(m).
  static_assert(!CONV || PTS / 8 == kFftThreads, "one middle-run group per thread");
  T gv[8];
  if (CONV) {
    const T *G = (const T *)p.green;
    const int lb = threadIdx.x & (B - 1), q = threadIdx.x >> log2B;
    const int line = line0 + lb;
    int i, j2;
    line_fs(line, p, i, j2);
    const bool live = line < nlines && i < p.nfv;
    const int jf = j2 <= p.my / 2 ? j2 : p.my - j2;
#pragma unroll
    for (int j = 0; j < 8; j++) {
      const int kz = bitrev((q << 3) + j, log2L);
      const int kf = kz <= (L >> 1) ? kz : L - kz;
      T g = (T)0;
      if (live) g = G[i + p.gkx * jf + p.gky * kf];
      gv[j] = g;
    }
  }
  // Complex lines walked across (unit line stride, element stride other
  // than one: the y passes and the fused z pass) skip the load's LDS round
  // trip: thread t loads the 8 points of its group of the first radix-8
  // run, positions q + j L/8 of line lb (lb = t mod B, q = t / B: lanes walk
  // across the block's neighbouring lines, so each run of B points is one
  // 128-byte line), straight from global memory and runs those three
  // stages in registers before its first LDS write.
  // The y passes (complex lines in and out, both walked across) run as a
  // decimation in time: the first radix-8 run takes its groups of
  // bit-reversed positions 8q .. 8q+7, points bitrev(q) + bitrev3(j) L/8,
  // straight from global memory, and the last leaves natural positions
  // q + j L/8, stored from registers, so the data passes through LDS only
  // between runs.
  constexpr bool kFuseLoad = !PAIR && LOAD == kLoadCplx;
  const bool fuse = kFuseLoad && p.se != 1 && p.sf == 1 && log2L >= 6;
  const bool dit = fuse && !CONV && STORE == kStoreCplx && p.df == 1;
  int first = 0;  // stages run before the data reaches LDS
  if (fuse) {
    const int lb = threadIdx.x & (B - 1), q = threadIdx.x >> log2B;
    const bool act = threadIdx.x < (PTS >> 3);  // one group per thread
    const int line = line0 + lb;
    int f = 0, sl = 0;
    line_fs(line, p, f, sl);
    const bool live = act && line < nlines && f < p.nfv;
    const int64_t base = f * p.sf + sl * p.ss;
    const int s8 = L >> 3;
    const int qr = dit ? bitrev(q, log2L - 3) : q;
    cx<T> v[8];
#pragma unroll
    for (int j = 0; j < 8; j++) {
      const int m = qr + (dit ? bitrev(j, 3) : j) * s8;
      T re = (T)0, im = (T)0;
      if (live && m < p.Lin) {
        const cx<T> x = ((const cx<T> *)p.src)[base + m * p.se];
        re = x.re; im = x.im;
      }
      v[j] = {re, im};
    }
#pragma unroll
    for (int it = 0; it < kTwPer; it++) {
      const int t = threadIdx.x + it * kFftThreads;
      if (t < (L >> 1)) tw[t] = twv[it];
    }
    __syncthreads();
    if (act && dit) {
      run_regs<T, true, 3>(v, 0, 0, log2L, tw, inverse != 0);
#pragma unroll
      for (int j = 0; j < 8; j++) buf[lb * LP + lds_pos((q << 3) + j, mask)] = v[j];
    } else if (act) {
      run_regs<T, false, 3>(v, log2L - 3, q, log2L, tw, inverse != 0);
#pragma unroll
      for (int j = 0; j < 8; j++) buf[lb * LP + lds_pos(q + j * s8, mask)] = v[j];
    }
    __syncthreads();
    first = 3;
  } else if constexpr (LOAD == kLoadIgf) {
    // ---- even lines of G: each value is formed once and written to both of
    // its places, m and L-m (thread m = 0 also takes m = L/2)
    static_assert(LOAD != kLoadIgf || PAIR, "even lines travel in pairs");
    const int half = L >> 1;
    const int near[3] = {p.box->near[0], p.box->near[1], p.box->near[2]};
    constexpr int kPer = PTS / 2 / kFftThreads;
#pragma unroll
    for (int it = 0; it < kPer; it++) {
      const int t = threadIdx.x + it * kFftThreads;
      const int lb = t >> (log2L - 1), m = t & (half - 1);
      const int l0 = 2 * (line0 + lb), l1 = l0 + 1;
      const bool has0 = l0 < nlines, has1 = l1 < nlines;
      int j0, k0, j1, k1;
      line_fs(has0 ? l0 : 0, p, j0, k0);
      line_fs(has1 ? l1 : 0, p, j1, k1);
      const T a = igf_value<T>(p, m, j0, k0, near);
      const T b = igf_value<T>(p, m, j1, k1, near);
      const cx<T> v = {has0 ? a : (T)0, has1 ? b : (T)0};
      cx<T> *row = buf + lb * LP;
      row[lds_pos(m, mask)] = v;
      if (m > 0) {
        row[lds_pos(L - m, mask)] = v;
      } else {
        const T ah = igf_value<T>(p, half, j0, k0, near);
        const T bh = igf_value<T>(p, half, j1, k1, near);
        row[lds_pos(half, mask)] = {has0 ? ah : (T)0, has1 ? bh : (T)0};
      }
    }
#pragma unroll
    for (int it = 0; it < kTwPer; it++) {
      const int t = threadIdx.x + it * kFftThreads;
      if (t < (L >> 1)) tw[t] = twv[it];
    }
    __syncthreads();
  } else {
    // ---- load (zero padding / even extension / Hermitian completion): all of
    // a thread's loads are issued before the first LDS write
    constexpr int kPer = PTS / kFftThreads;  // B * L == PTS
    cx<T> ld[kPer];
    int slot[kPer];
    int64_t at[kPer][2];  // kLoadFx: where the pair's values came from (-1: nowhere)
#pragma unroll
    for (int it = 0; it < kPer; it++) {
      const int t = threadIdx.x + it * kFftThreads;
      int lb, m;
      map_thread(t, p.se, log2L, log2B, lb, m);
      const int line = line0 + lb;
      slot[it] = lb * LP + lds_pos(m, mask);
      T re = (T)0, im = (T)0;
      if (LOAD == kLoadFx) at[it][0] = at[it][1] = -1;
      if (PAIR) {
        const int l0 = 2 * line, l1 = l0 + 1;
        const T *src = (const T *)p.src;
        const cx<T> *csrc = (const cx<T> *)p.src;
        if (l0 < nlines) {
          int f0, s0, f1, s1;
          line_fs(l0, p, f0, s0);
          line_fs(l1, p, f1, s1);
          const int64_t b0 = f0 * p.sf + s0 * p.ss;
          const bool has1 = l1 < nlines;
          const int64_t b1 = has1 ? f1 * p.sf + s1 * p.ss : b0;
          if (LOAD == kLoadEven) {
            const int mm = m <= (L >> 1) ? m : L - m;
            re = src[b0 + mm * p.se];
            im = has1 ? src[b1 + mm * p.se] : (T)0;
          } else if (LOAD == kLoadReal) {
            if (m < p.Lin) {
              re = src[b0 + m * p.se];
              im = has1 ? src[b1 + m * p.se] : (T)0;
            }
          } else if (LOAD == kLoadFx) {
            if (m < p.Lin) {
              const long long *fx = (const long long *)p.src;
              at[it][0] = b0 + m * p.se;
              re = (T)((double)fx[at[it][0]] * p.fx_inv);
              if (has1) {
                at[it][1] = b1 + m * p.se;
                im = (T)((double)fx[at[it][1]] * p.fx_inv);
              }
            }
          } else {  // kLoadHerm: Z = X + iY of the completed spectra
            const bool lo = m <= (L >> 1);
            const int mm = lo ? m : L - m;
            cx<T> x = csrc[b0 + mm * p.se];
            cx<T> y = has1 ? csrc[b1 + mm * p.se] : cx<T>{(T)0, (T)0};
            if (!lo) { x.im = -x.im; y.im = -y.im; }
            re = x.re - y.im;
            im = x.im + y.re;
          }
        }
      } else if (line < nlines) {
        int f, s;
        line_fs(line, p, f, s);
        const int64_t base = f * p.sf + s * p.ss;
        if (f >= p.nfv) {
          // a padding line: zeros
        } else if (LOAD == kLoadReal) {
          if (m < p.Lin) re = ((const T *)p.src)[base + m * p.se];
        } else if (LOAD == kLoadCplx) {
          if (m < p.Lin) {
            const cx<T> v = ((const cx<T> *)p.src)[base + m * p.se];
            re = v.re; im = v.im;
          }
        } else if (LOAD == kLoadEven) {
          const int mm = m <= (L >> 1) ? m : L - m;
          re = ((const T *)p.src)[base + mm * p.se];
        } else {  // kLoadHerm: first L/2+1 values stored
          const bool lo = m <= (L >> 1);
          const cx<T> v = ((const cx<T> *)p.src)[base + (lo ? m : L - m) * p.se];
          re = v.re; im = lo ? v.im : -v.im;
        }
      }
      ld[it] = {re, im};
    }
#pragma unroll
    for (int it = 0; it < kPer; it++) buf[slot[it]] = ld[it];
    if (LOAD == kLoadFx) {
      T *rho = (T *)p.rho;
      unsigned long long *fx = (unsigned long long *)const_cast<void *>(p.src);
#pragma unroll
      for (int it = 0; it < kPer; it++) {
        if (at[it][0] >= 0) { rho[at[it][0]] = ld[it].re; fx[at[it][0]] = 0ull; }
        if (at[it][1] >= 0) { rho[at[it][1]] = ld[it].im; fx[at[it][1]] = 0ull; }
      }
    }
#pragma unroll
    for (int it = 0; it < kTwPer; it++) {
      const int t = threadIdx.x + it * kFftThreads;
      if (t < (L >> 1)) tw[t] = twv[it];
    }
    __syncthreads();
  }
  // The last run of a decimation in time leaves positions q + j L/8 of
  // each line in natural order: with lanes walking across the lines, the
  // thread stores its group from registers (runs of B neighbouring x
  // lines), skipping the store's LDS round trip.
  auto last_run_store = [&](bool inv) {
    const int lb = threadIdx.x & (B - 1), q = threadIdx.x >> log2B;
    if (threadIdx.x >= (PTS >> 3)) return;  // one group per thread
    const int s8 = L >> 3;
    cx<T> v[8];
#pragma unroll
    for (int j = 0; j < 8; j++) v[j] = buf[lb * LP + lds_pos(q + j * s8, mask)];
    run_regs<T, true, 3>(v, log2L - 3, q, log2L, tw, inv);
    const int line = line0 + lb;
    if (line >= nlines) return;
    int f, sl;
    line_fs(line, p, f, sl);
    if (f >= p.nfv) return;
    const int64_t o = f * p.df + sl * p.ds;
#pragma unroll
    for (int j = 0; j < 8; j++) {
      const int m = q + j * s8;
      if (m < p.Lout)
        ((cx<T> *)p.dst)[o + m * p.de] = {(T)(v[j].re * p.out_scale),
                                          (T)(v[j].im * p.out_scale)};
    }
  };
  if (dit) {
    fft_stages<T, true>(buf, LP, log2L, B, tw, inverse != 0, mask, 3, log2L - 3);
    last_run_store(inverse != 0);
    return;
  }
  if (CONV) {
    fft_stages<T, false>(buf, LP, log2L, B, tw, inverse != 0, mask, first, log2L - 3);
    fft_conv_middle<T>(buf, LP, log2L, log2B, tw, inverse != 0, gv, mask);
    if (log2L >= 6 && p.df == 1 && STORE == kStoreCplx) {
      fft_stages<T, true>(buf, LP, log2L, B, tw, true, mask, 3, log2L - 3);
      last_run_store(true);
      return;
    }
    fft_stages<T, true>(buf, LP, log2L, B, tw, true, mask, 3);
  } else {
    fft_stages<T, false>(buf, LP, log2L, B, tw, inverse != 0, mask, first);
  }
  // ---- store the kept part of each line
  const int totout = B * L;
  for (int t = threadIdx.x; t < totout; t += kFftThreads) {
    int lb, m;
    map_thread(t, p.de, log2L, log2B, lb, m);
    if (m >= p.Lout) continue;
    if (PAIR) {
      const int l0 = 2 * (line0 + lb), l1 = l0 + 1;
      if (l0 >= nlines) continue;
      const bool has1 = l1 < nlines;
      int f0, s0, f1, s1;
      line_fs(l0, p, f0, s0);
      line_fs(l1, p, f1, s1);
      const int64_t o0 = f0 * p.df + s0 * p.ds + m * p.de;
      const int64_t o1 = has1 ? f1 * p.df + s1 * p.ds + m * p.de : o0;
      const cx<T> z = buf[lb * LP + lds_pos(bitrev(m, log2L), mask)];
      if (STORE == kStoreReal) {
        ((T *)p.dst)[o0] = (T)(z.re * p.out_scale);
        if (has1) ((T *)p.dst)[o1] = (T)(z.im * p.out_scale);
      } else {
        // X(m) = (Z(m) + conj Z(L-m)) / 2,  Y(m) = (Z(m) - conj Z(L-m)) / 2i
        const cx<T> w = buf[lb * LP + lds_pos(bitrev((L - m) & (L - 1), log2L), mask)];
        const T h = (T)(0.5 * p.out_scale);
        ((cx<T> *)p.dst)[o0] = {(z.re + w.re) * h, (z.im - w.im) * h};
        if (has1) ((cx<T> *)p.dst)[o1] = {(z.im + w.im) * h, (w.re - z.re) * h};
      }
      continue;
    }
    int line = line0 + lb;
    if (line >= nlines) continue;
    int f, s;
    line_fs(line, p, f, s);
    if (f >= p.nfv) continue;
    int64_t o = f * p.df + s * p.ds + m * p.de;
    cx<T> v = buf[lb * LP + lds_pos(CONV ? m : bitrev(m, log2L), mask)];
    if (STORE == kStoreCplx) {
      ((cx<T> *)p.dst)[o] = {(T)(v.re * p.out_scale), (T)(v.im * p.out_scale)};
    } else {
      ((T *)p.dst)[o] = (T)(v.re * p.out_scale);
    }
  }
}

template <typename T, int LOAD, int STORE, bool CONV, bool PAIR, int PTS, int LL>
__global__ void __launch_bounds__(kFftThreads)
k_fft_lines(Lines p, const cx<T> *__restrict__ twg, int inverse) {
  __shared__ cx<T> buf[kFftLds<PTS>];
  extern __shared__ __align__(16) unsigned char fft_dyn[];  // L/2 twiddles
  fft_lines_block<T, LOAD, STORE, CONV, PAIR, PTS, LL>(
      p, twg, inverse, (int)blockIdx.x, (int)gridDim.x, buf,
      reinterpret_cast<cx<T> *>(fft_dyn));
}

// Two independent forward passes along one axis in one launch: nba blocks of
// the Green function's lines (pairs of even real lines), then, from the next
// multiple of eight on (which keeps xcd_block's dealing), those of the charge.
// The Green function's transform and the charge's have the same depth, so a
// step's chain is as long as the charge's alone, with no second stream.
template <typename T, int LOADA, int LOADB, int STOREB, bool PAIRB, int LL>
__global__ void __launch_bounds__(kFftThreads)
k_fft_two(Lines a, Lines b, int nba, int nbb, const cx<T> *__restrict__ twg) {
  __shared__ cx<T> buf[kFftLds<kFftPoints>];
  extern __shared__ __align__(16) unsigned char fft_dyn[];
  cx<T> *tw = reinterpret_cast<cx<T> *>(fft_dyn);
  const int first_b = (nba + 7) & ~7, bid = (int)blockIdx.x;
  if (bid < first_b) {
    if (bid < nba)
      fft_lines_block<T, LOADA, kStoreReal, false, true, kFftPoints, LL>(a, twg, 0, bid, nba,
                                                                         buf, tw);
  } else {
    fft_lines_block<T, LOADB, STOREB, false, PAIRB, kFftPoints, LL>(b, twg, 0, bid - first_b,
                                                                    nbb, buf, tw);
  }
}

// ------------------------------------------------------ Green function
// Block bid of nb of the Green function's values: the corners of the box near
// the origin, and the series' values on the nodes outside of it (far: the grid
// of (nx+1)(ny+1)(nz+1) nodes; the x pass reads neither elsewhere).  The first
// block leaves the box for the x pass.  C: kIgfTerms doubles of LDS.
template <typename T>
__device__ inline void igf_block(double *__restrict__ out, T *__restrict__ far, int nx, int ny,
                                 int nz, const DevDom *__restrict__ dom,
                                 const double *__restrict__ tab, IgfBox *__restrict__ box,
                                 double *C, int bid, int nb) {
  const double hx = dom->msize[0], hy = dom->msize[1], hz = dom->msize[2];
  const double h2[3] = {hx * hx, hy * hy, hz * hz};
  const int gx = nx + 1, gy = ny + 1, gz = nz + 1;
  const bool series = (int64_t)gx * gy * gz > kIgfSeriesNodes;
  const double reach = kIgfFar * 0.5 * sqrt(h2[0] + h2[1] + h2[2]);
  const auto edge = [&](int g, double h) {
    return series ? (int)fmin((double)g, floor(reach / h) + 1.0) : g;
  };
  const int near[3] = {edge(gx, hx), edge(gy, hy), edge(gz, hz)};
  if (bid == 0 && threadIdx.x < 3) box->near[threadIdx.x] = near[threadIdx.x];
  // corners first (the longer chain), a thread each up to half the blocks;
  // the rest take the series, or the corners too where there is none
  const int bx = near[0] + 1, by = near[1] + 1, bz = near[2] + 1;
  const int ncorners = bx * by * bz;
  const bool all = near[0] == gx && near[1] == gy && near[2] == gz;
  const int nbc = all ? nb : min((ncorners + (int)blockDim.x - 1) / (int)blockDim.x, nb / 2);
  if (bid < nbc) {
    // IGF antiderivative (src/Appl/Field.f90:384-418)
    const double vol = hx * hy * hz;
    const int tx = nx + 2, ty = ny + 2;
    for (int c = bid * (int)blockDim.x + (int)threadIdx.x; c < ncorners;
         c += nbc * (int)blockDim.x) {
      const int k = c / (bx * by), rem = c - k * bx * by, j = rem / bx, i = rem - j * bx;
      double x = i * hx - hx / 2.0, y = j * hy - hy / 2.0, z = k * hz - hz / 2.0;
      double rr = sqrt(x * x + y * y + z * z);
      double aa = -z * z * atan(x * y / (z * rr)) / 2.0;
      double bb = -y * y * atan(x * z / (y * rr)) / 2.0;
      double cc = -x * x * atan(y * z / (x * rr)) / 2.0;
      double dd = y * z * log(x + rr);
      double ee = x * z * log(y + rr);
      double ff = x * y * log(z + rr);
      out[i + tx * (int64_t)(j + ty * k)] = (aa + bb + cc + dd + ee + ff) / vol;
    }
    return;
  }
  if ((int)threadIdx.x < kIgfTerms) {
    // term t: its row of the table times the monomials of the squared mesh
    // sizes (the table is zero between orders)
    double pw[3][kIgfOrder + 1];
#pragma unroll
    for (int a = 0; a < 3; a++) {
      pw[a][0] = 1.0;
#pragma unroll
      for (int q = 1; q <= kIgfOrder; q++) pw[a][q] = pw[a][q - 1] * h2[a];
    }
    const double *row = tab + (int)threadIdx.x * kIgfTerms;
    double c = 0.0;
#pragma unroll
    for (int i = 0; i <= kIgfOrder; i++)
#pragma unroll
      for (int j = 0; i + j <= kIgfOrder; j++)
#pragma unroll
        for (int k = 0; i + j + k <= kIgfOrder; k++)
          c += row[igf_term(i, j, k)] * (pw[0][i] * pw[1][j] * pw[2][k]);
    C[threadIdx.x] = c;
  }
  __syncthreads();
  // ---- the series.  Its coefficients move to scalar registers, so a node is
  // its 34 multiply-adds and a reciprocal root; the node's indexes split by
  // FP64 multiplies (exact: (c + 1/2) / g is at least 1/(2g) from an integer)
  {
    double U[kIgfTerms];
#pragma unroll
    for (int t = 0; t < kIgfTerms; t++) {
      const int lo = __builtin_amdgcn_readfirstlane(__double2loint(C[t]));
      const int hi = __builtin_amdgcn_readfirstlane(__double2hiint(C[t]));
      U[t] = __hiloint2double(hi, lo);
    }
    const int total = gx * gy * gz;
    const double igx = 1.0 / gx, igy = 1.0 / gy;
    for (int c = (bid - nbc) * (int)blockDim.x + (int)threadIdx.x; c < total;
         c += (nb - nbc) * (int)blockDim.x) {
      const int jk = (int)((c + 0.5) * igx), i = c - jk * gx;
      const int k = (int)((jk + 0.5) * igy), j = jk - k * gy;
      if (i < near[0] && j < near[1] && k < near[2]) continue;
      far[c] = (T)igf_far(U, (double)(i * i) * h2[0], (double)(j * j) * h2[1],
                          (double)(k * k) * h2[2]);
    }
  }
}

constexpr int kIgfBlocks = 768;  // as many as the deposit's LDS lets run at once (2048: 45 us)
template <typename T>
__global__ void __launch_bounds__(kBlock)
k_igf(double *__restrict__ out, T *__restrict__ far, int nx, int ny, int nz,
      const DevDom *__restrict__ dom, const double *__restrict__ tab,
      IgfBox *__restrict__ box) {
  __shared__ double C[kIgfTerms];
  igf_block<T>(out, far, nx, ny, nz, dom, tab, box, C, (int)blockIdx.x, (int)gridDim.x);
}

// --------------------------------------------------------------- deposit
// Lower-node cell (0-based) and CIC weights of deposit_BeamBunch
// (src/Appl/BeamBunch.f90:3737-3744) in the position type P.  The multiply and
// the add are fused by name, as the compiler fuses them: the kernels of one
// binned deposit then agree on every particle's cell by construction.
template <typename P>
struct Cic {
  int i, j, k;
  P ab, cd, ef;
};

template <typename P>
__device__ inline Cic<P> cic_of(P x, P y, P z, P xmin, P ymin, P zmin, P hx, P hy,
                                P hz, P hxi, P hyi, P hzi) {
  Cic<P> c;
  int ix = (int)fma(x - xmin, hxi, (P)1);
  c.ab = ((xmin - x) + ix * hx) * hxi;
  int jx = (int)fma(y - ymin, hyi, (P)1);
  c.cd = ((ymin - y) + jx * hy) * hyi;
  int kx = (int)fma(z - zmin, hzi, (P)1);
  c.ef = ((zmin - z) + kx * hz) * hzi;
  c.i = ix - 1;
  c.j = jx - 1;
  c.k = kx - 1;
  return c;
}

// x rounded to the nearest integer (ties to even), as __double2ll_rn.
// FAST: valid for |x| < 2^50 (the launch checks that every contribution is
// below it): adding 1.5 * 2^52 leaves round(x) in the low mantissa bits, one
// add and one integer subtract instead of the split conversion.
template <bool FAST>
__device__ inline long long fx_round(double x) {
  if constexpr (FAST) {
    const double t = __dadd_rn(x, 6755399441055744.0);
    return (long long)(__double_as_longlong(t) - 0x4338000000000000LL);
  } else {
    return __double2ll_rn(x);
  }
}

// Fixed-point contributions of one particle, in the reference's node order.
template <typename P, bool FAST = false>
__device__ inline void cic_contrib(const Cic<P> &c, double wq, long long v[8]) {
  // each product is rounded to FP64 before it is rounded to an integer: no
  // multiply may fuse with the short form's add
#pragma clang fp contract(off)
  const P one = (P)1;
  const P a = c.ab, b = c.cd, e = c.ef;
  v[0] = fx_round<FAST>((double)(a * b * e) * wq);
  v[1] = fx_round<FAST>((double)(a * (one - b) * e) * wq);
  v[2] = fx_round<FAST>((double)(a * (one - b) * (one - e)) * wq);
  v[3] = fx_round<FAST>((double)(a * b * (one - e)) * wq);
  v[4] = fx_round<FAST>((double)((one - a) * b * (one - e)) * wq);
  v[5] = fx_round<FAST>((double)((one - a) * (one - b) * (one - e)) * wq);
  v[6] = fx_round<FAST>((double)((one - a) * (one - b) * e) * wq);
  v[7] = fx_round<FAST>((double)((one - a) * b * e) * wq);
}

// Node offsets (di, dj, dk) in the order of cic_contrib.
__constant__ int kNode[8][3] = {{0, 0, 0}, {0, 1, 0}, {0, 1, 1}, {0, 0, 1},
                                {1, 0, 1}, {1, 1, 1}, {1, 1, 0}, {1, 0, 0}};

// ---- izh_charge: deposit_BeamBunch (src/Appl/BeamBunch.f90:3678-3768) for
// the bunch's own rows (t frame, FP64), which are in no spatial order.
// Particles with a NaN x and nodes outside the grid are skipped, as the
// reference skips them (:3746-3747).  Values are fixed point (int64, scale
// 2^e), so the result is exact and independent of the order of the additions,
// and every form below gives the same bits.
struct DepRows {
  const double *x, *y, *z;
  const uint32_t *orig;
  const double *w0;        // charge weights by original index, or w for all
  double w;
  int uniform;
  int64_t n;
  const DevDom *dom;
  int nx, ny, nz;
  double scale;
};

__device__ inline double row_weight(const DepRows &d, int64_t i) {
  return d.uniform ? d.w : d.w0[d.orig[i]];
}

// The particle's lower node and weights; false when it deposits nothing.
__device__ inline bool row_cic(const DepRows &d, double x, double y, double z, Cic<double> &c) {
  if (!(x == x)) return false;
  c = cic_of<double>(x, y, z, d.dom->range[0], d.dom->range[2], d.dom->range[4],
                     d.dom->msize[0], d.dom->msize[1], d.dom->msize[2], d.dom->hinv[0],
                     d.dom->hinv[1], d.dom->hinv[2]);
  return c.i >= 0 && c.i + 1 < d.nx && c.j >= 0 && c.j + 1 < d.ny && c.k >= 0 &&
         c.k + 1 < d.nz;
}

// One thread per particle, straight to the grid: a few thousand particles, or
// no memory for the bins.
__global__ void __launch_bounds__(kBlock)
k_deposit_direct(DepRows d, unsigned long long *__restrict__ rho) {
  const int64_t sy = d.nx, sz = (int64_t)d.nx * d.ny;
  for (int64_t i = blockIdx.x * (int64_t)kBlock + threadIdx.x; i < d.n;
       i += (int64_t)gridDim.x * kBlock) {
    Cic<double> c;
    if (!row_cic(d, d.x[i], d.y[i], d.z[i], c)) continue;
    long long v[8];
    cic_contrib<double>(c, row_weight(d, i) * d.scale, v);
    const int64_t g0 = c.i + sy * c.j + sz * c.k;
#pragma unroll
    for (int q = 0; q < 8; q++)
      atomicAdd(&rho[g0 + kNode[q][0] + sy * kNode[q][1] + sz * kNode[q][2]],
                (unsigned long long)v[q]);
  }
}

// A grid that fits LDS: each block accumulates all of it for its share of the
// particles and adds its nonzero nodes to the grid once.  On 16x16x32, us at
// kSmallPer 512 / 1024 / 2048 / 4096: 5k particles 9.9 / 10.0 / 11.1 / 12.5, 20k
// 8.8 / 10.0 / 11.6 / 16.3, 100k 12.9 / 11.4 / 12.1 / 16.6, 300k 20.0 / 20.4 /
// 16.7 / 17.8: shorter shares for few particles, fewer flushes for many.
constexpr int kSmallGrid = 8192;      // nodes: 64 KB, two blocks per CU
constexpr int kSmallPer = 1024;       // particles per block at least
constexpr int kSmallBlocks = 256;
__global__ void __launch_bounds__(kBlock)
k_deposit_small(DepRows d, unsigned long long *__restrict__ rho) {
  extern __shared__ __align__(16) unsigned long long small_win[];
  const int sy = d.nx, sz = d.nx * d.ny, g = sz * d.nz;  // g is even
  ulonglong2 *w2 = reinterpret_cast<ulonglong2 *>(small_win);
  for (int c = threadIdx.x; 2 * c < g; c += kBlock) w2[c] = make_ulonglong2(0ull, 0ull);
  __syncthreads();
  for (int64_t i = blockIdx.x * (int64_t)kBlock + threadIdx.x; i < d.n;
       i += (int64_t)gridDim.x * kBlock) {
    Cic<double> c;
    if (!row_cic(d, d.x[i], d.y[i], d.z[i], c)) continue;
    long long v[8];
    cic_contrib<double>(c, row_weight(d, i) * d.scale, v);
    const int l0 = c.i + sy * c.j + sz * c.k;
#pragma unroll
    for (int q = 0; q < 8; q++)
      atomicAdd(&small_win[l0 + kNode[q][0] + sy * kNode[q][1] + sz * kNode[q][2]],
                (unsigned long long)v[q]);
  }
  __syncthreads();
  for (int c = threadIdx.x; c < g; c += kBlock) {
    const unsigned long long v = small_win[c];
    if (v) atomicAdd(&rho[c], v);
  }
}

// Everything else is binned first: a counting sort of the positions by the
// tile of their lower node (count, scan, scatter), then one block per run of
// a tile accumulates in the tile's 9x9x9 nodes.  Straight to the grid, the
// int64 adds of scattered particles reach 17 G/s (2M on 64^3: 958 us, where
// the positions take 10 us to read).  The order the sort leaves within a tile
// varies from run to run and changes no bit of the sum.  The whole chain, us:
//   kBinPer 4 / 8 / 16        20k on 32^3 25.5 / 28.4 / 35.1, 300k on 64^3 41.6 /
//                             44.2 / 51.3, 2M on 64^3 86 / 85 / 88, 2M on 128^3
//                             143 / 139 / 136, 10M on 128x128x256 596 / 579 / 581
//   kBinChunk 1024 / 2048 /   100k on 32^3 28.9 / 31.9 / 38.6 / 49.2, 2M on 64^3
//   4096 / 8192               98 / 85 / 86 / 96, 10M on 128x128x256 612 / 579 /
//                             576 / 585
constexpr int kBinThreads = 512;
constexpr int kBinPer = 8;            // particles per thread of a scatter block
constexpr int kBinLdsTiles = 8192;    // tiles a block counts in LDS (32 KB)
constexpr int kBinCountBlocks = 512;
constexpr int kBinChunk = 2048;       // particles per deposit block at most

struct BinGrid {
  int s[3], tnx, tny, ntiles;         // tiles of 2^s nodes per axis
};

__device__ inline uint32_t bin_of(const BinGrid &b, const Cic<double> &c) {
  return (uint32_t)((c.i >> b.s[0]) +
                    b.tnx * ((c.j >> b.s[1]) + b.tny * (c.k >> b.s[2])));
}

template <bool LDS>
__global__ void __launch_bounds__(kBinThreads)
k_bin_count(DepRows d, BinGrid b, uint32_t *__restrict__ hist) {
  extern __shared__ uint32_t bin_lds[];
  if constexpr (LDS) {
    for (int t = threadIdx.x; t < b.ntiles; t += kBinThreads) bin_lds[t] = 0u;
    __syncthreads();
  }
  for (int64_t i = blockIdx.x * (int64_t)kBinThreads + threadIdx.x; i < d.n;
       i += (int64_t)gridDim.x * kBinThreads) {
    Cic<double> c;
    if (row_cic(d, d.x[i], d.y[i], d.z[i], c))
      atomicAdd(LDS ? &bin_lds[bin_of(b, c)] : &hist[bin_of(b, c)], 1u);
  }
  if constexpr (LDS) {
    __syncthreads();
    for (int t = threadIdx.x; t < b.ntiles; t += kBinThreads) {
      const uint32_t v = bin_lds[t];
      if (v) atomicAdd(&hist[t], v);
    }
  }
}

constexpr int kBinScanThreads = 1024;
__global__ void __launch_bounds__(kBinScanThreads)
k_bin_scan(uint32_t *hist, int ntiles, uint32_t *__restrict__ cursor,
           Chunk *__restrict__ chunks, int64_t *__restrict__ nchunks) {
  __shared__ uint32_t wsum[kBinScanThreads / 64][2];
  tile_scan<kBinScanThreads>(hist, ntiles, kBinChunk, cursor, chunks, nchunks, hist, wsum);
}

// A block ranks its 4096 particles within their tiles in LDS and takes each
// tile's slots with one add, so a tile's particles of a block land in one run.
template <bool LDS>
__global__ void __launch_bounds__(kBinThreads)
k_bin_scatter(DepRows d, BinGrid b, uint32_t *__restrict__ cursor, double *__restrict__ out,
              int64_t cap) {
  extern __shared__ uint32_t bin_lds[];
  const int64_t base = blockIdx.x * (int64_t)(kBinThreads * kBinPer);
  if constexpr (LDS) {
    for (int t = threadIdx.x; t < b.ntiles; t += kBinThreads) bin_lds[t] = 0u;
    __syncthreads();
  }
  double x[kBinPer], y[kBinPer], z[kBinPer];
  uint32_t key[kBinPer], rank[kBinPer];
#pragma unroll
  for (int u = 0; u < kBinPer; u++) {
    const int64_t i = base + u * kBinThreads + threadIdx.x;
    const int64_t j = i < d.n ? i : d.n - 1;
    x[u] = d.x[j]; y[u] = d.y[j]; z[u] = d.z[j];
  }
#pragma unroll
  for (int u = 0; u < kBinPer; u++) {
    const int64_t i = base + u * kBinThreads + threadIdx.x;
    Cic<double> c;
    key[u] = kDeadKey;
    rank[u] = 0u;
    if (i < d.n && row_cic(d, x[u], y[u], z[u], c)) {
      key[u] = bin_of(b, c);
      rank[u] = atomicAdd(LDS ? &bin_lds[key[u]] : &cursor[key[u]], 1u);
    }
  }
  if constexpr (LDS) {
    __syncthreads();
    for (int t = threadIdx.x; t < b.ntiles; t += kBinThreads) {
      const uint32_t v = bin_lds[t];
      if (v) bin_lds[t] = atomicAdd(&cursor[t], v);
    }
    __syncthreads();
  }
#pragma unroll
  for (int u = 0; u < kBinPer; u++) {
    if (key[u] == kDeadKey) continue;
    const int64_t q = (LDS ? bin_lds[key[u]] : 0u) + rank[u];
    out[q] = x[u];
    out[cap + q] = y[u];
    out[2 * cap + q] = z[u];
    if (!d.uniform)
      out[3 * cap + q] = row_weight(d, base + u * kBinThreads + threadIdx.x);
  }
}

// FAST: as k_deposit_tiles.  WE: nodes per axis of the window.
template <bool FAST, int WE>
__global__ void __launch_bounds__(kBlock)
k_deposit_binned(DepRows d, BinGrid b, const double *__restrict__ bin, int64_t cap,
                 const Chunk *__restrict__ chunks, const int64_t *__restrict__ nchunks,
                 unsigned long long *__restrict__ rho) {
  __shared__ unsigned long long win[WE * WE * WE];
  if (blockIdx.x >= *nchunks) return;
  const Chunk ch = chunks[blockIdx.x];
  const int txy = b.tnx * b.tny;
  const int tz = (int)ch.tile / txy, rem = (int)ch.tile - tz * txy;
  const int ty = rem / b.tnx, tx = rem - ty * b.tnx;
  const int bx = tx << b.s[0], by = ty << b.s[1], bz = tz << b.s[2];
  for (int c = threadIdx.x; c < WE * WE * WE; c += kBlock) win[c] = 0ull;
  __syncthreads();
  for (uint32_t t = threadIdx.x; t < ch.len; t += kBlock) {
    const int64_t i = (int64_t)ch.start + t;
    Cic<double> c;
    // binned particles all deposit, in this tile
    row_cic(d, bin[i], bin[cap + i], bin[2 * cap + i], c);
    const double w = d.uniform ? d.w : bin[3 * cap + i];
    long long v[8];
    cic_contrib<double, FAST>(c, w * d.scale, v);
    const int l0 = (c.i - bx) + WE * ((c.j - by) + WE * (c.k - bz));
#pragma unroll
    for (int q = 0; q < 8; q++)
      atomicAdd(&win[l0 + kNode[q][0] + WE * (kNode[q][1] + WE * kNode[q][2])],
                (unsigned long long)v[q]);
  }
  __syncthreads();
  const int64_t sy = d.nx, sz = (int64_t)d.nx * d.ny;
  for (int c = threadIdx.x; c < WE * WE * WE; c += kBlock) {
    const unsigned long long v = win[c];
    if (v == 0ull) continue;
    const int lx = c % WE, ly = (c / WE) % WE, lz = c / (WE * WE);
    atomicAdd(&rho[(bx + lx) + sy * (by + ly) + sz * (bz + lz)], v);
  }
}

// The fused run's deposit.  Each block takes one chunk of the sorted bunch:
// at most kChunk slots grouped under one sort tile (the tile of the
// particles' previous position, in the grid *kgrid that key was computed
// in).  The block accumulates in an LDS window of the tile's nodes, mapped
// into this step's grid and widened on every side (plus the upper CIC node)
// by kTileMarginT nodes across the beam and kTileMarginL along it, so no
// pass over the positions is needed to bound them; particles that moved
// further add to the grid directly and are counted in *spill.  The margins
// follow how far particles move in cells between the key and the deposit
// (one or two steps): transversely several cells in a drift step, along the
// bunch (the t-frame phase) about one.  Same fixed-point arithmetic and
// node order as izh_charge's.  A block of few particles is bound by
// clearing and flushing its window (5733 nodes): the window's pitch is fixed
// and it is cleared 16 bytes a lane, which took a flush's cell index from two
// integer divisions to multiplies (100k particles on 32^3: 9.4 -> 7.9 us).
// 512 threads a block gained where chunks are full (4M on 32^3: 38 -> 34 us)
// and lost more where tiles are sparse (10M on 128x128x256: 264 -> 300 us).
// The positions are read once and then rewritten by the next pass, so they are
// read past the caches, which keep the grid and the rows instead (16 steps:
// 2M on 64^3 3.74 -> 3.72 ms, 4M on 32^3 mixed 4.24 -> 4.17, 10M on 64^3 10.57
// -> 10.41, 50M on 128x128x256 61.7 -> 61.4; 137k and 1.2M unchanged).
constexpr int kTileMarginT = 6;
constexpr int kTileMarginL = 2;
constexpr int kTileWinEdgeT = (1 << kTileShift) + 1 + 2 * kTileMarginT;
constexpr int kTileWinEdgeL = (1 << kTileShift) + 1 + 2 * kTileMarginL;
constexpr int kTileWinCells = kTileWinEdgeT * kTileWinEdgeT * kTileWinEdgeL;

constexpr int kDepThreads = 256;
// Consecutive chunks one XCD takes in a row (a row of tiles at 128 nodes):
// their windows overlap, and one L2 then merges the flushes (100k on 32^3:
// 8.5 -> 7.9 us, 2M on 64^3 59 -> 57 us, 50M on 128x128x256 474 -> 470 us;
// runs of 64 unbalance the XCDs between core and halo: 507 us).
constexpr int kDepRun = 16;

// Chunk of physical block p of n: XCD p mod 8 takes every eighth run of
// kDepRun consecutive chunks.
__device__ inline int dep_chunk(int p, int n) {
  const int span = 8 * kDepRun, s = p / span;
  if ((s + 1) * span > n) return p;  // the incomplete last span: in order
  const int r = p - s * span;
  return s * span + (r & 7) * kDepRun + (r >> 3);
}

template <typename P, bool FAST>
__global__ void __launch_bounds__(kDepThreads)
k_deposit_tiles(const P *__restrict__ X, const P *__restrict__ Y,
                const P *__restrict__ Z, const uint32_t *__restrict__ orig,
                const double *__restrict__ w0, double w_uniform, int uniform,
                const Chunk *__restrict__ chunks, const int64_t *__restrict__ d_nchunks,
                const KeyGrid *__restrict__ kgrid, const DevDom *__restrict__ dom, int nx,
                int ny, int nz, int s0, int s1, int s2, int tnx, int tny, double scale,
                unsigned long long *__restrict__ rho, int64_t *__restrict__ spill,
                double *__restrict__ corner, P *__restrict__ far,
                const double *__restrict__ igf_tab, IgfBox *__restrict__ box, int ncorner) {
  __shared__ __align__(16) unsigned long long win[kTileWinCells + 1];
  // the first ncorner blocks (a multiple of eight) prepare the step's Green
  // function, which needs only the domain: arithmetic beside the deposit's
  // LDS traffic, and no launch of its own
  if ((int)blockIdx.x < ncorner) {
    igf_block<P>(corner, far, nx, ny, nz, dom, igf_tab, box, reinterpret_cast<double *>(win),
                 (int)blockIdx.x, ncorner);
    return;
  }
  const int bid = (int)blockIdx.x - ncorner;
  const int64_t nchunks = *d_nchunks;
  if (bid >= nchunks) return;
  const Chunk ch = chunks[dep_chunk(bid, (int)nchunks)];
  const int tz = (int)(ch.tile / ((uint32_t)tnx * (uint32_t)tny));
  const int rem = (int)(ch.tile % ((uint32_t)tnx * (uint32_t)tny));
  const int ty = rem / tnx, tx = rem % tnx;
  const int wx = min((1 << s0) + 1 + 2 * kTileMarginT, nx);
  const int wy = min((1 << s1) + 1 + 2 * kTileMarginT, ny);
  const int wz = min((1 << s2) + 1 + 2 * kTileMarginL, nz);
  const KeyGrid kg = *kgrid;
  const int bx = min(max(tile_first_node(tx << s0, kg.lo[0], kg.h[0], dom->range[0],
                                         dom->hinv[0]) - kTileMarginT, 0), nx - wx);
  const int by = min(max(tile_first_node(ty << s1, kg.lo[1], kg.h[1], dom->range[2],
                                         dom->hinv[1]) - kTileMarginT, 0), ny - wy);
  const int bz = min(max(tile_first_node(tz << s2, kg.lo[2], kg.h[2], dom->range[4],
                                         dom->hinv[2]) - kTileMarginL, 0), nz - wz);
  // the window's rows keep the full pitch on a smaller grid too, so the
  // flush splits a cell's index by constants
  constexpr int kWx = kTileWinEdgeT, kWy = kTileWinEdgeT;
  const int wcells = kWx * kWy * wz;
  {
    ulonglong2 *w2 = reinterpret_cast<ulonglong2 *>(win);
    for (int c = threadIdx.x; 2 * c < wcells; c += kDepThreads) w2[c] = make_ulonglong2(0ull, 0ull);
  }
  __syncthreads();
  const P xmin = (P)dom->range[0], ymin = (P)dom->range[2], zmin = (P)dom->range[4];
  const P hx = (P)dom->msize[0], hy = (P)dom->msize[1], hz = (P)dom->msize[2];
  const P hxi = (P)dom->hinv[0], hyi = (P)dom->hinv[1], hzi = (P)dom->hinv[2];
  const int64_t sy = nx, sz = (int64_t)nx * ny;
  uint32_t nspill = 0;
  // kDepBatch slots per thread per round: all their loads are issued first
  constexpr int kDepBatch = 4;
  for (uint32_t t0 = threadIdx.x; t0 < ch.len; t0 += kDepBatch * kDepThreads) {
    P px[kDepBatch], py[kDepBatch], pz[kDepBatch];
    double pw[kDepBatch];
#pragma unroll
    for (int u = 0; u < kDepBatch; u++) {
      const uint32_t t = t0 + u * kDepThreads;
      const int64_t i = (int64_t)ch.start + (t < ch.len ? t : ch.len - 1);
      const P xi = __builtin_nontemporal_load(X + i);
      px[u] = t < ch.len ? xi : (P)NAN;
      py[u] = __builtin_nontemporal_load(Y + i);
      pz[u] = __builtin_nontemporal_load(Z + i);
      pw[u] = uniform ? w_uniform : w0[orig[i]];
    }
#pragma unroll
    for (int u = 0; u < kDepBatch; u++) {
      const P x = px[u];
      if (!(x == x)) continue;
      const Cic<P> c = cic_of<P>(x, py[u], pz[u], xmin, ymin, zmin, hx, hy, hz, hxi,
                                 hyi, hzi);
      if (c.i < 0 || c.i + 1 >= nx || c.j < 0 || c.j + 1 >= ny || c.k < 0 ||
          c.k + 1 >= nz)
        continue;
      long long v[8];
      cic_contrib<P, FAST>(c, pw[u] * scale, v);
      const int li = c.i - bx, lj = c.j - by, lk = c.k - bz;
      if (li >= 0 && li + 1 < wx && lj >= 0 && lj + 1 < wy && lk >= 0 && lk + 1 < wz) {
        const int l0 = li + kWx * (lj + kWy * lk);
#pragma unroll
        for (int q = 0; q < 8; q++)
          atomicAdd(&win[l0 + kNode[q][0] + kWx * (kNode[q][1] + kWy * kNode[q][2])],
                    (unsigned long long)v[q]);
      } else {
        const int64_t g0 = c.i + sy * c.j + sz * c.k;
#pragma unroll
        for (int q = 0; q < 8; q++)
          atomicAdd(&rho[g0 + kNode[q][0] + sy * kNode[q][1] + sz * kNode[q][2]],
                    (unsigned long long)v[q]);
        nspill++;
      }
    }
  }
  __syncthreads();
  for (int c = threadIdx.x; c < wcells; c += kDepThreads) {
    const unsigned long long v = win[c];
    if (v == 0ull) continue;
    const int lx = c % kWx, ly = (c / kWx) % kWy, lz = c / (kWx * kWy);
    atomicAdd(&rho[(bx + lx) + sy * (by + ly) + sz * (bz + lz)], v);
  }
  if (spill) {
    int tot = (int)nspill;
    for (int off = 32; off > 0; off >>= 1) tot += __shfl_down(tot, off, 64);
    if ((threadIdx.x & 63) == 0 && tot > 0)
      atomicAdd((unsigned long long *)spill, (unsigned long long)tot);
  }
}

__global__ void k_fill_u32(uint32_t *__restrict__ p, int64_t n, uint32_t v) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    p[i] = v;
}

// The grid charge of one izh_charge, and the accumulator cleared for the next
// deposit (field_alloc clears it first; the fused run's forward x pass does
// both as it reads).
template <typename T>
__global__ void k_fx_to_grid(unsigned long long *__restrict__ fx, T *__restrict__ rho,
                             int64_t n, double inv) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    rho[i] = (T)((double)(long long)fx[i] * inv);
    fx[i] = 0ull;
  }
}

// ------------------------------------------------------------- E field
// kick1_BeamBunch one-process Flagbc=1 stencils (src/Appl/BeamBunch.f90:
// 1782-1794, 1885-1899, 1966-2005): central differences, one-sided at edges,
// written interleaved (Ex, Ey, Ez, 0) for the 8-node gather.
template <typename T>
__global__ void k_efield(const T *__restrict__ phi, E4<T> *__restrict__ e,
                         int nx, int ny, int nz, const DevDom *__restrict__ dom) {
  const int sy = nx, sz = nx * ny, n = sz * nz;
  const T hx = (T)dom->hinv[0], hy = (T)dom->hinv[1], hz = (T)dom->hinv[2];
  const T hx2 = (T)(0.5 * dom->hinv[0]), hy2 = (T)(0.5 * dom->hinv[1]),
          hz2 = (T)(0.5 * dom->hinv[2]);
  for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < n;
       c += gridDim.x * blockDim.x) {
    int i = c % nx;
    int j = (c / nx) % ny;
    int k = c / sz;
    E4<T> v;
    if (i == 0) v.x = hx * (phi[c] - phi[c + 1]);
    else if (i == nx - 1) v.x = hx * (phi[c - 1] - phi[c]);
    else v.x = hx2 * (phi[c - 1] - phi[c + 1]);
    if (j == 0) v.y = hy * (phi[c] - phi[c + sy]);
    else if (j == ny - 1) v.y = hy * (phi[c - sy] - phi[c]);
    else v.y = hy2 * (phi[c - sy] - phi[c + sy]);
    if (k == 0) v.z = hz * (phi[c] - phi[c + sz]);
    else if (k == nz - 1) v.z = hz * (phi[c - sz] - phi[c]);
    else v.z = hz2 * (phi[c - sz] - phi[c + sz]);
    v.w = (T)0;
    e[c] = v;
  }
}

int ilog2(int v) {
  int r = 0;
  while ((1 << r) < v) r++;
  return r;
}

// Completes a pass's description (block shape, index multiplier) and checks it
// against what the kernel assumes; *nblk: its blocks.
int lines_setup(Lines &p, int pts, bool pair, int64_t *nblk) {
  p.log2L = ilog2(p.L);
  if (p.nfv == 0) p.nfv = p.nf;
  if (p.L < kFftMinLine || p.L > pts || (1 << p.log2L) != p.L)
    return fail(IZH_ERR_ARG, "FFT line of %d points: not a power of two in %d..%d", p.L,
                kFftMinLine, pts);
  p.B = pts / p.L;
  p.log2B = ilog2(p.B);
  // line / nf is a multiply by ceil(2^40 / nf), exact below these bounds
  if (p.nf < 1 || p.nf >= (1 << 16) || 2 * p.nf * p.ns >= (1 << 24))
    return fail(IZH_ERR_ARG, "FFT of %lld x %lld lines outside the kernel's index range",
                (long long)p.nf, (long long)p.ns);
  p.nf_mul = ((1ull << 40) + (uint64_t)p.nf - 1) / (uint64_t)p.nf;
  const int64_t nlines = p.nf * p.ns;
  const int64_t nfft = pair ? (nlines + 1) / 2 : nlines;
  *nblk = (nfft + p.B - 1) / p.B;
  return IZH_OK;
}

template <typename T, int LOAD, int STORE, bool CONV, bool PAIR = false>
int run_lines(hipStream_t stream, Lines p, const void *tw, bool inverse) {
  // the fused z pass takes twice the lines per block: its rows of the
  // spectrum and of G^ are read across the lines
  constexpr int pts = CONV ? kFftPointsZ : kFftPoints;
  int64_t nblk = 0;
  IZH_CHECK(lines_setup(p, pts, PAIR, &nblk));
  const size_t tw_bytes = (size_t)(p.L / 2) * sizeof(cx<T>);
  const dim3 g((unsigned)nblk), b(kFftThreads);
  const cx<T> *twc = (const cx<T> *)tw;
  const int inv = inverse ? 1 : 0;
  // the line lengths of the 32^3 .. 128x128x256 grids as compile-time sizes
  switch (p.log2L) {
    case 6:
      hipLaunchKernelGGL((k_fft_lines<T, LOAD, STORE, CONV, PAIR, pts, 6>), g, b, tw_bytes,
                         stream, p, twc, inv);
      break;
    case 7:
      hipLaunchKernelGGL((k_fft_lines<T, LOAD, STORE, CONV, PAIR, pts, 7>), g, b, tw_bytes,
                         stream, p, twc, inv);
      break;
    case 8:
      hipLaunchKernelGGL((k_fft_lines<T, LOAD, STORE, CONV, PAIR, pts, 8>), g, b, tw_bytes,
                         stream, p, twc, inv);
      break;
    case 9:
      hipLaunchKernelGGL((k_fft_lines<T, LOAD, STORE, CONV, PAIR, pts, 9>), g, b, tw_bytes,
                         stream, p, twc, inv);
      break;
    default:
      hipLaunchKernelGGL((k_fft_lines<T, LOAD, STORE, CONV, PAIR, pts, 0>), g, b, tw_bytes,
                         stream, p, twc, inv);
      break;
  }
  IZH_HIP(hipGetLastError());
  return IZH_OK;
}

// k_fft_two: the Green function's lines ga and the charge's lines cb, of one
// length.
template <typename T, int LOADA, int LOADB, int STOREB, bool PAIRB>
int run_two(hipStream_t stream, Lines ga, Lines cb, const void *tw) {
  int64_t nba = 0, nbb = 0;
  if (ga.L != cb.L) return fail(IZH_ERR_ARG, "FFT passes of %d and %d points", ga.L, cb.L);
  IZH_CHECK(lines_setup(ga, kFftPoints, true, &nba));
  IZH_CHECK(lines_setup(cb, kFftPoints, PAIRB, &nbb));
  const size_t tw_bytes = (size_t)(ga.L / 2) * sizeof(cx<T>);
  const dim3 g((unsigned)(((nba + 7) & ~(int64_t)7) + nbb)), b(kFftThreads);
  const cx<T> *twc = (const cx<T> *)tw;
  const int na = (int)nba, nb = (int)nbb;
  switch (ga.log2L) {
    case 6:
      hipLaunchKernelGGL((k_fft_two<T, LOADA, LOADB, STOREB, PAIRB, 6>), g, b, tw_bytes,
                         stream, ga, cb, na, nb, twc);
      break;
    case 7:
      hipLaunchKernelGGL((k_fft_two<T, LOADA, LOADB, STOREB, PAIRB, 7>), g, b, tw_bytes,
                         stream, ga, cb, na, nb, twc);
      break;
    case 8:
      hipLaunchKernelGGL((k_fft_two<T, LOADA, LOADB, STOREB, PAIRB, 8>), g, b, tw_bytes,
                         stream, ga, cb, na, nb, twc);
      break;
    case 9:
      hipLaunchKernelGGL((k_fft_two<T, LOADA, LOADB, STOREB, PAIRB, 9>), g, b, tw_bytes,
                         stream, ga, cb, na, nb, twc);
      break;
    default:
      hipLaunchKernelGGL((k_fft_two<T, LOADA, LOADB, STOREB, PAIRB, 0>), g, b, tw_bytes,
                         stream, ga, cb, na, nb, twc);
      break;
  }
  IZH_HIP(hipGetLastError());
  return IZH_OK;
}

// The convolution: the transforms of G (from its corners) and of the charge,
// pass by pass in common launches, the fused z pass, inverse y, inverse x, on
// the field's stream.  FX: the charge is the deposit's fixed-point
// accumulator, converted (and cleared) as it is read; else the grid rho.
template <typename T, bool FX>
int convolve_t(izh_field *f) {
  const int nx = f->nx, ny = f->ny, nz = f->nz;
  const int mx = 2 * nx, my = 2 * ny, mz = 2 * nz, kx = nx + 1;
  const hipStream_t fs = f->stream;
  ScopedTimer tm_(IZH_T_FFT, fs);
  // The half spectra hold x rows of ld = f->ldx >= kx values.  The y and z
  // passes run over all ld x lines, so a block's run of neighbouring lines
  // starts on a 128-byte boundary; lines kx..ld-1 are padding.
  const int64_t ld = f->ldx;
  Lines g{}, p{};
  // ---- x: lines (j<=ny, k<=nz) of G as they are formed -> green, and
  // rho (nx,ny,nz) real -> A (kx of ld, ny, nz)
  g.src = f->corner; g.dst = f->green;
  g.tx = nx + 2; g.ty = ny + 2;
  g.far = f->green_t; g.box = f->igf_box;
  g.nf = ny + 1; g.ns = nz + 1;
  g.df = kx; g.ds = (int64_t)kx * (ny + 1); g.de = 1;
  g.L = mx; g.Lin = g.L; g.Lout = nx + 1; g.out_scale = 1.0;
  p.src = FX ? (const void *)f->rho_fx : f->rho; p.dst = f->spec_a;
  p.rho = f->rho; p.fx_inv = f->rho_scale / f->fixed_scale;
  p.nf = ny; p.ns = nz;
  p.sf = nx; p.ss = (int64_t)nx * ny; p.se = 1;
  p.df = ld; p.ds = ld * ny; p.de = 1;
  p.L = mx; p.Lin = nx; p.Lout = kx; p.out_scale = 1.0;
  IZH_CHECK((run_two<T, kLoadIgf, FX ? kLoadFx : kLoadReal, kStoreCplx, true>(fs, g, p,
                                                                            f->tw_x)));
  // ---- y: lines (i<=nx, k<=nz) of green -> green_t, and A -> B (kx of ld, my, nz)
  g.src = f->green; g.dst = f->green_t;
  g.nf = kx; g.ns = nz + 1;
  g.sf = 1; g.ss = (int64_t)kx * (ny + 1); g.se = kx;
  g.df = 1; g.ds = (int64_t)kx * (ny + 1); g.de = kx;
  g.L = my; g.Lin = g.L; g.Lout = ny + 1;
  p.src = f->spec_a; p.dst = f->spec_b;
  p.nf = ld; p.nfv = kx; p.ns = nz;
  p.sf = 1; p.ss = ld * ny; p.se = ld;
  p.df = 1; p.ds = ld * my; p.de = ld;
  p.L = my; p.Lin = ny; p.Lout = my;
  IZH_CHECK((run_two<T, kLoadEven, kLoadCplx, kStoreCplx, false>(fs, g, p, f->tw_y)));
  // ---- z of G: lines (i<=nx, j<=ny); green_t -> green, scaled by
  // 1/(mx my mz).  G^ is stored [j][k][i] with i rows at the spectra's pitch
  // ldx: the fused z pass of a block of x lines then reads, for its one y
  // index, aligned runs of neighbouring i at neighbouring k, one contiguous
  // region of ldx*(nz+1) values instead of one value run per z plane.
  g.src = f->green_t; g.dst = f->green;
  g.nf = kx; g.ns = ny + 1;
  g.sf = 1; g.ss = kx; g.se = (int64_t)kx * (ny + 1);
  g.df = 1; g.ds = ld * (nz + 1); g.de = ld;
  g.L = mz; g.Lin = g.L; g.Lout = nz + 1;
  g.out_scale = 1.0 / ((double)mx * my * mz);
  IZH_CHECK((run_lines<T, kLoadEven, kStoreReal, false, true>(fs, g, f->tw_z, false)));
  // ---- z: FFT, * G^, IFFT, keep k < nz; in place in B
  p.src = f->spec_b; p.dst = f->spec_b;
  p.nf = ld; p.nfv = kx; p.ns = my;
  p.sf = 1; p.ss = ld; p.se = ld * my;
  p.df = 1; p.ds = ld; p.de = ld * my;
  p.L = mz; p.Lin = nz; p.Lout = nz;
  p.green = f->green; p.gkx = ld * (nz + 1); p.gky = ld; p.my = my;
  IZH_CHECK((run_lines<T, kLoadCplx, kStoreCplx, true>(fs, p, f->tw_z, false)));
  // ---- inverse y: B -> A, keep j < ny
  p.green = nullptr;
  p.src = f->spec_b; p.dst = f->spec_a;
  p.nf = ld; p.nfv = kx; p.ns = nz;
  p.sf = 1; p.ss = ld * my; p.se = ld;
  p.df = 1; p.ds = ld * ny; p.de = ld;
  p.L = my; p.Lin = my; p.Lout = ny;
  IZH_CHECK((run_lines<T, kLoadCplx, kStoreCplx, false>(fs, p, f->tw_y, true)));
  // ---- inverse x (C2R): A -> phi, keep i < nx
  p.src = f->spec_a; p.dst = f->phi;
  p.nf = ny; p.nfv = ny; p.ns = nz;
  p.sf = ld; p.ss = ld * ny; p.se = 1;
  p.df = nx; p.ds = (int64_t)nx * ny; p.de = 1;
  p.L = mx; p.Lin = mx; p.Lout = nx;
  IZH_CHECK((run_lines<T, kLoadHerm, kStoreReal, false, true>(fs, p, f->tw_x, true)));
  return IZH_OK;
}

template <typename T>
void make_twiddles(cx<T> *tw, int L) {
  for (int t = 0; t < L / 2; t++) {
    long double a = -2.0L * 3.141592653589793238462643383279502884L * t / L;
    tw[t] = {(T)cosl(a), (T)sinl(a)};
  }
}

// The series' table: tab[t * kIgfTerms + u] is what the derivative of 1/r of
// orders (2i, 2j, 2k), u = igf_term(i, j, k), adds to term t per monomial
// hx^2i hy^2j hz^2k: the derivative's polynomial P / r^(2n+1) by
// d/dx (P r^-m) = (r^2 dP/dx - m x P) r^-(m+2), times the mean of s^2i / (2i)!
// over the cell, 1 / (4^i (2i+1)!), and alike for y and z.  P's term
// x^2p y^2q z^2r / r^(2n) is a^p b^q c^r.
std::vector<double> igf_table() {
  using Exps = std::array<int, 3>;
  std::vector<double> tab((size_t)kIgfTerms * kIgfTerms, 0.0);
  long double fact[2 * kIgfOrder + 2] = {1.0L};
  for (int q = 1; q < 2 * kIgfOrder + 2; q++) fact[q] = fact[q - 1] * q;
  for (int i = 0; i <= kIgfOrder; i++)
    for (int j = 0; i + j <= kIgfOrder; j++)
      for (int k = 0; i + j + k <= kIgfOrder; k++) {
        const int n[3] = {i, j, k}, u = igf_term(i, j, k);
        std::map<Exps, long double> P{{Exps{0, 0, 0}, 1.0L}};
        int m = 1;
        long double w = 1.0L;
        for (int a = 0; a < 3; a++) {
          w /= powl(4.0L, n[a]) * fact[2 * n[a] + 1];
          for (int d = 0; d < 2 * n[a]; d++, m += 2) {
            std::map<Exps, long double> Q;
            for (const auto &t : P) {
              Exps e = t.first;
              e[a]++;
              Q[e] -= m * t.second;
              if (t.first[a] == 0) continue;
              e = t.first;
              e[a]--;
              for (int c = 0; c < 3; c++) {
                Exps f = e;
                f[c] += 2;
                Q[f] += t.first[a] * t.second;
              }
            }
            P = Q;
          }
        }
        for (const auto &t : P)
          if (t.second != 0.0L)
            tab[(size_t)igf_term(t.first[0] / 2, t.first[1] / 2, t.first[2] / 2) * kIgfTerms +
                u] = (double)(w * t.second);
      }
  return tab;
}

// Twiddles of the three line lengths and the series' table, in one buffer.
template <typename T>
int upload_tables(izh_field *f) {
  static const std::vector<double> igf = igf_table();
  const int len[3] = {2 * f->nx, 2 * f->ny, 2 * f->nz};
  size_t at[4] = {0, 0, 0, 0}, bytes = igf.size() * sizeof(double);
  for (int a = 0; a < 3; a++) {
    at[a] = bytes;
    bytes = (bytes + len[a] / 2 * sizeof(cx<T>) + 255) / 256 * 256;
  }
  std::vector<char> host(bytes);
  std::memcpy(host.data(), igf.data(), igf.size() * sizeof(double));
  for (int a = 0; a < 3; a++) make_twiddles<T>((cx<T> *)(host.data() + at[a]), len[a]);
  IZH_HIP(dev_malloc((void **)&f->tables, bytes));
  IZH_HIP(hipMemcpy(f->tables, host.data(), bytes, hipMemcpyHostToDevice));
  f->igf_tab = (const double *)f->tables;
  f->tw_x = f->tables + at[0];
  f->tw_y = f->tables + at[1];
  f->tw_z = f->tables + at[2];
  return IZH_OK;
}

}  // namespace

// ================================================================ launchers

double fixed_point_scale(double wabs_sum) {
  // every cell holds at most sum|w| (CIC weights of a particle sum to one),
  // so 2^e * sum|w| <= 2^61 leaves headroom for the +-0.5 rounding per term
  double wsum = wabs_sum > 0 ? wabs_sum : 1.0;
  int e = 61 - (int)std::ceil(std::log2(wsum));
  return std::ldexp(1.0, e);
}

int field_alloc(izh_field *f) {
  const size_t es = f->precision == IZH_FP64 ? sizeof(double) : sizeof(float);
  const int64_t g = f->g, kx = f->nx + 1;
  const int64_t ghalf = kx * (f->ny + 1) * (f->nz + 1);
  // rows of whole 128-byte lines: the y and z passes read and write runs of
  // neighbouring x lines, which then start on a line boundary
  const int64_t row = 128 / (2 * (int64_t)es);
  f->ldx = (kx + row - 1) / row * row;
  IZH_HIP(dev_malloc((void **)&f->rho_fx, g * sizeof(unsigned long long)));
  IZH_HIP(hipMemset(f->rho_fx, 0, g * sizeof(unsigned long long)));
  IZH_HIP(dev_malloc(&f->rho, g * es));
  IZH_HIP(dev_malloc(&f->phi, g * es));
  IZH_HIP(dev_malloc(&f->e, 4 * g * es));
  IZH_HIP(dev_malloc(&f->spec_a, f->ldx * f->ny * f->nz * 2 * es));
  IZH_HIP(dev_malloc(&f->spec_b, f->ldx * 2 * f->ny * f->nz * 2 * es));
  // G^ at x pitch ldx ([j][k][i], written by its z pass; the x pass's
  // output at pitch kx fits as well)
  IZH_HIP(dev_malloc(&f->green, f->ldx * (f->ny + 1) * (f->nz + 1) * es));
  IZH_HIP(dev_malloc(&f->green_t, ghalf * es));
  IZH_HIP(dev_malloc((void **)&f->corner,
                    (size_t)(f->nx + 2) * (f->ny + 2) * (f->nz + 2) * sizeof(double)));
  IZH_HIP(dev_malloc((void **)&f->d_dom, sizeof(DevDom)));
  IZH_HIP(hipHostMalloc((void **)&f->h_dom, sizeof(DevDom), hipHostMallocDefault));
  IZH_HIP(hipMemset(f->d_dom, 0, sizeof(DevDom)));
  IZH_HIP(dev_malloc((void **)&f->igf_box, sizeof(IgfBox)));
  if (f->precision == IZH_FP64) return upload_tables<double>(f);
  return upload_tables<float>(f);
}

uint64_t next_stamp() {
  static std::atomic<uint64_t> last{0};
  return ++last;
}

int field_set_domain(izh_field *f, const izh_compdom *dom) {
  IZH_CHECK(field_fresh_e(f));
  f->dom_stamp = next_stamp();
  // the pinned staging buffer may still feed an earlier copy
  IZH_HIP(hipStreamSynchronize(f->stream));
  DevDom d{};
  for (int k = 0; k < 6; k++) d.range[k] = dom->range[k];
  for (int k = 0; k < 3; k++) {
    d.msize[k] = dom->msize[k];
    d.hinv[k] = 1.0 / dom->msize[k];
  }
  *f->h_dom = d;
  IZH_HIP(hipMemcpyAsync(f->d_dom, f->h_dom, sizeof(DevDom), hipMemcpyHostToDevice,
                         f->stream));
  return IZH_OK;
}

// The grid value of the charge a deposit accumulates, FP64: charge itself;
// mixed: charge / sum|w| (O(1) values).
static void deposit_scales(const izh_bunch *b, izh_field *f) {
  f->fixed_scale = fixed_point_scale(b->wabs_sum);
  const double wsum = b->wabs_sum > 0 ? b->wabs_sum : 1.0;
  f->rho_scale = f->precision == IZH_FP64 ? 1.0 : 1.0 / wsum;
}

// Whatever reads the accumulator clears it for the next deposit, unless the call
// failed in between: then this deposit clears it first.
static void begin_deposit(izh_field *f) {
  if (f->fx_dirty)
    hipLaunchKernelGGL(k_fill_u32, dim3(grid_for(2 * f->g)), dim3(kBlock), 0, f->stream,
                       (uint32_t *)f->rho_fx, 2 * f->g, 0u);
  f->fx_dirty = 1;
}

// The fused run's deposit: the t positions (T) of the tile-sorted bunch, by
// its chunk list, into the (cleared) fixed-point accumulator, and in the same
// launch the corners of the step's Green function; launch_convolve_fx
// follows and leaves rho, the cleared accumulator and phi.
int launch_deposit(izh_bunch *b, izh_field *f, const Chunk *chunks, const KeyGrid *kgrid,
                   const int64_t *d_nchunks, int64_t max_chunks) {
  if (!chunks || !kgrid || max_chunks < 1)
    return fail(IZH_ERR_ARG, "deposit: no chunk list or key grid");
  deposit_scales(b, f);
  begin_deposit(f);
  // every contribution is at most |w| * scale: below 2^50 the fused
  // deposit rounds with the short form
  const bool fast = b->wabs_max * f->fixed_scale < 0x1p50;
  ScopedTimer tm_(IZH_T_DEPOSIT, f->stream);
  const int s0 = tile_shift(f->nx), s1 = tile_shift(f->ny), s2 = tile_shift(f->nz);
  const int tnx = f->nx >> s0, tny = f->ny >> s1;
  int64_t *spill = b->d_scal ? &b->d_scal->overflow : nullptr;
  const int64_t nc = (int64_t)(f->nx + 2) * (f->ny + 2) * (f->nz + 2);
  const int ncorner = std::min((grid_for(nc, kDepThreads) + 7) & ~7, kIgfBlocks);
  const auto go = [&](auto kern, const auto *tp) {
    hipLaunchKernelGGL(kern, dim3((unsigned)(ncorner + max_chunks)), dim3(kDepThreads), 0,
                       f->stream, tp, tp + b->cap, tp + 2 * b->cap, b->orig, b->w0, b->w_value,
                       b->w_uniform, chunks, d_nchunks, kgrid, f->d_dom, f->nx, f->ny, f->nz,
                       s0, s1, s2, tnx, tny, f->fixed_scale, f->rho_fx, spill, f->corner,
                       const_cast<std::remove_const_t<std::remove_pointer_t<decltype(tp)>> *>(
                           (decltype(tp))f->green_t),
                       f->igf_tab, f->igf_box, ncorner);
  };
  if (f->precision == IZH_MIXED) {
    const float *tp = (const float *)b->tpos;
    if (fast) go(k_deposit_tiles<float, true>, tp);
    else go(k_deposit_tiles<float, false>, tp);
  } else {
    const double *tp = (const double *)b->tpos;
    if (fast) go(k_deposit_tiles<double, true>, tp);
    else go(k_deposit_tiles<double, false>, tp);
  }
  IZH_HIP(hipGetLastError());
  f->have_rho = 0;
  f->have_phi = 0;
  return IZH_OK;
}

// Scratch of the binned deposit in the field, grown to the largest bunch it
// has deposited: positions (and weights) in bin order, histogram, cursors and
// chunk list.  false: no memory for it.
static bool bins_ready(izh_field *f, int64_t n, bool weights, int ntiles) {
  const int64_t rows = weights ? 4 : 3, nch = n / kBinChunk + ntiles + 1;
  if (f->bin && n <= f->bin_cap && rows <= f->bin_rows && ntiles == f->bin_tiles) return true;
  (void)hipStreamSynchronize(f->stream);
  dev_release(f->bin);
  f->bin = nullptr;
  const size_t head = (size_t)2 * ntiles * sizeof(uint32_t) + (size_t)nch * sizeof(Chunk);
  const size_t at_rows = (head + sizeof(int64_t) + 255) / 256 * 256;
  if (dev_malloc((void **)&f->bin, at_rows + (size_t)rows * n * sizeof(double)) != hipSuccess)
    return false;
  // nchunks, cursors, histogram, chunks, then the rows
  f->bin_cap = n;
  f->bin_rows = (int)rows;
  f->bin_tiles = ntiles;
  f->bin_at_rows = (int64_t)at_rows;
  hipLaunchKernelGGL(k_fill_u32, dim3(grid_for(ntiles)), dim3(kBlock), 0, f->stream,
                     (uint32_t *)(f->bin + sizeof(int64_t)) + ntiles, (int64_t)ntiles, 0u);
  return true;
}

// izh_charge's deposit: straight to the grid up to kDirect particles (the
// adds of a few thousand take less than the launches of anything else), the
// whole grid in LDS up to kSmallGrid nodes, binned otherwise.  The line is the
// small grids': on 16x16x32 direct / in LDS 7.9 / 9.4 us at 1000 particles, 9.1 /
// 9.6 at 4096, 13.2 / 9.6 at 8192.  Against the bins direct adds would stay ahead
// longer (64^3: 8.8 / 24.6 at 4096, 12.3 / 26.7 at 16384, 958 / 85 at 2M).
constexpr int64_t kDirect = 4096;
int launch_deposit_granular(izh_bunch *b, izh_field *f) {
  deposit_scales(b, f);
  begin_deposit(f);
  const DepRows d{b->r[0], b->r[2], b->r[4], b->orig, b->w0, b->w_value, b->w_uniform, b->n,
                  f->d_dom, f->nx, f->ny, f->nz, f->fixed_scale};
  if (b->n > 0) {
    ScopedTimer tm_(IZH_T_DEPOSIT, f->stream);
    BinGrid bg{};
    // tiles of 8 nodes per axis, of 16 where those would not fit a block's LDS
    const int nn[3] = {f->nx, f->ny, f->nz};
    int wide = 0, tn[3];
    for (;; wide++) {
      for (int a = 0; a < 3; a++) {
        bg.s[a] = std::min(tile_shift(nn[a]) + wide, ilog2(nn[a]));
        tn[a] = nn[a] >> bg.s[a];
      }
      bg.ntiles = tn[0] * tn[1] * tn[2];
      if (bg.ntiles <= kBinLdsTiles || wide == 1) break;
    }
    bg.tnx = tn[0];
    bg.tny = tn[1];
    const bool lds = bg.ntiles <= kBinLdsTiles;
    if (b->n > kDirect && f->g <= kSmallGrid) {
      const int64_t nb = std::min<int64_t>((b->n + kSmallPer - 1) / kSmallPer, kSmallBlocks);
      hipLaunchKernelGGL(k_deposit_small, dim3((unsigned)nb), dim3(kBlock),
                         (size_t)f->g * sizeof(unsigned long long), f->stream, d, f->rho_fx);
    } else if (b->n > kDirect && bins_ready(f, b->n, !b->w_uniform, bg.ntiles)) {
      const int64_t cap = f->bin_cap;
      int64_t *nchunks = (int64_t *)f->bin;
      uint32_t *cursor = (uint32_t *)(f->bin + sizeof(int64_t));
      uint32_t *hist = cursor + bg.ntiles;
      Chunk *chunks = (Chunk *)(hist + bg.ntiles);
      double *rows = (double *)(f->bin + f->bin_at_rows);
      const size_t sh = lds ? (size_t)bg.ntiles * sizeof(uint32_t) : 0;
      const int64_t nbc = std::min<int64_t>((b->n + kBinThreads - 1) / kBinThreads,
                                            kBinCountBlocks);
      hipLaunchKernelGGL(lds ? k_bin_count<true> : k_bin_count<false>, dim3((unsigned)nbc),
                         dim3(kBinThreads), sh, f->stream, d, bg, hist);
      hipLaunchKernelGGL(k_bin_scan, dim3(1), dim3(kBinScanThreads), 0, f->stream, hist,
                         bg.ntiles, cursor, chunks, nchunks);
      const int64_t per = kBinThreads * kBinPer, nbs = (b->n + per - 1) / per;
      hipLaunchKernelGGL(lds ? k_bin_scatter<true> : k_bin_scatter<false>, dim3((unsigned)nbs),
                         dim3(kBinThreads), sh, f->stream, d, bg, cursor, rows, cap);
      const bool fast = b->wabs_max * f->fixed_scale < 0x1p50;
      const unsigned nbd = (unsigned)(b->n / kBinChunk + bg.ntiles + 1);
      const auto go = [&](auto kern) {
        hipLaunchKernelGGL(kern, dim3(nbd), dim3(kBlock), 0, f->stream, d, bg, rows, cap, chunks,
                           nchunks, f->rho_fx);
      };
      if (wide == 0) go(fast ? k_deposit_binned<true, 9> : k_deposit_binned<false, 9>);
      else go(fast ? k_deposit_binned<true, 17> : k_deposit_binned<false, 17>);
    } else {
      hipLaunchKernelGGL(k_deposit_direct, dim3(grid_for(b->n)), dim3(kBlock), 0, f->stream, d,
                         f->rho_fx);
    }
    IZH_HIP(hipGetLastError());
  }
  const double inv = f->rho_scale / f->fixed_scale;
  if (f->precision == IZH_FP64)
    hipLaunchKernelGGL(k_fx_to_grid<double>, dim3(grid_for(f->g)), dim3(kBlock), 0,
                       f->stream, f->rho_fx, (double *)f->rho, f->g, inv);
  else
    hipLaunchKernelGGL(k_fx_to_grid<float>, dim3(grid_for(f->g)), dim3(kBlock), 0,
                       f->stream, f->rho_fx, (float *)f->rho, f->g, inv);
  IZH_HIP(hipGetLastError());
  f->fx_dirty = 0;
  f->have_rho = 1;
  f->have_phi = 0;
  return IZH_OK;
}

int launch_convolve_fx(izh_field *f) {
  const int rc = f->precision == IZH_FP64 ? convolve_t<double, true>(f)
                                          : convolve_t<float, true>(f);
  if (rc == IZH_OK) {
    f->fx_dirty = 0;
    f->have_rho = f->have_phi = 1;
  }
  return rc;
}

int launch_solve(izh_field *f) {
  {
    ScopedTimer tm_(IZH_T_GREEN, f->stream);
    const int nc = (f->nx + 2) * (f->ny + 2) * (f->nz + 2);
    const dim3 g(std::min(grid_for(nc), kIgfBlocks)), t(kBlock);
    if (f->precision == IZH_FP64)
      hipLaunchKernelGGL(k_igf<double>, g, t, 0, f->stream, f->corner, (double *)f->green_t,
                         f->nx, f->ny, f->nz, f->d_dom, f->igf_tab, f->igf_box);
    else
      hipLaunchKernelGGL(k_igf<float>, g, t, 0, f->stream, f->corner, (float *)f->green_t,
                         f->nx, f->ny, f->nz, f->d_dom, f->igf_tab, f->igf_box);
    IZH_HIP(hipGetLastError());
  }
  const int rc = f->precision == IZH_FP64 ? convolve_t<double, false>(f)
                                          : convolve_t<float, false>(f);
  if (rc == IZH_OK) f->have_phi = 1;
  return rc;
}

int launch_efield(izh_field *f) {
  ScopedTimer tm_(IZH_T_EFIELD, f->stream);
  if (f->precision == IZH_FP64)
    hipLaunchKernelGGL(k_efield<double>, dim3(grid_for(f->g)), dim3(kBlock), 0,
                       f->stream, (const double *)f->phi, (E4<double> *)f->e,
                       f->nx, f->ny, f->nz, f->d_dom);
  else
    hipLaunchKernelGGL(k_efield<float>, dim3(grid_for(f->g)), dim3(kBlock), 0,
                       f->stream, (const float *)f->phi, (E4<float> *)f->e, f->nx,
                       f->ny, f->nz, f->d_dom);
  IZH_HIP(hipGetLastError());
  f->e_stale = 0;
  return IZH_OK;
}

}  // namespace izh

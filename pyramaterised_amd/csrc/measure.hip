// Measures of states on the GPU: Meyer-Wallach (reference measure.py:226-249)
// and the stabiliser Renyi sum (measure.py:268-349).
//
// Both kernels keep 16 amplitudes (or transform values) per thread in
// registers and bring further index bits into registers through one LDS
// round trip, so no index bit costs an LDS pass of its own.  All sums run in
// double precision in an order that depends on the width alone, so a result
// does not depend on what else is in the batch.
#include "measure.hpp"

#include <algorithm>
#include <string>

#include "plan.hpp"

namespace pqs {
void set_error(const std::string &s);
}

namespace {

template <typename R> struct CT;
template <> struct CT<double> { using V = double2; };
template <> struct CT<float> { using V = float2; };

// LDS slot of tile index j: spreads every 16-index group over the banks
__device__ __forceinline__ int swz(int j) { return j ^ (((j >> 4) ^ (j >> 8)) & 15); }

// Trade lane bit 5 (or 4) of the wave with a register bit: x holds the
// register bit's 0 half, y its 1 half.
template <int LB>
__device__ __forceinline__ void lane_swap(double &x, double &y) {
  unsigned xs[2], ys[2];
  __builtin_memcpy(xs, &x, 8);
  __builtin_memcpy(ys, &y, 8);
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    if constexpr (LB == 5) {
      const auto r = __builtin_amdgcn_permlane32_swap(xs[i], ys[i], false, false);
      xs[i] = r[0];
      ys[i] = r[1];
    } else {
      const auto r = __builtin_amdgcn_permlane16_swap(xs[i], ys[i], false, false);
      xs[i] = r[0];
      ys[i] = r[1];
    }
  }
  __builtin_memcpy(&x, xs, 8);
  __builtin_memcpy(&y, ys, 8);
}

// ------------------------------------------------------------ Meyer-Wallach
constexpr int MB = 256;         // threads per block
constexpr int MTILE = 16 * MB;  // amplitudes per block and pass

constexpr int mw_chunk_bits(int n) { return n < 12 ? (n < 4 ? 4 : n) : 12; }

// Sum 16 values over the 2^NB lanes of a group: each halving step hands half
// of the values to the partner lane, so lane l ends with the totals of the
// values starting at fold_first<NB>(l), 16 >> min(4, NB) of them.
template <int NB, int S = 0>
__device__ __forceinline__ void fold16(double (&v)[16], int lane) {
  constexpr int bit = NB - 1 - S;
  if constexpr (bit >= 0 && S < 4) {
    constexpr int half = 8 >> S;
    const bool up = (lane >> bit) & 1;
#pragma unroll
    for (int i = 0; i < half; ++i) {
      if constexpr (bit >= 4) {
        lane_swap<bit>(v[i], v[i + half]);
        v[i] += v[i + half];
      } else {
        const double keep = up ? v[i + half] : v[i], send = up ? v[i] : v[i + half];
        v[i] = keep + __shfl_xor(send, 1 << bit);
      }
    }
    fold16<NB, S + 1>(v, lane);
  } else if constexpr (bit >= 0) {
    v[0] += __shfl_xor(v[0], 1 << bit);
    fold16<NB, S + 1>(v, lane);
  }
}

template <int NB>
__device__ __forceinline__ int fold_first(int lane) {
  int f = 0;
#pragma unroll
  for (int s = 0; s < (NB < 4 ? NB : 4); ++s) f |= ((lane >> (NB - 1 - s)) & 1) << (3 - s);
  return f;
}

// v[4 b + c]: for register bit b >= LO the sums over this thread's
// amplitudes of |a|^2 with the bit clear, with the bit set, and of
// a0 conj(a1) (real, imaginary)
template <int LO, typename V>
__device__ __forceinline__ void bit_sums(const V (&a)[16], double (&v)[16]) {
  double p[16];
#pragma unroll
  for (int u = 0; u < 16; ++u) p[u] = fma(double(a[u].x), double(a[u].x), double(a[u].y) * a[u].y);
#pragma unroll
  for (int b = 3; b >= 0; --b) {
    double s0 = 0, s1 = 0, re = 0, im = 0;
    if (b >= LO) {
      // p holds the sums over the register bits above b
#pragma unroll
      for (int u = 0; u < (1 << b); ++u) {
        s0 += p[u];
        s1 += p[u | (1 << b)];
        p[u] += p[u | (1 << b)];
      }
#pragma unroll
      for (int u = 0; u < 16; ++u) {
        if ((u >> b) & 1) continue;
        const V x = a[u], y = a[u | (1 << b)];
        re = fma(double(x.x), double(y.x), fma(double(x.y), double(y.y), re));
        im = fma(double(x.y), double(y.x), fma(-double(x.x), double(y.y), im));
      }
    }
    v[4 * b] = s0;
    v[4 * b + 1] = s1;
    v[4 * b + 2] = re;
    v[4 * b + 3] = im;
  }
}

// One block works on 4096 contiguous amplitudes: 2^(12 - N) whole states of
// N <= 12 qubits (it then writes rho and Q itself), or for N = 12 < n one
// chunk after another of a larger state (PART: it writes partial sums).
// Each thread holds 16 amplitudes over 4 index bits; the top 4 come with the
// load, the lower ones through one LDS write and a read per further 4 bits.
// 13 FP64 operations per amplitude and 4 bits against 16 bytes read: the
// FP64 units and HBM are about equally busy.
// The bits of a state above the chunk, 4 at a time, are summed by blocks of
// their own that hold those bits in registers and read the state once more;
// all blocks of a state run on one XCD side by side, so those reads hit its
// L2.  A block takes two chunks, the second one's loads under the first one's
// sums (1000 states of 16 qubits in a loop over one tensor: 376 us against 441
// us with one chunk per block).  Measured: the entanglement call on 1000
// complex128 states of 16 qubits 1320 -> 309 us, 3.4 TB/s of state, the loop 376
// to 385 us (before: an LDS pass and a block tree per bit, partner chunks
// re-read); 16,000 of 12 qubits 247 us, 4.2 TB/s.
template <typename R, int N, bool PART>
__global__ __launch_bounds__(MB, 2) void k_mw(const typename CT<R>::V *__restrict__ states, int n, int64_t batch,
                                           int64_t ncg, int M, int groups, double *__restrict__ rho,
                                           double *__restrict__ q, double *__restrict__ part) {
  using V = typename CT<R>::V;
  constexpr int LT = N - 4;                     // thread bits of a state (chunk)
  constexpr int NB = LT < 6 ? LT : 6;           // of which lane bits
  constexpr int NL = (N + 3) / 4;               // register layouts
  constexpr int KEEP = 16 >> (NB < 4 ? NB : 4); // totals per lane after the fold
  constexpr int UNITS = MB >> NB;               // lane groups per block
  extern __shared__ __align__(16) unsigned char smem[];
  V *tile = reinterpret_cast<V *>(smem);
  double *red = reinterpret_cast<double *>(smem);  // [UNITS][NL * 16], after the last tile read
  const int tid = threadIdx.x, lane = tid & 63;
  const int glane = lane & ((1 << NB) - 1), unit = tid >> NB;

  int64_t b, cg = 0;
  int role = 0;
  if constexpr (PART) {
    const int64_t per = ncg * (1 + groups);
    int64_t sub;
    if (batch >= 8) {  // the dispatcher deals blocks round-robin to the 8 XCDs
      const int64_t slot = blockIdx.x >> 3;
      b = (blockIdx.x & 7) + 8 * (slot / per);
      sub = slot % per;
    } else {
      b = blockIdx.x / per;
      sub = blockIdx.x % per;
    }
    if (b >= batch) return;
    cg = sub / (1 + groups);
    role = int(sub % (1 + groups));
  } else {
    b = int64_t(blockIdx.x) << (12 - N);  // the block's first state
  }

  if (PART && role > 0) {
    // register bits p0 .. p0 + 3, thread bits 0 .. 7, the rest from the chunk id
    const int want = 12 + 4 * (role - 1);
    const int p0 = want < n - 4 ? want : n - 4;
    const V *st = states + (b << n);
    const int64_t lowm = (int64_t(1) << (p0 - 8)) - 1;
    auto fetch = [&](int m, V(&a)[16]) {
      const int64_t ch = cg * M + m;
      const V *src = st + (tid | ((ch & lowm) << 8) | ((ch & ~lowm) << 12));
#pragma unroll
      for (int u = 0; u < 16; ++u) a[u] = src[int64_t(u) << p0];
    };
    double acc = 0;
    auto add = [&](const V(&a)[16]) {
      double v[16];
      bit_sums<0>(a, v);
      fold16<6>(v, lane);
      acc += v[0];
    };
    V a0[16], a1[16];  // chunks in turn, one in flight under the other's sums
    fetch(0, a0);
    for (int m = 0; m < M; m += 2) {
      if (m + 1 < M) fetch(m + 1, a1);
      add(a0);
      if (m + 1 < M) {
        if (m + 2 < M) fetch(m + 2, a0);
        add(a1);
      }
    }
    if ((lane & 3) == 0) red[unit * 16 + fold_first<6>(lane)] = acc;
    __syncthreads();
    if (tid < 16 && p0 + (tid >> 2) >= want) {
      const int qq = n - 1 - (p0 + (tid >> 2));
      double s = red[tid];
#pragma unroll
      for (int w = 1; w < MB / 64; ++w) s += red[w * 16 + tid];
      part[((b * n + qq) * ncg + cg) * 4 + (tid & 3)] = s;
    }
    return;
  }

  double acc[NL][KEEP];
#pragma unroll
  for (int l = 0; l < NL; ++l)
#pragma unroll
    for (int i = 0; i < KEEP; ++i) acc[l][i] = 0;
  // this thread's state (N < 12: several per block) and its index in it
  const int t = tid & ((1 << LT) - 1), sl = tid >> LT;
  V a[16];
  auto fetch = [&](int m) {
    const V *src = PART ? states + (b << n) + ((cg * M + m) << N) : states + ((b + sl) << N);
    if (PART || b + sl < batch) {
#pragma unroll
      for (int u = 0; u < 16; ++u) a[u] = src[t + (u << LT)];
    } else {
#pragma unroll
      for (int u = 0; u < 16; ++u) a[u] = V{0, 0};
    }
  };
  fetch(0);
#pragma unroll 1
  for (int m = 0; m < M; ++m) {
    if constexpr (NL > 1) {
      if (m > 0) __syncthreads();
#pragma unroll
      for (int u = 0; u < 16; ++u) tile[swz((sl << N) | t | (u << LT))] = a[u];
    }
    double v[16];
    bit_sums<4 * (NL - 1) - LT>(a, v);
    if constexpr (NL > 1) {
      __syncthreads();
      // the next chunk's loads run under the lower layouts' sums
      if (m + 1 < M) fetch(m + 1);
    }
    fold16<NB>(v, lane);
#pragma unroll
    for (int i = 0; i < KEEP; ++i) acc[NL - 1][i] += v[i];
    if constexpr (NL > 1) {
#pragma unroll
      for (int l = NL - 2; l >= 0; --l) {
        const int lo = t & ((1 << (4 * l)) - 1), hi = t >> (4 * l);
        const int base = (sl << N) | lo | (hi << (4 * l + 4));
        V c[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) c[u] = tile[swz(base | (u << (4 * l)))];
        bit_sums<0>(c, v);
        fold16<NB>(v, lane);
#pragma unroll
        for (int i = 0; i < KEEP; ++i) acc[l][i] += v[i];
      }
    }
  }
  __syncthreads();
  if (NB <= 4 || (lane & ((1 << (NB > 4 ? NB - 4 : 0)) - 1)) == 0) {
    const int f = fold_first<NB>(glane);
#pragma unroll
    for (int l = 0; l < NL; ++l)
#pragma unroll
      for (int i = 0; i < KEEP; ++i) red[unit * (NL * 16) + l * 16 + f + i] = acc[l][i];
  }
  __syncthreads();
  // value c of bit position pos of state s of the block
  constexpr int W = LT > 6 ? 1 << (LT - 6) : 1;  // waves per state
  auto value = [&](int s, int pos, int c) {
    const int l = pos / 4;
    const int bit = l == NL - 1 ? pos - LT : pos - 4 * l;
    const double *r = red + s * W * (NL * 16) + l * 16 + 4 * bit + c;
    double x = r[0];
    for (int w = 1; w < W; ++w) x += r[w * NL * 16];
    return x;
  };
  if constexpr (PART) {
    if (tid < 48) {
      const int pos = tid >> 2;
      part[((b * n + (n - 1 - pos)) * ncg + cg) * 4 + (tid & 3)] = value(0, pos, tid & 3);
    }
  } else {
    constexpr int SB = MTILE >> N;
    double *pur = red + UNITS * NL * 16;
    for (int i = tid; i < SB * N; i += MB) {
      const int s = i / N, qq = i - s * N;
      if (b + s >= batch) break;
      double x[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) x[c] = value(s, N - 1 - qq, c);
      if (rho) {
#pragma unroll
        for (int c = 0; c < 4; ++c) rho[((b + s) * N + qq) * 4 + c] = x[c];
      }
      pur[i] = x[0] * x[0] + x[1] * x[1] + 2 * (x[2] * x[2] + x[3] * x[3]);
    }
    __syncthreads();
    if (q && tid < SB && b + tid < batch) {
      double p = 0;
      for (int i = 0; i < N; ++i) p += pur[tid * N + i];
      q[b + tid] = 2 * (1 - p / N);
    }
  }
}

// States of 1-3 qubits: one thread each.
template <typename R>
__global__ __launch_bounds__(MB) void k_mw_tiny(const typename CT<R>::V *__restrict__ states, int n, int64_t batch,
                                                double *__restrict__ rho, double *__restrict__ q) {
  const int64_t b = int64_t(blockIdx.x) * MB + threadIdx.x;
  if (b >= batch) return;
  const auto *a = states + (b << n);
  double purity = 0;
  for (int qq = 0; qq < n; ++qq) {
    const int bit = 1 << (n - 1 - qq);
    double x[4] = {0, 0, 0, 0};
    for (int u = 0; u < (1 << n); ++u) {
      if (u & bit) continue;
      const auto y0 = a[u], y1 = a[u | bit];
      x[0] += double(y0.x) * y0.x + double(y0.y) * y0.y;
      x[1] += double(y1.x) * y1.x + double(y1.y) * y1.y;
      x[2] += double(y0.x) * y1.x + double(y0.y) * y1.y;
      x[3] += double(y0.y) * y1.x - double(y0.x) * y1.y;
    }
    if (rho)
      for (int c = 0; c < 4; ++c) rho[(b * n + qq) * 4 + c] = x[c];
    purity += x[0] * x[0] + x[1] * x[1] + 2 * (x[2] * x[2] + x[3] * x[3]);
  }
  if (q) q[b] = 2 * (1 - purity / n);
}

// Totals of the chunk partials of one state (one block): 16 lanes of a wave
// per value and qubit, the purities in qubit order.
__global__ __launch_bounds__(MB) void k_mw_total(const double *__restrict__ part, int n, int64_t ncg,
                                                 double *__restrict__ rho, double *__restrict__ q) {
  __shared__ double pur[pqs::kMaxQubits];
  const int64_t b = blockIdx.x;
  const int lane = threadIdx.x & 63;
  for (int qq = threadIdx.x >> 6; qq < n; qq += MB / 64) {
    const double *p = part + (b * n + qq) * ncg * 4 + (lane & 3);
    double x = 0;
    for (int64_t c = lane >> 2; c < ncg; c += 16) x += p[c * 4];
#pragma unroll
    for (int o = 4; o < 64; o <<= 1) x += __shfl_xor(x, o);
    if (rho && lane < 4) rho[(b * n + qq) * 4 + lane] = x;
    double s = (lane & 2 ? 2 : 1) * x * x;
    s += __shfl_xor(s, 1);
    s += __shfl_xor(s, 2);
    if (lane == 0) pur[qq] = s;
  }
  __syncthreads();
  if (q && threadIdx.x == 0) {
    double s = 0;
    for (int qq = 0; qq < n; ++qq) s += pur[qq];
    q[b] = 2 * (1 - s / n);
  }
}

// Chunks per block and chunk groups of a state of n > 12 qubits: two chunks
// (the comment of k_mw), more where that would leave over 256 groups, so that
// the totals stay short; by the width alone (fixed order of the sums).
void mw_split(int n, int &M, int64_t &ncg, int &groups) {
  const int64_t nch = int64_t(1) << (n - 12);
  M = int(std::max<int64_t>(std::min<int64_t>(nch, 2), nch / 256));
  ncg = nch / M;
  groups = (n - 12 + 3) / 4;
}

// ------------------------------------------------------ stabiliser entropy
// For every X part j, f(m) = conj(c_m) c_{m^j} and its Walsh-Hadamard
// transform F(i) = sum_m (-1)^{i.m} f(m) = <psi|X^j Z^i|psi> up to a phase; the
// sum wanted is over i and j of (2^{-n} |F(i)|^2)^alpha.  f(m ^ j) = conj f(m),
// so F(i) is real where i.j is even and imaginary where it is odd: the
// transform of Im f vanishes on the first set and that of Re f on the second,
// and one real transform, of g = Re f + Im f, gives |F| everywhere.
//
// A transform of 2^N values runs in 2^(N-4) threads, 16 values each: the four
// top index bits in registers as loaded, lane bits 5 and 4 by cross-lane
// swaps, lane bits 3-0 by one LDS transpose within the wave; wave bits (N >
// 10) by one LDS round trip of the block.  Bound by FP64 adds (N per value).
// A block keeps its state's (Re c + Im c, Im c - Re c) in LDS (N <= 12) and
// its amplitudes in registers over the X parts it takes.  Measured: 200
// complex128 states of 10 qubits 1255 -> 180 us (before: complex transforms
// bit by bit in LDS, a barrier each), about half of the FP64 add rate.
enum { kSquare = 0, kRoot = 1, kPower = 2 };

template <int FORM>
__device__ __forceinline__ double magic_term(double f, double scale, double alpha) {
  if constexpr (FORM == kRoot) return fabs(f);  // 2^{-n/2} on the thread's sum
  const double a2 = f * f * scale;
  return FORM == kSquare ? a2 * a2 : pow(a2, alpha);
}

// acc + the terms of M values, the last one first, and the X parts likewise:
// the identity's term (f[0] of the first thread, j = 0) is about a quarter of a
// whole sum, and every addition after it would round at its size.
template <int FORM, int M>
__device__ __forceinline__ double magic_terms(double acc, const double (&f)[16], double scale, double alpha) {
#pragma unroll
  for (int u = M - 1; u >= 0; --u) acc += magic_term<FORM>(f[u], scale, alpha);
  return acc;
}

// 2^{-N/2} x: of odd N the rounding of sqrt(1/2) would be in every term alike,
// so its remainder is added (measured on 3 qubits, alpha = 1/2: 2.2e-16 off an
// 80-bit value without, 1.6e-16 with it).
template <int N>
__device__ __forceinline__ double root_scale(double x) {
  constexpr double p = 1.0 / (1 << (N / 2));
  if constexpr (N % 2 == 0) return x * p;
  return fma(x, p * 0.70710678118654757, x * (p * -4.8336466567264567e-17));
}

template <int LO, int HI>
__device__ __forceinline__ void wht_regs(double (&f)[16]) {
#pragma unroll
  for (int b = LO; b < HI; ++b)
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      if ((u >> b) & 1) continue;
      const double x = f[u], y = f[u | (1 << b)];
      f[u] = x + y;
      f[u | (1 << b)] = x - y;
    }
}

template <int LB>
__device__ __forceinline__ void wht_lane(double (&f)[16]) {
#pragma unroll
  for (int u = 0; u < 8; ++u) {
    lane_swap<LB>(f[u], f[u + 8]);
    const double x = f[u], y = f[u + 8];
    f[u] = x + y;
    f[u + 8] = x - y;
  }
}

constexpr int magic_block(int N) { return N >= 12 ? 512 : 256; }
// X parts of one block: enough to reuse its amplitudes, few enough that one
// state of 8 qubits and more still makes several blocks.  All 128 of 7 qubits in
// one block need no second kernel: 2000 states 35.8 us, in two blocks 41.3; one
// state 15 and 17.7
constexpr int magic_parts(int N) { return N == 7 ? 128 : N <= 9 ? 64 : 32; }

template <typename R, int N, int FORM>
__global__ __launch_bounds__(magic_block(N)) void k_magic(const typename CT<R>::V *__restrict__ states, double alpha,
                                                          double *__restrict__ part) {
  constexpr int BT = magic_block(N), LT = N - 4, T = 1 << LT, C = BT / T, D = 1 << N;
  constexpr int JPB = magic_parts(N), NBLK = D / JPB;
  constexpr bool STAGE = N <= 12;
  constexpr int NLOW = LT < 4 ? LT : 4;  // lane bits that the transpose brings in
  extern __shared__ __align__(16) unsigned char smem[];
  double2 *cs = reinterpret_cast<double2 *>(smem);                 // [D] (STAGE)
  double *xp = reinterpret_cast<double *>(smem) + (STAGE ? 2 * D : 0);  // [16 BT]
  __shared__ double wsum[BT / 64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t b = blockIdx.x / NBLK;
  const int j0 = int(blockIdx.x % NBLK) * JPB;
  const auto *c = states + (b << N);
  const int t = tid & (T - 1), grp = tid >> LT;
  double2 x[16];
#pragma unroll
  for (int u = 0; u < 16; ++u) {
    const auto y = c[t | (u << LT)];
    x[u] = double2{double(y.x), double(y.y)};
  }
  if constexpr (STAGE) {
    for (int m = tid; m < D; m += BT) {
      const auto y = c[m];
      cs[m] = double2{double(y.x) + double(y.y), double(y.y) - double(y.x)};
    }
    __syncthreads();
  }
  const double scale = 1.0 / D;
  double acc = 0;
  for (int it = JPB / C - 1; it >= 0; --it) {
    const int j = j0 + it * C + grp;
    double f[16];
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      const int m = (t | (u << LT)) ^ j;
      double2 y;
      if constexpr (STAGE) {
        y = cs[m];
      } else {
        const auto z = c[m];
        y = double2{double(z.x) + double(z.y), double(z.y) - double(z.x)};
      }
      f[u] = fma(x[u].x, y.x, x[u].y * y.y);
    }
    wht_regs<0, 4>(f);
    if constexpr (N > 10) {
      // wave bits: index bits 6 .. N - 5 into registers
      __syncthreads();
#pragma unroll
      for (int u = 0; u < 16; ++u) xp[(grp << N) | t | (u << LT)] = f[u];
      __syncthreads();
      const int base = (grp << N) | (t & 63) | ((t >> 6) << 10);
#pragma unroll
      for (int u = 0; u < 16; ++u) f[u] = xp[base | (u << 6)];
      wht_regs<0, N - 10>(f);
      __syncthreads();
    }
    if constexpr (LT >= 6) wht_lane<5>(f);
    if constexpr (LT >= 5) wht_lane<4>(f);
    // transpose lane bits 3-0 and the register bits within the wave
    const int w0 = wave * 1024 + (lane >> 4) * 256, lo = lane & 15;
#pragma unroll
    for (int u = 0; u < 16; ++u) xp[w0 + u * 16 + (lo ^ u)] = f[u];
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int u = 0; u < 16; ++u) f[u] = xp[w0 + lo * 16 + (u ^ lo)];
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    wht_regs<0, NLOW>(f);
    acc = magic_terms<FORM, 16>(acc, f, scale, alpha);
  }
  if constexpr (FORM == kRoot) acc = root_scale<N>(acc);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o);
  if (lane == 0) wsum[wave] = acc;
  __syncthreads();
  if (tid == 0) {
    double s = wsum[0];
    for (int w = 1; w < BT / 64; ++w) s += wsum[w];
    part[blockIdx.x] = s;
  }
}

// Re conj(x) y + Im conj(x) y, the imaginary part zero where y is x: few values
// of a small state average the rounding of (Re y + Im y) out.
__device__ __forceinline__ double re_plus_im(double2 x, double2 y) {
#pragma clang fp contract(off)
  return (x.x * y.x + x.y * y.y) + (x.x * y.y - x.y * y.x);
}

// N <= 5: one transform per thread (two threads for N = 5, over lane bit 0),
// the 2^N X parts of a state side by side in a wave.
template <typename R, int N, int FORM>
__global__ __launch_bounds__(256) void k_magic_small(const typename CT<R>::V *__restrict__ states, int64_t batch,
                                                     double alpha, double *__restrict__ out) {
  constexpr int LT = N > 4 ? N - 4 : 0, NR = 1 << (N - LT), GB = N + LT;
  const int64_t u0 = int64_t(blockIdx.x) * 256 + threadIdx.x;
  const int64_t b = u0 >> GB;
  const int t = int(u0) & ((1 << LT) - 1), j = int(u0 >> LT) & ((1 << N) - 1);
  double acc = 0;
  if (b < batch) {
    const auto *c = states + (b << N);
    double f[16];
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      f[u] = 0;
      if (u < NR) {
        const auto x = c[t | (u << LT)], y = c[(t | (u << LT)) ^ j];
        f[u] = re_plus_im(double2{double(x.x), double(x.y)}, double2{double(y.x), double(y.y)});
      }
    }
    wht_regs<0, N - LT>(f);
    const double scale = 1.0 / (1 << N);
#pragma unroll
    for (int u = 0; u < NR; ++u) {
      if constexpr (LT == 1) {  // the other thread of the transform is in this wave and takes this branch too
        const double o = __shfl_xor(f[u], 1);
        f[u] = t ? o - f[u] : f[u] + o;
      }
    }
    acc = magic_terms<FORM, NR>(acc, f, scale, alpha);
    if constexpr (FORM == kRoot) acc = root_scale<N>(acc);
  }
#pragma unroll
  for (int o = 1; o < (1 << GB); o <<= 1) acc += __shfl_xor(acc, o);
  if (b < batch && (u0 & ((1 << GB) - 1)) == 0) out[b] = acc;
}

__global__ __launch_bounds__(256) void k_magic_total(const double *__restrict__ part, int nblk, int64_t batch,
                                                     double *__restrict__ out) {
  const int64_t b = int64_t(blockIdx.x) * 4 + (threadIdx.x >> 6);
  if (b >= batch) return;
  double s = 0;
  for (int i = threadIdx.x & 63; i < nblk; i += 64) s += part[b * nblk + i];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
  if ((threadIdx.x & 63) == 0) out[b] = s;
}

int fail(const char *msg) {
  pqs::set_error(msg);
  return PQS_ERR_UNSUPPORTED;
}

int hip_status(const char *what) {
  const hipError_t e = hipGetLastError();
  if (e == hipSuccess) return PQS_OK;
  pqs::set_error(std::string(what) + " failed: " + hipGetErrorString(e));
  return PQS_ERR_HIP;
}

int allow_lds(const void *kernel, size_t lds) {
  const hipError_t e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, int(lds));
  if (e == hipSuccess) return PQS_OK;
  pqs::set_error(std::string("hipFuncSetAttribute failed: ") + hipGetErrorString(e));
  return PQS_ERR_HIP;
}

template <typename R, int N>
int mw_whole(const void *states, int64_t batch, double *rho, double *q, hipStream_t st) {
  using V = typename CT<R>::V;
  constexpr int LT = N - 4, NB = LT < 6 ? LT : 6, NL = (N + 3) / 4;
  constexpr size_t red = size_t(MB >> NB) * NL * 16 * 8 + size_t(MTILE >> N) * N * 8;
  constexpr size_t lds = std::max(NL > 1 ? MTILE * sizeof(V) : size_t(0), red);
  const int64_t grid = (batch + (MTILE >> N) - 1) >> (12 - N);
  if (grid > 0x7fffffff) return fail("batch too large");
  hipLaunchKernelGGL((k_mw<R, N, false>), dim3(unsigned(grid)), dim3(MB), lds, st, (const V *)states, N, batch,
                     int64_t(1), 1, 0, rho, q, (double *)nullptr);
  return hip_status("k_mw");
}

template <typename R>
int mw_run(const void *states, int n, int64_t batch, double *rho, double *q, double *part, hipStream_t st) {
  using V = typename CT<R>::V;
  switch (n) {
    case 4: return mw_whole<R, 4>(states, batch, rho, q, st);
    case 5: return mw_whole<R, 5>(states, batch, rho, q, st);
    case 6: return mw_whole<R, 6>(states, batch, rho, q, st);
    case 7: return mw_whole<R, 7>(states, batch, rho, q, st);
    case 8: return mw_whole<R, 8>(states, batch, rho, q, st);
    case 9: return mw_whole<R, 9>(states, batch, rho, q, st);
    case 10: return mw_whole<R, 10>(states, batch, rho, q, st);
    case 11: return mw_whole<R, 11>(states, batch, rho, q, st);
    case 12: return mw_whole<R, 12>(states, batch, rho, q, st);
    default: break;
  }
  if (n < 4) {
    if ((batch + MB - 1) / MB > 0x7fffffff) return fail("batch too large");
    hipLaunchKernelGGL((k_mw_tiny<R>), dim3(unsigned((batch + MB - 1) / MB)), dim3(MB), 0, st, (const V *)states, n,
                       batch, rho, q);
    return hip_status("k_mw_tiny");
  }
  int M, groups;
  int64_t ncg;
  mw_split(n, M, ncg, groups);
  const int64_t per = ncg * (1 + groups);
  const int64_t grid = (batch >= 8 ? (batch + 7) / 8 * 8 : batch) * per;
  if (grid > 0x7fffffff) return fail("batch too large");
  hipLaunchKernelGGL((k_mw<R, 12, true>), dim3(unsigned(grid)), dim3(MB), MTILE * sizeof(V), st, (const V *)states, n,
                     batch, ncg, M, groups, rho, q, part);
  if (const int rc = hip_status("k_mw")) return rc;
  hipLaunchKernelGGL(k_mw_total, dim3(unsigned(batch)), dim3(MB), 0, st, part, n, ncg, rho, q);
  return hip_status("k_mw_total");
}

template <typename R, int N, int FORM>
int magic_one(const void *states, int64_t batch, double alpha, double *out, double *part, hipStream_t st) {
  using V = typename CT<R>::V;
  if constexpr (N <= 5) {
    constexpr int GB = N + (N > 4 ? N - 4 : 0);
    const int64_t grid = ((batch << GB) + 255) / 256;
    if (grid > 0x7fffffff) return fail("batch too large");
    hipLaunchKernelGGL((k_magic_small<R, N, FORM>), dim3(unsigned(grid)), dim3(256), 0, st, (const V *)states, batch,
                       alpha, out);
    return hip_status("k_magic_small");
  } else {
    constexpr int nblk = (1 << N) / magic_parts(N);
    constexpr size_t lds = (N <= 12 ? sizeof(double2) << N : 0) + 16 * magic_block(N) * sizeof(double);
    if (batch * nblk > 0x7fffffff) return fail("batch too large");
    if constexpr (lds > 65536 - 64)  // with the block's wave sums over 64 KiB
      if (const int rc = allow_lds((const void *)k_magic<R, N, FORM>, lds)) return rc;
    double *to = nblk == 1 ? out : part;
    hipLaunchKernelGGL((k_magic<R, N, FORM>), dim3(unsigned(batch * nblk)), dim3(magic_block(N)), lds, st,
                       (const V *)states, alpha, to);
    if (const int rc = hip_status("k_magic")) return rc;
    if (nblk > 1) {
      hipLaunchKernelGGL(k_magic_total, dim3(unsigned((batch + 3) / 4)), dim3(256), 0, st, part, nblk, batch, out);
      return hip_status("k_magic_total");
    }
    return PQS_OK;
  }
}

template <typename R, int N>
int magic_form(const void *states, int64_t batch, double alpha, double *out, double *part, hipStream_t st) {
  if (alpha == 2.0) return magic_one<R, N, kSquare>(states, batch, alpha, out, part, st);
  if (alpha == 0.5) return magic_one<R, N, kRoot>(states, batch, alpha, out, part, st);
  return magic_one<R, N, kPower>(states, batch, alpha, out, part, st);
}

template <typename R>
int magic_run(const void *states, int n, int64_t batch, double alpha, double *out, double *part, hipStream_t st) {
  switch (n) {
    case 1: return magic_form<R, 1>(states, batch, alpha, out, part, st);
    case 2: return magic_form<R, 2>(states, batch, alpha, out, part, st);
    case 3: return magic_form<R, 3>(states, batch, alpha, out, part, st);
    case 4: return magic_form<R, 4>(states, batch, alpha, out, part, st);
    case 5: return magic_form<R, 5>(states, batch, alpha, out, part, st);
    case 6: return magic_form<R, 6>(states, batch, alpha, out, part, st);
    case 7: return magic_form<R, 7>(states, batch, alpha, out, part, st);
    case 8: return magic_form<R, 8>(states, batch, alpha, out, part, st);
    case 9: return magic_form<R, 9>(states, batch, alpha, out, part, st);
    case 10: return magic_form<R, 10>(states, batch, alpha, out, part, st);
    case 11: return magic_form<R, 11>(states, batch, alpha, out, part, st);
    case 12: return magic_form<R, 12>(states, batch, alpha, out, part, st);
    case 13: return magic_form<R, 13>(states, batch, alpha, out, part, st);
    default: return fail("stabiliser entropy is limited to 13 qubits (4^n work)");
  }
}

}  // namespace

namespace pqs {

size_t mw_ws(int n, int64_t batch) {
  if (n <= 12) return 0;
  int M, groups;
  int64_t ncg;
  mw_split(n, M, ncg, groups);
  return size_t(batch * n * ncg) * 4 * sizeof(double);
}

int mw_launch(int dtype, const void *states, int n, int64_t batch, double *rho, double *q, void *ws, hipStream_t st) {
  return dtype == PQS_C128 ? mw_run<double>(states, n, batch, rho, q, (double *)ws, st)
                           : mw_run<float>(states, n, batch, rho, q, (double *)ws, st);
}

size_t magic_ws(int n, int64_t batch) {
  return n <= 7 ? 0 : size_t(batch) * (size_t(1) << n) / magic_parts(n) * sizeof(double);
}

int magic_launch(int dtype, const void *states, int n, int64_t batch, double alpha, double *out, void *ws,
                 hipStream_t st) {
  return dtype == PQS_C128 ? magic_run<double>(states, n, batch, alpha, out, (double *)ws, st)
                           : magic_run<float>(states, n, batch, alpha, out, (double *)ws, st);
}

}  // namespace pqs

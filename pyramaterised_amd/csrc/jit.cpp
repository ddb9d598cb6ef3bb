// Run-time specialisation of sweeps (hiprtc).
//
// The interpreter kernel (engine.hip, k_sweep_reg) dispatches every op at run
// time on its kind and register bits; with a register array of 16 complex
// amplitudes per thread, the compiler has to bring every specialised variant
// back to one register assignment at each dispatch join, which costs about
// as many register moves as the arithmetic itself.  For a plan that will run
// many times (batched sampling, Jacobians, benchmarks) the planner instead
// emits one straight-line kernel per sweep: register bits, tile / global bit
// positions, op kinds and fixed matrices are compile-time constants, so the
// whole op sequence is SSA code with no joins and no moves, and each
// rotation costs one FMA per output component (scaled form, below).
//
// Rotations are applied as f * M with f = cos(a/2) and
// M = [[1, -t], [t, 1]] (R_y), [[1, -i t], [-i t, 1]] (R_x) or
// diag(1 -/+ i t) (R_z, R_zz), t = tan(a/2).  The scalar f is the same for
// every amplitude; it is accumulated over the sweep's phases and applied
// once at the end (or at the end of a phase that flips its sign per lane).
// |cos| is clamped below at cmin (sign kept), which changes an entry of the
// matrix by at most cmin, and only when |cos(a/2)| < cmin.  The scaled
// matrix has norm 1/|cos|, so amplitudes grow by at most 1/|f| since f was
// last applied; near a = pi that is up to 1/cmin per rotation.  Every K
// rotations within a phase the kernel therefore applies f early when |f|
// has fallen below T.  Between two such checks |f| stays above T * cmin^K,
// which bounds the growth and keeps f a normal number:
//   double: cmin 1e-20, K 10, T 1e-100 -> |f| >= 1e-300;
//   float:  cmin 1e-7,  K 4,  T 1e-9   -> |f| >= 1e-37.
// With random angles |f| halves per rotation on average, so the early
// application is rare; the check itself is one compare per K rotations.
//
// Sweeps with X(x)X, Y(x)Y and fSim gates, whose gates share angles, and sweeps
// with measurements multiply f by groups: every amplitude shares f, so the
// rounding of a product of hundreds of cosines does not average out.  The angle
// table's threads also work out by how much cos^2 (1 + t^2) misses one for the
// rounded cos and t, multiply the cosines of the rotations between two uses of
// f in higher precision and with that correction, and the sweep takes one
// product per group.  Error against an 80-bit evolution, rms, of matrices op by
// op / one product per rotation / groups: 12-qubit XXZ states of 10 layers
// 2.24e-15 / 2.81e-15 / 1.16e-15, 11-qubit HEA gradients of 8 layers 2.71e-15 /
// 3.45e-15 / 2.67e-15.  Time: 1000 of the XXZ states 178.7 -> 177.6 us, the
// 20-qubit gradient of 40 layers 1.93 -> 1.98 ms; in every sweep it would cost
// the 16-qubit HEA sweeps, which always had the plain product, up to 5%.
#include <hip/hiprtc.h>

#include <cmath>
#include <cstdio>
#include <sstream>
#include <string>
#include <vector>

#include "plan.hpp"

namespace pqs {

void set_error(const std::string &s);

static const char *kPrelude = R"PQS(
typedef unsigned long long u64;
struct InstDev {
  void *state;
  const void *src;
  const double *params;
  void *alt;
  int tangent, init, start_sweep, pingpong;
};
#define NA 16
__device__ __forceinline__ V cmul(V a, V b) { return V{a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x}; }
__device__ __forceinline__ V cadd(V a, V b) { return V{a.x + b.x, a.y + b.y}; }
__device__ __forceinline__ int swz(int j) { return j ^ (((j >> 4) ^ (j >> 8) ^ (j >> 12)) & 15); }
// LDS tile element at a byte offset (phase addresses are XORs of byte offsets)
#define LDSD(o) (*reinterpret_cast<double *>(reinterpret_cast<char *>(tile) + (o)))
#define LDSB(o) (*reinterpret_cast<V *>(reinterpret_cast<char *>(tile) + (o)))
template <int B> __device__ __forceinline__ void ry(V (&a)[NA], R t) {
#pragma unroll
  for (int v = 0; v < NA; ++v) {
    if (v & (1 << B)) continue;
    const V x = a[v], y = a[v | (1 << B)];
    a[v] = V{fma(-t, y.x, x.x), fma(-t, y.y, x.y)};
    a[v | (1 << B)] = V{fma(t, x.x, y.x), fma(t, x.y, y.y)};
  }
}
template <int B> __device__ __forceinline__ void rx(V (&a)[NA], R t) {
#pragma unroll
  for (int v = 0; v < NA; ++v) {
    if (v & (1 << B)) continue;
    const V x = a[v], y = a[v | (1 << B)];
    a[v] = V{fma(t, y.y, x.x), fma(-t, y.x, x.y)};
    a[v | (1 << B)] = V{fma(t, x.y, y.x), fma(-t, x.x, y.y)};
  }
}
// x (1 - i t)
__device__ __forceinline__ V pm(V x, R t) { return V{fma(t, x.y, x.x), fma(-t, x.x, x.y)}; }
template <int B> __device__ __forceinline__ void rz(V (&a)[NA], R t) {
#pragma unroll
  for (int v = 0; v < NA; ++v) a[v] = pm(a[v], (v & (1 << B)) ? -t : t);
}
template <int B0, int B1> __device__ __forceinline__ void rzz(V (&a)[NA], R t) {
#pragma unroll
  for (int v = 0; v < NA; ++v) a[v] = pm(a[v], (((v >> B0) ^ (v >> B1)) & 1) ? -t : t);
}
__device__ __forceinline__ void pall(V (&a)[NA], R t) {
#pragma unroll
  for (int v = 0; v < NA; ++v) a[v] = pm(a[v], t);
}
template <int B> __device__ __forceinline__ void mat1(V (&a)[NA], V m00, V m01, V m10, V m11) {
#pragma unroll
  for (int v = 0; v < NA; ++v) {
    if (v & (1 << B)) continue;
    const V x = a[v], y = a[v | (1 << B)];
    a[v] = cadd(cmul(m00, x), cmul(m01, y));
    a[v | (1 << B)] = cadd(cmul(m10, x), cmul(m11, y));
  }
}
__device__ __forceinline__ void scale(V (&a)[NA], V d) {
#pragma unroll
  for (int v = 0; v < NA; ++v) a[v] = cmul(a[v], d);
}
__device__ __forceinline__ void rscale(V (&a)[NA], R f) {
#pragma unroll
  for (int v = 0; v < NA; ++v) a[v] = V{a[v].x * f, a[v].y * f};
}
template <int BT, int BC> __device__ __forceinline__ void cxr(V (&a)[NA]) {
#pragma unroll
  for (int v = 0; v < NA; ++v) {
    if ((v & (1 << BT)) || !(v & (1 << BC))) continue;
    const V x = a[v];
    a[v] = a[v | (1 << BT)];
    a[v | (1 << BT)] = x;
  }
}
template <int BT> __device__ __forceinline__ void cxc(V (&a)[NA], int on) {
  // per-component selects (a select of whole structs can be lowered
  // through scratch memory)
#pragma unroll
  for (int v = 0; v < NA; ++v) {
    if (v & (1 << BT)) continue;
    const V x = a[v], y = a[v | (1 << BT)];
    a[v].x = on ? y.x : x.x;
    a[v].y = on ? y.y : x.y;
    a[v | (1 << BT)].x = on ? x.x : y.x;
    a[v | (1 << BT)].y = on ? x.y : y.y;
  }
}
template <int B0, int B1> __device__ __forceinline__ void czr(V (&a)[NA]) {
#pragma unroll
  for (int v = 0; v < NA; ++v)
    if ((v & (1 << B0)) && (v & (1 << B1))) a[v] = V{-a[v].x, -a[v].y};
}
template <int B> __device__ __forceinline__ void czc(V (&a)[NA], int on) {
  const R s = on ? R(-1) : R(1);
#pragma unroll
  for (int v = 0; v < NA; ++v)
    if (v & (1 << B)) a[v] = V{a[v].x * s, a[v].y * s};
}
// 1 - i t P on register bits B0, B1: P = X(x)X, or Y(x)Y (YY): -X(x)X on 00, 11
template <int B0, int B1, bool YY> __device__ __forceinline__ void rpp(V (&a)[NA], R t) {
#pragma unroll
  for (int v = 0; v < NA; ++v) {
    const int w = v ^ (1 << B0) ^ (1 << B1);
    if (w < v) continue;
    const R u = YY && !(((v >> B0) ^ (v >> B1)) & 1) ? -t : t;
    const V x = a[v], y = a[w];
    a[v] = V{fma(u, y.y, x.x), fma(-u, y.x, x.y)};
    a[w] = V{fma(u, x.y, y.x), fma(-u, x.x, y.y)};
  }
}
// [[d, -i o], [-i o, d]] on 01, 10 and p on 11
template <int B0, int B1> __device__ __forceinline__ void fsim(V (&a)[NA], R d, R o, V p) {
#pragma unroll
  for (int v = 0; v < NA; ++v) {
    if ((v >> B0) & 1) {
      if ((v >> B1) & 1) a[v] = cmul(a[v], p);
      continue;
    }
    if (!((v >> B1) & 1)) continue;
    const int w = v ^ (1 << B0) ^ (1 << B1);
    const V x = a[v], y = a[w];
    a[v] = V{fma(d, x.x, o * y.y), fma(d, x.y, -o * y.x)};
    a[w] = V{fma(d, y.x, o * x.y), fma(d, y.y, -o * x.x)};
  }
}
__device__ __forceinline__ void negall(V (&a)[NA], int on) { rscale(a, on ? R(-1) : R(1)); }
// Trade lane bit LB (5 or 4) with a register bit: x holds the register bit's
// 0 half, y its 1 half; y of a lane with the lane bit clear and x of its
// partner (the bit set) swap places (v_permlane32_swap / v_permlane16_swap
// on every 32-bit word).
template <int LB> __device__ __forceinline__ void lswap(V &x, V &y) {
  constexpr int nw = int(sizeof(V) / 4);
  unsigned xs[nw], ys[nw];
  __builtin_memcpy(xs, &x, sizeof(V));
  __builtin_memcpy(ys, &y, sizeof(V));
#pragma unroll
  for (int i = 0; i < nw; ++i) {
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
  __builtin_memcpy(&x, xs, sizeof(V));
  __builtin_memcpy(&y, ys, sizeof(V));
}
)PQS";

// Measurement plans: sums of per-lane values over the wave.
static const char *kMeasPrelude = R"PQS(
template <int LB> __device__ __forceinline__ void dswap(double &x, double &y) {
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
template <int B> __device__ __forceinline__ double dxor(double x) {
  int w[2];
  __builtin_memcpy(w, &x, 8);
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    if constexpr (B == 3) w[i] = __builtin_amdgcn_update_dpp(0, w[i], 0x128, 0xf, 0xf, true);
    else if constexpr (B == 2) {
      w[i] = __builtin_amdgcn_update_dpp(0, w[i], 0x141, 0xf, 0xf, true);
      w[i] = __builtin_amdgcn_update_dpp(0, w[i], 0x1b, 0xf, 0xf, true);
    } else if constexpr (B == 1) w[i] = __builtin_amdgcn_update_dpp(0, w[i], 0x4e, 0xf, 0xf, true);
    else w[i] = __builtin_amdgcn_update_dpp(0, w[i], 0xb1, 0xf, 0xf, true);
  }
  __builtin_memcpy(&x, w, 8);
  return x;
}
// Totals over the wave of M values per lane (a power of two up to 16): each
// step hands half of them to the lane across bit B; lane l ends with value
// mfirst<M>(l) in v[0].
template <int M, int B = 5> __device__ __forceinline__ void mfold(double *v, int lane) {
  if constexpr (B >= 0) {
    if constexpr (M > 1) {
      constexpr int H = M / 2;
      const bool up = (lane >> B) & 1;
#pragma unroll
      for (int i = 0; i < H; ++i) {
        if constexpr (B >= 4) {
          dswap<B>(v[i], v[i + H]);
          v[i] += v[i + H];
        } else {
          const double keep = up ? v[i + H] : v[i], send = up ? v[i] : v[i + H];
          v[i] = keep + dxor<B>(send);
        }
      }
      mfold<H, B - 1>(v, lane);
    } else {
      if constexpr (B >= 4) {
        double y = v[0];
        dswap<B>(v[0], y);
        v[0] += y;
      } else {
        v[0] += dxor<B>(v[0]);
      }
      mfold<1, B - 1>(v, lane);
    }
  }
}
template <int M> __device__ __forceinline__ int mfirst(int lane) {
  int f = 0;
#pragma unroll
  for (int m = M / 2, b = 5; m > 0; m >>= 1, --b) f += ((lane >> b) & 1) * m;
  return f;
}
)PQS";

static constexpr int NA_() { return 1 << kRegBits; }
// cmin, K and T of the scaled rotation form (comment at the top of this file)
static double cos_min(const pqs_plan &p) { return p.dtype == PQS_C128 ? 1e-20 : 1e-7; }
// Measurements take products of two scaled amplitudes times f^2, so their
// plans keep |f| >= 1e-60 * 1e-80: f^2 stays a normal number.
static int rot_per_check(const pqs_plan &p) { return p.dtype != PQS_C128 || p.n_meas ? 4 : 10; }
static double rescale_below(const pqs_plan &p) { return p.n_meas ? 1e-60 : p.dtype == PQS_C128 ? 1e-100 : 1e-9; }
static int swz_host(int j) { return j ^ (((j >> 4) ^ (j >> 8) ^ (j >> 12)) & 15); }

static std::string dbl(double v) {
  char b[64];
  std::snprintf(b, sizeof b, "%.17g", v);
  std::string s(b);
  if (s.find_first_of(".eEn") == std::string::npos) s += ".0";
  return s;
}

// bit expression of a qubit that is not a register bit in a phase
static std::string cbit_expr(const DevOp &d, int which) {
  const int t = which ? d.t1 : d.t0;
  const int g = which ? d.g1 : d.g0;
  std::ostringstream o;
  if (t >= 0) o << "((toff >> " << t << ") & 1)";
  else o << "int((base >> " << g << ") & 1ull)";
  return o.str();
}

// Two-qubit gates and LDS phases (Pauli-sum generators) are specialised in
// complex128 only: complex64 plans keep the interpreter there (plan.cpp).
// Measured: 1000 XXZ states of 12 qubits, 10 layers, 695 us interpreted and
// 242 us specialised; the 12-qubit TFIM Jacobian (20 shared parameters, a
// Pauli sum each) 227 and 65 us.
bool jit_sweep_ok(const pqs_plan &p, int s) {
  if (!p.reg_exec) return false;
  const DevSweep &ds = p.dev_sweeps[s];
  return !ds.n_coef || p.dtype == PQS_C128;
}

static void emit_sweep(const pqs_plan &p, int s, std::ostringstream &o);

static std::string prelude(const pqs_plan &p) {
  std::string t = p.dtype == PQS_C128 ? "typedef double R;\ntypedef double2 V;\n" : "typedef float R;\ntypedef float2 V;\n";
  return t + kPrelude + (p.n_meas ? kMeasPrelude : "");
}

std::string jit_source_sweep(const pqs_plan &p, int s) {
  std::ostringstream o;
  o << prelude(p);
  emit_sweep(p, s, o);
  return o.str();
}

std::string jit_source(const pqs_plan &p, std::vector<int> &sweeps_out) {
  std::ostringstream o;
  o << prelude(p);
  sweeps_out.clear();
  for (int s = 0; s < int(p.dev_sweeps.size()); ++s) {
    if (!jit_sweep_ok(p, s)) continue;
    sweeps_out.push_back(s);
    emit_sweep(p, s, o);
  }
  return o.str();
}

static bool can_halve(const pqs_plan &p, int s) {
  const DevSweep &ds = p.dev_sweeps[size_t(s)];
  if (p.dtype != PQS_C128 || (p.flags & PQS_PLAN_JIT_PERSISTENT) || ds.phase_end == ds.phase_begin) return false;
  for (int ph = ds.phase_begin; ph < ds.phase_end; ++ph)
    if (p.dev_phases[size_t(ph)].lds) return false;
  return true;
}

// Slots of a tile of doubles: linear in the tile index, the low five bits such
// that the first five lane bits of as many phases as possible reach 32
// different ones, so that 32 lanes read or write 8 bytes each from all banks.
struct Slots {
  int col[kMaxTileBits];
};
static Slots half_slots(const pqs_plan &p, const DevSweep &ds) {
  // tile bits of the first five lane bits: the load, the phases, the store
  std::vector<std::vector<int>> lanes;
  const int nl = std::min(5, ds.k - kRegBits);
  std::vector<int> v(static_cast<size_t>(nl));
  for (int i = 0; i < nl; ++i) v[size_t(i)] = i;
  if (!ds.direct_load) lanes.push_back(v);
  for (int ph = ds.phase_begin; ph < ds.phase_end; ++ph) {
    for (int i = 0; i < nl; ++i) v[size_t(i)] = p.dev_phases[size_t(ph)].tb[i];
    lanes.push_back(v);
  }
  for (int i = 0; i < nl; ++i) v[size_t(i)] = ds.rolling ? ds.sperm[i] : i;
  if (!ds.direct_store) lanes.push_back(v);
  auto conflicts = [&](const Slots &c) {
    int n = 0;
    for (const auto &l : lanes) {
      int basis[5] = {0, 0, 0, 0, 0}, rank = 0;
      for (int bit : l) {
        int v = c.col[bit] & 31;
        for (int b = 4; b >= 0 && v; --b) {
          if (!((v >> b) & 1)) continue;
          if (!basis[b]) {
            basis[b] = v;
            ++rank;
            v = 0;
          } else {
            v ^= basis[b];
          }
        }
      }
      n += nl - rank;
    }
    return n;
  };
  Slots best{}, c{};
  for (int b = 0; b < kMaxTileBits; ++b) best.col[b] = (1 << b) | (b >= 5 ? 1 << (b % 5) : 0);
  int least = conflicts(best);
  uint32_t seed = 12345;
  for (int t = 0; t < 4000 && least > 0; ++t) {
    for (int b = 0; b < kMaxTileBits; ++b) {
      seed = seed * 1664525u + 1013904223u;
      c.col[b] = (1 << b) | (b >= 5 ? int((seed >> 16) & 31) : 0);
    }
    const int n = conflicts(c);
    if (n < least) {
      least = n;
      best = c;
    }
  }
  return best;
}

static void emit_sweep(const pqs_plan &p, int s, std::ostringstream &o) {
  const int S_total = int(p.dev_sweeps.size());
  {
    const DevSweep &ds = p.dev_sweeps[s];
    const int k = ds.k;
    const int S = 1 << k;
    const int nthr = S >> kRegBits;
    const int kt = k - kRegBits;
    // angle ops of this sweep, in op order
    // (fSim: theta, then phi where it has one, both doubled, since the table
    // holds (tan, cos) of half of each angle, and of these (sin, cos))
    struct Angle {
      int slot;
      double scale, offset;
      int shift;
      bool plain = false;
    };
    std::vector<int> ang(ds.op_end - ds.op_begin, -1);
    std::vector<Angle> aops;
    bool shifts = false;  // rotations that carry their derivatives
    bool plains = false;  // fSim angles
    auto is_rot = [](int kd) {
      return kd == PQS_OP_RX || kd == PQS_OP_RY || kd == PQS_OP_RZ || kd == PQS_OP_RZZ || kd == PQS_OP_RXX ||
             kd == PQS_OP_RYY;
    };
    bool grouped = p.n_meas > 0;  // f by groups (comment at the top)
    for (int i = ds.op_begin; i < ds.op_end; ++i) {
      const DevOp &d = p.dev_ops[i];
      if (d.kind == PQS_OP_RXX || d.kind == PQS_OP_RYY) grouped = true;
      if (!is_rot(d.kind)) continue;
      ang[i - ds.op_begin] = int(aops.size());
      aops.push_back({d.slot, d.scale, d.offset, d.shift});
      if (d.shift >= 0) shifts = true;
    }
    const int nrots = int(aops.size());  // the rotations first: a group is a range of them
    for (int i = ds.op_begin; i < ds.op_end; ++i) {
      const DevOp &d = p.dev_ops[i];
      if (d.kind != PQS_OP_FSIM && d.kind != PQS_OP_GEN_FSIM) continue;
      ang[i - ds.op_begin] = int(aops.size());
      aops.push_back({d.slot, 2 * d.scale, 2 * d.offset, kNoShift, true});
      if (d.slot2 >= 0) aops.push_back({d.slot2, 2.0, 0.0, kNoShift, true});
      plains = grouped = true;
    }
    const int na = int(aops.size());
    grouped = grouped && nrots > 0;
    int last_reg = -1;  // the last register phase applies the accumulated scale
    for (int ph = ds.phase_begin; ph < ds.phase_end; ++ph)
      if (!p.dev_phases[ph].lds) last_reg = ph;
    // terms of the Pauli sums
    for (int i = ds.op_begin; i < ds.op_end; ++i) {
      const DevOp &d = p.dev_ops[i];
      if (d.kind != kPauliSum) continue;
      o << "struct PT" << i << " { unsigned xm, zm; u64 zg; double re, im; };\n__device__ const PT" << i << " PS" << i << "["
        << d.nterms << "] = {";
      for (int t = 0; t < d.nterms; ++t) {
        const DevTerm &m = p.dev_terms[size_t(d.term0 + t)];
        o << (t ? "," : "") << "{" << m.xm << "u," << m.zm_tile << "u," << m.zm_glob << "ull," << dbl(m.cre) << ","
          << dbl(m.cim) << "}";
      }
      o << "};\n";
    }
    if (na > 0) {
      o << "__device__ const int SL" << s << "[" << na << "] = {";
      for (int a = 0; a < na; ++a) o << (a ? "," : "") << aops[a].slot;
      o << "};\n__device__ const double SC" << s << "[" << na << "] = {";
      for (int a = 0; a < na; ++a) o << (a ? "," : "") << dbl(aops[a].scale);
      o << "};\n__device__ const double OF" << s << "[" << na << "] = {";
      for (int a = 0; a < na; ++a) o << (a ? "," : "") << dbl(aops[a].offset);
      o << "};\n";
      if (shifts) {
        o << "__device__ const int SH" << s << "[" << na << "] = {";
        for (int a = 0; a < na; ++a) o << (a ? "," : "") << aops[a].shift;
        o << "};\n";
      }
      if (plains) {
        o << "__device__ const unsigned char PL" << s << "[" << na << "] = {";
        for (int a = 0; a < na; ++a) o << (a ? "," : "") << int(aops[a].plain);
        o << "};\n";
      }
    }
    const bool persist = (p.flags & PQS_PLAN_JIT_PERSISTENT) != 0;
    // The last sweep of a plan also comes as a pair kernel (pqs_jit_pair_<s>)
    // when the plan has no tangent generators: block b evolves tile
    // (b mod n_tiles) of instances 2 (b / n_tiles) and 2 (b / n_tiles) + 1 one
    // after the other, keeps the first one's final amplitudes in registers
    // and writes the tile's share of <psi_2i|psi_2i+1> to pov[b].  Both
    // instances end in the same register / lane layout, so each thread pairs
    // its own amplitudes.
    const bool emit_pair = s == S_total - 1 && !persist && p.n_tangents == 0 && !p.n_meas;
    // measurements of this sweep, in op order: output indices
    std::vector<int> meas;
    for (int i = ds.op_begin; i < ds.op_end; ++i)
      if (p.dev_ops[i].kind == PQS_OP_MEAS) meas.push_back(p.dev_ops[i].term0);
    const int nm = int(meas.size()), nwaves = std::max(1, nthr / 64);
    if (nm) {
      o << "__device__ const int MI" << s << "[" << nm << "] = {";
      for (int i = 0; i < nm; ++i) o << (i ? "," : "") << meas[i];
      o << "};\n";
    }
  std::ostringstream &decl = o;
  for (int pm = 0; pm < (emit_pair ? 2 : 1); ++pm) {
    const bool pair = pm == 1;
    // the kernel's text; the groups it turns out to need are declared before it
    std::ostringstream o;
    std::vector<int> group_end;  // groups of rotations between two uses of f
    int turned = 0;              // rotations applied so far
    const std::string gname = std::to_string(s) + (pair ? "p" : "");
    // f of a rotation about to be applied
    auto turn = [&]() -> const char * {
      ++turned;
      return grouped ? "" : "fs *= c.y; ";
    };
    // f up to date
    auto settle = [&]() {
      if (!grouped || turned == (group_end.empty() ? 0 : group_end.back())) return;
      o << "    fs *= gp[" << group_end.size() << "];\n";
      group_end.push_back(turned);
    };
    // the groups, then the kernel
    auto finish = [&]() {
      if (grouped) {
        decl << "enum { NU" << gname << " = " << group_end.size() << " };\n__device__ const int GB" << gname << "["
             << group_end.size() + 1 << "] = {0";
        for (int e : group_end) decl << "," << e;
        decl << "};\n";
      }
      decl << o.str();
    };
    // Block b processes flat tile b (flat tile = instance * n_tiles + tile).
    // Persistent form (PQS_PLAN_JIT_PERSISTENT): block b processes tiles b,
    // b + G, b + 2G, ... and issues the loads of its next tile into
    // registers before the current tile's phases, so HBM traffic overlaps
    // compute when only one block fits per CU.
    // Halves: a transition trades the real parts through a tile of doubles,
    // then the imaginary ones, so a block holds half the LDS.  What bounds
    // these sweeps is FP64 issue (3/4 of the cycles at 2 waves per SIMD, the
    // most that whole tiles leave room for, and at the card's power limit: an
    // effective 1.9 GHz); 3 waves cover the LDS round trips and barriers
    // better: 10,000 16-qubit states of 20 HEA layers 47.5 -> 45.6 ms, one
    // 24-qubit state 1144 -> 1065 us; single tiles, which wait for their own
    // barriers alone, 126 -> 128 us.  The bound of 3 (168 registers): HEA sweeps
    // on 11 bits need 133-144, so it does nothing there; sweeps with two-qubit
    // gates, 13-bit tiles and some of the longest spill 8-24 registers under it.
    // Bound 2 against 3, halves in both: 1000 12-qubit XXZ states 210.5 / 196.5
    // us, fSim 129.9 / 124.9 us (one 12-bit tile each, all resident at once),
    // the 16-qubit Jacobian 1861 / 1851 us; slower under 3: 200 16-qubit XXZ
    // states 815 / 836 us, 500 13-qubit HEA states 157.8 / 160.6 us.  A bound of
    // 4 spills more: up to 2% faster at 16 qubits, 10% slower at 24.  Sweeps with
    // measurements keep the whole tile and run at one wave per SIMD: the
    // compiler holds the amplitudes of each measurement until its sums are
    // folded (370-512 registers; 20-qubit gradient bounded to 4 waves: 6.9
    // against 1.9 ms).  Pair kernels keep the whole tile for a second state.
    const bool halves = can_halve(p, s) && !pair && !nm;
    Slots slots;
    if (halves) slots = half_slots(p, ds);
    o << "extern \"C\" __global__ __launch_bounds__(" << nthr << (halves ? ", 3" : "") << ") void " << (pair ? "pqs_jit_pair_" : "pqs_jit_sweep_")
      << s << "(const InstDev *__restrict__ insts, long long n_active, const V *__restrict__ init_tab"
      << (pair ? ", double2 *__restrict__ pov" : p.n_meas ? ", double *__restrict__ mpart" : "") << ") {\n";
    o << "  __shared__ " << (halves ? "double" : "V") << " tile[" << S << "];\n";
    o << "  __shared__ double2 tf[" << (na > 0 ? na : 1) << "];\n";
    if (grouped) o << "  __shared__ double gp[NU" << gname << "];\n  __shared__ double tr[" << nrots << "];\n";
    o << "  const int tid = threadIdx.x;\n";
    if (nm) o << "  __shared__ double mred[" << nm * nwaves << "];\n";
    if (pair) {
      o << "  __shared__ double2 pred[" << std::max(1, nthr / 64) << "];\n";
      o << "  const long long total = (n_active >> 1) << " << (p.n - k) << ";\n";
      o << "  const long long pb = blockIdx.x;\n";
      o << "  if (pb >= total) return;\n";
      // keep: the first instance's final amplitudes; (ore, oim): this
      // thread's share of the overlap.  Each pass takes its thread index
      // through an empty asm, so that nothing derived from it (lane
      // offsets, addresses) is hoisted out of the loop and held in
      // registers across both passes.
      o << "  V keep[NA];\n  double ore = 0.0, oim = 0.0;\n";
      o << "#pragma unroll 1\n  for (int half = 0; half < 2; ++half) {\n";
      o << "  int tidv = threadIdx.x;\n  asm volatile(\"\" : \"+v\"(tidv));\n  const int tid = tidv;\n";
      o << "  const long long t = ((((pb >> " << (p.n - k) << ") << 1) | half) << " << (p.n - k) << ") | (pb & "
        << (ds.n_tiles - 1) << "ll);\n";
    } else {
      o << "  const long long total = n_active << " << (p.n - k) << ";\n";
      o << "  long long t = blockIdx.x;\n";
      o << "  if (t >= total) return;\n";
    }
    // address / source helpers for a flat tile index
    o << "  auto tile_base = [&](long long ft) -> u64 {\n";
    o << "    const u64 tile_id = u64(ft) & " << (ds.n_tiles - 1) << "ull;\n";
    o << "    return 0ull";
    for (int r = 0; r < ds.cnruns; ++r)
      o << " | (((tile_id >> " << ds.crun_shift[r] << ") & " << ((1ull << ds.crun_len[r]) - 1) << "ull) << "
        << ds.crun_pos[r] << ")";
    o << ";\n  };\n";
    int tpos[kMaxTileBits];
    for (int r = 0; r < ds.nruns; ++r)
      for (int b = 0; b < ds.run_len[r]; ++b) tpos[ds.run_shift[r] + b] = ds.run_pos[r] + b;
    o << "  const u64 dtid = 0ull";
    for (int i = 0; i < kt; ++i) o << " | (u64((tid >> " << i << ") & 1) << " << tpos[i] << ")";
    o << ";\n";
    auto hp = [&](int m) {
      unsigned long long g = 0;
      for (int b = 0; b < kRegBits; ++b)
        if (m & (1 << b)) g |= 1ull << tpos[kt + b];
      return g;
    };
    o << "  auto io = [&](const InstDev &in, const V *&src, V *&dst, int &init) {\n";
    o << "    init = 0;\n";
    o << "    if (in.pingpong) {\n";
    o << "      dst = " << (((S_total - 1 - s) & 1) == 0 ? "(V *)in.state" : "(V *)in.alt") << ";\n";
    o << "      if (" << s << " == in.start_sweep) { src = (const V *)in.src; init = in.src ? 0 : in.init; }\n";
    o << "      else src = " << (((S_total - s) & 1) == 0 ? "(const V *)in.state" : "(const V *)in.alt") << ";\n";
    o << "    } else {\n";
    o << "      dst = (V *)in.state;\n";
    o << "      if (" << s << " == in.start_sweep) { src = in.src ? (const V *)in.src : dst; init = in.src ? 0 : in.init; }\n";
    o << "      else src = dst;\n";
    o << "    }\n  };\n";
    // Direct load / store: the first (last) phase's registers come from (go
    // to) HBM without staging the tile in LDS; the planner made the tile
    // bits at read (write) positions 0 and 1 lane bits of that phase, so
    // every 4 lanes touch 64 contiguous bytes.  Otherwise the tile is staged
    // with thread bit i = tile bit i and register bit b = tile bit kt + b.
    const bool dload = ds.direct_load && !persist && ds.phase_end > ds.phase_begin;
    const bool dstore = ds.direct_store && !persist && ds.phase_end > ds.phase_begin;
    int lthr[kMaxTileBits], lreg[kRegBits];  // global positions of the load's thread / register bits
    for (int i = 0; i < kt; ++i) lthr[i] = tpos[dload ? p.dev_phases[ds.phase_begin].tb[i] : i];
    for (int b = 0; b < kRegBits; ++b) lreg[b] = tpos[dload ? p.dev_phases[ds.phase_begin].rb[b] : kt + b];
    auto lhp = [&](int m) {
      unsigned long long g = 0;
      for (int b = 0; b < kRegBits; ++b)
        if (m & (1 << b)) g |= 1ull << lreg[b];
      return g;
    };
    o << "  const u64 ltid = 0ull";
    for (int i = 0; i < kt; ++i) o << " | (u64((tid >> " << i << ") & 1) << " << lthr[i] << ")";
    o << ";\n";
    o << "  auto fetch = [&](long long ft, V (&pre)[NA]) {\n";
    o << "    const InstDev in = insts[ft >> " << (p.n - k) << "];\n";
    o << "    const V *src; V *dst; int init;\n    io(in, src, dst, init);\n";
    o << "    const u64 dl = tile_base(ft) | ltid;\n";
    o << "    if (init == 0) {\n";
    for (int m = 0; m < NA_(); ++m) o << "      pre[" << m << "] = src[dl | " << lhp(m) << "ull];\n";
    o << "    } else if (init == 1) {\n";
    for (int m = 0; m < NA_(); ++m)
      o << "      pre[" << m << "] = V{(dl | " << lhp(m) << "ull) == 0ull ? R(1) : R(0), R(0)};\n";
    o << "    } else {\n";
    o << "#pragma unroll\n      for (int m = 0; m < NA; ++m) {\n";
    o << "        u64 gi = dl;\n";
    for (int b = 0; b < kRegBits; ++b) o << "        if (m & " << (1 << b) << ") gi |= " << (1ull << lreg[b]) << "ull;\n";
    o << "        V v{R(1), R(0)};\n";
    o << "        for (int q = 0; q < " << p.n << "; ++q) v = cmul(v, init_tab[2 * q + int((gi >> (" << (p.n - 1)
      << " - q)) & 1ull)]);\n";
    o << "        pre[m] = v;\n      }\n    }\n  };\n";
    o << "  V pre[NA];\n  fetch(t, pre);\n";
    // the final amplitude w of register / slot m: kept (first instance) or
    // paired with the kept one (second instance)
    auto capture = [&](const std::string &m, const std::string &w) {
      if (!pair) return;
      o << "    if (half == 0) keep[" << m << "] = " << w << ";\n"
        << "    else {\n"
        << "      ore += double(keep[" << m << "].x) * double(" << w << ".x) + double(keep[" << m << "].y) * double(" << w
        << ".y);\n"
        << "      oim += double(keep[" << m << "].x) * double(" << w << ".y) - double(keep[" << m << "].y) * double(" << w
        << ".x);\n"
        << "    }\n";
    };
    if (persist) o << "  for (; t < total; t += gridDim.x) {\n";
    else o << "  {\n";
    o << "  const InstDev in = insts[t >> " << (p.n - k) << "];\n";
    o << "  const V *src; V *dst; int init;\n  io(in, src, dst, init);\n";
    o << "  const u64 base = tile_base(t);\n";
    o << "  const u64 dl = base | dtid;\n";
    o << "  const double *params = in.params;\n";
    o << "  __syncthreads();\n";
    // registers carried into a phase that takes its layout by an exchange, and
    // the imaginary parts between the two halves of a transition
    o << "  V areg[NA];\n";
    if (halves) o << "  int hb;\n";
    bool half_pending = false;
    std::string half_sync;
    int half_kv[NA_()];
    // the real parts are in the tile: read them, then trade the imaginary ones
    auto second_half = [&](const char *a, const int *kv) {
      for (int v = 0; v < NA_(); ++v) o << "    " << a << "[" << v << "].x = LDSD(ptb ^ " << 8 * kv[v] << ");\n";
      o << half_sync;
      for (int v = 0; v < NA_(); ++v) o << "    LDSD(hb ^ " << 8 * half_kv[v] << ") = areg[" << v << "].y;\n";
      o << half_sync;
      for (int v = 0; v < NA_(); ++v) o << "    " << a << "[" << v << "].y = LDSD(ptb ^ " << 8 * kv[v] << ");\n";
      half_pending = false;
    };
    // slot of a thread whose bit i is tile bit b[i] (halves), as an expression
    auto thread_slot = [&](const char *tid, auto bit, int n) {
      std::ostringstream e;
      e << "0";
      for (int i = 0; i < n; ++i) e << " ^ (-((" << tid << " >> " << i << ") & 1) & " << slots.col[bit(i)] << ")";
      return e.str();
    };
    if (!dload && halves) {
      o << "  hb = 8 * (" << thread_slot("tid", [](int i) { return i; }, kt) << ");\n";
      for (int v = 0; v < NA_(); ++v) {
        half_kv[v] = 0;
        for (int b = 0; b < kRegBits; ++b)
          if (v & (1 << b)) half_kv[v] ^= slots.col[kt + b];
        o << "  LDSD(hb ^ " << 8 * half_kv[v] << ") = pre[" << v << "].x;\n  areg[" << v << "].y = pre[" << v << "].y;\n";
      }
      half_sync = "    __syncthreads();\n";
      half_pending = true;
    } else if (!dload) {
      o << "#pragma unroll\n  for (int m = 0; m < NA; ++m) tile[swz(tid + m * " << nthr << ")] = pre[m];\n";
    }
    if (persist) o << "  if (t + gridDim.x < total) fetch(t + gridDim.x, pre);\n";
    if (grouped)  // fetched under the angles
      o << "  int gb = GB" << gname << "[tid < NU" << gname << " ? tid : 0], ge = GB" << gname << "[tid < NU" << gname
        << " ? tid + 1 : 0];\n";
    if (na > 0) {
      o << "  for (int i = tid; i < " << na << "; i += " << nthr << ") {\n";
      o << "    double sn, cs;\n";
      o << "    const int sl = SL" << s << "[i];\n";
      o << "    sincos(0.5 * (OF" << s << "[i] + (sl >= 0 ? SC" << s << "[i] * params[sl] : 0.0)), &sn, &cs);\n";
      if (shifts) {
        // the derivative's instance: the angle plus pi, and half its scale
        o << "    double f = 1.0;\n";
        o << "    if (SH" << s << "[i] == in.tangent) { const double u = sn; sn = cs; cs = -u; f = 0.5 * SC" << s
          << "[i]; }\n";
      }
      if (plains) o << "    if (PL" << s << "[i]) { tf[i] = double2{sn, cs}; continue; }\n";
      o << "    if (fabs(cs) < " << dbl(cos_min(p)) << ") cs = cs < 0.0 ? -" << dbl(cos_min(p)) << " : "
        << dbl(cos_min(p)) << ";\n";
      o << "    const double tn = sn / cs;\n    tf[i] = double2{tn, " << (shifts ? "f * cs" : "cs") << "};\n";
      if (grouped)
        // (of a rotation) half of 1 - cs^2 - (cs tn)^2, exact squares: the larger one is at
        // least 1/2, so the two differences are exact too
        o << "    const double q = cs * tn, ql = fma(cs, tn, -q), c2 = cs * cs, q2 = q * q;\n"
             "    tr[i] = 0.5 * (((1.0 - fmax(c2, q2)) - fmin(c2, q2)) - (fma(cs, cs, -c2) + (fma(q, q, -q2) + 2 * q * ql)));\n";
      o << "  }\n";
    }
    o << "  __syncthreads();\n";
    if (grouped) {
      const int most = rot_per_check(p);
      o << "  for (int g = tid; g < NU" << gname << "; g += " << nthr << ") {\n"
        << "    if (g != tid) { gb = GB" << gname << "[g]; ge = GB" << gname << "[g + 1]; }\n"
        << "    double f[" << most << "], r[" << most << "], h = 1.0, e = 0.0;\n"
        << "#pragma unroll\n    for (int j = 0; j < " << most << "; ++j) {\n"
           "      const int i = gb + j < ge ? gb + j : gb;\n"
           "      f[j] = gb + j < ge ? tf[i].y : 1.0;\n      r[j] = gb + j < ge ? tr[i] : 0.0;\n    }\n"
        << "#pragma unroll\n    for (int j = 0; j < " << most << "; ++j) {\n"
           "      const double x = h * f[j];\n"
           "      e = fma(h, f[j], -x) + fma(e, f[j], x * r[j]);\n      h = x;\n    }\n"
           "    gp[g] = h + e;\n  }\n  __syncthreads();\n";
    }
    // fs: the accumulated scale of the rotations (uniform over the block
    // unless a phase flips its sign per lane); it carries across phases and
    // is applied at the end of the sweep, at the end of a phase with
    // per-lane sign flips, or early by the growth check
    o << "  double fs = 1.0;\n";
    // (tan, cos) of the next phase's first rotations, read from the angle
    // table before this phase's LDS writes: LDS returns in issue order, so
    // a table read issued after the transition's 16 reads would hold the
    // next phase's first products until the whole transition has arrived
    constexpr int kPre = 4;
    o << "  double2 nxc[" << kPre << "];\n";
    std::vector<int> pre_ai;  // angle indices held in nxc for this phase
    auto aexpr = [&](int ai) {
      for (size_t j = 0; j < pre_ai.size(); ++j)
        if (pre_ai[j] == ai) return "nxc[" + std::to_string(j) + "]";
      return "tf[" + std::to_string(ai) + "]";
    };
    // emit the reads of the next register phase's first rotations
    auto preload = [&](int next) -> std::vector<int> {
      std::vector<int> v;
      if (next >= ds.phase_end) return v;
      const DevPhase &Q = p.dev_phases[next];
      for (int i = Q.op_begin; i < Q.op_end && int(v.size()) < kPre; ++i) {
        const int ai = ang[i - ds.op_begin];
        if (ai >= 0) v.push_back(ai);
      }
      for (size_t j = 0; j < v.size(); ++j) o << "    nxc[" << j << "] = tf[" << v[j] << "];\n";
      return v;
    };
    std::vector<int> next_pre;
    int n_meas_done = 0;  // measurements whose wave totals are in mred
    bool carry = false;
    int nrot = 0;  // rotations since the last check of the accumulated scale
    // phases
    for (int ph = ds.phase_begin; ph < ds.phase_end; ++ph) {
      const DevPhase &P = p.dev_phases[ph];
      pre_ai.swap(next_pre);
      next_pre.clear();
      if (P.lds) {
        // Pauli sums over the whole tile, in the instance of their tangent
        // (uniform per block); the tile is in LDS before and after
        for (int i = P.op_begin; i < P.op_end; ++i) {
          const DevOp &d = p.dev_ops[i];
          o << "  if (in.tangent == " << d.tangent << ") {\n    V acc[NA];\n"
            << "#pragma unroll\n    for (int m = 0; m < NA; ++m) acc[m] = V{R(0), R(0)};\n"
            << "#pragma unroll 1\n    for (int t = 0; t < " << d.nterms << "; ++t) {\n"
            << "      const PT" << i << " pt = PS" << i << "[t];\n"
            << "      const int gp = __popcll(base & pt.zg);\n"
            << "#pragma unroll\n      for (int m = 0; m < NA; ++m) {\n"
            << "        const int jj = (tid + m * " << nthr << ") ^ int(pt.xm);\n"
            << "        const R sg = ((__popc(unsigned(jj) & pt.zm) + gp) & 1) ? R(-1) : R(1);\n"
            << "        acc[m] = cadd(acc[m], cmul(V{R(pt.re) * sg, R(pt.im) * sg}, tile[swz(jj)]));\n"
            << "      }\n    }\n    __syncthreads();\n"
            << "#pragma unroll\n    for (int m = 0; m < NA; ++m) tile[swz(tid + m * " << nthr << ")] = acc[m];\n"
            << "    __syncthreads();\n  }\n";
        }
        next_pre = preload(ph + 1);
        continue;
      }
      bool lane_sign = false;  // this phase flips fs per lane
      o << "  {\n";
      // in a loop over tiles (persistent form, pair kernel) each phase takes
      // its lane index through an empty asm, so its lane offsets are not
      // hoisted out of the loop and held for the whole kernel; in one pass
      // the compiler may compute them early, before the previous phase's
      // LDS writes (12-bit headline plan -1.5%, others unchanged)
      if (persist || pair)
        o << "    int ptid = tid;\n    asm volatile(\"\" : \"+v\"(ptid));\n";
      else
        o << "    const int ptid = tid;\n";
      o << "    const int toff = 0";
      for (int i = 0; i < P.ntb; ++i) o << " | (((ptid >> " << i << ") & 1) << " << P.tb[i] << ")";
      o << ";\n";
      auto slot_of = [&](int bit) { return halves ? slots.col[bit] : swz_host(1 << bit); };
      if (halves) {
        o << "    const int pt = " << thread_slot("ptid", [&](int i) { return P.tb[i]; }, P.ntb) << ";\n";
      } else {
        o << "    const int pt = swz(toff);\n";
      }
      int kv[NA_()];
      for (int v = 0; v < NA_(); ++v) {
        int a = 0;
        for (int i = 0; i < kRegBits; ++i)
          if (v & (1 << i)) a ^= slot_of(P.rb[i]);
        kv[v] = a;
      }
      o << "    const int ptb = pt * int(sizeof(*tile));\n    V a[NA];\n";
      if (carry) {
        for (int v = 0; v < NA_(); ++v) o << "    a[" << v << "] = areg[" << v << "];\n";
        carry = false;
      } else if (dload && ph == ds.phase_begin) {
        for (int v = 0; v < NA_(); ++v) o << "    a[" << v << "] = pre[" << v << "];\n";
      } else if (half_pending) {
        second_half("a", kv);
      } else {
        for (int v = 0; v < NA_(); ++v)
          o << "    a[" << v << "] = LDSB(ptb ^ (" << kv[v] << " * int(sizeof(V))));\n";
      }
      // Pending X flips: a CNOT whose control is a thread or constant bit
      // does not move data; it XORs a per-lane flag xf<r> meaning "logical
      // register index bit r is stored flipped".  Later ops on r compensate
      // (X Ry(a) X = Ry(-a), X Rz(a) X = Rz(-a), X Rx X = Rx, CNOT with a
      // flipped control = CNOT then X on the target, X_a CZ X_a = CZ Z_b),
      // and the phase's LDS store addresses absorb the flips.
      bool fl[kRegBits] = {false, false, false, false};
      o << "    int xf0 = 0, xf1 = 0, xf2 = 0, xf3 = 0;\n";
      auto xf = [](int r) { return "xf" + std::to_string(r); };
      auto materialise = [&](int r) {  // apply a pending flip as data movement
        if (r >= 0 && fl[r]) {
          o << "    cxc<" << r << ">(a, " << xf(r) << ");\n    " << xf(r) << " = 0;\n";
          fl[r] = false;
        }
      };
      // Measurements: each leaves a per-thread value; up to 16 of them are
      // summed over the wave together.  conj(a) b per pair of amplitudes is
      // not changed by diagonal gates (both halves turn alike) and serves
      // every Z string until the next non-diagonal op ("wz<id>", "wt<id>").
      std::vector<std::string> mvals;
      int wz_id = -1, wz_count = 0;
      int wz_parts = 0;  // 1: real products there, 2: imaginary ones
      bool wz_total[2] = {false, false};
      auto flush_meas = [&]() {
        if (mvals.empty()) return;
        int M = 1;
        while (M < int(mvals.size())) M *= 2;
        o << "    { double mv[" << M << "] = {";
        for (int j = 0; j < M; ++j) o << (j ? ", " : "") << (j < int(mvals.size()) ? mvals[size_t(j)] : "0.0");
        o << "};\n      const int ln = ptid & 63;\n      mfold<" << M << ">(mv, ln);\n      const int f = mfirst<" << M
          << ">(ln);\n      if ((ln & " << (64 / M - 1) << ") == 0 && f < " << mvals.size() << ") mred[(ptid >> 6) * "
          << nm << " + " << n_meas_done << " + f] = mv[0]; }\n";
        n_meas_done += int(mvals.size());
        mvals.clear();
      };
      for (int i = P.op_begin; i < P.op_end; ++i) {
        const DevOp &d = p.dev_ops[i];
        const int ai = ang[i - ds.op_begin];
        const bool r0 = d.r0 >= 0, r1 = d.r1 >= 0;
        if (d.kind != PQS_OP_MEAS && d.kind != PQS_OP_RZ && d.kind != PQS_OP_RZZ && d.kind != PQS_OP_CZ) wz_id = -1;
        if (is_rot(d.kind)) {
          if (nrot == rot_per_check(p)) {
            settle();
            o << "    if (fabs(fs) < " << dbl(rescale_below(p)) << ") { rscale(a, R(fs)); fs = 1.0; }\n";
            nrot = 0;
          }
          ++nrot;
        }
        // "(xf) ? -t : t" for a rotation whose sign flips with pending X flips
        auto tsign = [&](const std::string &flip, const std::string &t) {
          return flip.empty() ? t : "((" + flip + ") ? -" + t + " : " + t + ")";
        };
        switch (d.kind) {
          case PQS_OP_RY:
            o << "    { const double2 c = " << aexpr(ai) << "; " << turn() << "ry<" << d.r0 << ">(a, "
              << tsign(fl[d.r0] ? xf(d.r0) : "", "R(c.x)") << "); }\n";
            break;
          case PQS_OP_RX:
            o << "    { const double2 c = " << aexpr(ai) << "; " << turn() << "rx<" << d.r0 << ">(a, R(c.x)); }\n";
            break;
          case PQS_OP_RZ:
            if (r0)
              o << "    { const double2 c = " << aexpr(ai) << "; " << turn() << "rz<" << d.r0 << ">(a, "
                << tsign(fl[d.r0] ? xf(d.r0) : "", "R(c.x)") << "); }\n";
            else
              o << "    { const double2 c = " << aexpr(ai) << "; " << turn() << "pall(a, " << cbit_expr(d, 0)
                << " ? R(-c.x) : R(c.x)); }\n";
            break;
          case PQS_OP_RZZ: {
            std::string flip;
            if (r0 && fl[d.r0]) flip = xf(d.r0);
            if (r1 && fl[d.r1]) flip = flip.empty() ? xf(d.r1) : "(" + flip + " ^ " + xf(d.r1) + ")";
            if (r0 && r1)
              o << "    { const double2 c = " << aexpr(ai) << "; " << turn() << "rzz<" << d.r0 << "," << d.r1 << ">(a, "
                << tsign(flip, "R(c.x)") << "); }\n";
            else if (r0 || r1) {
              const std::string cb = cbit_expr(d, r0 ? 1 : 0);
              o << "    { const double2 c = " << aexpr(ai) << "; " << turn() << "rz<" << (r0 ? d.r0 : d.r1) << ">(a, ("
                << (flip.empty() ? cb : "(" + cb + " ^ " + flip + ")") << ") ? R(-c.x) : R(c.x)); }\n";
            } else
              o << "    { const double2 c = " << aexpr(ai) << "; " << turn() << "pall(a, (" << cbit_expr(d, 0) << " ^ "
                << cbit_expr(d, 1) << ") ? R(-c.x) : R(c.x)); }\n";
            break;
          }
          case PQS_OP_MEAS: {
            // Re(c <a|P|b>): (P b)[j] = (-1)^{z.(j ^ x)} b[j ^ x], i^{#Y} in c
            int top = -1;  // register bit of the pair's qubit
            for (int r = 0; r < kRegBits; ++r)
              if (P.rb[r] == ds.pair_bit) top = r;
            const bool xx = d.pauli == 1 || d.pauli == 2, zz = d.pauli == 2 || d.pauli == 3;
            int xr = 0, zr = 0;
            std::string sign;  // the lane's part of the sign, as a bit expression
            auto add_sign = [&](const std::string &e) { sign += sign.empty() ? e : " ^ " + e; };
            for (int w = 0; w < (d.g1 >= 0 ? 2 : 1); ++w) {
              const int r = w ? d.r1 : d.r0;
              if (xx) xr |= 1 << r;
              if (!zz) continue;
              if (r >= 0) {
                zr |= 1 << r;
                if (fl[r]) add_sign(xf(r));
              } else {
                add_sign(cbit_expr(d, w));
              }
            }
            const bool want[2] = {d.m[0] != 0, d.m[1] != 0};
            const std::string id = std::to_string(ph - ds.phase_begin) + "_" + std::to_string(i - ds.op_begin);
            auto prod = [&](int part, int v) {  // conj(a) (P b) without the sign, one part
              const std::string A = "a[" + std::to_string(v) + "]", B = "a[" + std::to_string((v ^ xr) | (1 << top)) + "]";
              return part == 0 ? "fma(" + A + ".x, " + B + ".x, " + A + ".y * " + B + ".y)"
                               : "fma(" + A + ".x, " + B + ".y, -" + A + ".y * " + B + ".x)";
            };
            o << "    double me" << id << " = 0.0;\n";
            for (int part = 0; part < 2; ++part) {
              if (!want[part]) continue;
              const std::string c = dbl(part == 0 ? d.m[0] : -d.m[1]);
              if (!xx) {
                // products shared by the Z strings of this point, true scale
                if (wz_id < 0) {
                  wz_id = wz_count++;
                  wz_parts = 0;
                  wz_total[0] = wz_total[1] = false;
                }
                const std::string nm_ = std::to_string(ph - ds.phase_begin) + "_" + std::to_string(wz_id) + "_" + std::to_string(part);
                if (!((wz_parts >> part) & 1)) {
                  settle();
                  o << "    double wz" << nm_ << "[8]; { const double f2 = fs * fs;\n";
                  int q = 0;
                  for (int v = 0; v < NA_(); ++v)
                    if (!((v >> top) & 1)) o << "      wz" << nm_ << "[" << q++ << "] = (" << prod(part, v) << ") * f2;\n";
                  o << "    }\n";
                  wz_parts |= 1 << part;
                }
                std::string sum;
                if (zr == 0) {
                  if (!wz_total[part]) {
                    o << "    const double wt" << nm_ << " = ((wz" << nm_ << "[0] + wz" << nm_ << "[1]) + (wz" << nm_
                      << "[2] + wz" << nm_ << "[3])) + ((wz" << nm_ << "[4] + wz" << nm_ << "[5]) + (wz" << nm_
                      << "[6] + wz" << nm_ << "[7]));\n";
                    wz_total[part] = true;
                  }
                  sum = "wt" + nm_;
                } else {
                  int q = 0;
                  for (int v = 0; v < NA_(); ++v) {
                    if ((v >> top) & 1) continue;
                    sum += (__builtin_popcount(unsigned(v & zr)) & 1 ? " - wz" : q ? " + wz" : "wz") + nm_ + "[" + std::to_string(q) + "]";
                    ++q;
                  }
                }
                o << "    me" << id << " += " << c << " * (" << sum << ");\n";
              } else {
                settle();
                o << "    { double t = 0.0;\n";
                for (int v = 0; v < NA_(); ++v) {
                  if ((v >> top) & 1) continue;
                  const bool neg = __builtin_popcount(unsigned((v ^ xr) & zr)) & 1;
                  const std::string A = "a[" + std::to_string(v) + "]", B = "a[" + std::to_string((v ^ xr) | (1 << top)) + "]";
                  const std::string sA = (neg ? "-" : "") + A, nA = (neg ? "" : "-") + A;
                  if (part == 0) o << "      t = fma(" << sA << ".x, " << B << ".x, fma(" << sA << ".y, " << B << ".y, t));\n";
                  else o << "      t = fma(" << sA << ".x, " << B << ".y, fma(" << nA << ".y, " << B << ".x, t));\n";
                }
                o << "      me" << id << " += " << c << " * t * fs * fs; }\n";
              }
            }
            if (!sign.empty()) o << "    if (" << sign << ") me" << id << " = -me" << id << ";\n";
            mvals.push_back("me" + id);
            if (mvals.size() == 16) flush_meas();
            break;
          }
          case PQS_OP_RXX:  // X flips commute with X(x)X
            o << "    { const double2 c = " << aexpr(ai) << "; " << turn() << "rpp<" << d.r0 << "," << d.r1
              << ",false>(a, R(c.x)); }\n";
            break;
          case PQS_OP_RYY: {
            std::string flip;
            if (fl[d.r0]) flip = xf(d.r0);
            if (fl[d.r1]) flip = flip.empty() ? xf(d.r1) : "(" + flip + " ^ " + xf(d.r1) + ")";
            o << "    { const double2 c = " << aexpr(ai) << "; " << turn() << "rpp<" << d.r0 << "," << d.r1 << ",true>(a, "
              << tsign(flip, "R(c.x)") << "); }\n";
            break;
          }
          case PQS_OP_FSIM:
          case PQS_OP_GEN_FSIM: {
            // fSim, or a derivative matrix as the reference writes it
            // (gates.py:609-648, 719-737; pauli 1 d_theta, 2 d_phi, 3 fixed)
            materialise(d.r0);
            materialise(d.r1);
            const int sel = d.kind == PQS_OP_FSIM ? 0 : d.pauli;
            const bool dth = sel == 1 || sel == 3;
            if (sel) o << "    if (in.tangent == " << d.tangent << ")";
            o << "    { const double2 c = " << aexpr(ai) << ", f = "
              << (d.slot2 >= 0 ? "tf[" + std::to_string(ai + 1) + "]" : std::string("double2{0.0, 1.0}"))
              << "; const double st = c.x, ct = c.y, sp = f.x, cp = f.y; fsim<" << d.r0 << "," << d.r1
              << ">(a, R(" << (dth ? "-st" : "ct") << "), R(" << (dth ? "ct" : "st") << "), "
              << (sel == 3 ? "V{R(1), R(0)}" : sel == 2 ? "V{R(-sp), R(-cp)}" : "V{R(cp), R(-sp)}") << "); }\n";
            break;
          }
          case PQS_OP_MAT2: {
            // row by row, the zero entries left out
            materialise(d.r0);
            materialise(d.r1);
            for (int v = 0; v < NA_(); ++v) {
              if (((v >> d.r0) | (v >> d.r1)) & 1) continue;
              auto at = [&](int c) { return v | ((c >> 1) << d.r0) | ((c & 1) << d.r1); };
              o << "    {";
              for (int c = 0; c < 4; ++c) o << " const V x" << c << " = a[" << at(c) << "];";
              for (int r = 0; r < 4; ++r) {
                std::string e;
                for (int c = 0; c < 4; ++c) {
                  const double re = d.m[2 * (4 * r + c)], im = d.m[2 * (4 * r + c) + 1];
                  if (re == 0 && im == 0) continue;
                  const std::string x = "x" + std::to_string(c);
                  const std::string t = re == 1 && im == 0 ? x : "cmul(V{R(" + dbl(re) + "), R(" + dbl(im) + ")}, " + x + ")";
                  e = e.empty() ? t : "cadd(" + e + ", " + t + ")";
                }
                o << " a[" << at(r) << "] = " << (e.empty() ? "V{R(0), R(0)}" : e) << ";";
              }
              o << " }\n";
            }
            break;
          }
          case PQS_OP_MAT1: {
            auto cv = [&](int e) { return "V{R(" + dbl(d.m[2 * e]) + "), R(" + dbl(d.m[2 * e + 1]) + ")}"; };
            if (r0) {
              materialise(d.r0);
              o << "    mat1<" << d.r0 << ">(a, " << cv(0) << ", " << cv(1) << ", " << cv(2) << ", " << cv(3)
                << ");\n";
            } else
              o << "    scale(a, " << cbit_expr(d, 0) << " ? " << cv(3) << " : " << cv(0) << ");\n";
            break;
          }
          case kGen1: {
            // c * Pauli on q0, only in the instance carrying this tangent
            if (r0) materialise(d.r0);
            const double cr = d.m[0], ci = d.m[1];
            double m[8] = {0, 0, 0, 0, 0, 0, 0, 0};  // m00, m01, m10, m11 (re, im)
            if (d.pauli == 0) { m[0] = cr; m[1] = ci; m[6] = cr; m[7] = ci; }
            else if (d.pauli == 1) { m[2] = cr; m[3] = ci; m[4] = cr; m[5] = ci; }
            else if (d.pauli == 2) { m[2] = ci; m[3] = -cr; m[4] = -ci; m[5] = cr; }
            else { m[0] = cr; m[1] = ci; m[6] = -cr; m[7] = -ci; }
            auto cv = [&](int e) { return "V{R(" + dbl(m[2 * e]) + "), R(" + dbl(m[2 * e + 1]) + ")}"; };
            o << "    if (in.tangent == " << d.tangent << ") ";
            if (r0)
              o << "mat1<" << d.r0 << ">(a, " << cv(0) << ", " << cv(1) << ", " << cv(2) << ", " << cv(3) << ");\n";
            else
              o << "scale(a, " << cbit_expr(d, 0) << " ? " << cv(3) << " : " << cv(0) << ");\n";
            break;
          }
          case PQS_OP_CX:
            // q0 = control, q1 = target (a register bit)
            if (r0) {
              o << "    cxr<" << d.r1 << "," << d.r0 << ">(a);\n";
              if (fl[d.r0]) {  // flipped control: CNOT then X on the target
                o << "    " << xf(d.r1) << " ^= " << xf(d.r0) << ";\n";
                fl[d.r1] = true;
              }
            } else {
              o << "    " << xf(d.r1) << " ^= " << cbit_expr(d, 0) << ";\n";
              fl[d.r1] = true;
            }
            break;
          case PQS_OP_CZ:
            if (r0 && r1) {
              o << "    czr<" << d.r0 << "," << d.r1 << ">(a);\n";
              // X_a CZ X_a = CZ Z_b; both flipped: -CZ Z_a Z_b
              if (fl[d.r0]) o << "    czc<" << d.r1 << ">(a, " << xf(d.r0) << ");\n";
              if (fl[d.r1]) o << "    czc<" << d.r0 << ">(a, " << xf(d.r1) << ");\n";
              if (fl[d.r0] && fl[d.r1]) {
                o << "    if (" << xf(d.r0) << " & " << xf(d.r1) << ") fs = -fs;\n";
                lane_sign = true;
              }
            } else if (r0 || r1) {
              const int rr = r0 ? d.r0 : d.r1;
              const std::string cb = cbit_expr(d, r0 ? 1 : 0);
              o << "    czc<" << rr << ">(a, " << cb << ");\n";
              // X_r CZ(r, c) X_r = CZ Z_c: a sign where the constant bit is set
              if (fl[rr]) {
                o << "    if (" << xf(rr) << " & " << cb << ") fs = -fs;\n";
                lane_sign = true;
              }
            } else {
              o << "    negall(a, " << cbit_expr(d, 0) << " & " << cbit_expr(d, 1) << ");\n";
            }
            break;
          default:
            break;
        }
      }
      flush_meas();
      // Exchange into the next phase: its layout is this one with register
      // bits traded against lane bits 5 / 4, so the amplitudes move with
      // cross-lane swaps and stay in registers (no LDS round trip, no
      // barrier).  Pending flips are applied as data first.
      const bool xnext = ph + 1 < ds.phase_end && p.dev_phases[ph + 1].xchg > 0 && !p.dev_phases[ph + 1].lds;
      if (xnext) {
        for (int r = 0; r < kRegBits; ++r) materialise(r);
        if (lane_sign) {
          settle();
          o << "    rscale(a, R(fs));\n    fs = 1.0;\n";
          nrot = 0;
        }
        next_pre = preload(ph + 1);
        const DevPhase &Q = p.dev_phases[ph + 1];
        for (int j = 0; j < Q.xchg; ++j)
          for (int v = 0; v < NA_(); ++v)
            if (!(v & (1 << Q.xr[j])))
              o << "    lswap<" << Q.xb[j] << ">(a[" << v << "], a[" << (v | (1 << Q.xr[j])) << "]);\n";
        for (int v = 0; v < NA_(); ++v) o << "    areg[" << v << "] = a[" << v << "];\n";
        o << "  }\n";
        carry = true;
        continue;
      }
      // stores land where the flipped indices belong
      {
        bool any = false;
        for (int r = 0; r < kRegBits; ++r) any = any || fl[r];
        if (any) {
          o << "    const int pst = pt";
          for (int r = 0; r < kRegBits; ++r)
            if (fl[r]) o << " ^ (" << xf(r) << " ? " << slot_of(P.rb[r]) << " : 0)";
          o << ";\n";
        } else {
          o << "    const int pst = pt;\n";
        }
      }
      if (lane_sign || ph == last_reg) {
        settle();
        o << "    rscale(a, R(fs));\n    fs = 1.0;\n";
        nrot = 0;
      }
      if (dstore && ph + 1 == ds.phase_end) {
        // direct store: tile bit j goes to write position wp[j]; flipped
        // register bits flip their position bit per lane
        int wp[kMaxTileBits];
        for (int j = 0; j < k; ++j) wp[j] = ds.rolling ? ds.wpos[j] : tpos[j];
        if (ds.rolling) {
          o << "    const u64 wtid = u64(t) & " << (ds.n_tiles - 1) << "ull;\n";
          o << "    const u64 gb = 0ull";
          for (int j = 0; j < p.n - k; ++j) o << " | (((wtid >> " << j << ") & 1ull) << " << ds.cwpos[j] << ")";
          o << ";\n";
        } else {
          o << "    const u64 gb = tile_base(t);\n";
        }
        o << "    const u64 gt = gb";
        for (int i = 0; i < P.ntb; ++i) o << " | (u64((ptid >> " << i << ") & 1) << " << wp[P.tb[i]] << ")";
        for (int r = 0; r < kRegBits; ++r)
          if (fl[r]) o << " ^ (" << xf(r) << " ? " << (1ull << wp[P.rb[r]]) << "ull : 0ull)";
        o << ";\n";
        for (int v = 0; v < NA_(); ++v) {
          unsigned long long cm = 0;
          for (int b = 0; b < kRegBits; ++b)
            if (v & (1 << b)) cm |= 1ull << wp[P.rb[b]];
          o << "    dst[gt ^ " << cm << "ull] = a[" << v << "];\n";
        }
        for (int v = 0; v < NA_(); ++v) capture(std::to_string(v), "a[" + std::to_string(v) + "]");
        o << "  }\n";
        continue;
      }
      next_pre = preload(ph + 1);
      if (halves) {
        o << "    hb = pst * 8;\n";
        for (int v = 0; v < NA_(); ++v) {
          half_kv[v] = kv[v];
          o << "    LDSD(hb ^ " << 8 * kv[v] << ") = a[" << v << "].x;\n    areg[" << v << "].y = a[" << v << "].y;\n";
        }
      } else {
        o << "    const int pstb = pst * int(sizeof(V));\n";
        for (int v = 0; v < NA_(); ++v)
          o << "    LDSB(pstb ^ (" << kv[v] << " * int(sizeof(V)))) = a[" << v << "];\n";
      }
      // the next phase keeps the wave bits (thread bits 6..): its LDS reads
      // touch only this wave's amplitudes, which this wave's own earlier
      // LDS writes (executed in order) already hold
      bool wave_local = false;
      if (ph + 1 < ds.phase_end && !(p.flags & PQS_PLAN_NO_WAVE_LOCAL)) {
        const DevPhase &Q = p.dev_phases[ph + 1];
        wave_local = !Q.lds && Q.ntb == P.ntb;
        for (int i = 6; wave_local && i < P.ntb; ++i) wave_local = Q.tb[i] == P.tb[i];
      }
      half_sync = wave_local ? "    __builtin_amdgcn_fence(__ATOMIC_RELEASE, \"wavefront\");\n"
                               "    __builtin_amdgcn_wave_barrier();\n"
                               "    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, \"wavefront\");\n"
                             : "    __syncthreads();\n";
      half_pending = halves;
      o << half_sync << "  }\n";
    }
    if (halves && !dstore) {
      // the store's layout, read through the halves as a phase's
      auto bit = [&](int i) { return ds.rolling ? ds.sperm[i] : i; };
      int kv[NA_()];
      for (int v = 0; v < NA_(); ++v) {
        kv[v] = 0;
        for (int b = 0; b < kRegBits; ++b)
          if (v & (1 << b)) kv[v] ^= slots.col[bit(kt + b)];
      }
      o << "  V w[NA];\n  {\n    const int ptb = 8 * (" << thread_slot("tid", bit, kt) << ");\n";
      second_half("w", kv);
      o << "  }\n";
    }
    auto stored = [&](int m, const std::string &index) {
      return halves ? "w[" + std::to_string(m) + "]" : "tile[swz(" + index + ")]";
    };
    if (dstore) {
      // stored by the last phase
    } else if (!ds.rolling) {
      for (int m = 0; m < NA_(); ++m) {
        o << "  {\n    const V x = " << stored(m, "tid + " + std::to_string(m * nthr)) << ";\n    dst[dl | " << hp(m)
          << "ull] = x;\n";
        capture(std::to_string(m), "x");
        o << "  }\n";
      }
    } else {
      // write layout: store index bit i is tile bit sperm[i], at write
      // position wpos[sperm[i]] (ascending), complement bit j at cwpos[j]
      o << "  {\n    const u64 wtid = u64(t) & " << (ds.n_tiles - 1) << "ull;\n";
      o << "    const u64 wdl = 0ull";
      for (int j = 0; j < p.n - k; ++j) o << " | (((wtid >> " << j << ") & 1ull) << " << ds.cwpos[j] << ")";
      for (int i = 0; i < kt; ++i) o << " | (u64((tid >> " << i << ") & 1) << " << ds.wpos[ds.sperm[i]] << ")";
      o << ";\n    const int jdl = 0";
      for (int i = 0; i < kt; ++i) o << " | (((tid >> " << i << ") & 1) << " << ds.sperm[i] << ")";
      o << ";\n";
      for (int m = 0; m < NA_(); ++m) {
        unsigned long long cm = 0;
        int jm = 0;
        for (int b = 0; b < kRegBits; ++b)
          if (m & (1 << b)) {
            cm |= 1ull << ds.wpos[ds.sperm[kt + b]];
            jm |= 1 << ds.sperm[kt + b];
          }
        o << "    {\n    const V x = " << stored(m, "jdl | " + std::to_string(jm)) << ";\n    dst[wdl | " << cm
          << "ull] = x;\n";
        capture(std::to_string(m), "x");
        o << "    }\n";
      }
      o << "  }\n";
    }
    if (!pair) {
      if (nm) {
        o << "  __syncthreads();\n  for (int i = tid; i < " << nm << "; i += " << nthr << ") {\n    double x = mred[i];\n";
        for (int w = 1; w < nwaves; ++w) o << "    x += mred[" << w * nm << " + i];\n";
        o << "    mpart[t * " << p.n_meas << "ll + MI" << s << "[i]] = x;\n  }\n";
      }
      o << "  }\n}\n";
      finish();
      continue;
    }
    // close the tile scope and the loop over the pair; sum the threads'
    // shares in a fixed order (wave, then waves)
    o << "  }\n  }\n";
    o << "  for (int off = 32; off > 0; off >>= 1) {\n"
         "    ore += __shfl_xor(ore, off);\n    oim += __shfl_xor(oim, off);\n  }\n";
    o << "  if ((tid & 63) == 0) pred[tid >> 6] = double2{ore, oim};\n  __syncthreads();\n";
    o << "  if (tid == 0) {\n    double2 sum = pred[0];\n";
    if (nthr / 64 > 1)
      o << "    for (int w = 1; w < " << nthr / 64 << "; ++w) { sum.x += pred[w].x; sum.y += pred[w].y; }\n";
    o << "    pov[pb] = sum;\n  }\n}\n";
    finish();
  }
  }
}

static const char *kJitOpts[] = {"--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature",
                                 "-Xclang", "-packed-fp32-ops"};

// What besides the source decides the code object: the compile options and
// the hiprtc version (part of the on-disk cache key).
std::string jit_signature() {
  std::string sig;
  for (const char *o : kJitOpts) {
    sig += o;
    sig += ' ';
  }
  int major = 0, minor = 0;
  hiprtcVersion(&major, &minor);
  sig += "hiprtc " + std::to_string(major) + "." + std::to_string(minor);
  return sig;
}

int jit_compile(const std::string &src, std::vector<char> &code, std::string &log) {
  hiprtcProgram prog;
  if (hiprtcCreateProgram(&prog, src.c_str(), "pqs_jit.hip", 0, nullptr, nullptr) != HIPRTC_SUCCESS) {
    log = "hiprtcCreateProgram failed";
    return PQS_ERR_HIP;
  }
  hiprtcResult r = hiprtcCompileProgram(prog, int(sizeof kJitOpts / sizeof kJitOpts[0]), kJitOpts);
  size_t ls = 0;
  hiprtcGetProgramLogSize(prog, &ls);
  log.assign(ls, '\0');
  if (ls) hiprtcGetProgramLog(prog, &log[0]);
  if (r != HIPRTC_SUCCESS) {
    hiprtcDestroyProgram(&prog);
    return PQS_ERR_HIP;
  }
  size_t cs = 0;
  hiprtcGetCodeSize(prog, &cs);
  code.resize(cs);
  hiprtcGetCode(prog, code.data());
  hiprtcDestroyProgram(&prog);
  return PQS_OK;
}

}  // namespace pqs

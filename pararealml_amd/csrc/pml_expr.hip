// Device evaluation of symbolic right-hand sides compiled to a small
// register-machine program (the device form of what the reference's
// SymbolMapper builds with sympy.lambdify, pararealml/operators/
// symbol_mapper.py:160-253), and the batched ODE time loop that runs such a
// program (FDMOperator.solve on a system without a mesh,
// pararealml/operators/fdm/fdm_operator.py:48-77 with the explicit
// integrators of numerical_integrator.py:42-132).
//
// Program: n_instr instructions of four int32 {op, dst, a, b}; registers
// live in LDS, one column per thread (register r of thread i at
// regs[r * blockDim.x + i]), so an instruction's operands are dynamic
// indices without private-memory spills.  Every thread runs the same
// instruction stream, so the code and constants are read through uniform
// (scalar) loads.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <exception>
#include <string>
#include <vector>

#include "pml_common.h"

namespace pml {

enum ExprOp : int {
  OP_CONST = 0,  // r[dst] = consts[a]
  OP_LOAD = 1,   // r[dst] = input a at this element
  OP_TIME = 2,   // r[dst] = t
  OP_ADD = 3,
  OP_SUB = 4,
  OP_MUL = 5,
  OP_DIV = 6,
  OP_POW = 7,    // pow(r[a], r[b])
  OP_POWI = 8,   // r[a] ** b, b an integer (negative: 1 / r[a] ** -b)
  OP_NEG = 9,
  OP_STORE = 10,  // output dst at this element = r[a]
  OP_SQRT = 11,
  OP_EXP = 12,
  OP_LOG = 13,
  OP_SIN = 14,
  OP_COS = 15,
  OP_TAN = 16,
  OP_TANH = 17,
  OP_ABS = 18,
  OP_ASIN = 19,
  OP_ACOS = 20,
  OP_ATAN = 21,
  OP_SINH = 22,
  OP_COSH = 23,
  OP_ATAN2 = 24,
  OP_MIN = 25,
  OP_MAX = 26,
  OP_SIGN = 27,
  OP_POW3H = 28,  // r[a] ** 1.5
  OP_COUNT = 29
};

template <typename T>
__device__ __forceinline__ T powi(T x, int k) {
  const bool neg = k < 0;
  unsigned int e = neg ? static_cast<unsigned int>(-k) : static_cast<unsigned int>(k);
  // left-to-right binary powering: x^2 = x*x exactly as NumPy's square
  T r = T(1);
  bool started = false;
  for (int bit = 31; bit >= 0; --bit) {
    if (started) r = r * r;
    if ((e >> bit) & 1u) {
      r = started ? r * x : x;
      started = true;
    }
  }
  return neg ? T(1) / r : r;
}

// x^(3/2) as x sqrt(x) with the rounding errors of both operations added
// back: s = sqrt(x) is off by r / (2 s), r = x - s^2, and the product by
// pe, so x sqrt(x) = p + (pe + s r / 2).  Within 0.5005 ulp in FP64 on 400000
// arguments in [0, 8] and 1e-100 .. 1e100 (pow: 1.28), and some 25 dependent
// instructions where pow has hundreds.  Zero, infinities, negative values and
// NaN as pow (x sqrt(x) of -infinity is NaN, pow's limit there infinity).
__device__ __forceinline__ double pow3h(double x) {
  const double s = sqrt(x);
  const double p = x * s;
  const double r = __builtin_fma(-s, s, x);
  const double pe = __builtin_fma(x, s, -p);
  const double v = p + __builtin_fma(0.5 * s, r, pe);
  if (fabs(p) < __builtin_inf()) return v;
  return x == -__builtin_inf() ? -x : p;
}
__device__ __forceinline__ float pow3h(float x) {
  const double d = x;
  return x == -__builtin_inff() ? -x : static_cast<float>(d * sqrt(d));
}

// The operations on one or two values (every opcode that is neither a read
// of an input, a constant or the time, nor a store, nor POWI).
template <typename T>
__device__ __forceinline__ T alu(int op, T x, T y) {
  switch (op) {
    case OP_ADD: return x + y;
    case OP_SUB: return x - y;
    case OP_MUL: return x * y;
    case OP_DIV: return x / y;
    case OP_POW: return pow(x, y);
    case OP_NEG: return -x;
    case OP_SQRT: return sqrt(x);
    case OP_EXP: return exp(x);
    case OP_LOG: return log(x);
    case OP_SIN: return sin(x);
    case OP_COS: return cos(x);
    case OP_TAN: return tan(x);
    case OP_TANH: return tanh(x);
    case OP_ABS: return fabs(x);
    case OP_ASIN: return asin(x);
    case OP_ACOS: return acos(x);
    case OP_ATAN: return atan(x);
    case OP_SINH: return sinh(x);
    case OP_COSH: return cosh(x);
    case OP_ATAN2: return atan2(x, y);
    case OP_MIN: return (x != x || y != y) ? x + y : (y < x ? y : x);
    case OP_MAX: return (x != x || y != y) ? x + y : (y > x ? y : x);
    case OP_SIGN: return x > T(0) ? T(1) : (x < T(0) ? T(-1) : x);
    case OP_POW3H: return pow3h(x);
    default: return T(0);
  }
}

__host__ __device__ __forceinline__ bool two_operands(int op) {
  return (op >= OP_ADD && op <= OP_POW) || (op >= OP_ATAN2 && op <= OP_MAX);
}

// Runs the program for one element: load(k) gives input k, store(k, v)
// receives output k.
template <typename T, class Load, class Store>
__device__ __forceinline__ void run_program(const int4 *__restrict__ code, int n_instr,
                                            const double *__restrict__ consts, T *regs, int rs,
                                            T t, Load load, Store store) {
  for (int pc = 0; pc < n_instr; ++pc) {
    const int4 in = code[pc];
    T *d = regs + in.y * rs;
    // every operand index was range-checked when the program was created
    const T x = in.x >= OP_ADD ? regs[in.z * rs] : T(0);
    switch (in.x) {
      case OP_CONST: *d = static_cast<T>(consts[in.z]); break;
      case OP_LOAD: *d = load(in.z); break;
      case OP_TIME: *d = t; break;
      case OP_POWI: *d = powi(x, in.w); break;
      case OP_STORE: store(in.y, x); break;
      default: *d = alu<T>(in.x, x, two_operands(in.x) ? regs[in.w * rs] : T(0)); break;
    }
  }
}

struct ExprIO {
  const void *in[PML_EXPR_MAX_IO];
  int64_t in_stride[PML_EXPR_MAX_IO];
  void *out[PML_EXPR_MAX_IO];
  int64_t out_stride[PML_EXPR_MAX_IO];
};

template <typename T>
__global__ void __launch_bounds__(128) k_expr_eval(const int4 *code, int n_instr,
                                                   const double *consts, int n_regs, ExprIO io,
                                                   double t, int64_t count) {
  extern __shared__ unsigned char smem[];
  T *regs = reinterpret_cast<T *>(smem) + threadIdx.x;
  const int rs = blockDim.x;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < count;
       e += (int64_t)gridDim.x * blockDim.x) {
    auto load = [&](int k) -> T {
      return static_cast<const T *>(io.in[k])[e * io.in_stride[k]];
    };
    auto store = [&](int k, T v) { static_cast<T *>(io.out[k])[e * io.out_stride[k]] = v; };
    run_program<T>(code, n_instr, consts, regs, rs, static_cast<T>(t), load, store);
  }
  (void)n_regs;
}

// One thread per batch element; the whole time loop in registers + LDS.
// LDS per thread: the program's registers, then y, the stage input and the
// stage accumulator (n rows each), then the stage derivative (n rows).
template <typename T>
__global__ void __launch_bounds__(64) k_ode_solve(const int4 *code, int n_instr,
                                                  const double *consts, int n_regs, int n,
                                                  int integrator, int64_t batch,
                                                  const double *t0, const double *t_step,
                                                  double dt, int64_t n_steps, T *y, T *snaps,
                                                  int64_t snap_every) {
  extern __shared__ unsigned char smem[];
  const int rs = blockDim.x;
  T *regs = reinterpret_cast<T *>(smem) + threadIdx.x;
  T *ys = regs + static_cast<int64_t>(n_regs) * rs;  // y
  T *yt = ys + static_cast<int64_t>(n) * rs;         // stage input
  T *acc = yt + static_cast<int64_t>(n) * rs;        // k1 + 2 k2 + 2 k3 (RK4)
  T *kk = acc + static_cast<int64_t>(n) * rs;        // f(t, .) of the stage
  const int64_t b = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (b >= batch) return;
  for (int i = 0; i < n; ++i) ys[i * rs] = y[b * n + i];
  const T h = static_cast<T>(dt);
  const T half = h / T(2);
  const double tb = t0[b], step = t_step[b];
  int64_t snap = 0;
  auto f = [&](T t, const T *src) {
    auto load = [&](int k) -> T { return src[k * rs]; };
    auto store = [&](int k, T v) { kk[k * rs] = v; };
    run_program<T>(code, n_instr, consts, regs, rs, t, load, store);
  };
  for (int64_t s = 0; s < n_steps; ++s) {
    // the reference's time grid: linspace(t0, t0 + n dt, n + 1)
    const T t = static_cast<T>(static_cast<double>(s) * step + tb);
    if (integrator == PML_INT_FE) {
      f(t, ys);
      for (int i = 0; i < n; ++i) ys[i * rs] = ys[i * rs] + h * kk[i * rs];
    } else if (integrator == PML_INT_MIDPOINT) {
      f(t, ys);
      for (int i = 0; i < n; ++i) yt[i * rs] = ys[i * rs] + half * kk[i * rs];
      f(t + half, yt);
      for (int i = 0; i < n; ++i) ys[i * rs] = ys[i * rs] + h * kk[i * rs];
    } else {
      // k1 = h f(t, y); k2 = h f(t + h/2, y + k1/2); k3 = h f(t + h/2,
      // y + k2/2); k4 = h f(t + h, y + k3); y + (k1 + 2 k2 + 2 k3 + k4) / 6
      f(t, ys);
      for (int i = 0; i < n; ++i) {
        const T k1 = h * kk[i * rs];
        acc[i * rs] = k1;
        yt[i * rs] = ys[i * rs] + k1 / T(2);
      }
      f(t + half, yt);
      for (int i = 0; i < n; ++i) {
        const T k2 = h * kk[i * rs];
        acc[i * rs] = acc[i * rs] + T(2) * k2;
        yt[i * rs] = ys[i * rs] + k2 / T(2);
      }
      f(t + half, yt);
      for (int i = 0; i < n; ++i) {
        const T k3 = h * kk[i * rs];
        acc[i * rs] = acc[i * rs] + T(2) * k3;
        yt[i * rs] = ys[i * rs] + k3;
      }
      f(t + h, yt);
      for (int i = 0; i < n; ++i) {
        const T k4 = h * kk[i * rs];
        ys[i * rs] = ys[i * rs] + (acc[i * rs] + k4) / T(6);
      }
    }
    if (snaps && (s + 1) % snap_every == 0) {
      T *dst = snaps + (snap * batch + b) * n;
      for (int i = 0; i < n; ++i) dst[i] = ys[i * rs];
      ++snap;
    }
  }
  for (int i = 0; i < n; ++i) y[b * n + i] = ys[i * rs];
}

// ---------------------------------------------------------------------------
// The same time loop with the program's independent instructions side by
// side in the lanes of one wavefront per batch element.  A thread that runs
// a right-hand side alone pays an instruction fetch, an LDS round trip and
// the operation's latency for each of its instructions in turn (about 240
// cycles each), with 63 of 64 lanes idle when one system is solved.  Here
// the straight-line program is scheduled on the host into rounds of at most
// 64 instructions whose operands are ready and that share one uniform
// branch; a round costs that latency once.
//
// Values live in LDS slots in single assignment: the stage input y[0 .. n),
// the time, 1, -1, -0, the program's constants, then one slot per
// instruction and one that the idle lanes of a round write.  Lane i < n also
// keeps variable i's state and stage sums in registers.  Every operation
// rounds as the serial kernel's, so the results are the same to the bit.
//
// Bound by latency: a round is an LDS read, the operation and an LDS write,
// and a system's rounds follow one another.  Additions, subtractions,
// products and negations are one fused multiply-add of three slots (x 1 + z,
// z (-1) + x, x z + (-0), x (-1) + (-0): each rounds once, as the operation
// itself; integer powers are their products), so a run of such rounds has no branch and no selection; the other
// kinds are uniform branches between runs.  Measured on four bodies in space
// (206 instructions, 9 rounds), one system, 1000 RK4 steps in FP64 with
// every 10th state kept: 272 ms by the serial kernel (with pow for the cubed
// distances), 6.1 ms by this one (1.5 us a right-hand side).

// One lane's part of a round: operand slots and the result's.
struct WaveOp {
  uint16_t a, b, c, dst;
};
// Consecutive rounds of one kind: WK_FMA or an opcode.
struct WaveRun {
  int kind, rounds;
};
constexpr int WK_FMA = -1;
constexpr int kWaveLanes = 64;
constexpr int kMaxWaveSlots = 2048;  // 16 KiB of FP64 values
constexpr int kMaxWaveRounds = 95;   // 47.5 KiB of schedule
// Systems at once, per instruction of the program, up to which this kernel
// runs.  Its time grows with the batch from about 1024 systems on (4 to 5 us
// a step for each 1024 of four bodies), the serial kernel's with the number
// of instructions (64 systems per wavefront).  RK4 steps of FP64 systems, at
// once / serial: Lorenz (18 instructions) 4096 systems 8.4 / 20.4 us, 16384
// 30.5 / 20.4; two bodies (34) 8192 28 / 63; four bodies (206) 16384 76 / 278;
// Van der Pol (10) 2048 6.9 / 14.1, 8192 25.2 / 14.1.  With elementary
// functions (225 registers, 2 wavefronts per SIMD; 63 instructions) 4096 75 /
// 93, 8192 146 / 93.
// That holds for programs with several instructions a round.  The deeper a
// program, the less this kernel shares out: its time for a batch beyond what
// the chip holds at once is that of the batch's rounds, the serial kernel's
// that of the instructions.  Both are estimated (WaveCost) from chains of 2 to
// 40 operations, one and three side by side (FP64, us a right-hand side, at
// once / serial, 50 RK4 steps): 40 square roots and additions (80 rounds), 256
// systems 15 / 26, 1024 32 / 26, 21248 470 / 26; 16 instructions in 9 rounds,
// 2048 systems 2.8 / 4.6, 4096 5.5 / 4.5.
constexpr int64_t kWaveBatchPerInstr = 256, kWaveBatchPerInstrElementary = 64;

// Microseconds a right-hand side: rounds_us is one system's alone, system_us
// what each of many adds, serial_us the serial kernel's (up to 65536 systems).
struct WaveCost {
  double rounds_us = 0.4, system_us = 0.0, serial_us = 0.0;
  int64_t at_once = 0;  // systems that the 256 CUs hold

  void add_round(int kind) {
    const bool fma = kind == WK_FMA;
    const bool root = kind == OP_DIV || kind == OP_SQRT || kind == OP_POW3H;
    rounds_us += fma ? 0.12 : (root ? 0.30 : 0.35);
    system_us += fma ? 1.6e-4 : (root ? 2.6e-4 : 3.0e-4);
  }
  void add_instruction(int op) {
    const bool plain = op <= OP_DIV || op == OP_NEG || op == OP_STORE || op == OP_SQRT ||
                       op == OP_POW3H;
    serial_us += plain ? 0.28 : (op == OP_POWI ? 0.60 : 0.33);
  }
  bool pays(int64_t batch) const {
    const int64_t fills = (batch + at_once - 1) / at_once;
    return (fills == 1 || fills * rounds_us <= serial_us) && batch * system_us <= serial_us;
  }
};

// kAll false: programs of additions, products, divisions, square roots and
// integer and three-halves powers only (the kernel without the elementary
// functions needs a fifth of the registers).
template <typename T, bool kAll>
__global__ void __launch_bounds__(kWaveLanes)
    k_ode_wave(const WaveOp *__restrict__ rounds, int n_rounds, const WaveRun *__restrict__ runs,
               int n_runs, const double *__restrict__ consts, int n_consts, int n_slots,
               const int *__restrict__ out_slots, int n, int integrator, int64_t batch,
               const double *__restrict__ t0, const double *__restrict__ t_step, double dt,
               int64_t n_steps, T *y, T *snaps, int64_t snap_every) {
  extern __shared__ unsigned char smem[];
  WaveOp *code = reinterpret_cast<WaveOp *>(smem);
  // (one row more than the schedule: each round reads the next one's row)
  T *slot = reinterpret_cast<T *>(smem + sizeof(WaveOp) * kWaveLanes * (n_rounds + 1));
  const int lane = threadIdx.x;
  const int64_t b = blockIdx.x;
  for (int k = lane; k < n_rounds * kWaveLanes; k += kWaveLanes) code[k] = rounds[k];
  for (int k = lane; k < n_slots; k += kWaveLanes) {
    const int c = k - (n + 4);
    slot[k] = c >= 0 && c < n_consts ? static_cast<T>(consts[c])
              : k == n + 1           ? T(1)
              : k == n + 2           ? T(-1)
              : k == n + 3           ? -T(0)
                                     : T(0);
  }
  const bool own = lane < n;
  const int out = own ? out_slots[lane] : 0;
  T ys = own ? y[b * n + lane] : T(0);
  const T h = static_cast<T>(dt);
  const T half = h / T(2);
  const double tb = t0[b], step = t_step[b];
  __syncthreads();

  // f(t, src) of the lane's variable.  One wavefront: its LDS accesses
  // complete in order, the fences keep the compiler from moving them.
  auto f = [&](T t, T src) -> T {
    if (own) slot[lane] = src;
    if (lane == 0) slot[n] = t;
    const WaveOp *op = code + lane;
    WaveOp w = *op;
    for (int run = 0; run < n_runs; ++run) {
      const WaveRun R = runs[run];
      if (R.kind == WK_FMA) {
        for (int r = 0; r < R.rounds; ++r) {
          op += kWaveLanes;
          const WaveOp next = *op;
          __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
          slot[w.dst] = __builtin_elementwise_fma(slot[w.a], slot[w.b], slot[w.c]);
          w = next;
        }
      } else {
        for (int r = 0; r < R.rounds; ++r) {
          op += kWaveLanes;
          const WaveOp next = *op;
          __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
          const T x = slot[w.a], z = slot[w.b];
          T v;
          if (R.kind == OP_DIV) v = x / z;
          else if (R.kind == OP_POW3H) v = pow3h(x);
          else if (kAll) v = alu<T>(R.kind, x, z);
          else v = sqrt(x);
          slot[w.dst] = v;
          w = next;
        }
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    const T k = slot[out];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    return k;
  };

  int64_t snap = 0, until = snap_every;
  const int stages = integrator == PML_INT_FE ? 1 : (integrator == PML_INT_MIDPOINT ? 2 : 4);
  for (int64_t s = 0; s < n_steps; ++s) {
    const T t = static_cast<T>(static_cast<double>(s) * step + tb);
    T src = ys, acc = T(0), ts = t;
    for (int stage = 0; stage < stages; ++stage) {
      const T kk = f(ts, src);
      const T k = h * kk;
      if (stage == stages - 1) {
        ys = ys + (stages == 4 ? (acc + k) / T(6) : k);
      } else if (stages == 2) {
        src = ys + half * kk;
        ts = t + half;
      } else {
        acc = stage == 0 ? k : acc + T(2) * k;
        src = ys + (stage == 2 ? k : k / T(2));
        ts = t + (stage == 2 ? h : half);
      }
    }
    if (snaps && --until == 0) {
      if (own) snaps[(snap * batch + b) * n + lane] = ys;
      ++snap;
      until = snap_every;
    }
  }
  if (own) y[b * n + lane] = ys;
}

}  // namespace pml

using namespace pml;

// A validated program resident in device memory, with its wavefront schedule
// (n_rounds 0: it has none and runs serially).
struct pml_program_s {
  int4 *code = nullptr;
  double *consts = nullptr;
  int n_instr = 0, n_consts = 0, n_regs = 0, n_in = 0, n_out = 0;
  bool all_outputs_stored = false;
  int device = 0;
  WaveOp *rounds = nullptr;
  WaveRun *runs = nullptr;
  int *out_slots = nullptr;
  int n_rounds = 0, n_runs = 0, n_slots = 0;
  bool elementary = false;  // uses more than the short kernel's operations
  WaveCost cost;
};

static size_t wave_lds(const pml_program_s *p, size_t value_bytes) {
  return sizeof(WaveOp) * kWaveLanes * (p->n_rounds + 1) + value_bytes * p->n_slots;
}

// Schedules a validated program into rounds for k_ode_wave: slots in single
// assignment, then, round by round, the instructions that share the branch
// of the ready one with the longest way to an output (in rough latencies),
// the longest ways first.  Returns no rounds where the program does not fit.
static void wave_schedule(const int32_t *code, int n_instr, int n_consts, int n_vars,
                          int n_outputs, std::vector<WaveOp> *rounds, std::vector<WaveRun> *runs,
                          std::vector<int> *out_slots, int *n_slots) {
  struct Node {
    int kind;  // instructions of one kind may share a round
    int s[3];  // operand slots
    int ways = 0, waits = 0;
    std::vector<int> users;
  };
  rounds->clear();
  runs->clear();
  const int time = n_vars, one = n_vars + 1, minus_one = n_vars + 2, minus_zero = n_vars + 3;
  const int first = n_vars + 4 + n_consts;
  std::vector<Node> nodes;
  std::vector<int> reg(PML_EXPR_MAX_REGS, 0);
  auto node = [&](int kind, int a, int b, int c) {  // returns the result's slot
    Node nd{kind, {a, b, c}};
    nodes.push_back(std::move(nd));
    return first + static_cast<int>(nodes.size()) - 1;
  };
  out_slots->assign(n_outputs, 0);
  for (int pc = 0; pc < n_instr; ++pc) {
    const int op = code[4 * pc], dst = code[4 * pc + 1], a = code[4 * pc + 2],
              b = code[4 * pc + 3];
    if (op == OP_CONST) {
      reg[dst] = n_vars + 4 + a;
    } else if (op == OP_LOAD) {
      reg[dst] = a;
    } else if (op == OP_TIME) {
      reg[dst] = time;
    } else if (op == OP_STORE) {
      (*out_slots)[dst] = reg[a];
    } else {
      const int x = reg[a], z = two_operands(op) ? reg[b] : x;
      if (op == OP_ADD) {
        reg[dst] = node(WK_FMA, x, one, z);
      } else if (op == OP_SUB) {
        reg[dst] = node(WK_FMA, z, minus_one, x);
      } else if (op == OP_MUL) {
        reg[dst] = node(WK_FMA, x, z, minus_zero);
      } else if (op == OP_NEG) {
        reg[dst] = node(WK_FMA, x, minus_one, minus_zero);
      } else if (op == OP_POWI) {  // powi()'s products
        const unsigned e = b < 0 ? 0u - static_cast<unsigned>(b) : static_cast<unsigned>(b);
        int r = one;
        bool started = false;
        for (int bit = 31; bit >= 0; --bit) {
          if (started) r = node(WK_FMA, r, r, minus_zero);
          if ((e >> bit) & 1u) {
            r = started ? node(WK_FMA, r, x, minus_zero) : x;
            started = true;
          }
        }
        reg[dst] = b < 0 ? node(OP_DIV, one, r, r) : r;
      } else {
        reg[dst] = node(op, x, z, x);
      }
      if (first + static_cast<int>(nodes.size()) >= kMaxWaveSlots) return;
    }
  }
  const int count = static_cast<int>(nodes.size());
  *n_slots = first + count + 1;
  const auto idle_dst = static_cast<uint16_t>(first + count);
  for (int k = 0; k < count; ++k) {
    std::vector<int> from(nodes[k].s, nodes[k].s + 3);
    std::sort(from.begin(), from.end());
    from.erase(std::unique(from.begin(), from.end()), from.end());
    for (int slot : from) {
      if (slot < first) continue;
      nodes[slot - first].users.push_back(k);
      ++nodes[k].waits;
    }
  }
  for (int k = count - 1; k >= 0; --k) {
    const int kind = nodes[k].kind;
    const int cost = kind == WK_FMA ? 1
                     : kind == OP_DIV || kind == OP_SQRT || kind == OP_POW3H ? 2
                                                                             : 6;
    int below = 0;
    for (int u : nodes[k].users) below = std::max(below, nodes[u].ways);
    nodes[k].ways = cost + below;
  }
  std::vector<int> ready;
  for (int k = 0; k < count; ++k)
    if (!nodes[k].waits) ready.push_back(k);
  while (!ready.empty()) {
    std::stable_sort(ready.begin(), ready.end(),
                     [&](int x, int y) { return nodes[x].ways > nodes[y].ways; });
    const int kind = nodes[ready.front()].kind;
    std::vector<int> taken, rest;
    for (int k : ready) {
      const bool fits =
          nodes[k].kind == kind && taken.size() < static_cast<size_t>(kWaveLanes);
      (fits ? taken : rest).push_back(k);
    }
    const size_t base = rounds->size();
    if (base / kWaveLanes >= static_cast<size_t>(kMaxWaveRounds)) {
      rounds->clear();
      return;
    }
    rounds->resize(base + kWaveLanes, WaveOp{0, 0, 0, idle_dst});
    for (size_t l = 0; l < taken.size(); ++l) {
      const Node &nd = nodes[taken[l]];
      (*rounds)[base + l] =
          WaveOp{static_cast<uint16_t>(nd.s[0]), static_cast<uint16_t>(nd.s[1]),
                 static_cast<uint16_t>(nd.s[2]), static_cast<uint16_t>(first + taken[l])};
    }
    if (!runs->empty() && runs->back().kind == kind)
      ++runs->back().rounds;
    else
      runs->push_back(WaveRun{kind, 1});
    ready = std::move(rest);
    for (int k : taken)
      for (int u : nodes[k].users)
        if (--nodes[u].waits == 0) ready.push_back(u);
  }
}

extern "C" int pml_program_create(const int32_t *code, int n_instr, const double *consts,
                                  int n_consts, int n_regs, int n_inputs, int n_outputs,
                                  pml_program *out) {
  if (!out) return fail(PML_E_INVALID, "null program handle");
  *out = nullptr;
  if (!code || n_instr <= 0 || n_instr > (1 << 20)) return fail(PML_E_INVALID, "empty program");
  if (n_regs <= 0 || n_regs > PML_EXPR_MAX_REGS)
    return fail(PML_E_INVALID, "program register count out of range");
  if (n_consts < 0 || (n_consts && !consts)) return fail(PML_E_INVALID, "bad constants");
  if (n_inputs < 0 || n_inputs > PML_EXPR_MAX_IO || n_outputs <= 0 ||
      n_outputs > PML_EXPR_MAX_IO)
    return fail(PML_E_INVALID, "program input/output count out of range");
  std::vector<char> stored(n_outputs, 0);
  for (int pc = 0; pc < n_instr; ++pc) {
    const int op = code[4 * pc], dst = code[4 * pc + 1], a = code[4 * pc + 2],
              b = code[4 * pc + 3];
    auto reg = [&](int r) { return r >= 0 && r < n_regs; };
    bool ok = op >= 0 && op < OP_COUNT;
    if (ok) {
      switch (op) {
        case OP_CONST: ok = reg(dst) && a >= 0 && a < n_consts; break;
        case OP_LOAD: ok = reg(dst) && a >= 0 && a < n_inputs; break;
        case OP_TIME: ok = reg(dst); break;
        case OP_STORE:
          ok = dst >= 0 && dst < n_outputs && reg(a);
          if (ok) stored[dst] = 1;
          break;
        case OP_POWI: ok = reg(dst) && reg(a); break;
        case OP_ADD: case OP_SUB: case OP_MUL: case OP_DIV: case OP_POW: case OP_ATAN2:
        case OP_MIN: case OP_MAX:
          ok = reg(dst) && reg(a) && reg(b);
          break;
        default: ok = reg(dst) && reg(a); break;
      }
    }
    if (!ok) return fail(PML_E_INVALID, "invalid instruction " + std::to_string(pc));
  }
  auto *p = new pml_program_s();
  p->n_instr = n_instr;
  p->n_consts = n_consts;
  p->n_regs = n_regs;
  p->n_in = n_inputs;
  p->n_out = n_outputs;
  p->all_outputs_stored = true;
  for (char c : stored) p->all_outputs_stored = p->all_outputs_stored && c;
  hipError_t e = hipGetDevice(&p->device);
  if (e == hipSuccess) e = hipMalloc(&p->code, sizeof(int4) * n_instr);
  if (e == hipSuccess) e = hipMalloc(&p->consts, sizeof(double) * (n_consts > 0 ? n_consts : 1));
  if (e == hipSuccess)
    e = hipMemcpy(p->code, code, sizeof(int4) * n_instr, hipMemcpyHostToDevice);
  if (e == hipSuccess && n_consts)
    e = hipMemcpy(p->consts, consts, sizeof(double) * n_consts, hipMemcpyHostToDevice);
  // an ODE system's program also gets its wavefront schedule
  std::vector<WaveOp> rounds;
  std::vector<WaveRun> runs;
  std::vector<int> out_slots;
  int n_slots = 0;
  try {
    if (n_inputs <= n_outputs && p->all_outputs_stored)
      wave_schedule(code, n_instr, n_consts, n_outputs, n_outputs, &rounds, &runs, &out_slots,
                    &n_slots);
  } catch (const std::exception &) {
    rounds.clear();
  }
  if (!rounds.empty()) {
    if (e == hipSuccess) e = hipMalloc(&p->rounds, sizeof(WaveOp) * rounds.size());
    if (e == hipSuccess) e = hipMalloc(&p->runs, sizeof(WaveRun) * runs.size());
    if (e == hipSuccess) e = hipMalloc(&p->out_slots, sizeof(int) * n_outputs);
    if (e == hipSuccess)
      e = hipMemcpy(p->runs, runs.data(), sizeof(WaveRun) * runs.size(), hipMemcpyHostToDevice);
    if (e == hipSuccess)
      e = hipMemcpy(p->rounds, rounds.data(), sizeof(WaveOp) * rounds.size(),
                    hipMemcpyHostToDevice);
    if (e == hipSuccess)
      e = hipMemcpy(p->out_slots, out_slots.data(), sizeof(int) * n_outputs,
                    hipMemcpyHostToDevice);
    p->n_rounds = static_cast<int>(rounds.size() / kWaveLanes);
    p->n_runs = static_cast<int>(runs.size());
    p->n_slots = n_slots;
    for (const WaveRun &r : runs)
      p->elementary |= !(r.kind == WK_FMA || r.kind == OP_DIV || r.kind == OP_SQRT ||
                         r.kind == OP_POW3H);
    for (const WaveRun &r : runs)
      for (int k = 0; k < r.rounds; ++k) p->cost.add_round(r.kind);
    for (int pc = 0; pc < n_instr; ++pc) p->cost.add_instruction(code[4 * pc]);
    // by LDS, and by the registers: 8 wavefronts a SIMD, 2 with elementary functions
    p->cost.at_once = 256 * std::min<int64_t>(p->elementary ? 8 : 32,
                                              160 * 1024 / wave_lds(p, sizeof(double)));
  }
  if (e != hipSuccess) {
    if (p->code) (void)hipFree(p->code);
    if (p->consts) (void)hipFree(p->consts);
    if (p->rounds) (void)hipFree(p->rounds);
    if (p->runs) (void)hipFree(p->runs);
    if (p->out_slots) (void)hipFree(p->out_slots);
    delete p;
    return fail(PML_E_HIP, std::string("program upload: ") + hipGetErrorString(e));
  }
  *out = p;
  return PML_OK;
}

extern "C" int pml_program_destroy(pml_program p) {
  if (!p) return PML_OK;
  // a launch reading the program may still be in flight
  hipError_t e = hipDeviceSynchronize();
  (void)hipFree(p->code);
  (void)hipFree(p->consts);
  if (p->rounds) (void)hipFree(p->rounds);
  if (p->runs) (void)hipFree(p->runs);
  if (p->out_slots) (void)hipFree(p->out_slots);
  delete p;
  if (e != hipSuccess) return fail(PML_E_HIP, std::string("hipDeviceSynchronize: ") +
                                                 hipGetErrorString(e));
  return PML_OK;
}

static int check_device(const pml_program_s *p) {
  int dev = -1;
  PML_HIP_CHECK(hipGetDevice(&dev));
  if (dev != p->device) return fail(PML_E_INVALID, "program created on another device");
  return PML_OK;
}

extern "C" int pml_expr_eval(int precision, pml_program p, const void *const *inputs,
                             const int64_t *in_strides, void *const *outputs,
                             const int64_t *out_strides, double t, int64_t count,
                             void *stream) {
  if (!p) return fail(PML_E_INVALID, "null program");
  if (int rc = check_device(p); rc != PML_OK) return rc;
  if (count <= 0) return fail(PML_E_INVALID, "count must be positive");
  if ((p->n_in && (!inputs || !in_strides)) || !outputs || !out_strides)
    return fail(PML_E_INVALID, "null input/output tables");
  ExprIO io{};
  for (int k = 0; k < p->n_in; ++k) {
    if (!inputs[k] || in_strides[k] < 0) return fail(PML_E_INVALID, "bad program input");
    io.in[k] = inputs[k];
    io.in_stride[k] = in_strides[k];
  }
  for (int k = 0; k < p->n_out; ++k) {
    if (!outputs[k] || out_strides[k] < 0) return fail(PML_E_INVALID, "bad program output");
    io.out[k] = outputs[k];
    io.out_stride[k] = out_strides[k];
  }
  const int nt = 128;
  int64_t nb = (count + nt - 1) / nt;
  if (nb > 65536) nb = 65536;
  hipStream_t st = as_stream(stream);
  if (precision == PML_F64) {
    const size_t lds = static_cast<size_t>(p->n_regs) * nt * sizeof(double);
    hipLaunchKernelGGL(k_expr_eval<double>, dim3(nb), dim3(nt), lds, st, p->code, p->n_instr,
                       p->consts, p->n_regs, io, t, count);
  } else if (precision == PML_F32) {
    const size_t lds = static_cast<size_t>(p->n_regs) * nt * sizeof(float);
    hipLaunchKernelGGL(k_expr_eval<float>, dim3(nb), dim3(nt), lds, st, p->code, p->n_instr,
                       p->consts, p->n_regs, io, t, count);
  } else {
    return fail(PML_E_INVALID, "programs run in FP32 or FP64");
  }
  PML_LAUNCH_CHECK();
  return PML_OK;
}

extern "C" int pml_ode_wave_rounds(pml_program p, int64_t batch) {
  if (!p) return 0;
  const int64_t most =
      p->n_instr * (p->elementary ? kWaveBatchPerInstrElementary : kWaveBatchPerInstr);
  return p->n_rounds && batch <= most && p->cost.pays(batch) ? p->n_rounds : 0;
}

extern "C" int pml_ode_solve(int precision, pml_program p, int integrator_id, int64_t batch,
                             const double *t0, const double *t_step, double dt, int64_t n_steps,
                             void *y, void *snapshots, int64_t snapshot_every, void *stream) {
  if (!p) return fail(PML_E_INVALID, "null program");
  if (int rc = check_device(p); rc != PML_OK) return rc;
  const int n = p->n_out;
  if (p->n_in > n || !p->all_outputs_stored)
    return fail(PML_E_INVALID, "an ODE program reads y[0..n) and writes all n derivatives");
  if (batch <= 0 || !t0 || !t_step || !y || n_steps < 0)
    return fail(PML_E_INVALID, "bad ODE arguments");
  if (integrator_id != PML_INT_FE && integrator_id != PML_INT_MIDPOINT &&
      integrator_id != PML_INT_RK4)
    return fail(PML_E_UNSUPPORTED, "the ODE kernel runs the explicit integrators");
  if (snapshots && snapshot_every <= 0)
    return fail(PML_E_INVALID, "snapshot_every must be positive");
  if (n_steps == 0) return PML_OK;
  const size_t esz = precision == PML_F64 ? 8 : 4;
  if (pml_ode_wave_rounds(p, batch) && (precision == PML_F64 || precision == PML_F32)) {
    const size_t lds = wave_lds(p, esz);
    hipStream_t st = as_stream(stream);
    auto launch = [&](auto kernel, auto *yp, auto *sp) {
      hipLaunchKernelGGL(kernel, dim3(batch), dim3(kWaveLanes), lds, st, p->rounds, p->n_rounds,
                         p->runs, p->n_runs, p->consts, p->n_consts, p->n_slots, p->out_slots, n,
                         integrator_id, batch, t0, t_step, dt, n_steps, yp, sp, snapshot_every);
    };
    if (precision == PML_F64)
      launch(p->elementary ? k_ode_wave<double, true> : k_ode_wave<double, false>,
             static_cast<double *>(y), static_cast<double *>(snapshots));
    else
      launch(p->elementary ? k_ode_wave<float, true> : k_ode_wave<float, false>,
             static_cast<float *>(y), static_cast<float *>(snapshots));
    PML_LAUNCH_CHECK();
    return PML_OK;
  }
  const int nt = 64;
  const size_t lds = (static_cast<size_t>(p->n_regs) + 4 * static_cast<size_t>(n)) * nt * esz;
  if (lds > 160 * 1024)
    return fail(PML_E_UNSUPPORTED, "ODE system too large for the LDS-resident kernel");
  const dim3 grid((batch + nt - 1) / nt);
  hipStream_t st = as_stream(stream);
  if (precision == PML_F64)
    hipLaunchKernelGGL(k_ode_solve<double>, grid, dim3(nt), lds, st, p->code, p->n_instr,
                       p->consts, p->n_regs, n, integrator_id, batch, t0, t_step, dt, n_steps,
                       static_cast<double *>(y), static_cast<double *>(snapshots),
                       snapshot_every);
  else if (precision == PML_F32)
    hipLaunchKernelGGL(k_ode_solve<float>, grid, dim3(nt), lds, st, p->code, p->n_instr,
                       p->consts, p->n_regs, n, integrator_id, batch, t0, t_step, dt, n_steps,
                       static_cast<float *>(y), static_cast<float *>(snapshots),
                       snapshot_every);
  else
    return fail(PML_E_INVALID, "the ODE kernel runs in FP32 or FP64");
  PML_LAUNCH_CHECK();
  return PML_OK;
}

// xg_cf.hpp -- coefficient functions evaluated on the device.
//
// NGSolve evaluates a CoefficientFunction at the mapped integration points
// of a rule (symboliccutbfi.cpp:229-287 multiplies the proxies by the
// coefficient's values there; python_cutint.cpp:66-98 sums cf * weight).
// Here a coefficient is a small postfix program over the physical point x
// and the element's P1 grid functions, built on the host from the
// expression tree and interpreted per point: every lane of a wave runs the
// same program, so the dispatch on the opcode is wave-uniform.
//
// The header is shared with host builds (tests compile it with g++ and
// define XG_CF_FN themselves).
#pragma once
#include <math.h>
#include <stdint.h>

#ifndef XG_CF_FN
#include <hip/hip_runtime.h>
#define XG_CF_FN __device__ __forceinline__
#define XG_CF_HD __host__ __device__ inline
#endif
#ifndef XG_CF_HD
#define XG_CF_HD inline
#endif

namespace xg {
namespace cf {

// opcodes (the values are part of the C ABI, include/xg_abi.h)
enum Op : int32_t {
  END = 0,
  CONST = 1,   // + index into the constants: push c[k]
  COORD = 2,   // + coordinate d: push x_d (physical)
  ADD = 3,     // a b -> a + b
  SUB = 4,     // a b -> a - b
  MUL = 5,     // a b -> a * b
  DIV = 6,     // a b -> a / b
  NEG = 7,     // a -> -a
  POWI = 8,    // + integer exponent n: a -> a^n (n < 0: 1 / a^-n)
  POW = 9,     // a b -> pow(a, b)
  SQRT = 10,
  SIN = 11,
  COS = 12,
  TAN = 13,
  EXP = 14,
  LOG = 15,
  ATAN = 16,
  TANH = 17,
  ABS = 18,
  GF1 = 19,    // + grid function slot s: push sum_k lam_k u_s[v_k] (P1 nodal values)
  IFPOS = 20,  // a b c -> (a > 0 ? b : c)  (NGSolve IfPos)
  MAX = 21,    // a b -> max(a, b)
  MIN = 22,    // a b -> min(a, b)
  EL0 = 23,    // + grid function slot s: push u_s[e] (piecewise constant, one value per element)
  NOPS = 24
};

constexpr int MAXCODE = 192;  // program words
constexpr int MAXCONST = 48;  // constants
constexpr int MAXGF = 4;      // P1 grid functions
constexpr int MAXSTACK = 16;  // evaluation stack depth

// the operations as the kernels read them: by their effect on the stack, so
// that few comparisons lead to one
enum Ins : int32_t {
  I_CONST, I_COORD, I_GF1, I_EL0,                                // push
  I_ADD, I_SUB, I_MUL, I_DIV, I_MAX, I_MIN, I_POW, I_IFPOS,      // take one, IFPOS two
  I_NEG, I_ABS, I_SQRT, I_POWI, I_SIN, I_COS, I_TAN, I_EXP, I_LOG, I_ATAN, I_TANH
};
inline int32_t ins_of(int32_t op) {  // host
  constexpr int32_t t[NOPS] = {-1,    I_CONST, I_COORD, I_ADD,   I_SUB, I_MUL, I_DIV, I_NEG,  I_POWI,
                               I_POW, I_SQRT,  I_SIN,   I_COS,   I_TAN, I_EXP, I_LOG, I_ATAN, I_TANH,
                               I_ABS, I_GF1,   I_IFPOS, I_MAX,   I_MIN, I_EL0};
  return t[op];
}

// a validated program, passed to the kernels by value (kernel arguments are
// read through the scalar cache: wave-uniform)
struct Prog {
  int32_t n;      // operations
  int32_t depth;  // deepest stack
  int32_t math;   // has a function of the math library (POW .. TANH but SQRT)
  struct {
    int32_t op, a;                 // Ins, its immediate operand
  } ins[MAXCODE + 1];              // (one past the last may be read)
  double c[MAXCONST];
  const double *gf[MAXGF];
};

// words taken by an opcode (itself and its immediate operand)
inline int op_words(int32_t op) {
  return (op == CONST || op == COORD || op == POWI || op == GF1 || op == EL0) ? 2 : 1;
}

// stack effect of an opcode
inline int op_delta(int32_t op) {
  switch (op) {
    case CONST: case COORD: case GF1: case EL0: return 1;
    case ADD: case SUB: case MUL: case DIV: case POW: case MAX: case MIN: return -1;
    case IFPOS: return -2;
    default: return 0;
  }
}

// host: checks a program (known opcodes, operand ranges, stack depth within
// MAXSTACK, exactly one value left) and copies it into p.  Returns 0 or a
// message.
inline const char *validate(int32_t ncode, const int32_t *code, int32_t nconst, const double *consts, int32_t ngf,
                            const double *const *gf, Prog &p) {
  if (ncode <= 0 || ncode > MAXCODE || !code) return "coefficient program: 1 .. 192 code words";
  if (nconst < 0 || nconst > MAXCONST || (nconst > 0 && !consts)) return "coefficient program: at most 48 constants";
  if (ngf < 0 || ngf > MAXGF || (ngf > 0 && !gf)) return "coefficient program: at most 4 grid functions";
  int depth = 0;
  p.n = 0;
  p.depth = 1;
  p.math = 0;
  for (int pc = 0; pc < ncode;) {
    const int32_t op = code[pc];
    if (op <= END || op >= NOPS) return "coefficient program: unknown opcode";
    const int w = op_words(op);
    if (pc + w > ncode) return "coefficient program: missing operand";
    const int32_t a = w == 2 ? code[pc + 1] : 0;
    if (op == CONST && (a < 0 || a >= nconst)) return "coefficient program: constant index out of range";
    if (op == COORD && (a < 0 || a > 2)) return "coefficient program: coordinate out of range";
    if ((op == GF1 || op == EL0) && (a < 0 || a >= ngf || !gf[a]))
      return "coefficient program: grid function slot out of range";
    const int need = (op == IFPOS) ? 3 : (op_delta(op) == -1 ? 2 : (op_delta(op) == 0 ? 1 : 0));
    if (depth < need) return "coefficient program: stack underflow";
    depth += op_delta(op);
    if (depth > MAXSTACK) return "coefficient program: stack deeper than 16";
    if (depth > p.depth) p.depth = depth;
    if (op == POW || (op >= SIN && op <= TANH)) p.math = 1;
    p.ins[p.n].op = ins_of(op);
    p.ins[p.n++].a = a;
    pc += w;
  }
  if (depth != 1) return "coefficient program: must leave exactly one value";
  for (int k = p.n; k <= MAXCODE; ++k) p.ins[k].op = p.ins[k].a = 0;
  for (int k = 0; k < MAXCONST; ++k) p.c[k] = k < nconst ? consts[k] : 0.0;
  for (int k = 0; k < MAXGF; ++k) p.gf[k] = k < ngf ? gf[k] : nullptr;
  return nullptr;
}

// true when the program reads piecewise constant grid functions (EL0)
inline bool uses_elements(const Prog &p) {
  for (int pc = 0; pc < p.n; ++pc)
    if (p.ins[pc].op == I_EL0) return true;
  return false;
}

// the value that an operation pushes
template <int D>
XG_CF_FN double pushed(const Prog &P, int32_t op, int32_t a, const double *x, const double *lam, const int32_t *vv,
                       int e) {
  if (op == I_CONST) return P.c[a];
  if (op == I_COORD) return a == 0 ? x[0] : (a == 1 ? x[1] : x[2]);
  if (op == I_EL0) return P.gf[a][e];
  const double *u = P.gf[a];
  double v = 0.0;
#pragma unroll
  for (int k = 0; k <= D; ++k) v += lam[k] * u[vv[k]];
  return v;
}
// s op t (IFPOS aside)
template <bool MATH>
XG_CF_FN double binary(int32_t op, double s, double t) {
  switch (op) {
    case I_ADD: return s + t;
    case I_SUB: return s - t;
    case I_MUL: return s * t;
    case I_DIV: return s / t;
    case I_MAX: return fmax(s, t);
    case I_MIN: return fmin(s, t);
    default: break;
  }
  if constexpr (MATH) return pow(s, t);
  return t;
}
template <bool MATH>
XG_CF_FN double unary(int32_t op, int32_t a, double t) {
  switch (op) {
    case I_NEG: return -t;
    case I_ABS: return fabs(t);
    case I_SQRT: return sqrt(t);
    case I_POWI: {
      int n = a < 0 ? -a : a;
      double r = 1.0, q = t;
      while (n) {  // square and multiply
        if (n & 1) r *= q;
        q *= q;
        n >>= 1;
      }
      return a < 0 ? 1.0 / r : r;
    }
    default: break;
  }
  if constexpr (MATH) switch (op) {
      case I_SIN: return sin(t);
      case I_COS: return cos(t);
      case I_TAN: return tan(t);
      case I_EXP: return exp(t);
      case I_LOG: return log(t);
      case I_ATAN: return atan(t);
      case I_TANH: return tanh(t);
      default: break;
    }
  return t;
}

// Value of the program at the physical point x of element e with vertices
// vv (D + 1 of them) and barycentrics lam (lam_k of vertex k).  The stack is
// DEPTH registers with the top first: a push or pop moves the others, so no
// entry is addressed by a run-time index (an indexed private array lives in
// scratch memory: every operation of every point went through it).  MATH =
// false: for programs without library functions, whose registers (over 200)
// the others would pay for with their waves.
template <int D, int DEPTH = MAXSTACK, bool MATH = true>
XG_CF_FN double eval(const Prog &P, const double *x, const double *lam, const int32_t *vv, int e) {
  double st[DEPTH + 1];
#pragma unroll
  for (int k = 0; k <= DEPTH; ++k) st[k] = 0.0;
  int32_t op = P.ins[0].op, a = P.ins[0].a;
  for (int pc = 0; pc < P.n; ++pc) {
    // the next operation is under way while this one runs
    const int32_t op1 = P.ins[pc + 1].op, a1 = P.ins[pc + 1].a;
    if (op < I_ADD) {
      const double v = pushed<D>(P, op, a, x, lam, vv, e);
#pragma unroll
      for (int k = DEPTH; k > 0; --k) st[k] = st[k - 1];
      st[0] = v;
    } else if (op < I_IFPOS) {
      st[0] = binary<MATH>(op, st[1], st[0]);
#pragma unroll
      for (int k = 1; k < DEPTH; ++k) st[k] = st[k + 1];
    } else if (op == I_IFPOS) {
      st[0] = st[DEPTH > 1 ? 2 : 1] > 0.0 ? st[1] : st[0];
#pragma unroll
      for (int k = 1; k + 1 < DEPTH; ++k) st[k] = st[k + 2];
    } else {
      st[0] = unary<MATH>(op, a, st[0]);
    }
    op = op1;
    a = a1;
  }
  return st[0];
}

// The same with the entries below the top in memory (LDS on the device): entry
// k at st[k * stride], P.depth - 1 of them.  For deep programs, whose pushes and
// pops would move 16 registers each, and for programs with library functions,
// whose registers leave none for a stack.
template <int D, bool MATH>
XG_CF_FN double eval_mem(const Prog &P, const double *x, const double *lam, const int32_t *vv, int e, double *st,
                         int stride) {
  double t = 0.0;
  double *sp = st - stride;  // the entry below the top (before st: none)
  int32_t op = P.ins[0].op, a = P.ins[0].a;
  for (int pc = 0; pc < P.n; ++pc) {
    const int32_t op1 = P.ins[pc + 1].op, a1 = P.ins[pc + 1].a;
    if (op < I_ADD) {
      if (pc > 0) {
        sp += stride;
        *sp = t;
      }
      t = pushed<D>(P, op, a, x, lam, vv, e);
    } else if (op < I_IFPOS) {
      t = binary<MATH>(op, *sp, t);
      sp -= stride;
    } else if (op == I_IFPOS) {
      t = *(sp - stride) > 0.0 ? *sp : t;
      sp -= 2 * stride;
    } else {
      t = unary<MATH>(op, a, t);
    }
    op = op1;
    a = a1;
  }
  return t;
}

}  // namespace cf
}  // namespace xg

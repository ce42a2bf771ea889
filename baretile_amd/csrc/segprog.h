// A bt_program as the segment kernels (elementwise.hip) run it: split into what is one value a row and what differs
// along it, the second as a chain through an accumulator.
//
// The evaluator of program.h keeps a register file of 16 values for each of a segment's 8 columns and picks registers by
// index: 241 registers a thread, so two waves a SIMD, three moves around every operand of every column, and a broadcast
// operand's arithmetic (a row's mean, its reciprocal root) done again for each column. Here the host translates the
// program first (SegProgram::make): instructions whose operands are constants or inputs with a column stride of 0 run
// once a row, on one value; the others take operands from the accumulator (the instruction before, which most read), an
// input, one of a few stored values, or a row value, chosen by a uniform branch, and leave their result in the
// accumulator. The arithmetic of each instruction is program.h's, so the results are the same to the bit. Programs that
// need more inputs, stored values or row values than there are slots for run on the general evaluator.
//
// 2048 x 4096 bf16, back to back (the register file's times first): x * 2 29.9 -> 15.4 us, x + y 40 -> 16.5, silu 69 ->
// 26, the last step of a layer normalization ((x - m) * rsqrt(v + eps) * w + b) 111 -> 33; row sums 19.8 -> 9.7 and of
// (x - m)^2 36.6 -> 14.7. What is left is the dispatch: some 60 instructions an operation, on 4 waves a SIMD.
#pragma once
#include "program.h"

namespace bt {

constexpr int SEG_IN = 4, SEG_TMP = 4, SEG_ROW = 8;  // inputs that vary along a row, stored values, row values
// Operand codes: the accumulator, then the slots of each kind.
constexpr int SRC_ACC = 0, SRC_IN = 1, SRC_TMP = SRC_IN + SEG_IN, SRC_ROW = SRC_TMP + SEG_TMP;
constexpr uint8_t NO_SLOT = 255;
typedef uint32_t words4 __attribute__((ext_vector_type(4)));

struct SegInst {
  uint8_t op, x, y, z;  // operand codes
  uint8_t st, pad_[3];  // the stored-value slot that also takes the result, or NO_SLOT
};
struct RowInst {
  uint8_t op, dst, a, b, c;
  uint8_t st;  // the row-value slot that also takes the result, or NO_SLOT
  uint8_t pad_[2];
  uint32_t imm;
};

struct SegProgram {
  int32_t n_row, n_vec, n_in, n_tmp;
  uint8_t in_at[SEG_IN];  // the operand behind each input slot
  uint8_t wide[SEG_IN];   // its columns are contiguous and 1: every row starts on 16 bytes, 2 (4-byte values): some may
  RowInst row[BT_MAX_INST];
  SegInst vec[BT_MAX_INST + 1];
  bt_operand in[BT_MAX_INPUTS];

  // Translates prog for segments of rows of [batch, rows, cols]; false when it doesn't fit the slots.
  inline bool make(const bt_program &prog, int64_t batch, int64_t rows);
};

static inline int op_arity(int op) {
  switch (op) {
    case BT_OP_LOAD: case BT_OP_CONST: return 0;
    case BT_OP_ADD: case BT_OP_SUB: case BT_OP_MUL: case BT_OP_DIV: case BT_OP_MAX: case BT_OP_MIN:
    case BT_OP_CMPLT: case BT_OP_CMPLE: case BT_OP_CMPNE: case BT_OP_CMPEQ: return 2;
    case BT_OP_WHERE: return 3;
    default: return 1;
  }
}

// The lowest free slot of `n`, taken; -1 when there is none.
static inline int take_slot(uint32_t &used, int n) {
  for (int i = 0; i < n; i++)
    if (!(used >> i & 1u)) {
      used |= 1u << i;
      return i;
    }
  return -1;
}

inline bool SegProgram::make(const bt_program &prog, int64_t batch, int64_t rows) {
  // every instruction as a value of its own: its operands are the values last written to the registers it names
  struct Value {
    bool row, in, need;
    int src[3], slot, at, last, last_row;  // slot: input or row-value slot; at: place in vec; last: last reader in vec
    bool far;                              // read by a vec instruction other than the next
  } v[BT_MAX_INST];
  int reg[BT_MAX_REGS];
  for (int &r : reg) r = -1;
  n_in = n_row = n_vec = n_tmp = 0;
  for (int i = 0; i < prog.n_inst; i++) {
    const bt_inst &in = prog.inst[i];
    Value &u = v[i];
    u = Value{true, false, false, {-1, -1, -1}, -1, -1, -1, -1, false};
    if (in.op == BT_OP_MOV) {  // another name for its operand
      if (reg[in.a] < 0) return false;
      reg[in.dst] = reg[in.a];
      continue;
    }
    if (prog.dtype != BT_INT32 && (in.op == BT_OP_SIN || in.op == BT_OP_COS || in.op == BT_OP_TANH || in.op == BT_OP_GELU))
      return false;  // the longest operations stay out of line, in the general evaluator
    const uint8_t regs[3] = {in.a, in.b, in.c};
    for (int k = 0; k < op_arity(in.op); k++) {
      u.src[k] = reg[regs[k]];
      if (u.src[k] < 0) return false;  // a register that nothing wrote
      if (!v[u.src[k]].row) u.row = false;
    }
    if (in.op == BT_OP_LOAD && prog.in[in.a].sc != 0) u.row = false, u.in = true;
    reg[in.dst] = i;
  }
  const int result = reg[prog.result];
  if (result < 0) return false;
  v[result].need = true;
  for (int i = prog.n_inst - 1; i >= 0; i--)
    if (v[i].need)
      for (int s : v[i].src)
        if (s >= 0) v[s].need = true;
  // the row's instructions, on registers of their own; those that the rest reads also go to a row-value slot
  uint32_t row_slots = 0;
  auto keep_row = [&](int s) {
    if (v[s].slot < 0) v[s].slot = take_slot(row_slots, SEG_ROW);
    return v[s].slot >= 0;
  };
  for (int i = 0; i < prog.n_inst; i++) {
    if (!v[i].need || prog.inst[i].op == BT_OP_MOV) continue;
    for (int s : v[i].src)
      if (s >= 0 && v[s].row) {
        if (v[i].row) v[s].last_row = i;
        else if (!keep_row(s)) return false;
      }
    if (v[i].in) {
      const uint8_t at = prog.inst[i].a;
      for (int k = 0; k < n_in; k++)
        if (in_at[k] == at) v[i].slot = k;
      if (v[i].slot < 0) {
        if (n_in == SEG_IN) return false;
        v[i].slot = n_in;
        in_at[n_in++] = at;
      }
    } else if (!v[i].row) {
      for (int s : v[i].src)
        if (s >= 0 && !v[s].row && !v[s].in) {
          v[s].last = n_vec;
          if (n_vec != v[s].at + 1) v[s].far = true;
        }
      v[i].at = n_vec++;
    }
  }
  if (v[result].row && !keep_row(result)) return false;
  const bool mov = v[result].row || v[result].in || v[result].at != n_vec - 1;  // the result has to come last
  if (mov && !v[result].row && !v[result].in) v[result].last = n_vec, v[result].far = true;
  uint32_t regs = 0;
  int where[BT_MAX_INST];
  for (int i = 0; i < prog.n_inst; i++) {
    if (!v[i].need || !v[i].row || prog.inst[i].op == BT_OP_MOV) continue;
    const bt_inst &in = prog.inst[i];
    RowInst &o = row[n_row++];
    o = RowInst{in.op, 0, in.a, 0, 0, v[i].slot < 0 ? NO_SLOT : (uint8_t)v[i].slot, {0, 0}, in.imm};
    uint8_t *to[3] = {&o.a, &o.b, &o.c};
    for (int k = 0; k < op_arity(in.op); k++) *to[k] = (uint8_t)where[v[i].src[k]];
    for (int k = 0; k < op_arity(in.op); k++)
      if (v[v[i].src[k]].last_row == i) regs &= ~(1u << where[v[i].src[k]]);
    where[i] = take_slot(regs, BT_MAX_REGS);
    if (where[i] < 0) return false;
    o.dst = (uint8_t)where[i];
    if (v[i].last_row < 0) regs &= ~(1u << where[i]);  // no row instruction reads it
  }
  // the rest, in order
  uint32_t tmps = 0;
  int tmp[BT_MAX_INST];
  auto code = [&](int s, int at) -> uint8_t {
    if (v[s].row) return (uint8_t)(SRC_ROW + v[s].slot);
    if (v[s].in) return (uint8_t)(SRC_IN + v[s].slot);
    return (uint8_t)(v[s].at + 1 == at ? SRC_ACC : SRC_TMP + tmp[s]);
  };
  int at = 0;
  for (int i = 0; i < prog.n_inst; i++) {
    if (v[i].at < 0) continue;
    SegInst &o = vec[at];
    o = SegInst{prog.inst[i].op, SRC_ACC, SRC_ACC, SRC_ACC, NO_SLOT, {0, 0, 0}};
    uint8_t *to[3] = {&o.x, &o.y, &o.z};
    for (int k = 0; k < 3; k++)
      if (v[i].src[k] >= 0) *to[k] = code(v[i].src[k], at);
    for (int s : v[i].src)
      if (s >= 0 && v[s].far && v[s].last == at) tmps &= ~(1u << tmp[s]);
    if (v[i].far) {
      tmp[i] = take_slot(tmps, SEG_TMP);
      if (tmp[i] < 0) return false;
      o.st = (uint8_t)tmp[i];
      n_tmp = tmp[i] >= n_tmp ? tmp[i] + 1 : n_tmp;
    }
    at++;
  }
  if (mov) vec[n_vec++] = SegInst{BT_OP_MOV, code(result, at), SRC_ACC, SRC_ACC, NO_SLOT, {0, 0, 0}};
  for (int i = 0; i < prog.n_inputs; i++) in[i] = prog.in[i];
  for (int k = 0; k < n_in; k++) {
    const bt_operand &o = in[in_at[k]];
    const uint64_t size = o.dtype == BT_BF16 ? 2 : 4;
    uint64_t starts = o.ptr;
    if (rows > 1) starts |= (uint64_t)o.sr * size;
    if (batch > 1) starts |= (uint64_t)o.sb * size;
    wide[k] = o.sc != 1 ? 0 : starts % 16 == 0 ? 1 : size == 4 ? 2 : 0;
  }
  return true;
}

// A segment's 8 values. Vectors held in named variables, never arrays of them picked in loops: with those the compiler
// merges the branches' stores into one through a chosen address, and the values live in memory.
typedef uint32_t seg_t __attribute__((ext_vector_type(SEG)));
static_assert(SEG == 8, "a segment is one 8-wide vector");

template <class F> __device__ __forceinline__ seg_t seg_map(const seg_t &a, F f) {
  return seg_t{f(a[0]), f(a[1]), f(a[2]), f(a[3]), f(a[4]), f(a[5]), f(a[6]), f(a[7])};
}
template <class F> __device__ __forceinline__ seg_t seg_map(const seg_t &a, const seg_t &b, F f) {
  return seg_t{f(a[0], b[0]), f(a[1], b[1]), f(a[2], b[2]), f(a[3], b[3]),
               f(a[4], b[4]), f(a[5], b[5]), f(a[6], b[6]), f(a[7], b[7])};
}

// The operations up to SILU that expand to many instructions, in line (a call would have the registers that live across
// it saved to memory); make() leaves the longest to the general evaluator.
#define BT_LONG_OPS(BT_LONG)                        \
  BT_LONG(BT_OP_EXP, expf(A))                       \
  BT_LONG(BT_OP_EXP2, exp2f(A))                     \
  BT_LONG(BT_OP_LOG, logf(A))                       \
  BT_LONG(BT_OP_LOG2, log2f(A))                     \
  BT_LONG(BT_OP_SQRT, sqrtf(A))                     \
  BT_LONG(BT_OP_RECIP, 1.0f / A)                    \
  BT_LONG(BT_OP_RSQRT, 1.0f / sqrtf(A))             \
  BT_LONG(BT_OP_SIGMOID, 1.0f / (1.0f + expf(-A)))  \
  BT_LONG(BT_OP_SILU, A / (1.0f + expf(-A)))

// One instruction of two operands at most over a segment, as apply_op: the same arithmetic and rounding.
template <int DT>
__device__ __forceinline__ seg_t seg_op(int op, const seg_t &a, const seg_t &b) {
  if (DT == BT_INT32) return seg_map(a, b, [&](uint32_t x, uint32_t y) { return (uint32_t)int_op(op, (int32_t)x, (int32_t)y); });
  seg_t o;
#define BT_OP(code, expr)                                                    \
  case code:                                                                 \
    o = seg_map(a, b, [](uint32_t x, uint32_t y) {                           \
      const float A = __uint_as_float(x), B = __uint_as_float(y);            \
      (void)B;                                                               \
      return __float_as_uint(expr);                                          \
    });                                                                      \
    break;
  switch (op) {
    BT_OP(BT_OP_ADD, A + B)
    BT_OP(BT_OP_SUB, A - B)
    BT_OP(BT_OP_MUL, A * B)
    BT_OP(BT_OP_DIV, A / B)
    BT_OP(BT_OP_MAX, (A != A || B != B) ? __builtin_nanf("") : fmaxf(A, B))
    BT_OP(BT_OP_MIN, (A != A || B != B) ? __builtin_nanf("") : fminf(A, B))
    BT_OP(BT_OP_CMPLT, A < B ? 1.0f : 0.0f)
    BT_OP(BT_OP_CMPLE, A <= B ? 1.0f : 0.0f)
    BT_OP(BT_OP_CMPNE, A != B ? 1.0f : 0.0f)
    BT_OP(BT_OP_CMPEQ, A == B ? 1.0f : 0.0f)
    BT_OP(BT_OP_NEG, -A)
    BT_OP(BT_OP_RELU, A > 0.0f ? A : 0.0f)
    BT_OP(BT_OP_FTOB, round_packed(A))
    BT_LONG_OPS(BT_OP)
    default: o = a;
  }
#undef BT_OP
  if (DT == BT_BF16) o = seg_map(o, [](uint32_t x) { return __float_as_uint(round_packed(__uint_as_float(x))); });
  return o;
}

// The same on one value.
template <int DT>
__device__ __forceinline__ uint32_t row_op(int op, uint32_t a, uint32_t b) {
  Vals<1> x{{a}}, y{{b}};
  if (DT == BT_INT32 || op < BT_OP_EXP || op > BT_OP_SILU) return apply_op<DT, 1, false, false>(op, x, y).x[0];
  const float A = __uint_as_float(a);
  float f = A;
#define BT_OP(code, expr) case code: f = (expr); break;
  switch (op) { BT_LONG_OPS(BT_OP) }
#undef BT_OP
  return __float_as_uint(DT == BT_BF16 ? round_packed(f) : f);
}
#undef BT_LONG_OPS

// The row values of row (b, r): inputs with a column stride of 0, constants, and what follows from them.
template <int DT>
__device__ __forceinline__ seg_t run_row(const SegProgram &p, int64_t b, int64_t r) {
  static_assert(SEG_ROW == SEG, "row values are held as a segment is");
  regfile regs = (regfile)(0u);
  seg_t rv = (seg_t)(0u);
#pragma unroll 1
  for (int i = 0; i < p.n_row; i++) {
    const RowInst in = p.row[i];
    uint32_t o;
    if (in.op == BT_OP_LOAD) o = load_operand<DT>(p.in[in.a], b, r, 0);
    else if (in.op == BT_OP_CONST) o = in.imm;
    else if (in.op == BT_OP_WHERE) {
      const uint32_t cnd = regs[in.a];
      o = (DT == BT_INT32 ? cnd != 0 : __uint_as_float(cnd) != 0.0f) ? regs[in.b] : regs[in.c];
    } else {
      o = row_op<DT>(in.op, regs[in.a], regs[in.b]);
    }
    regs[in.dst] = o;
    if (in.st != NO_SLOT) rv[in.st & (SEG_ROW - 1)] = o;
  }
  return rv;
}

// The segment's 8 values of one input as they are stored: wide bf16 as 4 words of two values, anything else a value
// each, 0 past the row's end (n values to it). Wide segments but a row's last take 16-byte loads.
__device__ __forceinline__ seg_t seg_load(const bt_operand &o, bool wide, int64_t b, int64_t r, int64_t c0, int n) {
  const int64_t at = operand_matrix(o, b) * o.sb + r * o.sr + c0 * o.sc;
  if (o.dtype == BT_BF16) {
    const uint16_t *s = (const uint16_t *)o.ptr + at;
    if (wide && n == SEG) {
      const words4 w = gload((const words4 *)s);
      return seg_t{w[0], w[1], w[2], w[3], 0u, 0u, 0u, 0u};
    }
    auto get = [&](int v) -> uint32_t { return v < n ? gload(s + v * o.sc) : 0u; };
    const seg_t x = seg_t{get(0), get(1), get(2), get(3), get(4), get(5), get(6), get(7)};
    return wide ? seg_t{x[0] | x[1] << 16, x[2] | x[3] << 16, x[4] | x[5] << 16, x[6] | x[7] << 16, 0u, 0u, 0u, 0u} : x;
  }
  const uint32_t *s = (const uint32_t *)o.ptr + at;
  if (wide && n == SEG) {
    const words4 w0 = gload((const words4 *)s), w1 = gload((const words4 *)s + 1);
    return seg_t{w0[0], w0[1], w0[2], w0[3], w1[0], w1[1], w1[2], w1[3]};
  }
  auto get = [&](int v) -> uint32_t { return v < n ? gload(s + v * o.sc) : 0u; };
  return seg_t{get(0), get(1), get(2), get(3), get(4), get(5), get(6), get(7)};
}
template <int DT>
__device__ __forceinline__ seg_t seg_convert(const seg_t &x, int dtype, bool wide) {
  if (dtype == BT_BF16 && wide) {
    auto lo = [](uint32_t w) { return convert_raw<DT>(w & 0xFFFFu, BT_BF16); };
    auto hi = [](uint32_t w) { return convert_raw<DT>(w >> 16, BT_BF16); };
    return seg_t{lo(x[0]), hi(x[0]), lo(x[1]), hi(x[1]), lo(x[2]), hi(x[2]), lo(x[3]), hi(x[3])};
  }
  return seg_map(x, [&](uint32_t w) { return convert_raw<DT>(w, dtype); });
}

// Whether input k of row (b, r) is wide. ROWS: a wave's lanes share the row, so that where only some rows start on 16
// bytes (of rows of 1643 floats every fourth) this row's start counts, in a uniform branch; otherwise every row's. (With whole
// segments of aligned rows alone taking wide loads, 423 x 3628 int32 x + y took 12.6 us, 3 x 40 x 7898 fp32 9.5; so 7.3 and
// 8.9; 11.2 and 9.0 on the general evaluator.)
template <bool ROWS>
__device__ __forceinline__ bool seg_wide(const SegProgram &p, int k, int64_t b, int64_t r) {
  if (p.wide[k] != 2) return p.wide[k];
  const bt_operand &o = p.in[p.in_at[k]];
  return ROWS && (o.ptr + 4 * (uint64_t)(operand_matrix(o, b) * o.sb + r * o.sr)) % 16 == 0;
}
// The program's inputs over a segment, in its dtype, every load issued before the first is converted. FULL: a program
// of any number of inputs and stored values; otherwise three inputs at most and no stored value, on fewer registers
// (106 against 162: four waves a SIMD, not three).
struct SegInputs {
  seg_t x0, x1, x2, x3;
};
static_assert(SEG_IN == 4 && SEG_TMP == 4, "SegInputs and run_seg name four of each");
inline bool seg_small(const SegProgram &p) { return p.n_in <= 3 && p.n_tmp == 0; }
template <int DT, bool FULL, bool ROWS>
__device__ __forceinline__ void fetch_seg(const SegProgram &p, int64_t b, int64_t r, int64_t c0, int n, SegInputs &i) {
  const bool w0 = p.n_in > 0 && seg_wide<ROWS>(p, 0, b, r), w1 = p.n_in > 1 && seg_wide<ROWS>(p, 1, b, r);
  const bool w2 = p.n_in > 2 && seg_wide<ROWS>(p, 2, b, r), w3 = FULL && p.n_in > 3 && seg_wide<ROWS>(p, 3, b, r);
  i.x0 = i.x1 = i.x2 = i.x3 = (seg_t)(0u);
  if (p.n_in > 0) i.x0 = seg_load(p.in[p.in_at[0]], w0, b, r, c0, n);
  if (p.n_in > 1) i.x1 = seg_load(p.in[p.in_at[1]], w1, b, r, c0, n);
  if (p.n_in > 2) i.x2 = seg_load(p.in[p.in_at[2]], w2, b, r, c0, n);
  if (FULL && p.n_in > 3) i.x3 = seg_load(p.in[p.in_at[3]], w3, b, r, c0, n);
  if (p.n_in > 0) i.x0 = seg_convert<DT>(i.x0, p.in[p.in_at[0]].dtype, w0);
  if (p.n_in > 1) i.x1 = seg_convert<DT>(i.x1, p.in[p.in_at[1]].dtype, w1);
  if (p.n_in > 2) i.x2 = seg_convert<DT>(i.x2, p.in[p.in_at[2]].dtype, w2);
  if (FULL && p.n_in > 3) i.x3 = seg_convert<DT>(i.x3, p.in[p.in_at[3]].dtype, w3);
}

// Runs the instructions that vary along the row: the result's bits.
template <int DT, bool FULL>
__device__ __forceinline__ seg_t run_seg(const SegProgram &p, const SegInputs &in, const seg_t &rv) {
  seg_t acc = (seg_t)(0u), t0 = acc, t1 = acc, t2 = acc, t3 = acc;
  // BT_ARM keeps each arm a branch of its own: as selects (what the compiler makes of arms without side effects) an
  // operand costs a move for every slot there is
#define BT_ARM(cond, act) if (cond) { asm volatile(""); act; }
  auto pick = [&](int src) {
    seg_t o = acc;
    if (src != SRC_ACC) {
      if (src < SRC_TMP) {
        if (!FULL) BT_ARM(src == SRC_IN, o = in.x0) else BT_ARM(src == SRC_IN + 1, o = in.x1) else o = in.x2;
        else BT_ARM(src == SRC_IN, o = in.x0) else BT_ARM(src == SRC_IN + 1, o = in.x1) else BT_ARM(src == SRC_IN + 2, o = in.x2)
        else o = in.x3;
      } else if (FULL && src < SRC_ROW) {
        BT_ARM(src == SRC_TMP, o = t0) else BT_ARM(src == SRC_TMP + 1, o = t1) else BT_ARM(src == SRC_TMP + 2, o = t2)
        else o = t3;
      } else {
        o = (seg_t)(rv[(src - SRC_ROW) & (SEG_ROW - 1)]);
      }
    }
    return o;
  };
#pragma unroll 1
  for (int i = 0; i < p.n_vec; i++) {
    const SegInst in_ = p.vec[i];
    const seg_t a = pick(in_.x);
    if (in_.op == BT_OP_MOV) acc = a;
    else if (in_.op == BT_OP_WHERE) {
      const seg_t t = pick(in_.y), e = pick(in_.z);
      auto on = [](uint32_t c) { return DT == BT_INT32 ? c != 0 : __uint_as_float(c) != 0.0f; };
      acc = seg_t{on(a[0]) ? t[0] : e[0], on(a[1]) ? t[1] : e[1], on(a[2]) ? t[2] : e[2], on(a[3]) ? t[3] : e[3],
                  on(a[4]) ? t[4] : e[4], on(a[5]) ? t[5] : e[5], on(a[6]) ? t[6] : e[6], on(a[7]) ? t[7] : e[7]};
    } else {
      acc = seg_op<DT>(in_.op, a, pick(in_.y));
    }
    if (FULL && in_.st != NO_SLOT) {
      BT_ARM(in_.st == 0, t0 = acc) else BT_ARM(in_.st == 1, t1 = acc) else BT_ARM(in_.st == 2, t2 = acc) else t3 = acc;
    }
  }
#undef BT_ARM
  return acc;
}

}  // namespace bt

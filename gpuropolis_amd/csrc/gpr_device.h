// Device building blocks shared by the config and reference kernels: wave-level
// primitives (DPP reductions and scans, readlane), FP32 op semantics, the wave-uniform
// tape interpreter (handlers in one asm block, value stack in LDS under two VGPR entries),
// the Gaussian log-likelihood, its forward-mode and adjoint gradients, and the
// description-length prior of a wave-resident program.
#pragma once
#include "gpr_index.h"
#include "gpr_internal.h"

#define GPR_INF (__builtin_inf())

// ---------------------------------------------------------------- wave primitives
__device__ __forceinline__ int lane_id() { return (int)(threadIdx.x & 63); }
__device__ __forceinline__ int rl_i(int v, int l) { return __builtin_amdgcn_readlane(v, l); }
__device__ __forceinline__ float rl_f(float v, int l) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), l));
}
__device__ __forceinline__ double rl_d(double v, int l) {
    uint64_t b = __builtin_bit_cast(uint64_t, v);
    int lo = __builtin_amdgcn_readlane((int)(uint32_t)b, l);
    int hi = __builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), l);
    return __builtin_bit_cast(double, ((uint64_t)(uint32_t)hi << 32) | (uint32_t)lo);
}
__device__ __forceinline__ int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ double uni_d(double v) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    const unsigned long long hi = (uint32_t)uni((int)(b >> 32)), lo = (uint32_t)uni((int)(uint32_t)b);
    return __longlong_as_double((long long)((hi << 32) | lo));
}
// A dataset record with every field wave-uniform (scalar registers): a record loaded by
// the whole wave otherwise lands in vector registers, where values used at every step
// take registers from the step loop.
__device__ __forceinline__ GprDataset uni_dataset(const GprDataset &g) {
    GprDataset d;
    d.n = uni(g.n);
    d.off = uni(g.off);
    d.chain0 = uni(g.chain0);
    d.nchains = uni(g.nchains);
    d.cap = uni(g.cap);
    d.kc = uni(g.kc);
    d.lconst = uni_d(g.lconst);
    d.wconst = uni_d(g.wconst);
    return d;
}
// A copy of a wave-uniform value that the compiler cannot prove equal to the original:
// an address computed from it at a late use is computed there, instead of being kept
// live (and spilled) from an earlier use of the same address.
__device__ __forceinline__ uint32_t opaque_u32(uint32_t v) { __asm__ volatile("" : "+s"(v)); return v; }
__device__ __forceinline__ int opaque_lane_i32(int v) { __asm__ volatile("" : "+v"(v)); return v; }

// Lane gathers that stay in wave-uniform control flow: lane l receives v of lane
// src mod 64 (ds_bpermute reads the byte address' lane bits, so no index masking is
// needed).  ds_bpermute only sees the values of lanes active when it executes; the
// empty asm pins the result at this point so the compiler cannot sink the gather into a
// branch that deactivates source lanes.
__device__ __forceinline__ int shfl_all(int v, int src) {
    int r = __builtin_amdgcn_ds_bpermute(src << 2, v);
    __asm__ volatile("" : "+v"(r));
    return r;
}
__device__ __forceinline__ float shfl_all(float v, int src) {
    return __builtin_bit_cast(float, shfl_all(__builtin_bit_cast(int, v), src));
}
__device__ __forceinline__ double shfl_all_d(double v, int src) {
    const uint64_t b = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = (uint32_t)shfl_all((int)(uint32_t)b, src), hi = (uint32_t)shfl_all((int)(uint32_t)(b >> 32), src);
    return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}
__device__ __forceinline__ uint64_t ballot(bool p) { return __ballot(p); }

// DPP controls (gfx9 encoding): quad_perm, row_shr:n, row_mirror, row_half_mirror,
// row_bcast:15, row_bcast:31.  DPP moves are VALU operand modifiers: no LDS round trip.
#define DPP_QP_1032 0xB1
#define DPP_QP_2301 0x4E
#define DPP_ROW_SHR(n) (0x110 + (n))
#define DPP_ROW_MIRROR 0x140
#define DPP_ROW_HALF_MIRROR 0x141
#define DPP_ROW_BCAST15 0x142
#define DPP_ROW_BCAST31 0x143

template <int CTRL>
__device__ __forceinline__ int dpp_i(int v) {
    return __builtin_amdgcn_mov_dpp(v, CTRL, 0xf, 0xf, false);
}

// Sum over the 64 lanes, returned uniform.  Butterflies inside each 16-lane row, then rows 0
// and 1, rows 2 and 3, and the pairs, in lane 63: one add a step, with the other lane's value
// as its DPP operand (s_nop: that operand is read two wait states after the vector unit wrote
// it, and the lane one after).
__device__ __forceinline__ float wave_sum_f(float v) {
#define GPR_DPP_ADD(CTRL) "s_nop 1\n\tv_add_f32_dpp %0, %0, %0 " CTRL " bank_mask:0xf\n\t"
    __asm__(GPR_DPP_ADD("quad_perm:[1,0,3,2] row_mask:0xf") GPR_DPP_ADD("quad_perm:[2,3,0,1] row_mask:0xf")
            GPR_DPP_ADD("row_half_mirror row_mask:0xf") GPR_DPP_ADD("row_mirror row_mask:0xf")
            GPR_DPP_ADD("row_bcast:15 row_mask:0xa") GPR_DPP_ADD("row_bcast:31 row_mask:0xc") "s_nop 0"
            : "+v"(v));
#undef GPR_DPP_ADD
    return rl_f(v, 63);
}
template <int CTRL>
__device__ __forceinline__ double dpp_d(double v) {
    const uint64_t b = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)b, CTRL, 0xf, 0xf, false);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)(b >> 32), CTRL, 0xf, 0xf, false);
    return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}
__device__ __forceinline__ double wave_sum_d(double v) {
    v += dpp_d<DPP_QP_1032>(v);
    v += dpp_d<DPP_QP_2301>(v);
    v += dpp_d<DPP_ROW_HALF_MIRROR>(v);
    v += dpp_d<DPP_ROW_MIRROR>(v);
    return (rl_d(v, 0) + rl_d(v, 16)) + (rl_d(v, 32) + rl_d(v, 48));
}
__device__ __forceinline__ int wave_max_i(int v) {
    v = max(v, dpp_i<DPP_QP_1032>(v));
    v = max(v, dpp_i<DPP_QP_2301>(v));
    v = max(v, dpp_i<DPP_ROW_HALF_MIRROR>(v));
    v = max(v, dpp_i<DPP_ROW_MIRROR>(v));
    return max(max(rl_i(v, 0), rl_i(v, 16)), max(rl_i(v, 32), rl_i(v, 48)));
}
// Inclusive prefix sum over the 64 lanes: Kogge-Stone inside rows (row_shr with zero
// fill), then row 15 -> row 1,3 and lane 31 -> rows 2,3 broadcasts.
__device__ __forceinline__ int wave_scan_i(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, DPP_ROW_SHR(1), 0xf, 0xf, true);
    v += __builtin_amdgcn_update_dpp(0, v, DPP_ROW_SHR(2), 0xf, 0xf, true);
    v += __builtin_amdgcn_update_dpp(0, v, DPP_ROW_SHR(4), 0xf, 0xf, true);
    v += __builtin_amdgcn_update_dpp(0, v, DPP_ROW_SHR(8), 0xf, 0xf, true);
    v += __builtin_amdgcn_update_dpp(0, v, DPP_ROW_BCAST15, 0xa, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, DPP_ROW_BCAST31, 0xc, 0xf, false);
    return v;
}

// ---------------------------------------------------------------- op semantics (FP32)
// Values of dispatch_eval (main.cu:397-444) with IEEE division and accurate libm.
__device__ __forceinline__ float op_bin(int op, float a, float b) {
    switch (op) {
    case GPR_OP_ADD: return a + b;
    case GPR_OP_SUB: return a - b;
    case GPR_OP_MUL: return a * b;
    case GPR_OP_DIV: return a / b;
    case GPR_OP_POW: return powf(a, b);
    case GPR_OP_RSUB: return b - a;
    case GPR_OP_RDIV: return b / a;
    default: return powf(b, a);  // RPOW
    }
}
__device__ __forceinline__ float op_un(int op, float a, float c) {
    switch (op) {
    case GPR_OP_NEG: return -a;
    case GPR_OP_EXP: return expf(a);
    case GPR_OP_LOG: return logf(a);
    case GPR_OP_INV: return 1.0f / a;
    case GPR_OP_SQRT: return sqrtf(a);
    case GPR_OP_SIN: return sinf(a);
    case GPR_OP_ASIN: return asinf(a);
    case GPR_OP_COS: return cosf(a);
    case GPR_OP_ACOS: return acosf(a);
    case GPR_OP_TAN: return tanf(a);
    case GPR_OP_ATAN: return atanf(a);
    case GPR_OP_ABS: return fabsf(a);
    case GPR_OP_CADD: return a + c;
    case GPR_OP_CMUL: return c * a;
    case GPR_OP_CPOW: return powf(a, c);
    case GPR_OP_CRPOW: return powf(c, a);
    default: return __builtin_nanf("");
    }
}

// The dataset of a chain: the last one that starts at or before it.
__device__ __forceinline__ int chain_dataset(const GprDataset *ds, int nd, int chain) {
    int lo = 0, hi = nd;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (ds[mid].chain0 <= chain) lo = mid;
        else hi = mid;
    }
    return lo;
}

// ---------------------------------------------------------------- wave program state
// Lane l holds token l in (o0, c0) and token l+64 in (o1, c1); tokens >= len are 0.
struct WaveProg {
    int o0, o1;
    float c0, c1;
    int len;
};

#define GPR_KLOOP(expr)                              \
    do {                                             \
        _Pragma("unroll") for (int k = 0; k < KC; k++) T[k] = (expr); \
    } while (0)

// Token classes as wave-uniform bit masks (bit t of the low word, bit t-64 of the high
// word): the common classes dispatch on a scalar bit test, with no vector-to-scalar
// read of the op on their path.
// (x and constant leaves; +, -, *; every other op takes the generic path)
struct OpMasks {
    uint64_t leaf[2], x[2], cheap[2], mul[2], sub[2];
};
template <bool HI>
__device__ __forceinline__ OpMasks op_masks(const WaveProg &p) {
    const int l = lane_id();
    OpMasks m;
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const bool v = (h == 0 || HI) && l + 64 * h < p.len;
        const int o = h ? p.o1 : p.o0;
        m.leaf[h] = ballot(v && o <= GPR_OP_CONST);
        m.x[h] = ballot(v && o == GPR_OP_X);
        m.cheap[h] = ballot(v && o >= GPR_OP_ADD && o <= GPR_OP_MUL);
        m.mul[h] = ballot(v && o == GPR_OP_MUL);
        m.sub[h] = ballot(v && o == GPR_OP_SUB);
    }
    return m;
}

// ---------------------------------------------------------------- wave interpreter
// The tape is interpreted once per chunk of points; the program is wave-uniform, so every
// token is one scalar dispatch for all 64 lanes.  That dispatch is what bounds the sampler
// (the scalar unit, which the four SIMDs of a CU share): tests of token-class masks, as the
// compiler lays them out, took some 22 scalar instructions and 8 branches a token.  Here
// the hot tokens (x, constant, + - * with a leaf or a stack operand, negation) are handlers
// of equal size in one asm block, and a token's word, held in its lane like the token itself
// (prog_code), is the byte offset of its handler: a dispatch is one v_readlane, an add with
// carry and s_setpc, and a handler ends in the dispatch of the next token.  A leaf followed
// by +, - or * is one handler, and so are two leaves with their operator.  Division, exp and
// log, the frequent ones of the remaining operators, are larger handlers at the end of the table.
// The others (and the last lane's token, and exp where a value is not below 88) leave the
// block; the caller runs them and enters again at the next token with a handler.
//
// The value stack's top two entries stay in VGPRs (T, U) and the rest live in this wave's
// LDS slab, [level][k][lane] with GPR_MAX_DEPTH + 2 levels for any program; levels 0 and 1
// take the stores and loads of an empty U, so pushes and pops need no test.  p is this
// lane's LDS address of the level that the next push stores U to.  The tape must be well
// formed with stack depth at most GPR_MAX_DEPTH: the sampler's programs are (init,
// proposals and gpr_write_state check it).
//
// Against the mask tests, whole runs with their set-up and state copies: random walk,
// 131072 chains at n = 250 and cap 64, 150.5 -> 123.0 ms; 48 uneven datasets of 2048 chains,
// 47.1 -> 41.3 ms; MALA, whose gradients have interpreters of their own, 107.8 -> 103.0 ms.
// Two leaves and their operator in one handler, with the branch-free words below: 122.8 ->
// 120.3 ms and 39.6 -> 39.1 ms on those two random walks; division, exp and log inside the
// block, where each left it through some ten branches and thirty scalar instructions:
// 120.5 -> 103.0 ms, 39.3 -> 36.4 ms, MALA 102.9 -> 98.5 ms, and 100003 tapes at n = 250
// evaluated in 185 -> 161 us.
enum {
    GPR_U_EXIT = 0, GPR_U_X, GPR_U_C, GPR_U_XADD, GPR_U_XSUB, GPR_U_XMUL, GPR_U_CADD, GPR_U_CSUB, GPR_U_CMUL, GPR_U_ADD,
    GPR_U_SUB, GPR_U_MUL, GPR_U_NEG, GPR_U_XXADD, GPR_U_XCADD = GPR_U_XXADD + 3, GPR_U_CXADD = GPR_U_XCADD + 3,
    GPR_U_EXP = GPR_U_CXADD + 3
};
// (the last three handlers take two or three places of the table; .org stops the assembler
// at one that has outgrown its place)
template <int KC>
constexpr int GPR_U_DIV = GPR_U_EXP + (KC == 4 ? 3 : 2);
template <int KC>
constexpr int GPR_U_LOG = GPR_U_DIV<KC> + (KC == 4 ? 3 : 2);
static_assert(GPR_U_X == 1 && GPR_U_XADD == 3 && GPR_U_CADD == 6 && GPR_U_ADD == 9 && GPR_U_NEG == 12 && GPR_U_XXADD == 13 &&
                  GPR_U_CXADD == 19 && GPR_U_EXP == 22 && GPR_U_DIV<1> == 24 && GPR_U_LOG<1> == 26 && GPR_U_DIV<2> == 24 &&
                  GPR_U_LOG<2> == 26 && GPR_U_DIV<4> == 25 && GPR_U_LOG<4> == 28,
              "the places written in the tables");
// Handler words of a half tape: lane l holds token l's.  Lanes past the program, and lane
// 63 (whose successor the block could not read), hold the exit; so does every token
// without a handler.  A handler advances by the one, two (a leaf and its operator) or three
// tokens (two leaves, not both constants, and their operator) it stands for, all of them
// before min(n, 63), so the block always reaches an exit.  No branches: per lane they would
// cost more than the arithmetic.
template <int KC>
__device__ __forceinline__ int half_code(int o, int n) {
    const int l = lane_id(), end = min(n, 63);
    const int n1 = shfl_all(o, l + 1), n2 = shfl_all(o, l + 2);
    // the handler of a token by itself, five bits an op: x, constant, (one), + - * /, (four
    // operators), negation; nothing from op 12 on but exp and log
    constexpr uint64_t ALONE = (uint64_t)GPR_U_X | ((uint64_t)GPR_U_C << 5) | ((uint64_t)GPR_U_ADD << 15) |
                               ((uint64_t)GPR_U_SUB << 20) | ((uint64_t)GPR_U_MUL << 25) |
                               ((uint64_t)GPR_U_DIV<KC> << 30) | ((uint64_t)GPR_U_NEG << 55);
    int u = (int)(ALONE >> (5 * min(o, 12))) & 31;
    u = o == GPR_OP_EXP ? GPR_U_EXP : o == GPR_OP_LOG ? GPR_U_LOG<KC> : u;
    const bool leaf = o <= GPR_OP_CONST;
    const bool one = leaf & (l + 1 < end) & ((unsigned)(n1 - GPR_OP_ADD) < 3u);
    const bool two = leaf & (l + 2 < end) & (o + n1 < 2) & ((unsigned)(n2 - GPR_OP_ADD) < 3u);
    u = one ? GPR_U_XADD - GPR_OP_ADD + 3 * o + n1 : u;
    u = two ? GPR_U_XXADD - GPR_OP_ADD + 3 * (2 * o + n1) + n2 : u;
    u = l < end ? u : GPR_U_EXIT;
    return u << (KC == 1 ? 6 : 7);
}
static_assert(GPR_OP_X == 0 && GPR_OP_CONST == 1 && GPR_OP_ONE == 2 && GPR_OP_SUB == GPR_OP_ADD + 1 &&
                  GPR_OP_MUL == GPR_OP_ADD + 2 && GPR_OP_DIV == 6 && GPR_OP_NEG == 11,
              "half_code's arithmetic on op codes");
struct ProgCode {
    int w0, w1;
};
template <int KC, bool HI>
__device__ __forceinline__ ProgCode prog_code(const WaveProg &p) {
    ProgCode c;
    c.w0 = half_code<KC>(p.o0, p.len);
    c.w1 = 0;
    if (HI && p.len > 64) c.w1 = half_code<KC>(p.o1, p.len - 64);
    return c;
}

// LDS by byte address, as the asm blocks use it
typedef __attribute__((address_space(3))) float *gpr_lds_f;
__device__ __forceinline__ uint32_t lds_addr(const float *q) {
    return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const float *)q;
}
__device__ __forceinline__ float lds_ld(uint32_t a) { return *(gpr_lds_f)(uintptr_t)a; }
__device__ __forceinline__ void lds_st(uint32_t a, float v) { *(gpr_lds_f)(uintptr_t)a = v; }

// Pieces of the handlers.  GT_NEXT reads the next token's word early; GT_JUMP adds it to
// the handlers' base.  Wait states (the compiler does not look into the block): a lane read
// into a scalar register and its use by a vector instruction are two instructions apart; a
// vector register written by the vector unit is read by v_readlane only after others
// (nothing in the block writes the word and constant registers, and the entry runs four
// scalar instructions first).  Every LDS load is waited for before its register is used,
// and before the block ends.  v_exp and v_rcp are one instruction away from the use of their
// result, v_div_scale's vcc six from v_div_fmas, and a compare's vcc two from a select.
#define GT_NEXT(N) "s_add_i32 %[t], %[t], " #N "\n\tv_readlane_b32 %[w], %[word], %[t]\n\t"
#define GT_JUMP "s_add_u32 vcc_lo, %[blo], %[w]\n\ts_addc_u32 vcc_hi, %[bhi], 0\n\ts_setpc_b64 vcc\n\t"
#define GT_CONST "v_readlane_b32 %[s], %[c], %[t]\n\t"
// the constant of the token after this one
#define GT_CONST2 "s_add_i32 %[s], %[t], 1\n\tv_readlane_b32 %[s], %[c], %[s]\n\t"
#define GT_WAIT "s_waitcnt lgkmcnt(0)\n\t"
// entry: the base of the handlers, then the dispatch of token t
#define GT_ENTRY                                                                            \
    "s_getpc_b64 vcc\n.Lp%=:\n\t"                                                           \
    "s_add_u32 %[blo], vcc_lo, .Lh%=-.Lp%=\n\t"                                             \
    "s_addc_u32 %[bhi], vcc_hi, 0\n\t"                                                      \
    "v_readlane_b32 %[w], %[word], %[t]\n\t" GT_JUMP
#define GT_EXIT GT_WAIT "s_branch .Lx%=\n\t"

// exp of T: 2^k e^r from the product with log2(e), its rounding error and the constant's
// low part in one correction; for |T| < 88 neither end of the range needs a test, and every
// such value gives the bits of expf (all 2^32 inputs compared).  The steps and constants of
// exp, log and the division are those of the code that the AMD compiler emits for expf, logf
// and a float division on this target: the other paths of a program's value (tape_slow, the
// adjoint, the forward-mode pass, the lane schedule) call those, and the bits must not differ.
#define GT_LOG2E "s_mov_b32 %[s], 0x3fb8aa3b\n\t"
#define GT_EXP(T)                                                                                               \
    "v_mul_f32 %[q0], %[s], " T "\n\tv_rndne_f32 %[q1], %[q0]\n\tv_fma_f32 %[q2], " T ", %[s], -%[q0]\n\t"      \
    "v_sub_f32 %[q0], %[q0], %[q1]\n\tv_fmac_f32 %[q2], 0x32a5705f, " T "\n\tv_add_f32 %[q0], %[q0], %[q2]\n\t" \
    "v_exp_f32 %[q0], %[q0]\n\tv_cvt_i32_f32 %[q1], %[q1]\n\tv_ldexp_f32 " T ", %[q0], %[q1]\n\t"
// leave at this token when the largest magnitude M is not below 88
#define GT_EXP_TEST(M)                                                                                          \
    "s_mov_b32 %[s], 0x42b00000\n\tv_cmp_nlt_f32 vcc, |" M "|, %[s]\n\ts_cbranch_vccnz .Lh%=\n\t"
// log of T: log2 (of T 2^32 below the normal range, less 32 log(2) at the end) times log(2)
// in two parts, where it is finite.  Bits of logf for all 2^32 inputs.
#define GT_LOG(T)                                                                                               \
    "s_mov_b32 %[s], 0x800000\n\tv_cmp_gt_f32 vcc, %[s], " T "\n\ts_mov_b32 %[s], 0x3f317217\n\t"                 \
    "v_mov_b32 %[q2], 0x41b17218\n\tv_cndmask_b32 %[q0], 0, 32, vcc\n\tv_ldexp_f32 %[q0], " T ", %[q0]\n\t"       \
    "v_log_f32 %[q0], %[q0]\n\tv_cndmask_b32 %[q2], 0, %[q2], vcc\n\tv_mul_f32 %[q1], %[s], %[q0]\n\t"          \
    "v_fma_f32 %[q1], %[q0], %[s], -%[q1]\n\ts_mov_b32 %[s], 0x7f800000\n\tv_cmp_lt_f32 vcc, |%[q0]|, %[s]\n\t" \
    "v_fmac_f32 %[q1], 0x3377d1cf, %[q0]\n\tv_fmac_f32 %[q1], 0x3f317217, %[q0]\n\t"                            \
    "v_cndmask_b32 %[q0], %[q0], %[q1], vcc\n\tv_sub_f32 " T ", %[q0], %[q2]\n\t"
// U / T, correctly rounded: scaled operands, a reciprocal with one step, a quotient with two
#define GT_DIV(U, T)                                                                                            \
    "v_div_scale_f32 %[q0], vcc, " T ", " T ", " U "\n\tv_rcp_f32 %[q1], %[q0]\n\t"                             \
    "v_div_scale_f32 %[q2], vcc, " U ", " T ", " U "\n\tv_fma_f32 %[q3], -%[q0], %[q1], 1.0\n\t"                \
    "v_fmac_f32 %[q1], %[q3], %[q1]\n\tv_mul_f32 %[q3], %[q2], %[q1]\n\t"                                       \
    "v_fma_f32 %[q4], -%[q0], %[q3], %[q2]\n\tv_fmac_f32 %[q3], %[q4], %[q1]\n\t"                               \
    "v_fma_f32 %[q0], -%[q0], %[q3], %[q2]\n\tv_div_fmas_f32 %[q0], %[q0], %[q1], %[q3]\n\t"                    \
    "v_div_fixup_f32 " T ", %[q0], " T ", " U "\n\t"
#define GT_TEMPS float q0, q1, q2, q3, q4
#define GT_TEMP_OUT [q0] "=&v"(q0), [q1] "=&v"(q1), [q2] "=&v"(q2), [q3] "=&v"(q3), [q4] "=&v"(q4)

#define GT1(OP, A, B) OP " %[T0], " A ", " B "\n\t"
#define GT1_PUSH GT_WAIT "ds_write_b32 %[p], %[U0]\n\tv_add_u32 %[p], 0x100, %[p]\n\tv_mov_b32 %[U0], %[T0]\n\t"
#define GT1_POP "v_add_u32 %[p], 0xffffff00, %[p]\n\tds_read_b32 %[U0], %[p]\n\t"
// one point per lane, handlers of 64 bytes
__device__ __forceinline__ void tape_run(int word, float c, const float (&x)[1], float (&T)[1], float (&U)[1], uint32_t &p,
                                         int &t) {
    uint32_t blo, bhi, w, s;
    GT_TEMPS;
#define GT_H(N, BODY) ".org .Lh%=+64*" #N "\n\t" BODY
    __asm__ volatile(
        GT_ENTRY
        ".p2align 6\n.Lh%=:\n\t" GT_EXIT
        GT_H(1, GT_NEXT(1) GT1_PUSH "v_mov_b32 %[T0], %[x0]\n\t" GT_JUMP)
        GT_H(2, GT_CONST GT_NEXT(1) GT1_PUSH "v_mov_b32 %[T0], %[s]\n\t" GT_JUMP)
        GT_H(3, GT_NEXT(2) GT1("v_add_f32", "%[x0]", "%[T0]") GT_JUMP)
        GT_H(4, GT_NEXT(2) GT1("v_sub_f32", "%[T0]", "%[x0]") GT_JUMP)
        GT_H(5, GT_NEXT(2) GT1("v_mul_f32", "%[x0]", "%[T0]") GT_JUMP)
        GT_H(6, GT_CONST GT_NEXT(2) GT1("v_add_f32", "%[s]", "%[T0]") GT_JUMP)
        GT_H(7, GT_CONST GT_NEXT(2) GT1("v_subrev_f32", "%[s]", "%[T0]") GT_JUMP)
        GT_H(8, GT_CONST GT_NEXT(2) GT1("v_mul_f32", "%[s]", "%[T0]") GT_JUMP)
        GT_H(9, GT_NEXT(1) GT_WAIT GT1("v_add_f32", "%[U0]", "%[T0]") GT1_POP GT_JUMP)
        GT_H(10, GT_NEXT(1) GT_WAIT GT1("v_sub_f32", "%[U0]", "%[T0]") GT1_POP GT_JUMP)
        GT_H(11, GT_NEXT(1) GT_WAIT GT1("v_mul_f32", "%[U0]", "%[T0]") GT1_POP GT_JUMP)
        GT_H(12, GT_NEXT(1) "v_xor_b32 %[T0], 0x80000000, %[T0]\n\t" GT_JUMP)
        GT_H(13, GT_NEXT(3) GT1_PUSH GT1("v_add_f32", "%[x0]", "%[x0]") GT_JUMP)
        GT_H(14, GT_NEXT(3) GT1_PUSH GT1("v_sub_f32", "%[x0]", "%[x0]") GT_JUMP)
        GT_H(15, GT_NEXT(3) GT1_PUSH GT1("v_mul_f32", "%[x0]", "%[x0]") GT_JUMP)
        GT_H(16, GT_CONST2 GT_NEXT(3) GT1_PUSH GT1("v_add_f32", "%[s]", "%[x0]") GT_JUMP)
        GT_H(17, GT_CONST2 GT_NEXT(3) GT1_PUSH GT1("v_subrev_f32", "%[s]", "%[x0]") GT_JUMP)
        GT_H(18, GT_CONST2 GT_NEXT(3) GT1_PUSH GT1("v_mul_f32", "%[s]", "%[x0]") GT_JUMP)
        GT_H(19, GT_CONST GT_NEXT(3) GT1_PUSH GT1("v_add_f32", "%[s]", "%[x0]") GT_JUMP)
        GT_H(20, GT_CONST GT_NEXT(3) GT1_PUSH GT1("v_sub_f32", "%[s]", "%[x0]") GT_JUMP)
        GT_H(21, GT_CONST GT_NEXT(3) GT1_PUSH GT1("v_mul_f32", "%[s]", "%[x0]") GT_JUMP)
        GT_H(22, GT_EXP_TEST("%[T0]") GT_NEXT(1) GT_LOG2E GT_EXP("%[T0]") GT_JUMP)
        GT_H(24, GT_WAIT GT_NEXT(1) GT_DIV("%[U0]", "%[T0]") GT1_POP GT_JUMP)
        GT_H(26, GT_WAIT GT_NEXT(1) GT_LOG("%[T0]") GT_JUMP)
        ".Lx%=:"
        : [T0] "+&v"(T[0]), [U0] "+&v"(U[0]), [p] "+&v"(p), [t] "+&s"(t), [blo] "=&s"(blo), [bhi] "=&s"(bhi), [w] "=&s"(w),
          [s] "=&s"(s), GT_TEMP_OUT
        : [word] "v"(word), [c] "v"(c), [x0] "v"(x[0])
        : "vcc", "scc", "memory");
#undef GT_H
}

#define GT_H_(N, BODY) ".org .Lh%=+128*" #N "\n\t" BODY
#define GT_H(N, BODY) GT_H_(N, BODY)
#define GT2(OP, A, B) OP " %[T0], " A(0) ", " B(0) "\n\t" OP " %[T1], " A(1) ", " B(1) "\n\t"
#define GT4(OP, A, B) GT2(OP, A, B) OP " %[T2], " A(2) ", " B(2) "\n\t" OP " %[T3], " A(3) ", " B(3) "\n\t"
#define GT_T(k) "%[T" #k "]"
#define GT_U(k) "%[U" #k "]"
#define GT_X(k) "%[x" #k "]"
#define GT_S(k) "%[s]"
#define GT_NEGMASK(k) "0x80000000"
#define GT2_MOV(D, S) "v_mov_b32 " D(0) ", " S(0) "\n\tv_mov_b32 " D(1) ", " S(1) "\n\t"
#define GT4_MOV(D, S) GT2_MOV(D, S) "v_mov_b32 " D(2) ", " S(2) "\n\tv_mov_b32 " D(3) ", " S(3) "\n\t"
#define GT2_PUSH GT_WAIT "ds_write2_b32 %[p], %[U0], %[U1] offset1:64\n\tv_add_u32 %[p], 0x200, %[p]\n\t" GT2_MOV(GT_U, GT_T)
#define GT2_POP "v_add_u32 %[p], 0xfffffe00, %[p]\n\tds_read_b32 %[U0], %[p]\n\tds_read_b32 %[U1], %[p] offset:256\n\t"
#define GT4_PUSH                                                                                             \
    GT_WAIT "ds_write2_b32 %[p], %[U0], %[U1] offset1:64\n\tds_write2_b32 %[p], %[U2], %[U3] offset0:128 offset1:192\n\t" \
            "v_add_u32 %[p], 0x400, %[p]\n\t" GT4_MOV(GT_U, GT_T)
#define GT4_POP                                                                                              \
    "v_add_u32 %[p], 0xfffffc00, %[p]\n\tds_read_b32 %[U0], %[p]\n\tds_read_b32 %[U1], %[p] offset:256\n\t"     \
    "ds_read_b32 %[U2], %[p] offset:512\n\tds_read_b32 %[U3], %[p] offset:768\n\t"
#define GT2_EXP                                                                                              \
    "v_max_f32 %[q0], |%[T0]|, |%[T1]|\n\t" GT_EXP_TEST("%[q0]") GT_NEXT(1) GT_LOG2E GT_EXP("%[T0]") GT_EXP("%[T1]")
#define GT4_EXP                                                                                              \
    "v_max_f32 %[q0], |%[T0]|, |%[T1]|\n\tv_max3_f32 %[q0], %[q0], |%[T2]|, |%[T3]|\n\t" GT_EXP_TEST("%[q0]")  \
        GT_NEXT(1) GT_LOG2E GT_EXP("%[T0]") GT_EXP("%[T1]") GT_EXP("%[T2]") GT_EXP("%[T3]")
#define GT2_DIV GT_DIV("%[U0]", "%[T0]") GT_DIV("%[U1]", "%[T1]")
#define GT4_DIV GT2_DIV GT_DIV("%[U2]", "%[T2]") GT_DIV("%[U3]", "%[T3]")
#define GT2_LOG GT_LOG("%[T0]") GT_LOG("%[T1]")
#define GT4_LOG GT2_LOG GT_LOG("%[T2]") GT_LOG("%[T3]")
// several points per lane, handlers of 128 bytes
#define GT_TABLE(GT, MOV, PUSH, POP, EXP, DIV, LOG, DIVP, LOGP)                                             \
    GT_ENTRY                                                                     \
    ".p2align 7\n.Lh%=:\n\t" GT_EXIT                                             \
    GT_H(1, GT_NEXT(1) PUSH MOV(GT_T, GT_X) GT_JUMP)                                \
    GT_H(2, GT_CONST GT_NEXT(1) PUSH MOV(GT_T, GT_S) GT_JUMP)                       \
    GT_H(3, GT_NEXT(2) GT("v_add_f32", GT_X, GT_T) GT_JUMP)                         \
    GT_H(4, GT_NEXT(2) GT("v_sub_f32", GT_T, GT_X) GT_JUMP)                         \
    GT_H(5, GT_NEXT(2) GT("v_mul_f32", GT_X, GT_T) GT_JUMP)                         \
    GT_H(6, GT_CONST GT_NEXT(2) GT("v_add_f32", GT_S, GT_T) GT_JUMP)                \
    GT_H(7, GT_CONST GT_NEXT(2) GT("v_subrev_f32", GT_S, GT_T) GT_JUMP)             \
    GT_H(8, GT_CONST GT_NEXT(2) GT("v_mul_f32", GT_S, GT_T) GT_JUMP)                \
    GT_H(9, GT_NEXT(1) GT_WAIT GT("v_add_f32", GT_U, GT_T) POP GT_JUMP)             \
    GT_H(10, GT_NEXT(1) GT_WAIT GT("v_sub_f32", GT_U, GT_T) POP GT_JUMP)             \
    GT_H(11, GT_NEXT(1) GT_WAIT GT("v_mul_f32", GT_U, GT_T) POP GT_JUMP)             \
    GT_H(12, GT_NEXT(1) GT("v_xor_b32", GT_NEGMASK, GT_T) GT_JUMP)                   \
    GT_H(13, GT_NEXT(3) PUSH GT("v_add_f32", GT_X, GT_X) GT_JUMP)                    \
    GT_H(14, GT_NEXT(3) PUSH GT("v_sub_f32", GT_X, GT_X) GT_JUMP)                    \
    GT_H(15, GT_NEXT(3) PUSH GT("v_mul_f32", GT_X, GT_X) GT_JUMP)                    \
    GT_H(16, GT_CONST2 GT_NEXT(3) PUSH GT("v_add_f32", GT_S, GT_X) GT_JUMP)          \
    GT_H(17, GT_CONST2 GT_NEXT(3) PUSH GT("v_subrev_f32", GT_S, GT_X) GT_JUMP)       \
    GT_H(18, GT_CONST2 GT_NEXT(3) PUSH GT("v_mul_f32", GT_S, GT_X) GT_JUMP)          \
    GT_H(19, GT_CONST GT_NEXT(3) PUSH GT("v_add_f32", GT_S, GT_X) GT_JUMP)           \
    GT_H(20, GT_CONST GT_NEXT(3) PUSH GT("v_sub_f32", GT_S, GT_X) GT_JUMP)           \
    GT_H(21, GT_CONST GT_NEXT(3) PUSH GT("v_mul_f32", GT_S, GT_X) GT_JUMP)           \
    GT_H(22, EXP GT_JUMP)                                                            \
    GT_H(DIVP, GT_WAIT GT_NEXT(1) DIV POP GT_JUMP)                                     \
    GT_H(LOGP, GT_NEXT(1) LOG GT_JUMP)                                                 \
    ".Lx%=:"
__device__ __forceinline__ void tape_run(int word, float c, const float (&x)[2], float (&T)[2], float (&U)[2], uint32_t &p,
                                         int &t) {
    uint32_t blo, bhi, w, s;
    GT_TEMPS;
    __asm__ volatile(GT_TABLE(GT2, GT2_MOV, GT2_PUSH, GT2_POP, GT2_EXP, GT2_DIV, GT2_LOG, 24, 26)
                     : [T0] "+&v"(T[0]), [T1] "+&v"(T[1]), [U0] "+&v"(U[0]), [U1] "+&v"(U[1]), [p] "+&v"(p), [t] "+&s"(t),
                       [blo] "=&s"(blo), [bhi] "=&s"(bhi), [w] "=&s"(w), [s] "=&s"(s), GT_TEMP_OUT
                     : [word] "v"(word), [c] "v"(c), [x0] "v"(x[0]), [x1] "v"(x[1])
                     : "vcc", "scc", "memory");
}
__device__ __forceinline__ void tape_run(int word, float c, const float (&x)[4], float (&T)[4], float (&U)[4], uint32_t &p,
                                         int &t) {
    uint32_t blo, bhi, w, s;
    GT_TEMPS;
    __asm__ volatile(GT_TABLE(GT4, GT4_MOV, GT4_PUSH, GT4_POP, GT4_EXP, GT4_DIV, GT4_LOG, 25, 28)
                     : [T0] "+&v"(T[0]), [T1] "+&v"(T[1]), [T2] "+&v"(T[2]), [T3] "+&v"(T[3]), [U0] "+&v"(U[0]),
                       [U1] "+&v"(U[1]), [U2] "+&v"(U[2]), [U3] "+&v"(U[3]), [p] "+&v"(p), [t] "+&s"(t), [blo] "=&s"(blo),
                       [bhi] "=&s"(bhi), [w] "=&s"(w), [s] "=&s"(s), GT_TEMP_OUT
                     : [word] "v"(word), [c] "v"(c), [x0] "v"(x[0]), [x1] "v"(x[1]), [x2] "v"(x[2]), [x3] "v"(x[3])
                     : "vcc", "scc", "memory");
}
#undef GT_H

// One token outside the block (any op: the last lane's token may be a cheap one).
template <int KC>
__device__ __forceinline__ void tape_slow(int op, float c, const float (&xs)[KC], float (&T)[KC], float (&U)[KC],
                                          uint32_t &p) {
    if (op <= GPR_OP_ONE) {
#pragma unroll
        for (int k = 0; k < KC; k++) { lds_st(p + 256 * k, U[k]); U[k] = T[k]; }
        p += 256 * KC;
        const float sv = op == GPR_OP_CONST ? c : 1.0f;
        const bool isx = op == GPR_OP_X;
        GPR_KLOOP(isx ? xs[k] : sv);
    } else if (op <= GPR_OP_RPOW) {
        if (op <= GPR_OP_MUL) {
            const bool mul = op == GPR_OP_MUL;
            const float sgn = op == GPR_OP_SUB ? -1.0f : 1.0f;
#pragma unroll
            for (int k = 0; k < KC; k++) {
                const float pm = __builtin_fmaf(sgn, T[k], U[k]);
                const float pr = U[k] * T[k];
                T[k] = mul ? pr : pm;
            }
        } else {
            switch (op) {
            case GPR_OP_DIV: GPR_KLOOP(U[k] / T[k]); break;
            case GPR_OP_RSUB: GPR_KLOOP(T[k] - U[k]); break;
            case GPR_OP_RDIV: GPR_KLOOP(T[k] / U[k]); break;
            case GPR_OP_POW: GPR_KLOOP(powf(U[k], T[k])); break;
            default: GPR_KLOOP(powf(T[k], U[k])); break;
            }
        }
        p -= 256 * KC;
#pragma unroll
        for (int k = 0; k < KC; k++) U[k] = lds_ld(p + 256 * k);   // the new second entry
    } else {
        switch (op) {
        case GPR_OP_NEG: GPR_KLOOP(-T[k]); break;
        case GPR_OP_EXP: GPR_KLOOP(expf(T[k])); break;
        case GPR_OP_LOG: GPR_KLOOP(logf(T[k])); break;
        case GPR_OP_INV: GPR_KLOOP(1.0f / T[k]); break;
        case GPR_OP_SQRT: GPR_KLOOP(sqrtf(T[k])); break;
        case GPR_OP_SIN: GPR_KLOOP(sinf(T[k])); break;
        case GPR_OP_ASIN: GPR_KLOOP(asinf(T[k])); break;
        case GPR_OP_COS: GPR_KLOOP(cosf(T[k])); break;
        case GPR_OP_ACOS: GPR_KLOOP(acosf(T[k])); break;
        case GPR_OP_TAN: GPR_KLOOP(tanf(T[k])); break;
        case GPR_OP_ATAN: GPR_KLOOP(atanf(T[k])); break;
        case GPR_OP_ABS: GPR_KLOOP(fabsf(T[k])); break;
        case GPR_OP_CADD: GPR_KLOOP(T[k] + c); break;
        case GPR_OP_CMUL: GPR_KLOOP(c * T[k]); break;
        case GPR_OP_CPOW: GPR_KLOOP(powf(T[k], c)); break;
        case GPR_OP_CRPOW: GPR_KLOOP(powf(c, T[k])); break;
        default: GPR_KLOOP(__builtin_nanf("")); break;
        }
    }
}

// Values of the tape at KC points per lane.  ls: this wave's slab, levels of 64 * KC floats.
template <int KC, bool HI>
__device__ __forceinline__ void wave_eval_ls(const WaveProg &p, const float (&xs)[KC], float (&T)[KC], float *ls,
                                             const ProgCode &m) {
    float U[KC];
    uint32_t a = lds_addr(ls) + 4u * (uint32_t)lane_id();   // level -2 of the stack below T, U
#pragma unroll
    for (int k = 0; k < KC; k++) { T[k] = 0.0f; U[k] = 0.0f; }
    // one copy of the block and of the slow path for both halves of the tape
#pragma unroll 1
    for (int h = 0; h == 0 || (HI && 64 * h < p.len); h++) {
        // (uni: wave-uniform in any case, but the block needs it in a scalar register)
        const int n = uni(min(p.len - 64 * h, 64)), word = HI && h ? m.w1 : m.w0, o = HI && h ? p.o1 : p.o0;
        const float c = HI && h ? p.c1 : p.c0;
        for (int t = 0; t < n;) {
            t = uni(t);
            tape_run(word, c, xs, T, U, a, t);
            t = uni(t);
            // tokens without a handler, until one that has one
            while (t < n) {
                tape_slow<KC>(rl_i(o, t), rl_f(c, t), xs, T, U, a);
                t++;
                if (rl_i(word, t & 63) != GPR_U_EXIT) break;
            }
        }
    }
}

// Dataset points of one chunk: point index base + k*64 + lane, the last point again past the
// data (the sums take no term of these lanes).  A clamped 32-bit offset for the three loads costs
// a quarter of a mask and three 64-bit addresses; with the sums' DPP adds, 99.5 -> 96.6 ms
// on 131072 chains at n = 250, MALA 97.2 -> 94.7 ms.  base < n is wave-uniform: it goes to
// the scalar addresses.
template <int KC>
struct Chunk {
    float x[KC], y[KC], w[KC];
    __device__ __forceinline__ void load(const float *dx, const float *dy, const float *dw, int n, int base) {
        const int l = opaque_lane_i32(lane_id());   // the point's offset is computed here, not kept live
        const float *px = dx + base, *py = dy + base, *pw = dw + base;
#pragma unroll
        for (int k = 0; k < KC; k++) {
            const uint32_t o = gpr_point_offset(k * 64 + l, n - 1 - base);
            x[k] = *(const float *)((const char *)px + o);
            y[k] = *(const float *)((const char *)py + o);
            w[k] = *(const float *)((const char *)pw + o);
        }
    }
};

// Work-counter values of a program: operator tokens + 4 (the per-point FP32 ops of its
// evaluation and Gaussian term) and its constant-carrying tokens.
template <bool HI>
__device__ __forceinline__ void prog_counts(const WaveProg &p, int &opq, int &nc) {
    const int l = lane_id();
    const int nleaf = __popcll(ballot(l < p.len && p.o0 <= GPR_OP_ONE)) +
                      (HI ? __popcll(ballot(l + 64 < p.len && p.o1 <= GPR_OP_ONE)) : 0);
    nc = __popcll(ballot(l < p.len && gpr_has_const(p.o0))) +
         (HI ? __popcll(ballot(l + 64 < p.len && gpr_has_const(p.o1))) : 0);
    opq = p.len - nleaf + 4;
}

// Constant tokens of a program.
template <bool HI>
__device__ __forceinline__ int const_count(const WaveProg &p) {
    const int l = lane_id();
    return __popcll(ballot(l < p.len && p.o0 == GPR_OP_CONST)) +
           (HI ? __popcll(ballot(l + 64 < p.len && p.o1 == GPR_OP_CONST)) : 0);
}

// Random-walk moves of a program can be batched (four steps per Philox block) when
// BATCH holds, the chain has no proposal metric (mk = 0), the tape fits the low half (at
// most 64 tokens), it has at most 16 constant tokens and no constant-operand token.
template <bool BATCH, bool HI>
__device__ __forceinline__ bool batch_ok(const WaveProg &p, int mk) {
    if (!BATCH || mk != 0 || (HI && p.len > 64)) return false;
    const int l = lane_id();
    const uint64_t m = ballot(l < p.len && p.o0 == GPR_OP_CONST);
    return __popcll(m) <= 16 && ballot(l < p.len && gpr_has_const(p.o0)) == m;
}

// Gaussian log-likelihood of the wave's program: lconst - sum_i (f_i - y_i)^2 w_i.
// Per-lane Kahan sums, wave tree reduction; -inf if any term is not finite.
// ls: this wave's value-stack slab, pc: the program's handler words for KC points per lane.
// reject_below: the caller rejects the proposal whenever the LL lies below this value.
// Every term of the sum is >= 0, so after each chunk but the last the sum so far bounds
// the LL from above; when that bound (with a relative margin of 1e-4 on the partial sum,
// far above its FP32 rounding) is below reject_below, or the partial sum is not finite,
// the evaluation stops and returns -inf: the proposal is rejected either way.  *points
// receives the number of data points evaluated.
template <int KC, bool HI>
__device__ __forceinline__ double wave_loglik(const WaveProg &p, const GprDataset &d, const float *dx, const float *dy,
                              const float *dw, const Chunk<KC> &c0, int nchunks, float *ls, const ProgCode &pc,
                              double reject_below = -GPR_INF, int *points = nullptr) {
    float acc = 0.0f, comp = 0.0f;
    const int l = lane_id();
    const double wc = d.wconst > 0.0 ? d.wconst : 1.0;
    if (points) *points = d.n;
    for (int ch = 0; ch < nchunks; ch++) {
        Chunk<KC> c;
        if (ch == 0) c = c0; else c.load(dx, dy, dw, d.n, ch * 64 * KC);
        float T[KC];
        wave_eval_ls<KC, HI>(p, c.x, T, ls, pc);
#pragma unroll
        for (int k = 0; k < KC; k++) {
            const float r = T[k] - c.y[k];
            const float term = (ch * 64 * KC + k * 64 + l < d.n) ? (r * r) * c.w[k] : 0.0f;
            const float yv = term - comp;
            const float tv = acc + yv;
            comp = (tv - acc) - yv;
            acc = tv;
        }
        if (ch + 1 < nchunks && reject_below > -GPR_INF) {
            const double lb = (double)wave_sum_f(acc - comp) * (1.0 - 1e-4);
            const double ub = d.lconst - wc * lb;
            if (!(ub >= reject_below)) {
                if (points) *points = (ch + 1) * 64 * KC;
                return -GPR_INF;
            }
        }
    }
    // each lane's compensated partial, combined across the wave in FP64
    const double s = wave_sum_d((double)acc - (double)comp);
    if (!__builtin_isfinite(s)) return -GPR_INF;
    return d.lconst - (d.wconst > 0.0 ? d.wconst * s : s);
}

// ---------------------------------------------------------------- forward-mode gradient
// The MALA proposals of short programs with few constants get their gradient in the same
// interpreter pass as their likelihood: every stack entry carries the value and its
// tangents with respect to the program's constant tokens (constant of rank j: tangent j),
// W = 1 + NT floats, pushed to the wave's LDS stack as one 16-byte store (NT =
// GPR_DUAL_NT = 3, and NT = 2 in the same layout), one 8-byte store (NT = 1, programs of a
// single constant), for programs of four constants (NT = GPR_DUAL_NT4) a 16-byte store of
// the value and the first three tangents and a 4-byte store of the fourth into a second
// plane, and for five or six (NT = GPR_DUAL_NT6) a 16-byte, an 8-byte and a 4-byte store
// into three planes.  Programs of up to GPR_DUAL_NTMAX constants that fit none of these take
// two passes of four tangents each (constants of rank 0-3, then 4-7: the second pass only
// when the first completes).  The values take the same
// operations on the same operands as wave_eval_ls, so the LL is
// bit-identical to it (and early rejection stops a pass at the same chunk); each lane
// adds the per-point gradient (-2 r w) f' of its points, and one wave sum per constant
// ends the pass.  Programs qualify when they use only the config grammar (x, constant,
// one, + - * / pow exp log neg), hold no constant-operand token, and hold at most
// GPR_DUAL_NT constant tokens within stack depth GPR_DUAL_DEPTH or at most GPR_DUAL_NTMAX
// within GPR_DUAL_DEPTH4 (dual_nt: one pass of GPR_DUAL_NT4 tangents for four constants,
// of GPR_DUAL_NT6 for five or six within GPR_DUAL_DEPTH6, else two passes).
#define GPR_DUAL_NT 3
#define GPR_DUAL_NT4 4
#define GPR_DUAL_NT6 6
#define GPR_DUAL_NTMAX 8
#define GPR_DUAL_DEPTH 9
#define GPR_DUAL_DEPTH4 8
#define GPR_DUAL_DEPTH6 6
#define GPR_DUAL_W (1 + GPR_DUAL_NT)
// Stack levels: a push at stack size sp stores U at level sp - 2 and a binary op at sp
// loads level sp - 3, so a program of depth at most D uses levels -1 .. D - 3 (D - 1 of
// them), stored from offset 0 (level -1): token 0, always a leaf, starts the stack in T
// without the store of level -2 (U holds no entry yet).  Levels -1 and below hold no
// stack entry (the store at sp = 1 and the load at sp = 2 move the empty U).
#define GPR_DUAL_PACKED_FLOATS ((GPR_DUAL_DEPTH - 1) * 64 * GPR_DUAL_W)
#define GPR_DUAL_SPLIT_FLOATS ((GPR_DUAL_DEPTH4 - 1) * 64 * (GPR_DUAL_NT4 + 1))
#define GPR_DUAL_SPLIT6_FLOATS ((GPR_DUAL_DEPTH6 - 1) * 64 * (GPR_DUAL_NT6 + 1))
// floats of the dual stack of one wave
#define GPR_DUAL_LDS_FLOATS \
    (GPR_DUAL_PACKED_FLOATS > GPR_DUAL_SPLIT_FLOATS                                      \
         ? (GPR_DUAL_PACKED_FLOATS > GPR_DUAL_SPLIT6_FLOATS ? GPR_DUAL_PACKED_FLOATS : GPR_DUAL_SPLIT6_FLOATS) \
         : (GPR_DUAL_SPLIT_FLOATS > GPR_DUAL_SPLIT6_FLOATS ? GPR_DUAL_SPLIT_FLOATS : GPR_DUAL_SPLIT6_FLOATS))

template <int N>
__device__ __forceinline__ void ls_store(float *q, const float (&v)[N]) {
    if constexpr (N == 4) *(float4 *)q = make_float4(v[0], v[1], v[2], v[3]);
    else *(float2 *)q = make_float2(v[0], v[1]);
}
template <int N>
__device__ __forceinline__ void ls_load(const float *q, float (&v)[N]) {
    if constexpr (N == 4) { const float4 f = *(const float4 *)q; v[0] = f.x; v[1] = f.y; v[2] = f.z; v[3] = f.w; }
    else { const float2 f = *(const float2 *)q; v[0] = f.x; v[1] = f.y; }
}

// One stack entry of the dual stack at level lv >= -2 (lane, laneb, lanec: this lane's
// level 0 in each plane): packed W floats per lane; for NT = 4 four floats per lane in the
// first plane and the last tangent in laneb's; for NT = 6 also two in lanec's.
template <int NT>
__device__ __forceinline__ void dual_st(float *lane, float *laneb, float *lanec, int lv, const float (&v)[1 + NT]) {
    if constexpr (NT == GPR_DUAL_NT6) {
        *(float4 *)(lane + lv * 256) = make_float4(v[0], v[1], v[2], v[3]);
        *(float2 *)(lanec + lv * 128) = make_float2(v[4], v[5]);
        laneb[lv * 64] = v[NT];
    } else if constexpr (NT == GPR_DUAL_NT4) {
        *(float4 *)(lane + lv * 256) = make_float4(v[0], v[1], v[2], v[3]);
        laneb[lv * 64] = v[NT];
    } else if constexpr (NT == 2) {
        *(float4 *)(lane + lv * 256) = make_float4(v[0], v[1], v[NT], 0.0f);   // the NT = 3 layout
    } else {
        ls_store<1 + NT>(lane + lv * 64 * (1 + NT), v);
    }
}
template <int NT>
__device__ __forceinline__ void dual_ld(const float *lane, const float *laneb, const float *lanec, int lv,
                                        float (&v)[1 + NT]) {
    if constexpr (NT == GPR_DUAL_NT6) {
        const float4 f = *(const float4 *)(lane + lv * 256);
        const float2 e = *(const float2 *)(lanec + lv * 128);
        v[0] = f.x; v[1] = f.y; v[2] = f.z; v[3] = f.w;
        v[4] = e.x; v[5] = e.y;
        v[NT] = laneb[lv * 64];
    } else if constexpr (NT == GPR_DUAL_NT4) {
        const float4 f = *(const float4 *)(lane + lv * 256);
        v[0] = f.x; v[1] = f.y; v[2] = f.z; v[3] = f.w;
        v[NT] = laneb[lv * 64];
    } else if constexpr (NT == 2) {
        const float4 f = *(const float4 *)(lane + lv * 256);
        v[0] = f.x; v[1] = f.y; v[NT] = f.z;
    } else {
        ls_load<1 + NT>(lane + lv * 64 * (1 + NT), v);
    }
}

// a^(b-1), the partial derivative of a^b in a over b, given v = a^b: v / a where a is
// finite and non-zero and v finite on every lane of the wave (a division instead of a
// second pow), else the pow itself.
__device__ __forceinline__ float pow_bm1(float a, float b, float v) {
    if (ballot(a == 0.0f || !__builtin_isfinite(a) || !__builtin_isfinite(v))) return powf(a, b - 1.0f);
    return v / a;
}

// A zero tangent contributes nothing, whatever the partial derivative (an infinite or NaN
// partial of a constant-free operand must not reach the constants, as in the adjoint):
// the vector unit's legacy multiply, whose product is +0 when either factor is 0 and the
// IEEE product otherwise, one instruction for the test, the product and the select.
__device__ __forceinline__ float tmul(float t, float partial) {
    float r;
    __asm__("v_mul_legacy_f32 %0, %1, %2" : "=v"(r) : "v"(t), "v"(partial));
    return r;
}

// tangents of the forward-mode pass of a program of k constant tokens and stack depth dmax
// (GPR_DUAL_NTMAX: two passes of GPR_DUAL_NT4)
__device__ __forceinline__ int dual_nt(int k, int dmax) {
    return k <= 2 ? (k <= 1 ? 1 : 2)
                  : (k <= GPR_DUAL_NT ? GPR_DUAL_NT
                                      : (k <= GPR_DUAL_NT4 ? GPR_DUAL_NT4
                                                           : (k <= GPR_DUAL_NT6 && dmax <= GPR_DUAL_DEPTH6 ? GPR_DUAL_NT6
                                                                                                            : GPR_DUAL_NTMAX)));
}

template <bool HI>
__device__ __forceinline__ bool dual_ok(const WaveProg &p, int dmax) {
    constexpr uint32_t GRAMMAR = (1u << GPR_OP_X) | (1u << GPR_OP_CONST) | (1u << GPR_OP_ONE) | (1u << GPR_OP_ADD) |
                                 (1u << GPR_OP_SUB) | (1u << GPR_OP_MUL) | (1u << GPR_OP_DIV) | (1u << GPR_OP_POW) |
                                 (1u << GPR_OP_EXP) | (1u << GPR_OP_LOG) | (1u << GPR_OP_NEG);
    const int l = lane_id();
    const bool v0 = l < p.len, v1 = HI && l + 64 < p.len;
    const bool bad = (v0 && !((GRAMMAR >> (p.o0 & 31)) & 1u)) || (v1 && !((GRAMMAR >> (p.o1 & 31)) & 1u));
    const int k = const_count<HI>(p);
    return ballot(bad) == 0 && ((k <= GPR_DUAL_NT && dmax <= GPR_DUAL_DEPTH) || (k <= GPR_DUAL_NTMAX && dmax <= GPR_DUAL_DEPTH4));
}

// One token (two for a leaf fused with the next +, - or *) of the forward-mode
// interpreter, tokens of half H of the tape (t < 64 for H = 0): the half is a
// compile-time constant, so the token-class masks and the tape words are read without
// per-token selects.  NT tangents (1, 2, GPR_DUAL_NT, GPR_DUAL_NT4 or GPR_DUAL_NT6) for the
// constants of rank j0 .. j0 + NT - 1.  lane, laneb: this lane's level 0 of the stack (dual_st).
template <int H, int NT>
__device__ __forceinline__ void dual_token(const WaveProg &p, const OpMasks &m, const uint64_t (&cm)[2], int nlo,
                                           int j0, float xv, float *lane, float *laneb, float *lanec, float (&T)[1 + NT],
                                           float (&U)[1 + NT], int &sp, int &t) {
    constexpr int W = 1 + NT;
    const int li = t & 63;
    constexpr int h = H;
    const uint64_t bit = 1ull << li;
    if (m.leaf[h] & bit) {
        // the leaf's value and tangent: x (0), or constant of rank j0 + rk (e_rk)
        const bool isx = (m.x[h] & bit) != 0;
        const float cv = h ? rl_f(p.c1, li) : rl_f(p.c0, li);
        const int rk = isx ? -1 : (h ? nlo : 0) + __popcll(cm[h] & (bit - 1)) - j0;
        const float b = isx ? xv : cv;
        if (m.cheap[h] & (bit << 1)) {
            // leaf followed by +, - or *: T = T op leaf, stack untouched
            const uint64_t nb = bit << 1;
            if (m.mul[h] & nb) {
                const float tv = T[0];
                T[0] = T[0] * b;
#pragma unroll
                for (int j = 1; j < W; j++) T[j] = tmul(T[j], b);
                if (!isx) {
#pragma unroll
                    for (int j = 1; j < W; j++)
                        if (rk == j - 1) T[j] = T[j] + tv;
                }
            } else {
                const float sgn = (m.sub[h] & nb) ? -1.0f : 1.0f;
                T[0] = __builtin_fmaf(sgn, b, T[0]);
                if (!isx) {
#pragma unroll
                    for (int j = 1; j < W; j++)
                        if (rk == j - 1) T[j] = T[j] + sgn;
                }
            }
            t++;
            return;
        }
        dual_st<NT>(lane, laneb, lanec, sp - 2, U);
#pragma unroll
        for (int j = 0; j < W; j++) U[j] = T[j];
        sp++;
        T[0] = b;
#pragma unroll
        for (int j = 1; j < W; j++) T[j] = rk == j - 1 ? 1.0f : 0.0f;
        return;
    }
    if (m.cheap[h] & bit) {
        // U op T for +, -, *
        if (m.mul[h] & bit) {
            const float uv = U[0], tv = T[0];
            T[0] = U[0] * T[0];
#pragma unroll
            for (int j = 1; j < W; j++) T[j] = tmul(U[j], tv) + tmul(T[j], uv);
        } else {
            const float sgn = (m.sub[h] & bit) ? -1.0f : 1.0f;
            T[0] = __builtin_fmaf(sgn, T[0], U[0]);
#pragma unroll
            for (int j = 1; j < W; j++) T[j] = __builtin_fmaf(sgn, T[j], U[j]);
        }
        dual_ld<NT>(lane, laneb, lanec, sp - 3, U);
        sp--;
        return;
    }
    const int op = h ? rl_i(p.o1, li) : rl_i(p.o0, li);
    if (op == GPR_OP_ONE) {
        dual_st<NT>(lane, laneb, lanec, sp - 2, U);
#pragma unroll
        for (int j = 0; j < W; j++) { U[j] = T[j]; T[j] = j == 0 ? 1.0f : 0.0f; }
        sp++;
    } else if (op == GPR_OP_DIV) {
        const float a = U[0], b = T[0];
        const float q = a / b;
        const float ib = 1.0f / b, nq = -(a / (b * b));
#pragma unroll
        for (int j = 1; j < W; j++) T[j] = tmul(U[j], ib) + tmul(T[j], nq);
        T[0] = q;
        dual_ld<NT>(lane, laneb, lanec, sp - 3, U);
        sp--;
    } else if (op == GPR_OP_POW) {
        const float a = U[0], b = T[0];
        const float v = powf(a, b);
        const float pa = b * pow_bm1(a, b, v), pb = v * logf(a);
#pragma unroll
        for (int j = 1; j < W; j++) T[j] = tmul(U[j], pa) + tmul(T[j], pb);
        T[0] = v;
        dual_ld<NT>(lane, laneb, lanec, sp - 3, U);
        sp--;
    } else if (op == GPR_OP_EXP) {
        const float v = expf(T[0]);
#pragma unroll
        for (int j = 1; j < W; j++) T[j] = tmul(T[j], v);
        T[0] = v;
    } else if (op == GPR_OP_LOG) {
        const float a = T[0];
        const float ia = 1.0f / a;
        T[0] = logf(a);
#pragma unroll
        for (int j = 1; j < W; j++) T[j] = tmul(T[j], ia);
    } else {   // GPR_OP_NEG (dual_ok admits no other op)
#pragma unroll
        for (int j = 0; j < W; j++) T[j] = -T[j];
    }
}

// LL of the wave's program (as wave_loglik<1, HI, true>) and, when the pass completes,
// gs[j] = sum over points of (-2 r w) df/dc_{j0+j} for the constant token of rank j0 + j
// (token order; cm = the constant-token masks).  ls: the wave's dual stack region.
// NT: tangents carried (1, 2, GPR_DUAL_NT, GPR_DUAL_NT4 or GPR_DUAL_NT6), at least the
// program's constant count less j0 unless a second pass follows; gs[j] is 0 for j >= NT
// and for ranks past the program's constants.
template <bool HI, int NT>
__device__ __forceinline__ double wave_loglik_dual(const WaveProg &p, const GprDataset &d, const float *dx, const float *dy,
                                   const float *dw, const Chunk<1> &c0, int nchunks, float *ls, const OpMasks &m,
                                   const uint64_t (&cm)[2], double reject_below, int *points, int j0,
                                   float (&gs)[GPR_DUAL_NTMAX]) {
    static_assert(NT == 1 || NT == 2 || NT == GPR_DUAL_NT || NT == GPR_DUAL_NT4 || NT == GPR_DUAL_NT6, "tangent count");
    constexpr int W = 1 + NT;
    const int l = lane_id();
    // this lane's level 0 of the stack below T, U (dual_st); level -1 lies below it
    // NT = 4: planes of 4 and 1 floats, GPR_DUAL_DEPTH4 - 1 levels each; NT = 6: planes of
    // 4, 2 and 1 floats, GPR_DUAL_DEPTH6 - 1 levels each
    constexpr int LV = NT == GPR_DUAL_NT6 ? GPR_DUAL_DEPTH6 - 1 : GPR_DUAL_DEPTH4 - 1;
    float *lane = (NT >= GPR_DUAL_NT4 || NT == 2) ? ls + 256 + l * 4 : ls + 64 * W + l * W;
    float *lanec = ls + LV * 256 + 128 + l * 2;
    float *laneb = ls + LV * (NT == GPR_DUAL_NT6 ? 384 : 256) + 64 + l;
    float acc = 0.0f, comp = 0.0f;
    float ga[NT];
#pragma unroll
    for (int j = 0; j < NT; j++) ga[j] = 0.0f;
    const bool folded = d.wconst > 0.0;
    const float wf = (float)d.wconst;
    const double wc = folded ? d.wconst : 1.0;
    const int nlo = __popcll(cm[0]);
    if (points) *points = d.n;
    for (int ch = 0; ch < nchunks; ch++) {
        Chunk<1> c;
        if (ch == 0) c = c0; else c.load(dx, dy, dw, d.n, ch * 64);
        const int i = ch * 64 + l;
        const bool valid = i < d.n;
        // (0 past the data: pow_bm1 looks at every lane)
        const float xv = valid ? c.x[0] : 0.0f;
        float T[W], U[W];
        // token 0 (x, a constant of rank 0 or one) starts the stack in T
        const bool t0x = (m.x[0] & 1ull) != 0, t0c = (cm[0] & 1ull) != 0;
        T[0] = t0x ? xv : (t0c ? rl_f(p.c0, 0) : 1.0f);
#pragma unroll
        for (int j = 1; j < W; j++) T[j] = (t0c && j0 == 0 && j == 1) ? 1.0f : 0.0f;
#pragma unroll
        for (int j = 0; j < W; j++) U[j] = 0.0f;
        int sp = 1;
        // tokens of the low half, then (two-register tapes) the high half
        const int lo_end = HI ? min(p.len, 64) : p.len;
        for (int t = 1; t < lo_end; t++) dual_token<0, NT>(p, m, cm, nlo, j0, xv, lane, laneb, lanec, T, U, sp, t);
        if (HI)
            for (int t = 64; t < p.len; t++) dual_token<1, NT>(p, m, cm, nlo, j0, xv, lane, laneb, lanec, T, U, sp, t);
        const float r = T[0] - c.y[0];
        const float term = valid ? (r * r) * c.w[0] : 0.0f;
        const float yv = term - comp;
        const float tv = acc + yv;
        comp = (tv - acc) - yv;
        acc = tv;
        const float G = (-2.0f * r) * (folded ? wf : c.w[0]);
#pragma unroll
        for (int j = 0; j < NT; j++) ga[j] = valid ? __builtin_fmaf(G, T[j + 1], ga[j]) : ga[j];
        if (ch + 1 < nchunks && reject_below > -GPR_INF) {
            const double lb = (double)wave_sum_f(acc - comp) * (1.0 - 1e-4);
            const double ub = d.lconst - wc * lb;
            if (!(ub >= reject_below)) {
                if (points) *points = (ch + 1) * 64;
                return -GPR_INF;
            }
        }
    }
#pragma unroll
    for (int j = 0; j < GPR_DUAL_NTMAX; j++)
        gs[j] = (j < NT && j0 + j < nlo + (HI ? __popcll(cm[1]) : 0)) ? wave_sum_f(ga[j < NT ? j : 0]) : 0.0f;
    const double s = wave_sum_d((double)acc - (double)comp);
    if (!__builtin_isfinite(s)) return -GPR_INF;
    return d.lconst - (d.wconst > 0.0 ? d.wconst * s : s);
}

// npass (1 or 2) passes of GPR_DUAL_NT4 tangents: the constants of rank 0-3, then, when the
// first pass completes, those of rank 4-7 (its LL is the first's: same values, same
// order).
template <bool HI>
__device__ __forceinline__ double dual_passes4(const WaveProg &p, const GprDataset &d, const float *dx, const float *dy,
                                               const float *dw, const Chunk<1> &c0, int nchunks, float *ls,
                                               const OpMasks &m, const uint64_t (&cm)[2], double reject_below,
                                               int *points, int npass, float (&gs)[GPR_DUAL_NTMAX]) {
    const double ll =
        wave_loglik_dual<HI, GPR_DUAL_NT4>(p, d, dx, dy, dw, c0, nchunks, ls, m, cm, reject_below, points, 0, gs);
    if (npass > 1 && __builtin_isfinite(ll)) {
        float g[GPR_DUAL_NTMAX];
        (void)wave_loglik_dual<HI, GPR_DUAL_NT4>(p, d, dx, dy, dw, c0, nchunks, ls, m, cm, -GPR_INF, nullptr,
                                                 GPR_DUAL_NT4, g);
#pragma unroll
        for (int j = 0; j < GPR_DUAL_NT4; j++) gs[GPR_DUAL_NT4 + j] = g[j];
    }
    return ll;
}

// The gradient of the log posterior in the lane layout of wave_loglik_grad: lane t of g0
// (token t < 64) or g1 holds d/dc_t (from gs by the constant's rank) plus the Cauchy
// prior's -2c/(1+c^2); ok is false when one of them is not finite.
template <bool HI>
__device__ __forceinline__ void dual_grad_lanes(const WaveProg &p, const uint64_t (&cm)[2],
                                                const float (&gs)[GPR_DUAL_NTMAX], double &g0, double &g1, bool &ok) {
    const int l = lane_id();
    const uint64_t below = (1ull << l) - 1ull;
    const int r0 = __popcll(cm[0] & below);
    const int r1 = __popcll(cm[0]) + (HI ? __popcll(cm[1] & below) : 0);
    const bool c0 = (cm[0] >> l) & 1ull, c1 = HI && ((cm[1] >> l) & 1ull);
    float s0 = 0.0f, s1 = 0.0f;
#pragma unroll
    for (int j = 0; j < GPR_DUAL_NTMAX; j++) {
        s0 = r0 == j ? gs[j] : s0;
        s1 = r1 == j ? gs[j] : s1;
    }
    g0 = c0 ? (double)s0 - 2.0 * (double)p.c0 / (1.0 + (double)p.c0 * (double)p.c0) : 0.0;
    g1 = c1 ? (double)s1 - 2.0 * (double)p.c1 / (1.0 + (double)p.c1 * (double)p.c1) : 0.0;
    ok = ballot((c0 && !__builtin_isfinite(g0)) || (c1 && !__builtin_isfinite(g1))) == 0;
}

// As tape_run for one point per lane, with a lane's constants taken from cb in token order:
// ca is the byte index (ds_bpermute) of the lane holding the next one.  T may still be
// loading when a handler ends, so every handler waits first.
__device__ __forceinline__ void tape_run_groups(int word, float cb, float x, float &T, float &U, uint32_t &p, uint32_t &ca,
                                                int &t) {
    uint32_t blo, bhi, w, s;
    float v;
    GT_TEMPS;
#define GT_H(N, BODY) ".org .Lh%=+64*" #N "\n\t" BODY
#define GG_TAKE(D) "ds_bpermute_b32 " D ", %[ca], %[cb]\n\tv_add_u32 %[ca], 4, %[ca]\n\t"
    __asm__ volatile(
        GT_ENTRY
        ".p2align 6\n.Lh%=:\n\t" GT_EXIT
        GT_H(1, GT_NEXT(1) GT1_PUSH "v_mov_b32 %[T0], %[x]\n\t" GT_JUMP)
        GT_H(2, GT_NEXT(1) GT1_PUSH GG_TAKE("%[T0]") GT_JUMP)
        GT_H(3, GT_NEXT(2) GT_WAIT GT1("v_add_f32", "%[x]", "%[T0]") GT_JUMP)
        GT_H(4, GT_NEXT(2) GT_WAIT GT1("v_sub_f32", "%[T0]", "%[x]") GT_JUMP)
        GT_H(5, GT_NEXT(2) GT_WAIT GT1("v_mul_f32", "%[x]", "%[T0]") GT_JUMP)
        GT_H(6, GT_NEXT(2) GG_TAKE("%[v]") GT_WAIT GT1("v_add_f32", "%[v]", "%[T0]") GT_JUMP)
        GT_H(7, GT_NEXT(2) GG_TAKE("%[v]") GT_WAIT GT1("v_sub_f32", "%[T0]", "%[v]") GT_JUMP)
        GT_H(8, GT_NEXT(2) GG_TAKE("%[v]") GT_WAIT GT1("v_mul_f32", "%[v]", "%[T0]") GT_JUMP)
        GT_H(9, GT_NEXT(1) GT_WAIT GT1("v_add_f32", "%[U0]", "%[T0]") GT1_POP GT_JUMP)
        GT_H(10, GT_NEXT(1) GT_WAIT GT1("v_sub_f32", "%[U0]", "%[T0]") GT1_POP GT_JUMP)
        GT_H(11, GT_NEXT(1) GT_WAIT GT1("v_mul_f32", "%[U0]", "%[T0]") GT1_POP GT_JUMP)
        GT_H(12, GT_NEXT(1) GT_WAIT "v_xor_b32 %[T0], 0x80000000, %[T0]\n\t" GT_JUMP)
        GT_H(13, GT_NEXT(3) GT1_PUSH GT1("v_add_f32", "%[x]", "%[x]") GT_JUMP)
        GT_H(14, GT_NEXT(3) GT1_PUSH GT1("v_sub_f32", "%[x]", "%[x]") GT_JUMP)
        GT_H(15, GT_NEXT(3) GT1_PUSH GT1("v_mul_f32", "%[x]", "%[x]") GT_JUMP)
        GT_H(16, GT_NEXT(3) GG_TAKE("%[v]") GT1_PUSH GT1("v_add_f32", "%[v]", "%[x]") GT_JUMP)
        GT_H(17, GT_NEXT(3) GG_TAKE("%[v]") GT1_PUSH GT1("v_sub_f32", "%[x]", "%[v]") GT_JUMP)
        GT_H(18, GT_NEXT(3) GG_TAKE("%[v]") GT1_PUSH GT1("v_mul_f32", "%[v]", "%[x]") GT_JUMP)
        GT_H(19, GT_NEXT(3) GG_TAKE("%[v]") GT1_PUSH GT1("v_add_f32", "%[v]", "%[x]") GT_JUMP)
        GT_H(20, GT_NEXT(3) GG_TAKE("%[v]") GT1_PUSH GT1("v_sub_f32", "%[v]", "%[x]") GT_JUMP)
        GT_H(21, GT_NEXT(3) GG_TAKE("%[v]") GT1_PUSH GT1("v_mul_f32", "%[v]", "%[x]") GT_JUMP)
        GT_H(22, GT_WAIT GT_EXP_TEST("%[T0]") GT_NEXT(1) GT_LOG2E GT_EXP("%[T0]") GT_JUMP)
        GT_H(24, GT_WAIT GT_NEXT(1) GT_DIV("%[U0]", "%[T0]") GT1_POP GT_JUMP)
        GT_H(26, GT_WAIT GT_NEXT(1) GT_LOG("%[T0]") GT_JUMP)
        ".Lx%=:"
        : [T0] "+&v"(T), [U0] "+&v"(U), [p] "+&v"(p), [ca] "+&v"(ca), [t] "+&s"(t), [blo] "=&s"(blo), [bhi] "=&s"(bhi),
          [w] "=&s"(w), [s] "=&s"(s), [v] "=&v"(v), GT_TEMP_OUT
        : [word] "v"(word), [cb] "v"(cb), [x] "v"(x)
        : "vcc", "scc", "memory");
#undef GG_TAKE
#undef GT_H
}

// ---------------------------------------------------------------- speculative constant steps
// Datasets of at most 32 points fill a fraction of a wave.  The random-walk kernel then
// evaluates the proposals of G consecutive constant steps in one interpreter pass, one
// per lane group (G = 4 groups of 16 lanes for n <= 16, 2 of 32 for n <= 32): lane l
// takes point l mod (64 / G) of the proposal of step u0 + l / (64 / G).  All of them are
// proposals from the same current state, which is the state each step sees as long as
// the steps before it reject; the kernel uses them in step order and drops the rest
// after an accept.  The dispatch of every token serves the G proposals.
//
// Proposal constants come from the draw batch: the constant of rank r of step u is lane
// ks u + r of cb.  The value of each proposal is bit-identical to its own evaluation by
// wave_loglik<1, false>: the same operations per point, a one-chunk Kahan sum (the term
// itself), and a group sum whose FP64 additions are those of wave_sum_d over the lanes
// it would occupy alone (rows of 16 lanes summed by the same DPP steps; a group of two
// rows adds them as wave_sum_d adds rows 0 and 1, and adding the zero rows of a lone
// evaluation changes nothing).  ls: the wave's value-stack region (KC = 1 layout).
// out[g] receives the LL of group g's proposal, for g < gn (groups g >= gn repeat the
// proposal of group gn - 1).
__device__ __forceinline__ void wave_loglik_groups(const WaveProg &p, const GprDataset &d, const float *dx,
                                                   const float *dy, const float *dw, float *ls, const ProgCode &m,
                                                   float cb, int ks, int u0, int G, int gn, double (&out)[4]) {
    const int l = opaque_lane_i32(lane_id());       // what follows is computed here, not kept live
    const int lgs = G == 4 ? 4 : 5;                  // log2 of the group size
    const int gl = l >> lgs;
    const int i = l & ((1 << lgs) - 1);
    const bool valid = i < d.n;
    const float xv = valid ? dx[i] : 0.0f, yv = valid ? dy[i] : 0.0f, wv = valid ? dw[i] : 0.0f;
    uint32_t ca = 4u * (uint32_t)(ks * (u0 + min(gl, gn - 1)));   // lane of cb holding rank 0 of this group's step
    uint32_t a = lds_addr(ls) + 4u * (uint32_t)l;                 // level -2 of the stack below T, U
    float Ts[1] = {0.0f}, U[1] = {0.0f};
    const float xs[1] = {xv};
    const int n = uni(p.len);
    for (int t = 0; t < n; t++) {
        t = uni(t);
        tape_run_groups(m.w0, cb, xv, Ts[0], U[0], a, ca, t);
        t = uni(t);
        if (t >= n) break;
        // (no constant reaches this: the last lane's token of a full tape is an operator, and a
        // batched program has no constant-operand token)
        tape_slow<1>(rl_i(p.o0, t), 0.0f, xs, Ts, U, a);
    }
    const float T = Ts[0];
    const float r = T - yv;
    const float term = valid ? (r * r) * wv : 0.0f;
    double v = (double)term;
    v += dpp_d<DPP_QP_1032>(v);
    v += dpp_d<DPP_QP_2301>(v);
    v += dpp_d<DPP_ROW_HALF_MIRROR>(v);
    v += dpp_d<DPP_ROW_MIRROR>(v);
#pragma unroll
    for (int g = 0; g < 4; g++) {
        double s;
        if (G == 4) s = rl_d(v, 16 * g);
        else s = g < 2 ? rl_d(v, 32 * g) + rl_d(v, 32 * g + 16) : 0.0;
        out[g] = !__builtin_isfinite(s) ? -GPR_INF : d.lconst - (d.wconst > 0.0 ? d.wconst * s : s);
    }
}

// Description-length prior plus Cauchy(0,1) on every constant token, summed in token
// order in FP64 (the same order as the oracle, so the value is bit-reproducible).
template <bool HI>
__device__ __forceinline__ double wave_prior(const WaveProg &p, double lnsym) {
    const int l = lane_id();
    const bool v0 = l < p.len, v1 = HI && (l + 64) < p.len;
    int dl = p.len + __popcll(ballot(v0 && p.o0 >= GPR_OP_CADD)) + (HI ? __popcll(ballot(v1 && p.o1 >= GPR_OP_CADD)) : 0);
    uint64_t m0 = ballot(v0 && gpr_has_const(p.o0));
    const double lc0 = gpr_lcauchy(p.c0);
    double s = 0.0;
    while (m0) {
        const int b = __builtin_ctzll(m0);
        m0 &= m0 - 1;
        s += rl_d(lc0, b);
    }
    if (HI) {
        uint64_t m1 = ballot(v1 && gpr_has_const(p.o1));
        if (m1) {
            const double lc1 = gpr_lcauchy(p.c1);
            while (m1) {
                const int b = __builtin_ctzll(m1);
                m1 &= m1 - 1;
                s += rl_d(lc1, b);
            }
        }
    }
    return gpr_dl_prior(dl, lnsym, s);
}

// Subtree [s0, j] ending at token j: s0-1 is the last u < j whose stack depth after u is
// below the depth after j.  Also returns the maximum depth of the tape.
template <bool HI>
__device__ __forceinline__ void wave_depths(const WaveProg &p, int &D0, int &D1, int &dmax) {
    const int l = lane_id();
    const int d0 = l < p.len ? 1 - gpr_arity(p.o0) : 0;
    D0 = wave_scan_i(d0);
    dmax = wave_max_i(l < p.len ? D0 : 0);
    D1 = 0;
    if (HI && p.len > 64) {
        const int tot = rl_i(D0, 63);
        const int d1 = l + 64 < p.len ? 1 - gpr_arity(p.o1) : 0;
        D1 = wave_scan_i(d1) + tot;
        dmax = max(dmax, wave_max_i(l + 64 < p.len ? D1 : 0));
    }
}

template <bool HI>
__device__ __forceinline__ int subtree_start(int j, int D0, int D1) {
    const int l = lane_id();
    const int Dj = (HI && j >= 64) ? rl_i(D1, j - 64) : rl_i(D0, j);
    uint64_t m1 = HI ? ballot(l + 64 < j && D1 < Dj) : 0;
    if (m1) return 64 + (63 - __builtin_clzll(m1)) + 1;
    uint64_t m0 = ballot(l < j && D0 < Dj);
    if (m0) return (63 - __builtin_clzll(m0)) + 1;
    return 0;
}

// ---------------------------------------------------------------- subtree generation
// A structure move draws its new subtree one symbol per lane.  Symbol k of the
// right-child-first prefix order takes word 0 of the Philox block at counter
// {chain, step, GPR_P_STRUCT << 24, k} and, when it is CONST, its value from word 1 of
// that block; word 2 of block 0 picks the node to replace.  The subtree ends at the
// first symbol after which no operand is missing: a prefix sum of (arity - 1) over the
// lanes finds it.
//
// gpr_gen_symbol per lane: the top 6 bits of a word pick X (16 of 64 buckets), CONST
// (16), then ADD SUB MUL DIV POW EXP LOG NEG (4 each), packed one code per byte.
__device__ __forceinline__ int gen_symbol_lane(uint32_t r) {
    constexpr uint64_t ORDER = (uint64_t)GPR_OP_ADD | ((uint64_t)GPR_OP_SUB << 8) | ((uint64_t)GPR_OP_MUL << 16) |
                               ((uint64_t)GPR_OP_DIV << 24) | ((uint64_t)GPR_OP_POW << 32) |
                               ((uint64_t)GPR_OP_EXP << 40) | ((uint64_t)GPR_OP_LOG << 48) |
                               ((uint64_t)GPR_OP_NEG << 56);
    const int k = (int)(r >> 26);
    const int op = (int)((ORDER >> (8 * ((k >> 2) & 7))) & 0xff);
    return k < 16 ? GPR_OP_X : (k < 32 ? GPR_OP_CONST : op);
}
// gpr_gen_logp per lane: log 1/4 for the leaves, log 1/16 for the generated operators,
// -inf for ops the table never draws.
__device__ __forceinline__ double gen_logp_lane(int op) {
    constexpr uint32_t LEAF = (1u << GPR_OP_X) | (1u << GPR_OP_CONST);
    constexpr uint32_t GEN = (1u << GPR_OP_ADD) | (1u << GPR_OP_SUB) | (1u << GPR_OP_MUL) | (1u << GPR_OP_DIV) |
                             (1u << GPR_OP_POW) | (1u << GPR_OP_EXP) | (1u << GPR_OP_LOG) | (1u << GPR_OP_NEG);
    const uint32_t b = 1u << (op & 31);
    return (b & LEAF) ? GPR_LOG_QUARTER : ((b & GEN) ? GPR_LOG_SIXTEENTH : -__builtin_inf());
}
// generation term of one token: its symbol's log probability and, for CONST, the
// standard normal log density of its value
__device__ __forceinline__ double gen_term_lane(int op, float c) {
    return gen_logp_lane(op) + (op == GPR_OP_CONST ? gpr_lphi(c) : 0.0);
}

// value of a 128-token lane array at token index src (src may differ per lane)
__device__ __forceinline__ int gather_i(int v0, int v1, int src, bool hi) {
    const int a = shfl_all(v0, src & 63);
    if (!hi) return a;
    const int b = shfl_all(v1, src & 63);
    return src >= 64 ? b : a;
}
__device__ __forceinline__ float gather_f(float v0, float v1, int src, bool hi) {
    const float a = shfl_all(v0, src & 63);
    if (!hi) return a;
    const float b = shfl_all(v1, src & 63);
    return src >= 64 ? b : a;
}

// ---------------------------------------------------------------- reverse-mode adjoint
// KC points per lane and sweep pair.  The forward sweep stores the value of every operator
// token in the wave's rows, lv[row][k][lane], at the row of its rank among the operators;
// leaves (x, constant, one) are not stored, their values come from the token.  A binary
// token finds its left operand through a per-structure plan (its right operand is the token
// before it, whose value the sweep carries).  The reverse sweep walks the tape backwards
// carrying the adjoint of the current token.  Reverse postfix order visits a node, then its
// right subtree (ending at t-1), then its left subtree, so a binary token carries its right
// operand's adjoint on and pushes its left operand's onto a stack in the rows after the
// operators'; a leaf pops the next one.  The adjoint of a constant is summed over the wave as
// soon as it is known.  A program needs fewer rows than it has tokens: operators and pending
// left operands are at most len - 1.

// Per-structure plan of the two sweeps.  Word t (lane t of w0, lane t-64 of w1): a gpr_gtok, its
// operands a row, or GPR_G_X, GPR_G_ONE or GPR_G_C + token for a leaf.  rows: rows of the sweeps.
#define GPR_G_X 127
#define GPR_G_C 128
#define GPR_G_ONE 255
static_assert(GPR_NUM_OPS <= 31, "gpr_gtok keeps 31 for an unknown op");
struct GradPlan {
    int w0, w1;
    int nops, rows;
};

template <bool HI>
__device__ __forceinline__ GradPlan grad_plan(const WaveProg &p) {
    const int l = lane_id();
    GradPlan g;
    int D0, D1, dm;
    wave_depths<HI>(p, D0, D1, dm);
    const bool v0 = l < p.len, v1 = HI && l + 64 < p.len;
    const uint64_t m0 = ballot(v0 && p.o0 > GPR_OP_ONE), m1 = HI ? ballot(v1 && p.o1 > GPR_OP_ONE) : 0;
    const uint64_t below = (1ull << l) - 1ull;
    const int s0 = __popcll(m0 & below), s1 = __popcll(m0) + __popcll(m1 & below);
    // this token as an operand
    const int r0 = p.o0 == GPR_OP_X ? GPR_G_X : (p.o0 == GPR_OP_ONE ? GPR_G_ONE : (p.o0 == GPR_OP_CONST ? GPR_G_C + l : s0));
    const int r1 = p.o1 == GPR_OP_X ? GPR_G_X
                                    : (p.o1 == GPR_OP_ONE ? GPR_G_ONE : (p.o1 == GPR_OP_CONST ? GPR_G_C + 64 + l : s1));
    // the left operand of a binary token is the last token before it whose stack depth is its
    // own: the tokens between them, the right operand's, lie deeper
    int lc0 = 0, lc1 = 0;
    for (int k = 1; k <= min(dm, GPR_MAX_DEPTH); k++) {
        const uint64_t d0 = ballot(v0 && D0 == k), d1 = HI ? ballot(v1 && D1 == k) : 0;
        const uint64_t q0 = d0 & below, q1 = d1 & below;
        if (D0 == k) lc0 = q0 ? 63 - __builtin_clzll(q0) : 0;
        if (HI && D1 == k) lc1 = q1 ? 127 - __builtin_clzll(q1) : (d0 ? 63 - __builtin_clzll(d0) : 0);
    }
    const int left0 = gather_i(r0, r1, lc0, HI), right0 = gather_i(r0, r1, max(l - 1, 0), HI);
    g.w0 = gpr_gtok(p.o0, s0, left0, right0);
    g.w1 = 0;
    if (HI) {
        const int left1 = gather_i(r0, r1, lc1, HI), right1 = gather_i(r0, r1, l + 63, HI);
        g.w1 = gpr_gtok(p.o1, s1, left1, right1);
    }
    g.nops = __popcll(m0) + __popcll(m1);
    // pending left operands: at most one per level above the first
    g.rows = g.nops + max(dm - 1, 0);
    return g;
}

// operand r (a row or a leaf) at this lane's points
template <int KC, bool HI>
__device__ __forceinline__ void grad_val(const WaveProg &p, int r, const float (&x)[KC], const float *lvl, float (&v)[KC]) {
    if (r < GPR_G_X) {
#pragma unroll
        for (int k = 0; k < KC; k++) v[k] = lvl[(r * KC + k) * 64];
    } else {
        const int u = r - GPR_G_C;
        const float c = r == GPR_G_ONE ? 1.0f : ((HI && u >= 64) ? rl_f(p.c1, u & 63) : rl_f(p.c0, max(u, 0) & 63));
        const bool isx = r == GPR_G_X;
#pragma unroll
        for (int k = 0; k < KC; k++) v[k] = isx ? x[k] : c;
    }
}

// Forward sweep: the same operations on the same operands as wave_eval_ls, so the value is
// bit-identical.  P: the value before the last leaf, the left operand of a binary token
// right after a leaf.
template <int KC, bool HI>
__device__ __forceinline__ void grad_forward(const WaveProg &p, const GradPlan &g, const float (&x)[KC], float *lvl,
                                             float (&T)[KC]) {
    float P[KC];
#pragma unroll
    for (int k = 0; k < KC; k++) T[k] = P[k] = 0.0f;
    for (int t = 0; t < p.len; t++) {
        const int li = t & 63;
        const bool h = HI && t >= 64;
        const int w = h ? rl_i(g.w1, li) : rl_i(g.w0, li);
        const int op = gpr_gtok_op(w);
        if (op <= GPR_OP_ONE) {
            float L[KC];
            if (op == GPR_OP_X) {
#pragma unroll
                for (int k = 0; k < KC; k++) L[k] = x[k];
            } else {
                const float cv = h ? rl_f(p.c1, li) : rl_f(p.c0, li);
#pragma unroll
                for (int k = 0; k < KC; k++) L[k] = op == GPR_OP_CONST ? cv : 1.0f;
            }
            // with the +, - or * after it in one step, no copies of the stack's top: MALA with a
            // metric on a rational of 7 constants, n = 37, 2.95e8 -> 3.20e8 steps/s.  At several
            // points per lane the copies are a smaller share and the branches cost 1.5 %
            const int w2 = HI && t >= 63 ? rl_i(g.w1, (t + 1) & 63) : rl_i(g.w0, (t + 1) & 63), op2 = gpr_gtok_op(w2);
            if (KC == 1 && t + 1 < p.len && (unsigned)(op2 - GPR_OP_ADD) < 3u) {
                const int row = gpr_gtok_row(w2);
#pragma unroll
                for (int k = 0; k < KC; k++) {
                    if (op2 == GPR_OP_ADD) T[k] = T[k] + L[k];
                    else if (op2 == GPR_OP_SUB) T[k] = T[k] - L[k];
                    else T[k] = T[k] * L[k];
                    lvl[(row * KC + k) * 64] = T[k];
                }
                t++;
                continue;
            }
#pragma unroll
            for (int k = 0; k < KC; k++) { P[k] = T[k]; T[k] = L[k]; }
            continue;
        }
        if (op <= GPR_OP_RPOW) {
            float A[KC];
            if (gpr_gtok_right(w) >= GPR_G_X) {
#pragma unroll
                for (int k = 0; k < KC; k++) A[k] = P[k];
            } else {
                grad_val<KC, HI>(p, gpr_gtok_left(w), x, lvl, A);
            }
            if (op == GPR_OP_ADD) GPR_KLOOP(A[k] + T[k]);
            else if (op == GPR_OP_SUB) GPR_KLOOP(A[k] - T[k]);
            else if (op == GPR_OP_MUL) GPR_KLOOP(A[k] * T[k]);
            else GPR_KLOOP(op_bin(op, A[k], T[k]));
        } else {
            const float c = op >= GPR_OP_CADD ? (h ? rl_f(p.c1, li) : rl_f(p.c0, li)) : 0.0f;
            GPR_KLOOP(op_un(op, T[k], c));
        }
        const int row = gpr_gtok_row(w);
#pragma unroll
        for (int k = 0; k < KC; k++) lvl[(row * KC + k) * 64] = T[k];
    }
}

// Reverse sweep from the adjoints G of the program's value.  The wave sums of the constants'
// adjoints over the lanes with a valid point land at lane t of s0[k] (token t < 64) or s1[k].
template <int KC, bool HI>
__device__ __forceinline__ void grad_reverse(const WaveProg &p, const GradPlan &g, const float (&x)[KC], float *lvl,
                                             float (&G)[KC], const bool (&valid)[KC], float (&s0)[KC], float (&s1)[KC]) {
    const int l = lane_id();
    int top = g.nops;   // row of the next push
    auto constant = [&](int t, const float (&v)[KC]) {
#pragma unroll
        for (int k = 0; k < KC; k++) {
            const float s = wave_sum_f(valid[k] ? v[k] : 0.0f);
            if (HI && t >= 64) s1[k] = l == t - 64 ? s : s1[k];
            else s0[k] = l == t ? s : s0[k];
        }
    };
    for (int t = p.len - 1; t >= 0; t--) {
        const int li = t & 63;
        const bool h = HI && t >= 64;
        const int w = h ? rl_i(g.w1, li) : rl_i(g.w0, li);
        const int op = gpr_gtok_op(w);
        if (op <= GPR_OP_ONE) {
            if (op == GPR_OP_CONST) constant(t, G);
            // the next token roots a left operand: its adjoint waits on the stack
            if (t > 0) {
                top--;
#pragma unroll
                for (int k = 0; k < KC; k++) G[k] = lvl[(top * KC + k) * 64];
            }
            continue;
        }
        const int lr = gpr_gtok_left(w), rr = gpr_gtok_right(w);
        if (op <= GPR_OP_RPOW) {
            float ga[KC], gb[KC];
            if (op <= GPR_OP_SUB) {
                const bool sub = op == GPR_OP_SUB;
#pragma unroll
                for (int k = 0; k < KC; k++) { ga[k] = G[k]; gb[k] = sub ? -G[k] : G[k]; }
            } else {
                float A[KC], B[KC];
                grad_val<KC, HI>(p, lr, x, lvl, A);
                grad_val<KC, HI>(p, rr, x, lvl, B);
                const int row = gpr_gtok_row(w);
#pragma unroll
                for (int k = 0; k < KC; k++) {
                    const float a = A[k], b = B[k], q = G[k];
                    if (op == GPR_OP_MUL) {
                        ga[k] = q * b;
                        gb[k] = q * a;
                        continue;
                    }
                    switch (op) {
                    case GPR_OP_DIV: ga[k] = q / b; gb[k] = -(q * a) / (b * b); break;
                    case GPR_OP_RSUB: ga[k] = -q; gb[k] = q; break;
                    case GPR_OP_RDIV: gb[k] = q / a; ga[k] = -(q * b) / (a * a); break;
                    case GPR_OP_POW: {
                        const float v = lvl[(row * KC + k) * 64];
                        ga[k] = q * b * pow_bm1(a, b, v);
                        gb[k] = q * v * logf(a);
                        break;
                    }
                    default: {  // RPOW: b^a
                        const float v = lvl[(row * KC + k) * 64];
                        gb[k] = q * a * pow_bm1(b, a, v);
                        ga[k] = q * v * logf(b);
                        break;
                    }
                    }
                }
            }
            if (rr >= GPR_G_X) {
                // right operand is a leaf: its adjoint is final now, and the left operand's
                // subtree ends at t-2 and comes next, so its adjoint is carried
                if (rr >= GPR_G_C && rr != GPR_G_ONE) constant(t - 1, gb);
#pragma unroll
                for (int k = 0; k < KC; k++) G[k] = ga[k];
                t--;
                continue;
            }
#pragma unroll
            for (int k = 0; k < KC; k++) { lvl[(top * KC + k) * 64] = ga[k]; G[k] = gb[k]; }
            top++;
        } else {
            const float c = op >= GPR_OP_CADD ? (h ? rl_f(p.c1, li) : rl_f(p.c0, li)) : 0.0f;
            float A[KC], gc[KC];
            grad_val<KC, HI>(p, rr, x, lvl, A);
            const int row = gpr_gtok_row(w);
#pragma unroll
            for (int k = 0; k < KC; k++) {
                const float a = A[k], v = lvl[(row * KC + k) * 64], q = G[k];
                gc[k] = 0.0f;
                switch (op) {
                case GPR_OP_NEG: G[k] = -q; break;
                case GPR_OP_EXP: G[k] = q * v; break;
                case GPR_OP_LOG: G[k] = q / a; break;
                case GPR_OP_INV: G[k] = -q / (a * a); break;
                case GPR_OP_SQRT: G[k] = q * 0.5f / v; break;
                case GPR_OP_SIN: G[k] = q * cosf(a); break;
                case GPR_OP_COS: G[k] = -q * sinf(a); break;
                case GPR_OP_TAN: G[k] = q * (1.0f + v * v); break;
                case GPR_OP_ASIN: G[k] = q / sqrtf(1.0f - a * a); break;
                case GPR_OP_ACOS: G[k] = -q / sqrtf(1.0f - a * a); break;
                case GPR_OP_ATAN: G[k] = q / (1.0f + a * a); break;
                case GPR_OP_ABS: G[k] = a < 0.0f ? -q : q; break;
                case GPR_OP_CADD: gc[k] = q; break;
                case GPR_OP_CMUL: G[k] = q * c; gc[k] = q * a; break;
                case GPR_OP_CPOW: G[k] = q * c * pow_bm1(a, c, v); gc[k] = q * v * logf(a); break;
                case GPR_OP_CRPOW: G[k] = q * v * logf(c); gc[k] = q * a * pow_bm1(c, a, v); break;
                default: G[k] = __builtin_nanf(""); break;
                }
            }
            if (op >= GPR_OP_CADD) constant(t, gc);
        }
    }
}

// Both sweeps over KC chunks of 64 points from point `base`: their terms of the LL
// ((f - y)^2 w, 0 past the last point) and the constants' sums of each chunk.
template <int KC, bool HI>
__device__ __forceinline__ void grad_sweeps(const WaveProg &p, const GradPlan &g, const GprDataset &d, const float *dx,
                                            const float *dy, const float *dw, int base, float *lvl, float (&term)[KC],
                                            float (&s0)[KC], float (&s1)[KC]) {
    const int l = lane_id();
    const bool folded = d.wconst > 0.0;
    const float wf = (float)d.wconst;
    float x[KC], T[KC], G[KC];
    bool valid[KC];
#pragma unroll
    for (int k = 0; k < KC; k++) {
        const int i = base + 64 * k + l;
        valid[k] = i < d.n;
        x[k] = valid[k] ? dx[i] : 0.0f;
    }
    grad_forward<KC, HI>(p, g, x, lvl, T);
#pragma unroll
    for (int k = 0; k < KC; k++) {
        const int i = base + 64 * k + l;
        const float y = valid[k] ? dy[i] : 0.0f, w = valid[k] ? dw[i] : 0.0f;
        const float r = T[k] - y;
        term[k] = valid[k] ? (r * r) * w : 0.0f;
        // d/df of -(f - y)^2 w, with w = wconst when the weights are folded into it
        G[k] = valid[k] ? (-2.0f * r) * (folded ? wf : w) : 0.0f;
        s0[k] = s1[k] = 0.0f;
    }
    grad_reverse<KC, HI>(p, g, x, lvl, G, valid, s0, s1);
}

// the prior's -2c/(1+c^2) on the constant tokens of g0, g1; false when a gradient is not finite
template <bool HI>
__device__ __forceinline__ bool grad_prior(const WaveProg &p, double &g0, double &g1) {
    const int l = lane_id();
    const bool c0 = l < p.len && gpr_has_const(p.o0), c1 = HI && l + 64 < p.len && gpr_has_const(p.o1);
    if (c0) g0 += -2.0 * (double)p.c0 / (1.0 + (double)p.c0 * (double)p.c0);
    if (c1) g1 += -2.0 * (double)p.c1 / (1.0 + (double)p.c1 * (double)p.c1);
    return ballot((c0 && !__builtin_isfinite(g0)) || (c1 && !__builtin_isfinite(g1))) == 0;
}

// Log-likelihood and d(log posterior)/d(constant) of the wave's program (g: its plan).
// The LL is bit-identical to wave_loglik<KC, HI> for every KC: lane l visits points
// c*64 + l in increasing c, the same per-lane order and Kahan updates.  The gradient
// holds the wave sums of the per-point adjoints (FP32) accumulated over chunks in FP64,
// plus the Cauchy prior's -2c/(1+c^2); token t sits at lane t of g0 (t < 64) or g1.
// lv: this wave's slab of at least g.rows * 64 floats.  Returns false in ok when the
// LL or a constant's gradient is not finite.
template <bool HI>
__device__ __forceinline__ double wave_loglik_grad(const WaveProg &p, const GradPlan &g, const GprDataset &d, const float *dx,
                                   const float *dy, const float *dw, float *lv, double &g0, double &g1, bool &ok) {
    float *lvl = lv + lane_id();
    g0 = 0.0;
    g1 = 0.0;
    float acc = 0.0f, comp = 0.0f;
    for (int base = 0; base < d.n; base += 64) {
        float term[1], s0[1], s1[1];
        grad_sweeps<1, HI>(p, g, d, dx, dy, dw, base, lvl, term, s0, s1);
        const float yv = term[0] - comp;
        const float tv = acc + yv;
        comp = (tv - acc) - yv;
        acc = tv;
        g0 += (double)s0[0];
        if (HI) g1 += (double)s1[0];
    }
    const double s = wave_sum_d((double)acc - (double)comp);
    ok = grad_prior<HI>(p, g0, g1) && __builtin_isfinite(s);
    if (!__builtin_isfinite(s)) return -GPR_INF;
    return d.lconst - (d.wconst > 0.0 ? d.wconst * s : s);
}

// FP64 sum of the Gaussian log-density terms -f^2 r2 (r2 = 1 / (2 e^2)) over the lanes where m holds, in
// token order (lanes of the low half, then the high half), as a serial loop over tokens
// would add them.  A half without such lanes computes no terms.
template <bool HI>
__device__ __forceinline__ double wave_gauss_sum_d(double f0, bool m0, double f1, bool m1, double r2) {
    double s = 0.0;
    uint64_t b0 = ballot(m0);
    if (b0) {
        const double v0 = -f0 * f0 * r2;
        while (b0) {
            const int b = __builtin_ctzll(b0);
            b0 &= b0 - 1;
            s += rl_d(v0, b);
        }
    }
    if (HI) {
        uint64_t b1 = ballot(m1);
        if (b1) {
            const double v1 = -f1 * f1 * r2;
            while (b1) {
                const int b = __builtin_ctzll(b1);
                b1 &= b1 - 1;
                s += rl_d(v1, b);
            }
        }
    }
    return s;
}

// ---------------------------------------------------------------- proposal metric
// Lanes 0..k-1 hold metric rows; the matrices are row-major in global memory, and each
// lane reads its row with 16-byte loads issued together, before the products.  Products
// accumulate in FP32 in increasing index order, the density's forward substitution in
// FP64, both without contraction (the oracle's operation order).

// lane l's row of a 16-wide float matrix, columns below k (lanes past k read row k-1)
__device__ __forceinline__ void metric_row(const float *A, int k, float (&r)[GPR_METRIC_MAX]) {
    // (the row address is computed here, not kept live across the steps)
    const float4 *q = (const float4 *)(A + min(opaque_lane_i32(lane_id()), k - 1) * GPR_METRIC_MAX);
#pragma unroll
    for (int j = 0; j < GPR_METRIC_MAX; j += 4) {
        float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (j < k) v = q[j / 4];
        r[j] = v.x; r[j + 1] = v.y; r[j + 2] = v.z; r[j + 3] = v.w;
    }
}

// d_i = sum_{j <= i} L_ij v_j, v and d at lanes 0..k-1
__device__ __forceinline__ float metric_Lv(const float *L, int k, float v) {
    const int l = lane_id();
    float r[GPR_METRIC_MAX];
    metric_row(L, k, r);
    float acc = 0.0f;
#pragma unroll
    for (int j = 0; j < GPR_METRIC_MAX; j++) {
        if (j < k) {
            const float vj = rl_f(v, j);
            if (l < k && j <= l) acc = gpr_axpy(r[j], vj, acc);
        }
    }
    return acc;
}
// v_i = sum_j M_ij g_j, g and v at lanes 0..k-1
__device__ __forceinline__ float metric_Mv(const float *M, int k, float g) {
    const int l = lane_id();
    float r[GPR_METRIC_MAX];
    metric_row(M, k, r);
    float acc = 0.0f;
#pragma unroll
    for (int j = 0; j < GPR_METRIC_MAX; j++) {
        if (j < k) {
            const float gj = rl_f(g, j);
            if (l < k) acc = gpr_axpy(r[j], gj, acc);
        }
    }
    return acc;
}
// log density of a Gaussian proposal with covariance e^2 L L^T at offset r (lanes
// 0..k-1), up to its constant: -|w|^2 / (2 e^2) with w = L^-1 r; |w|^2 is summed in row
// order, then divided once.  The row of Li is read in two halves of 8 columns.
__device__ __forceinline__ double metric_logq(const double *Li, int k, double r, double two_e2) {
#pragma clang fp contract(off)
    const int l = lane_id();
    const double2 *q = (const double2 *)(Li + min(opaque_lane_i32(l), k - 1) * GPR_METRIC_MAX);
    double w = 0.0;
#pragma unroll
    for (int half = 0; half < 2; half++) {
        if (half * 8 >= k) continue;
        double row[8];
#pragma unroll
        for (int j = 0; j < 8; j += 2) {
            double2 v = make_double2(0.0, 0.0);
            if (half * 8 + j < k) v = q[(half * 8 + j) / 2];
            row[j] = v.x;
            row[j + 1] = v.y;
        }
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const int jj = half * 8 + j;
            if (jj < k) {
                const double rj = rl_d(r, jj);
                if (l < k && jj <= l) w = w + row[j] * rj;
            }
        }
    }
    const double w2 = w * w;
    double s = 0.0;
    for (int i = 0; i < k; i++) s += rl_d(w2, i);
    return -s / two_e2;
}

// config accept rule: invalid current always moves; log u < a otherwise.  u lies on the
// grid ((k + 1/2) 2^-23), so log u >= -16.64: any a < -17 rejects without drawing.
// The accept draw of step s is word s & 3 of the ACCEPT block s >> 2, so one Philox
// block serves four consecutive steps: a chain loop keeps the last block it computed.
struct AcceptDraws {
    gpr_u4 w;
    uint32_t blk;
    __device__ __forceinline__ AcceptDraws() : w{0, 0, 0, 0}, blk(0xffffffffu) {}
};
__device__ __forceinline__ bool cfg_accept(uint64_t seed, uint32_t chain, uint32_t step, double cur, double prop,
                                           double a, AcceptDraws &ad) {
    if (!__builtin_isfinite(cur)) return true;
    if (!__builtin_isfinite(prop)) return false;
    if (a >= 0.0) return true;
    if (a < -17.0) return false;
    if ((step >> 2) != ad.blk) {
        ad.w = gpr_step_block(seed, chain, step, GPR_P_ACCEPT, 0, 0);
        ad.blk = step >> 2;
    }
    const float u = gpr_u01(gpr_u4_word(ad.w, (int)(step & 3)));
    return (double)gpr_logf(u) < a;
}
__device__ __forceinline__ bool cfg_accept(uint64_t seed, uint32_t chain, uint32_t step, double cur, double prop,
                                           double a) {
    AcceptDraws ad;
    return cfg_accept(seed, chain, step, cur, prop, a, ad);
}


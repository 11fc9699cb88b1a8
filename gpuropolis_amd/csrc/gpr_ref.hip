// Reference-semantics kernels: the reference's own sampler (MH_simple_kernel,
// main.cu:679-813) on heap-31 programs, with its proposals, quirks and median
// resampling (main.cu:1215-1234), on the GPU.
//
// Draw sources: Philox substreams {chain, step, purpose, slot} (default) or the
// reference's 31-bit LCG seeded block_seed + chain (main.cu:213-216, 691), which
// replays the reference's per-thread draw sequence.  The draw transforms restate
// random_int / random_float / random_normal / random_geometric (main.cu:218-254) and
// the host variants (main.cu:262-284) with the shared spec math.
//
// Two kernels, both one wave per chain: heap in VGPRs (lane = slot), lane-parallel
// heap -> postfix decode of the reachable tree, the shared wave interpreter, per-constant
// proposals in parallel lanes.
//   k_mh_ref_literal  the lane schedule: the reference's likelihood arithmetic (FP64 terms
//                     of every point, main.cu:454-468) and its order of draws; Philox or LCG.
//   k_mh_ref_wave     the wave schedule: FP32 compensated terms with early rejection.
#include <algorithm>

#include "gpr_device.h"

// gpr_logf of the node counts 0 .. 31 (-inf at 0), filled once per device by
// gpr_launch_fill_ref_logint: the wave kernel's -log count terms become scalar loads.
static __device__ float gpr_ref_logint[GPR_REF_SLOTS + 1];
__global__ void k_fill_ref_logint() {
    const int i = (int)threadIdx.x;
    if (i <= GPR_REF_SLOTS) gpr_ref_logint[i] = gpr_logf((float)i);
}
hipError_t gpr_launch_fill_ref_logint(hipStream_t s) {
    hipLaunchKernelGGL(k_fill_ref_logint, dim3(1), dim3(64), 0, s);
    return hipGetLastError();
}

#define R_LOG01_F (-0x1.26bb1cp+1f)        /* logf(PROPOSE_GEOM_R = 0.1f) */
#define R_LOG015_F (-0x1.e5a9a8p+0f)       /* logf(PROPOSE_INT = 0.15f) */
#define R_LOG1M01_D (-0x1.af8e82826b325p-4) /* log(1.0 - 0.1f) */
#define R_LOG1M015_D (-0x1.4cd6ba6a55088p-3)/* log(1.0 - 0.15f) */
#define R_LOG2_D 0x1.62e42fefa39efp-1
#define R_LOG28_D 0x1.aa85ad6964a23p+1    /* log(NOPS + 1) of the default op set */
#define R_LOG2PI_F 0x1.d67f1ep+0f

__device__ __forceinline__ float r_pow10(int order) {  // powf(10, order), order in [-4, 3]
    switch (order) {
    case -4: return 0x1.a36e2ep-14f;
    case -3: return 0x1.0624dep-10f;
    case -2: return 0x1.47ae14p-7f;
    case -1: return 0x1.99999ap-4f;
    case 0: return 1.0f;
    case 1: return 10.0f;
    case 2: return 100.0f;
    default: return 1000.0f;
    }
}

// ---------------------------------------------------------------- draw sources
struct PhiloxSrc {
    gpr_rstream st;
    __device__ __forceinline__ uint32_t rand31() { return st.next() >> 1; }
};

template <class S> __device__ __forceinline__ int r_random_int(int n, S &s) {
    const uint32_t div = (uint32_t)(0x7fffffff / (n + 1));
    int r;
    do { r = (int)(s.rand31() / div); } while (r >= n);
    return r;
}
// random_float of random_int(1000000) = r: the reference divides in double and rounds to
// float; the product with the double 1e-6 rounds to the same float for every one of the
// million values of r (tests/test_gpu_ref_edges.py), in one instruction instead of a division
#define R_FLOAT_N 1000000
#define R_FLOAT_DIV (0x7fffffffu / (R_FLOAT_N + 1))
__device__ __forceinline__ float r_float_of(int r) { return (float)((double)r * 1e-6); }
template <class S> __device__ __forceinline__ float r_random_float(S &s) { return r_float_of(r_random_int(R_FLOAT_N, s)); }
__device__ __forceinline__ float r_box_muller(float u, float v) {
#pragma clang fp contract(off)
    return sqrtf(-2.0f * gpr_logf(u)) * gpr_sin2pi(v);
}
template <class S> __device__ __forceinline__ float r_random_normal(S &s) {
    const float u = r_random_float(s);
    const float v = r_random_float(s);
    return r_box_muller(u, v);
}
__device__ __forceinline__ float r_geometric_of(float u) { return ceilf(gpr_logf(u) / R_LOG01_F); }
template <class S> __device__ __forceinline__ float r_random_geometric(S &s) { return r_geometric_of(r_random_float(s)); }
template <class S> __device__ __forceinline__ int r_host_random_int(int limit, S &s) {
    const uint32_t div = (uint32_t)(0x7fffffff / limit);
    int r;
    do { r = (int)(s.rand31() / div); } while (r > limit - 1);
    return r;
}
template <class S> __device__ __forceinline__ float r_host_random_float(S &s) {
    return (float)s.rand31() / (float)0x7fffffff;
}
template <class S> __device__ __forceinline__ float r_host_random_normal(S &s) {
#pragma clang fp contract(off)
    const float u = r_host_random_float(s);
    const float v = r_host_random_float(s);
    return sqrtf(-2.0f * gpr_logf(u)) * gpr_sin2pi(v);
}

// Orders this wave's LDS accesses before the call against those after it (LDS operations
// of one wave execute in order; this keeps the compiler from moving them).
__device__ __forceinline__ void r_lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// One serial stream of 31-bit words, 64 of them at a time: lane k holds word k of the
// current batch and pos is the next word.  A draw that rejects values (random_int) makes
// the number of words it takes depend on them; take() finds the accepted ones by ballot, so
// that the words go where the serial loop over the stream would put them.
template <class Words>
struct WaveDraws {
    Words src;
    uint32_t raw;   // this lane's word of the batch
    int pos;
    __device__ __forceinline__ void refill() { raw = src.batch(); pos = 0; }
    // the next random_int(N)
    template <int N> __device__ __forceinline__ int next_int() {
        constexpr uint32_t div = 0x7fffffffu / (N + 1);
        int r;
        do {
            if (pos == 64) refill();
            r = (int)((uint32_t)rl_i((int)raw, pos++) / div);
        } while (r >= N);
        return r;
    }
    // buf[0 .. m-1] = the next m values of random_int(n), div = 0x7fffffff / (n + 1); every
    // iteration of the loop consumes the rest of a batch or ends it
    __device__ __forceinline__ void take(int m, int n, uint32_t div, int *buf) {
        const int l = lane_id();
        int got = 0;
        while (got < m) {
            if (pos == 64) refill();
            const int r = (int)(raw / div);
            const uint64_t ok = ballot(l >= pos && r < n);
            const int at = got + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(ok >> 32),
                                                                __builtin_amdgcn_mbcnt_lo((uint32_t)ok, 0u));
            const bool mine = ((ok >> l) & 1ull) != 0 && at < m;
            if (mine) buf[at] = r;
            const uint64_t last = ballot(mine && at == m - 1);
            pos = last ? __builtin_ctzll(last) + 1 : 64;
            got += __popcll(ok);
        }
    }
};

// words of a Philox substream, in order
struct PhiloxWords {
    uint64_t seed;
    uint32_t chain, step, c2, base;
    __device__ __forceinline__ uint32_t batch() {
        const int k = lane_id();
        const gpr_u4 b = gpr_philox(chain, step, c2, 16u * base + (uint32_t)(k >> 2), (uint32_t)seed, (uint32_t)(seed >> 32));
        base++;
        return gpr_u4_word(b, k & 3) >> 1;
    }
};
__device__ __forceinline__ WaveDraws<PhiloxWords> philox_draws(uint64_t seed, uint32_t chain, uint32_t step, uint32_t purpose) {
    return {{seed, chain, step, purpose << 24, 0u}, 0u, 64};
}
// the reference's LCG (main.cu:213-216): lane k jumps k + 1 steps ahead of the batch's
// start, x -> mul x + add (mod 2^31)
struct LcgWords {
    uint32_t x, mul, add;
    __device__ __forceinline__ uint32_t batch() {
        const uint32_t w = (mul * x + add) & 0x7fffffffu;
        x = (uint32_t)rl_i((int)w, 63);
        return w;
    }
};
__device__ __forceinline__ WaveDraws<LcgWords> lcg_draws(uint32_t seed) {
    uint32_t m = 1, c = 0, pm = 1103515245u, pc = 12345u;
    for (int e = lane_id() + 1; e; e >>= 1) {
        if (e & 1) { m *= pm; c = c * pm + pc; }
        pc = pc * pm + pc;
        pm *= pm;
    }
    return {{seed, m, c}, 0u, 64};
}

// ---------------------------------------------------------------- densities (main.cu:299-309)
__device__ __forceinline__ double r_lgeom(float n) {
#pragma clang fp contract(off)
    return (double)((n - 1.0f) * R_LOG01_F) + R_LOG1M01_D;
}
__device__ __forceinline__ double r_lnormal1(float x) {  // lnormalpdf(x, 1)
#pragma clang fp contract(off)
    return -(double)(x * x) / 2.0 - 0.5 * ((double)R_LOG2PI_F + 2.0 * (double)0.0f);
}
__device__ __forceinline__ bool r_is_int(float x) {      // main.cu:192
    if (!__builtin_isfinite(x)) return false;
    return (double)fabsf(x - roundf(x)) < 1.0e-6;
}
__device__ __forceinline__ double r_logplusexp(double a, double b) {  // main.cu:190
#pragma clang fp contract(off)
    const double m = a > b ? a : b;
    return (double)gpr_logf(gpr_expf((float)(a - m)) + gpr_expf((float)(b - m))) + m;
}
__device__ __forceinline__ bool r_valid(double x) { return __builtin_isfinite(x); }

// One constant proposal of the constant step (main.cu:746-785) from its four random_float
// draws: the first decides for the mixture (always: P_PROPOSE_C_GEOMETRIC = 1), the second
// for an integer (PROPOSE_INT), the others make the value.  A proposal does not depend on
// the constant it replaces.  ft: its forward term.
__device__ __forceinline__ float r_const_prop(float f1, float f2, float f3, double &ft) {
#pragma clang fp contract(off)
    if (f1 < 0.15f) {
        const float c = (f2 < 0.5f ? -1.0f : 1.0f) * r_geometric_of(f3) - 1.0f;
        ft = r_lgeom(c + 1.0f) + (c == 0.0f ? 0.0 : R_LOG2_D) + (double)R_LOG015_F;
        return c;
    }
    const float c = 1.0f * r_box_muller(f2, f3);
    ft = r_lnormal1(c / 1.0f) + R_LOG1M015_D;
    return c;
}
// The backward terms of a constant: for a proposal other than 0, and for 0 (main.cu:768-778).
__device__ __forceinline__ void r_const_back(float oldC, double &bt, double &bt0) {
#pragma clang fp contract(off)
    bt = bt0 = r_lnormal1(oldC / 1.0f) + R_LOG1M015_D;
    if (r_is_int(oldC)) {
        const double g = r_lgeom(oldC + 1.0f);
        bt = r_logplusexp(g + R_LOG2_D + (double)R_LOG015_F, bt0);
        bt0 = r_logplusexp(g + 0.0 + (double)R_LOG015_F, bt0);
    }
}
// The four random_float draws of a constant's Philox substream (chain, step, CPROP, slot):
// one block, unless a word is rejected (about 1 in 4400).
__device__ __forceinline__ void r_const_floats(uint64_t seed, uint32_t chain, uint32_t step, uint32_t slot, float (&f)[4]) {
    const gpr_u4 b = gpr_philox(chain, step, ((uint32_t)GPR_P_CPROP << 24) | slot, 0u, (uint32_t)seed, (uint32_t)(seed >> 32));
    const int r0 = (int)((b.x >> 1) / R_FLOAT_DIV), r1 = (int)((b.y >> 1) / R_FLOAT_DIV), r2 = (int)((b.z >> 1) / R_FLOAT_DIV),
              r3 = (int)((b.w >> 1) / R_FLOAT_DIV);
    f[0] = r_float_of(r0); f[1] = r_float_of(r1); f[2] = r_float_of(r2); f[3] = r_float_of(r3);
    if (max(max(r0, r1), max(r2, r3)) >= R_FLOAT_N) {
        PhiloxSrc pc;
        pc.st.init(seed, chain, step, GPR_P_CPROP, slot);
        for (int k = 0; k < 4; k++) f[k] = r_random_float(pc);
    }
}

// Is slot k (0-based) the slot n or one of its descendants (main.cu:660-677)?  Slot numbers
// from 1 shifted right by the difference of their bit lengths.
__device__ __forceinline__ bool r_is_descendant(int n, int k) {
    const int n1 = n + 1, k1 = k + 1, d = __builtin_clz(n1) - __builtin_clz(k1);
    return d >= 0 && (k1 >> d) == n1;
}

// reference op code -> postfix op code (A, B: -1, pass-through)
__device__ __forceinline__ int r_to_tape(int o) {
    switch (o) {
    case GPR_REF_ONE: return GPR_OP_ONE;
    case GPR_REF_CONST: return GPR_OP_CONST;
    case GPR_REF_INV: return GPR_OP_INV;
    case GPR_REF_PLUS: return GPR_OP_ADD;
    case GPR_REF_MINUS: return GPR_OP_SUB;
    case GPR_REF_RMINUS: return GPR_OP_RSUB;
    case GPR_REF_CPLUS: return GPR_OP_CADD;
    case GPR_REF_TIMES: return GPR_OP_MUL;
    case GPR_REF_CTIMES: return GPR_OP_CMUL;
    case GPR_REF_DIV: return GPR_OP_DIV;
    case GPR_REF_RDIV: return GPR_OP_RDIV;
    case GPR_REF_LOG: return GPR_OP_LOG;
    case GPR_REF_EXP: return GPR_OP_EXP;
    case GPR_REF_POW: return GPR_OP_POW;
    case GPR_REF_CPOW: return GPR_OP_CPOW;
    case GPR_REF_RPOW: return GPR_OP_RPOW;
    case GPR_REF_CRPOW: return GPR_OP_CRPOW;
    case GPR_REF_SQRT: return GPR_OP_SQRT;
    case GPR_REF_SIN: return GPR_OP_SIN;
    case GPR_REF_ASIN: return GPR_OP_ASIN;
    case GPR_REF_COS: return GPR_OP_COS;
    case GPR_REF_ACOS: return GPR_OP_ACOS;
    case GPR_REF_TAN: return GPR_OP_TAN;
    case GPR_REF_ATAN: return GPR_OP_ATAN;
    case GPR_REF_ABS: return GPR_OP_ABS;
    case GPR_REF_HALF: return GPR_OP_CMUL;     // a/2.0 in double, then float == 0.5f * a
    default: return gpr_ref_is_physical(o) ? GPR_OP_CONST : -1;
    }
}
// the constant a token of heap op o carries: its heap constant, a physical constant's
// value, or the factor of halving
__device__ __forceinline__ float r_tape_const(int o, float hc) {
    return gpr_ref_is_physical(o) ? gpr_ref_physical_value(o) : (o == GPR_REF_HALF ? 0.5f : hc);
}

// ---------------------------------------------------------------- heap decode
__device__ __forceinline__ int r_len_kind(int o) {  // 0 leaf, 1 A, 2 B, 3 unary, 4 C-op, 5 binary
    if (gpr_ref_is_physical(o)) return 0;              // PHYSICAL_CONSTANT_LENGTH_PRIOR = 1
    switch (o) {
    case GPR_REF_ONE: case GPR_REF_CONST: return 0;
    case GPR_REF_A: return 1;
    case GPR_REF_B: return 2;
    case GPR_REF_CPLUS: case GPR_REF_CTIMES: case GPR_REF_CPOW: case GPR_REF_CRPOW: return 4;
    case GPR_REF_PLUS: case GPR_REF_MINUS: case GPR_REF_RMINUS: case GPR_REF_TIMES: case GPR_REF_DIV:
    case GPR_REF_RDIV: case GPR_REF_POW: case GPR_REF_RPOW: return 5;
    default: return 3;
    }
}
// Lane-parallel decode of the heap held one slot per lane (lane i = slot i+1, i < 31)
// into the postfix tape of the reachable tree, one token per lane.  Subtree token
// counts are folded bottom-up and start positions pushed top-down, level by level;
// every emitted token (the op last in its subtree, x leaves below slots 16..31) is
// scattered to its lane with ds_permute.
struct RefTape {
    WaveProg p;     // ops and constants of the tape, o0/c0 per lane
    int slot;       // heap slot of each token (255 for x)
    int src;        // heap slot whose constant the token carries, or -1: its constant does
                    // not change with the heap's (none, a physical constant, halving's 0.5)
    int count;      // reachable non-pass-through ops: count_nodes (main.cu:604-608)
    int dl;         // description length: tokens + C-op tokens (dispatch_length fold)
};

__device__ RefTape r_decode_wave(int hop, float hc) {
    const int l = lane_id();
    const int s = l + 1;                                // 1-based slot
    const bool live = l < GPR_REF_SLOTS;
    const int k = live ? r_len_kind(hop) : 0;           // 0 leaf 1 A 2 B 3 unary 4 C-op 5 binary
    const bool bottom = s >= 16;                        // children are x leaves
    // subtree token counts, bottom-up (5 levels)
    // children of bottom slots are x leaves: they read lane 63, which always holds 1
    const int li = bottom ? 63 : 2 * s - 1, ri = bottom ? 63 : 2 * s;
    int size = 1;
#pragma unroll
    for (int it = 0; it < 5; it++) {
        const int lc = shfl_all(size, li);
        const int rc = shfl_all(size, ri);
        switch (k) {
        case 0: size = 1; break;
        case 1: size = lc; break;
        case 2: size = rc; break;
        case 3: case 4: size = 1 + lc; break;
        default: size = 1 + lc + rc; break;
        }
    }
    // start positions and reachability, top-down (4 levels below the root)
    int start = 0, reach = s == 1 ? 1 : 0;
#pragma unroll
    for (int it = 0; it < 4; it++) {
        const int par = (s >> 1) - 1;                   // parent lane
        const int pk = shfl_all(k, par & 63), ps = shfl_all(start, par & 63), pr = shfl_all(reach, par & 63);
        const int sib = shfl_all(size, (s - 2) & 63);   // left sibling size (for right children)
        if (s >= 2 && live) {
            const bool left = (s & 1) == 0;
            int r = 0, st = 0;
            if (pk == 1) { r = left; st = ps; }
            else if (pk == 2) { r = !left; st = ps; }
            else if (pk == 3 || pk == 4) { r = left; st = ps; }
            else if (pk == 5) { r = 1; st = left ? ps : ps + sib; }
            reach = pr && r;
            start = st;
        }
    }
    const int len = rl_i(size, 0);
    // scatter: op token at start + size - 1; x leaves below bottom slots
    const int top = r_to_tape(hop);
    const bool emit_op = live && reach && k != 1 && k != 2;
    const int v_op = emit_op ? (((top + 1) << 8) | (s - 1)) : 0;
    const int t_op = emit_op ? start + size - 1 : 63;
    const bool x1 = live && reach && bottom && k != 0;                // first x child
    const bool x2 = live && reach && bottom && k == 5;                // second x child
    const int v_x = (GPR_OP_X + 1) << 8 | 255;
    int t1 = __builtin_amdgcn_ds_permute(t_op * 4, v_op);
    int t2 = __builtin_amdgcn_ds_permute((x1 ? start : 63) * 4, x1 ? v_x : 0);
    int t3 = __builtin_amdgcn_ds_permute((x2 ? start + 1 : 63) * 4, x2 ? v_x : 0);
    __asm__ volatile("" : "+v"(t1), "+v"(t2), "+v"(t3));
    const int tok = t1 | t2 | t3;
    RefTape rt;
    const bool valid = l < len;
    rt.p.len = len;
    rt.p.o0 = valid ? (tok >> 8) - 1 : 0;
    rt.slot = valid ? (tok & 255) : 255;
    rt.p.o1 = 0;
    rt.p.c1 = 0.0f;
    const float cs = shfl_all(r_tape_const(hop, hc), rt.slot & 31);
    const int ho = shfl_all(hop, rt.slot & 31);
    const bool holds = valid && gpr_has_const(rt.p.o0);
    rt.p.c0 = holds ? cs : 0.0f;
    rt.src = holds && !gpr_ref_is_physical(ho) && ho != GPR_REF_HALF ? rt.slot : -1;
    rt.count = len - __popcll(ballot(valid && rt.p.o0 == GPR_OP_X));
    // description length: tokens plus the C-op tokens (dispatch_length kind 4; halving is
    // a c* token of length 1 + a)
    const int tk = shfl_all(k, rt.slot & 31);
    rt.dl = len + __popcll(ballot(valid && tk == 4));
    return rt;
}

// the tape with other heap constants: slot c's at lane base + c of v
__device__ __forceinline__ float r_tape_consts(const RefTape &rt, float v, int base) {
    const float cv = shfl_all(v, base + max(rt.src, 0));
    return rt.src >= 0 ? cv : rt.p.c0;
}

// ---------------------------------------------------------------- serial sums
// The prior and the proposal densities add 31 terms each in slot order (FP64, the order is
// part of the result).  A sum by lane reads costs two readlanes and an add per term; here
// the terms go through LDS, S[row][slot] with 32 doubles a row, and one lane does one
// serial sum, so that the sums of a step (or of the four constant steps between two structure
// moves) share every instruction.  Only the lanes that sum may be active: with the other
// lanes reading along (one address for all of them) the LDS took about 80 cycles an
// instruction, and a block of the batch of NIST sizes 7.4 ms instead of 3.9.
#define R_ROW 32
__device__ __forceinline__ double r_add_row(const double *row, double acc) {
#pragma clang fp contract(off)
#pragma unroll
    for (int c = 0; c < 24; c += 8) {
        double v[8];
#pragma unroll
        for (int k = 0; k < 8; k++) v[k] = row[c + k];
#pragma unroll
        for (int k = 0; k < 8; k++) acc += v[k];
    }
    double v[7];
#pragma unroll
    for (int k = 0; k < 7; k++) v[k] = row[24 + k];
#pragma unroll
    for (int k = 0; k < 7; k++) acc += v[k];
    return acc;
}
__device__ __forceinline__ double r_prior_start(int dl, double lnops) {
#pragma clang fp contract(off)
    return -(double)(1.0f * (float)dl) * lnops;
}
// prior: -length*log(NOPS+1) + sum over all 31 constants in slot order (main.cu:529-544);
// lc: slot c's term at lane c.
__device__ __forceinline__ double r_prior_wave(int dl, double lc, double lnops, double *S) {
    r_lds_order();
    if (lane_id() < R_ROW) S[lane_id()] = lc;
    r_lds_order();
    double acc = r_prior_start(dl, lnops);
    if (lane_id() == 0) acc = r_add_row(S, acc);
    return rl_d(acc, 0);
}

// LDS of one wave: the interpreter's stack for programs of depth at most 6 (heap-31 programs
// are trees of at most five levels; levels -2 .. 3 of wave_eval_ls), then the sums' rows
// and results (the random_int buffers of a structure move share the rows)
#define R_LEVELS 6
#define R_SUM_ROWS 12
#define R_SUM_DOUBLES (R_SUM_ROWS * R_ROW + 12)
__host__ __device__ constexpr size_t r_lds_floats(int kc) { return (size_t)R_LEVELS * 64 * kc + 2 * R_SUM_DOUBLES; }
extern __shared__ float r_lds[];

// The structure move's new ops (main.cu:717-730): a node drawn from the slots (the root when
// the current state is invalid), then a new op for it and each of its descendants in slot order.
template <class D>
__device__ __forceinline__ int r_struct_draw(D &dr, bool valid, int hop, int opset, int nops, int *buf) {
    const int l = lane_id();
    const int nn = valid ? dr.template next_int<GPR_REF_SLOTS>() : 0;
    const bool desc = l < GPR_REF_SLOTS && r_is_descendant(nn, l);
    const uint64_t dm = ballot(desc);
    r_lds_order();
    dr.take(__popcll(dm), nops, (uint32_t)(0x7fffffff / (nops + 1)), buf);
    r_lds_order();
    const int k = (int)__builtin_amdgcn_mbcnt_lo((uint32_t)dm, 0u);   // slots lie in the low lanes
    return desc ? gpr_opset_code(opset, buf[min(k, GPR_REF_SLOTS)]) : hop;
}

// ---------------------------------------------------------------- lane schedule
// Likelihood as main.cu:454-468: per point an FP64 term -(f - y)^2 / (2 sd^2) - lnc with the
// float square, -inf as soon as a value or a term is not finite.  Lanes compute their
// points' terms; the sum runs over them in point order, as the reference adds them (a
// program with an LL near -1e22 is accepted or not by the last bit of it), through the 64
// doubles of S.
template <int KC>
__device__ __forceinline__ double r_loglik64(const WaveProg &p, const ProgCode &m, float *ls, double *S, const float *x,
                                             const float *y, const float *sd, const double *lnc, int n) {
#pragma clang fp contract(off)
    const int l = lane_id();
    double s = 0.0;
    for (int base = 0; base < n; base += 64 * KC) {
        float xs[KC], T[KC];
#pragma unroll
        for (int k = 0; k < KC; k++) {
            const int i = base + 64 * k + l;
            xs[k] = i < n ? x[i] : 0.0f;
        }
        wave_eval_ls<KC, false>(p, xs, T, ls, m);
#pragma unroll
        for (int k = 0; k < KC; k++) {
            const int i = base + 64 * k + l, left = n - (base + 64 * k);
            if (left <= 0) break;
            double t = 0.0;              // adding +0 past the last point changes nothing
            if (i < n) {
                const float r = T[k] - y[i];
                const double e = (double)sd[i];
                t = __builtin_isfinite(T[k]) ? -(double)(r * r) / (2.0 * e * e) - lnc[i] : -GPR_INF;
            }
            r_lds_order();
            S[l] = t;
            r_lds_order();
            if (l == 0) for (int c = 0; c < min(left, 64); c += 8) {
                double v[8];
#pragma unroll
                for (int q = 0; q < 8; q++) v[q] = S[c + q];
#pragma unroll
                for (int q = 0; q < 8; q++) s += v[q];
            }
        }
    }
    s = rl_d(s, 0);
    return __builtin_isfinite(s) ? s : -GPR_INF;
}

// One wave per chain, one wave per workgroup, chains blockIdx.x, blockIdx.x + gridDim.x, ...
// The draws of a step depend on the step before it (a rejected value and the accept test
// take a varying number of LCG words), so steps are serial and only the work inside a step
// is spread over the lanes: 64 words of the stream at once, a constant per lane, a point per
// lane, the three serial sums in three lanes.  Bound by the latency of that chain at the
// command line's default of 1024 chains (four waves per CU).  One lane per chain, folding
// all 31 slots at every point with every lane's own ops, took 4600 us a step on 37 points
// at 1024 chains; this takes 11.
template <int KC, int RNG>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4))) k_mh_ref_literal(GprMHArgs a) {
    const uint32_t step0 = a.clock ? a.clock[0] : a.step0;
    const int nops = gpr_opset_nops(a.opset);
    const int l = lane_id();
    const int N = a.nchains;
    const bool live = l < GPR_REF_SLOTS;
    float *ls = r_lds;
    double *S = (double *)(r_lds + R_LEVELS * 64 * KC);
    int *buf = (int *)S;
    unsigned long long n_sprop = 0, n_sacc = 0, n_cprop = 0, n_cacc = 0, n_steps = 0, n_evals = 0;
    for (int ch = (int)blockIdx.x; ch < N; ch += (int)gridDim.x) {
        const uint32_t chain = (uint32_t)ch;
        int di = 0;
        while (a.ds[di].chain0 + a.ds[di].nchains <= ch) di++;
        const int n = a.ds[di].n, off = a.ds[di].off;
        const float *x = a.dx + off, *y = a.dy + off, *sdv = a.dsd + off;
        const double *lc = a.lnc + off;
        int hop = live ? a.ops[(size_t)l * N + chain] : 0;
        float hc = live ? a.cs[(size_t)l * N + chain] : 0.0f;
        RefTape cur = r_decode_wave(hop, hc);
        ProgCode cm = prog_code<KC, false>(cur.p);
        double cur_prior = r_prior_wave(cur.dl, gpr_lcauchy(hc), a.ref_lnops, S);
        double cur_ll = r_loglik64<KC>(cur.p, cm, ls, S, x, y, sdv, lc, n);
        double cur_post = cur_prior + cur_ll;
        double bt, bt0;
        r_const_back(hc, bt, bt0);
        WaveDraws<LcgWords> lcg = lcg_draws((uint32_t)a.block_seed + chain);
        double forward = 0.0, backward = 0.0;
        int phase = 0;
        for (int mcmci = 0; mcmci < a.steps; mcmci++) {
            const uint32_t step = step0 + (uint32_t)mcmci;
            int php = hop;
            float phc = hc;
            RefTape prop = cur;
            ProgCode pm = cm;
            double pp;
            const bool structural = phase == 0;
            phase = phase == 4 ? 0 : phase + 1;
            if (structural) {
                n_sprop++;
                forward = -(double)gpr_ref_logint[cur.count];
                if (RNG == GPR_RNG_LCG) {
                    php = r_struct_draw(lcg, r_valid(cur_post), hop, a.opset, nops, buf);
                } else {
                    WaveDraws<PhiloxWords> ph = philox_draws(a.seed, chain, step, GPR_P_STRUCT);
                    php = r_struct_draw(ph, r_valid(cur_post), hop, a.opset, nops, buf);
                }
                prop = r_decode_wave(php, hc);
                pm = prog_code<KC, false>(prop.p);
                backward = -(double)gpr_ref_logint[prop.count];
                pp = r_prior_wave(prop.dl, gpr_lcauchy(hc), a.ref_lnops, S);
            } else {
                n_cprop++;
                float f[4];
                if (RNG == GPR_RNG_LCG) {
                    r_lds_order();
                    lcg.take(4 * GPR_REF_SLOTS, R_FLOAT_N, R_FLOAT_DIV, buf);
                    r_lds_order();
#pragma unroll
                    for (int k = 0; k < 4; k++) f[k] = r_float_of(buf[min(4 * l, 4 * GPR_REF_SLOTS) + k]);
                } else {
                    r_const_floats(a.seed, chain, step, (uint32_t)(l & 31), f);
                }
                double ft;
                phc = r_const_prop(f[1], f[2], f[3], ft);
                if (!live) phc = 0.0f;
                // rows: prior, forward, backward; lane q sums row q
                r_lds_order();
                if (l < R_ROW) {
                    S[l] = gpr_lcauchy(phc);
                    S[R_ROW + l] = ft;
                    S[2 * R_ROW + l] = phc == 0.0f ? bt0 : bt;
                }
                r_lds_order();
                double acc = l == 0 ? r_prior_start(cur.dl, a.ref_lnops) : (l == 1 ? forward : backward);
                if (l < 3) acc = r_add_row(S + l * R_ROW, acc);
                pp = rl_d(acc, 0);
                forward = rl_d(acc, 1);
                backward = rl_d(acc, 2);
                prop.p.c0 = r_tape_consts(cur, phc, 0);
            }
            const double pl = r_loglik64<KC>(prop.p, pm, ls, S, x, y, sdv, lc, n);
            const double ppost = pp + pl;
            const double acc = ppost - cur_post + backward - forward;
            bool ok = !r_valid(cur_post);
            if (r_valid(ppost)) {
                if (acc > 0.0) {
                    ok = true;
                } else {
                    float u;
                    if (RNG == GPR_RNG_LCG) {
                        u = r_float_of(lcg.next_int<R_FLOAT_N>());
                    } else {
                        PhiloxSrc pa;
                        pa.st.init(a.seed, chain, step, GPR_P_ACCEPT, 0);
                        u = r_random_float(pa);
                    }
                    ok = ok || u < gpr_expf((float)acc);
                }
            }
            if (uni(ok)) {
                cur_post = ppost; cur_ll = pl; cur_prior = pp;
                hop = php; hc = phc; cur = prop; cm = pm;
                if (structural) n_sacc++;
                else { n_cacc++; r_const_back(hc, bt, bt0); }
            }
        }
        n_steps += (unsigned long long)a.steps;
        n_evals += (unsigned long long)a.steps * (unsigned long long)(GPR_REF_SLOTS * n);
        if (live) { a.ops[(size_t)l * N + chain] = (uint8_t)hop; a.cs[(size_t)l * N + chain] = hc; }
        if (l == 0) { a.prior[chain] = cur_prior; a.ll[chain] = cur_ll; }
    }
    if (l == 0 && a.counters) {
        atomicAdd(&a.counters[GPR_CNT_SPROP], n_sprop);
        atomicAdd(&a.counters[GPR_CNT_SACC], n_sacc);
        atomicAdd(&a.counters[GPR_CNT_CPROP], n_cprop);
        atomicAdd(&a.counters[GPR_CNT_CACC], n_cacc);
        atomicAdd(&a.counters[GPR_CNT_STEPS], n_steps);
        atomicAdd(&a.counters[GPR_CNT_EVALS], n_evals);
    }
}

// kc: points per lane per pass of the interpreter, 1 or 4 (the largest dataset's: a pass
// over at most 64 points with four per lane would interpret three empty ones)
hipError_t gpr_launch_mh_ref_lane(const GprMHArgs &a, int kc, hipStream_t s) {
    // a bounded grid: 64 lanes per chain would pass the 2^32 threads of a launch
    const dim3 grid(std::min(a.nchains, 1 << 20));
    const bool lcg = a.rng == GPR_RNG_LCG;
#define R_L(K, R) hipLaunchKernelGGL((k_mh_ref_literal<K, R>), grid, dim3(64), sizeof(float) * r_lds_floats(K), s, a)
    if (kc == 1) { if (lcg) R_L(1, GPR_RNG_LCG); else R_L(1, GPR_RNG_PHILOX); }
    else { if (lcg) R_L(4, GPR_RNG_LCG); else R_L(4, GPR_RNG_PHILOX); }
#undef R_L
    return hipGetLastError();
}

// ---------------------------------------------------------------- wave schedule
// One wave per chain, persistent over the tiles of a size class.  Bound by instruction
// issue.  A constant proposal does not depend on the constants it replaces, so the moves of
// the (up to four) constant steps between two structure steps are drawn together: a lane per
// constant and step (two steps a pass), the accept draws of all five steps in one Philox
// evaluation, and the steps' priors and running forward and backward sums by six lanes side
// by side.  Only the backward terms depend on the current constants; they are computed when
// those change (two per constant: for a proposal of 0 and for any other) and summed again
// for the steps that are left.  16384 chains x 100 steps: 2.9 ms at n = 20 and 4.1 at 236,
// where one step at a time, its sums by lane reads and the value stack in indexed registers
// took 4.4 and 7.6 (VALU instructions per chain-step halved).  Four waves per SIMD: the
// compiler takes 140 VGPRs (three waves) when left alone.
template <int KC>
__global__ void __launch_bounds__(GPR_WG) __attribute__((amdgpu_waves_per_eu(4))) k_mh_ref_wave(GprMHArgs a) {
    const uint32_t step0 = a.clock ? a.clock[0] : a.step0;
    const int nops = gpr_opset_nops(a.opset);
    const int wave = uni((int)(threadIdx.x >> 6));
    const int l = lane_id();
    const int N = a.nchains;
    const int slot = l & 31, half = l >> 5;
    float *ls = r_lds + (size_t)wave * r_lds_floats(KC);
    double *S = (double *)(ls + R_LEVELS * 64 * KC), *R = S + R_SUM_ROWS * R_ROW;
    unsigned long long n_sprop = 0, n_sacc = 0, n_cprop = 0, n_cacc = 0, n_evals = 0, n_steps = 0, n_flops = 0;
    for (;;) {
        __shared__ int s_tile;
        if (threadIdx.x == 0) s_tile = atomicAdd(a.tile_counter, 1);
        __syncthreads();
        const int tile_idx = uni(s_tile);
        __syncthreads();
        if (tile_idx >= a.ntiles) break;
        const GprTile tile = a.tiles[tile_idx];
        if (wave >= tile.count) continue;
        const GprDataset d = uni_dataset(a.ds[uni(tile.dataset)]);
        const uint32_t chain = (uint32_t)uni(tile.chain0 + wave);
        const float *dx = a.dx + d.off, *dy = a.dy + d.off, *dw = a.dw + d.off;
        const int nchunks = (d.n + 64 * KC - 1) / (64 * KC);
        Chunk<KC> c0;
        c0.load(dx, dy, dw, d.n, 0);
        // slot c's constant sits at lanes c and 32 + c
        const bool live = slot < GPR_REF_SLOTS;
        int hop = l < GPR_REF_SLOTS ? a.ops[(size_t)l * N + chain] : 0;
        float hc = live ? a.cs[(size_t)slot * N + chain] : 0.0f;
        RefTape cur = r_decode_wave(hop, hc);
        ProgCode cm = prog_code<KC, false>(cur.p);
        int opq, nconst;
        prog_counts<false>(cur.p, opq, nconst);
        double cur_prior = r_prior_wave(cur.dl, gpr_lcauchy(hc), a.ref_lnops, S);
        double cur_ll = wave_loglik<KC, false>(cur.p, d, dx, dy, dw, c0, nchunks, ls, cm);
        double cur_post = cur_prior + cur_ll;
        double bt, bt0;
        r_const_back(hc, bt, bt0);
        double forward = 0.0, backward = 0.0;
        float pc[2] = {0.0f, 0.0f};   // proposals of constant steps 0, 1 (halves) and 2, 3
        double sums = 0.0;            // lane u, 4 + u, 8 + u: prior, forward, backward of constant step u
        float au = 0.0f, alu = 0.0f;  // lane u: accept draw of step u of the five, and its log
        int phase = 0;
        for (int mcmci = 0; mcmci < a.steps; mcmci++) {
            const uint32_t step = step0 + (uint32_t)mcmci;
            int php = hop;
            RefTape prop = cur;
            ProgCode pm = cm;
            double pp;
            int p_opq = opq, p_nconst = nconst;
            const int ph5 = phase;
            const bool structural = ph5 == 0;
            phase = phase == 4 ? 0 : phase + 1;
            if (structural) {
                n_sprop++;
                forward = -(double)gpr_ref_logint[cur.count];
                WaveDraws<PhiloxWords> ph = philox_draws(a.seed, chain, step, GPR_P_STRUCT);
                php = r_struct_draw(ph, r_valid(cur_post), hop, a.opset, nops, (int *)S);
                prop = r_decode_wave(php, hc);
                pm = prog_code<KC, false>(prop.p);
                prog_counts<false>(prop.p, p_opq, p_nconst);
                backward = -(double)gpr_ref_logint[prop.count];
                pp = r_prior_wave(prop.dl, gpr_lcauchy(hc), a.ref_lnops, S);
                // the accept draw of step u is the first random_float of its ACCEPT substream
                {
                    const uint32_t st = step + (uint32_t)min(l, 4);
                    int r = (int)((gpr_first(a.seed, chain, st, GPR_P_ACCEPT, 0) >> 1) / R_FLOAT_DIV);
                    if (r >= R_FLOAT_N) {
                        PhiloxSrc pa;
                        pa.st.init(a.seed, chain, st, GPR_P_ACCEPT, 0);
                        r = r_random_int(R_FLOAT_N, pa);
                    }
                    au = r_float_of(r);
                    alu = gpr_logf(au);
                }
            } else {
                n_cprop++;
                const int u = ph5 - 1;
                if (u == 0) {
                    // every constant step up to the next structure step or the block's end
                    const int nw = min(4, a.steps - mcmci);
                    r_lds_order();
#pragma unroll
                    for (int p = 0; p < 2; p++) {
                        if (2 * p >= nw) break;
                        const int v = 2 * p + half;
                        float f[4];
                        r_const_floats(a.seed, chain, step + (uint32_t)v, (uint32_t)slot, f);
                        double ft;
                        pc[p] = r_const_prop(f[1], f[2], f[3], ft);
                        S[v * R_ROW + slot] = gpr_lcauchy(pc[p]);
                        S[(4 + v) * R_ROW + slot] = ft;
                        S[(8 + v) * R_ROW + slot] = pc[p] == 0.0f ? bt0 : bt;
                    }
                    r_lds_order();
                    // lanes 0-3: the steps' priors; lane 4: forward, lane 5: backward, running
                    // over the steps
                    double acc = l < 4 ? r_prior_start(cur.dl, a.ref_lnops) : (l == 4 ? forward : backward);
                    if (l < 6) {
                        for (int v = 0; v < nw; v++) {
                            acc = r_add_row(S + (l < 4 ? l : (l == 4 ? 4 + v : 8 + v)) * R_ROW, acc);
                            if (l >= 4) R[(l - 3) * 4 + v] = acc;
                            else if (v == 0) R[l] = acc;
                        }
                    }
                    r_lds_order();
                    if (l < 12) sums = R[l];
                }
                pp = rl_d(sums, u);
                forward = rl_d(sums, 4 + u);
                backward = rl_d(sums, 8 + u);
                prop.p.c0 = r_tape_consts(cur, (u & 2) ? pc[1] : pc[0], (u & 1) * 32);
            }
            // A valid current state accepts only if acc > 0 or u < expf(acc), and either needs
            // acc >= log u - 1 (u > 0) or acc >= -105 (u = 0: expf(acc) underflows to 0 below
            // -103.98).  That bounds the proposal's LL from below: the evaluation stops once
            // its partial sum proves the LL under the bound (wave_loglik), and the proposal is
            // rejected as it would be after the full sum.
            const float u01 = rl_f(au, ph5);
            double reject_below = -GPR_INF;
            if (r_valid(cur_post)) {
                const double amin = u01 > 0.0f ? (double)rl_f(alu, ph5) - 1.0 : -105.0;
                if (r_valid(pp) && r_valid(forward) && r_valid(backward))
                    reject_below = cur_post - backward + forward - pp + amin -
                                   1e-12 * (__builtin_fabs(cur_post) + __builtin_fabs(backward) +
                                            __builtin_fabs(forward) + __builtin_fabs(pp));
            }
            int pts = d.n;
            const double pl = wave_loglik<KC, false>(prop.p, d, dx, dy, dw, c0, nchunks, ls, pm, reject_below, &pts);
            pts = min(pts, d.n);
            n_evals += (unsigned long long)prop.p.len * (unsigned long long)pts;
            n_flops += (unsigned long long)p_opq * (unsigned long long)pts + (unsigned long long)p_nconst;
            const double ppost = pp + pl;
            const double acc = ppost - cur_post + backward - forward;
            if ((r_valid(ppost) && (acc > 0.0 || u01 < gpr_expf((float)acc))) || !r_valid(cur_post)) {
                cur_post = ppost; cur_ll = pl; cur_prior = pp;
                cur = prop;
                if (structural) {
                    n_sacc++;
                    hop = php;
                    cm = pm;
                    opq = p_opq;
                    nconst = p_nconst;
                } else {
                    n_cacc++;
                    const int u = ph5 - 1, nw = min(4, a.steps - (mcmci - u));
                    hc = shfl_all((u & 2) ? pc[1] : pc[0], (u & 1) * 32 + slot);
                    if (!live) hc = 0.0f;
                    r_const_back(hc, bt, bt0);
                    if (u + 1 < nw) {
                        // backward terms and sums of the steps that are left
                        r_lds_order();
#pragma unroll
                        for (int p = 0; p < 2; p++)
                            if (2 * p + half > u) S[(8 + 2 * p + half) * R_ROW + slot] = pc[p] == 0.0f ? bt0 : bt;
                        r_lds_order();
                        if (l == 0) {
                            double back = backward;
                            for (int v = u + 1; v < nw; v++) R[8 + v] = back = r_add_row(S + (8 + v) * R_ROW, back);
                        }
                        r_lds_order();
                        if (l < 12) sums = R[l];
                    }
                }
            }
        }
        n_steps += (unsigned long long)a.steps;
        if (l < GPR_REF_SLOTS) { a.ops[(size_t)l * N + chain] = (uint8_t)hop; a.cs[(size_t)l * N + chain] = hc; }
        if (l == 0) { a.prior[chain] = cur_prior; a.ll[chain] = cur_ll; }
    }
    if (l == 0 && a.counters) {
        atomicAdd(&a.counters[GPR_CNT_SPROP], n_sprop);
        atomicAdd(&a.counters[GPR_CNT_SACC], n_sacc);
        atomicAdd(&a.counters[GPR_CNT_CPROP], n_cprop);
        atomicAdd(&a.counters[GPR_CNT_CACC], n_cacc);
        atomicAdd(&a.counters[GPR_CNT_EVALS], n_evals);
        atomicAdd(&a.counters[GPR_CNT_STEPS], n_steps);
        atomicAdd(&a.counters[GPR_CNT_FLOPS], n_flops);
    }
}

hipError_t gpr_launch_mh_ref_wave(const GprMHArgs &a, int kc, int grid, hipStream_t s) {
    const dim3 wg(64 * a.wpg);
    const size_t sh = sizeof(float) * r_lds_floats(kc) * (size_t)a.wpg;
    if (kc == 1) hipLaunchKernelGGL((k_mh_ref_wave<1>), dim3(grid), wg, sh, s, a);
    else if (kc == 2) hipLaunchKernelGGL((k_mh_ref_wave<2>), dim3(grid), wg, sh, s, a);
    else hipLaunchKernelGGL((k_mh_ref_wave<4>), dim3(grid), wg, sh, s, a);
    return hipGetLastError();
}

// ---------------------------------------------------------------- init and median resampling
// initial draw (main.cu:1133-1137): 31 ops ~ U{0..NOPS-2}, then 31 constants
// 10^U{-4..3} N(0,1), host transforms, stream (chain, step, purpose, 0)
// The op set is a template parameter: the draw sees a constant table row.
// Word k of the stream, halved as rand31 does.
struct WordSrc {
    uint32_t chain, step, purpose, klo, khi, k;
    __device__ __forceinline__ uint32_t at(uint32_t i) const {
        return gpr_u4_word(gpr_philox(chain, step, purpose << 24, i >> 2, klo, khi), (int)(i & 3)) >> 1;
    }
    __device__ __forceinline__ uint32_t rand31() { return at(k++); }
};
template <int SET>
__device__ __forceinline__ void r_draw_serial(WordSrc s, uint8_t *ops, float *cs, int stride) {
#pragma clang fp contract(off)
    for (int i = 0; i < GPR_REF_SLOTS; i++)
        ops[i * stride] = (uint8_t)gpr_opset_code(SET, r_host_random_int(gpr_opset_nops(SET) - 1, s));
    for (int i = 0; i < GPR_REF_SLOTS; i++) {
        const int order = r_host_random_int(8, s) - 4;
        cs[i * stride] = 1.0f * r_pow10(order) * r_host_random_normal(s);
    }
}

// The draws of the chains of one workgroup (32 of them, from c0 on; those in `who`).  Drawn by
// one thread a chain waits for 31 Philox blocks and 31 normals in a row (1024 chains drawn in 50
// us with the call; 20 us this way).  Here
// a half wave draws a chain, a slot per lane: unless one of the 62 integer draws is
// rejected, op i takes word i of the stream and constant i the words 31 + 3 i .. 33 + 3 i.
// After a rejection (some 3e-7 of chains) the words move, and one lane draws in order.  The
// tapes are staged in LDS so that the state's rows are written 32 chains at a time.
#define R_DRAW_WG 512
#define R_DRAW_CHAINS 32
#define R_DRAW_STRIDE (R_DRAW_CHAINS + 1)
template <int SET>
__device__ void r_draw_chains(uint64_t seed, int c0, uint32_t who, uint32_t step, uint32_t purpose, uint8_t *ops,
                              float *cs, int N) {
#pragma clang fp contract(off)
    __shared__ float lc[GPR_REF_SLOTS * R_DRAW_STRIDE];
    __shared__ uint8_t lo[GPR_REF_SLOTS * R_DRAW_STRIDE];
    const int i = threadIdx.x & 31;
    const uint32_t klo = (uint32_t)uni((int)(uint32_t)seed), khi = (uint32_t)uni((int)(uint32_t)(seed >> 32));
    for (int p = 0; p < R_DRAW_CHAINS / (R_DRAW_WG / 32); p++) {
        const int h = p * (R_DRAW_WG / 32) + (int)(threadIdx.x >> 5);
        const bool drawn = (who >> h) & 1u;
        const WordSrc src{(uint32_t)(c0 + h), step, purpose, klo, khi, 0u};
        const uint32_t NOPS = (uint32_t)gpr_opset_nops(SET) - 1, ODIV = 0x7fffffffu / NOPS, EDIV = 0x7fffffffu / 8u;
        const int slot = min(i, GPR_REF_SLOTS - 1);
        const uint32_t op = src.at((uint32_t)slot) / ODIV, e = src.at((uint32_t)(GPR_REF_SLOTS + 3 * slot)) / EDIV;
        const float u = (float)src.at((uint32_t)(GPR_REF_SLOTS + 3 * slot + 1)) / (float)0x7fffffff;
        const float v = (float)src.at((uint32_t)(GPR_REF_SLOTS + 3 * slot + 2)) / (float)0x7fffffff;
        const uint64_t rejected = ballot(op >= NOPS || e >= 8u);
        if (((uint32_t)(rejected >> (threadIdx.x & 32))) == 0) {
            if (drawn && i < GPR_REF_SLOTS) {
                lo[i * R_DRAW_STRIDE + h] = (uint8_t)gpr_opset_code(SET, (int)op);
                lc[i * R_DRAW_STRIDE + h] = 1.0f * r_pow10((int)e - 4) * (sqrtf(-2.0f * gpr_logf(u)) * gpr_sin2pi(v));
            }
        } else if (drawn && i == 0) {
            r_draw_serial<SET>(src, lo + h, lc + h, R_DRAW_STRIDE);
        }
    }
    __syncthreads();
    if (!((who >> i) & 1u)) return;
    for (int t = threadIdx.x >> 5; t < GPR_REF_SLOTS; t += R_DRAW_WG / 32) {
        ops[(size_t)t * N + c0 + i] = lo[t * R_DRAW_STRIDE + i];
        cs[(size_t)t * N + c0 + i] = lc[t * R_DRAW_STRIDE + i];
    }
}

template <int SET>
__global__ void __launch_bounds__(R_DRAW_WG) k_init_ref(GprMHArgs a, int first) {
    const int c0 = (first + (int)blockIdx.x) * R_DRAW_CHAINS, n = min(R_DRAW_CHAINS, a.nchains - c0);
    r_draw_chains<SET>(a.seed, c0, n == 32 ? ~0u : (1u << n) - 1u, 0, GPR_P_INIT, a.ops, a.cs, a.nchains);
}

// KERNEL over the chains, R_DRAW_CHAINS a workgroup (16 threads a chain: from 2^28 chains on
// they pass the size of one launch)
#define GPR_DRAW_LAUNCH(KERNEL, SET, S, ARGS)                                                                     \
    return (hipError_t)gpr_launches((ARGS.nchains + R_DRAW_CHAINS - 1) / R_DRAW_CHAINS, R_DRAW_WG, [&](int first, int count) { \
        const dim3 grid(count), wg(R_DRAW_WG);                                                                    \
        switch (SET) {                                                                                            \
        case GPR_OPS_SIMPLIFIED: hipLaunchKernelGGL(KERNEL<GPR_OPS_SIMPLIFIED>, grid, wg, 0, S, ARGS, first); break; \
        case GPR_OPS_POLYNOMIAL: hipLaunchKernelGGL(KERNEL<GPR_OPS_POLYNOMIAL>, grid, wg, 0, S, ARGS, first); break; \
        case GPR_OPS_LINEAR: hipLaunchKernelGGL(KERNEL<GPR_OPS_LINEAR>, grid, wg, 0, S, ARGS, first); break;        \
        case GPR_OPS_PHYSICAL: hipLaunchKernelGGL(KERNEL<GPR_OPS_PHYSICAL>, grid, wg, 0, S, ARGS, first); break;    \
        default: hipLaunchKernelGGL(KERNEL<GPR_OPS_DEFAULT>, grid, wg, 0, S, ARGS, first); break;                   \
        }                                                                                                         \
        return (int)hipGetLastError();                                                                            \
    })

hipError_t gpr_launch_init_ref(const GprMHArgs &a, hipStream_t s) {
    GPR_DRAW_LAUNCH(k_init_ref, a.opset, s, a);
}

// Order-preserving key of a double with NaN below everything (cmp, main.cu:987-995).
__device__ __forceinline__ uint64_t r_key(double v) {
    if (v != v) return 0;
    const uint64_t b = __builtin_bit_cast(uint64_t, v);
    return (b >> 63) ? ~b : (b | 0x8000000000000000ull);
}
__device__ __forceinline__ double r_unkey(uint64_t k) {
    if (k == 0) return __builtin_nan("");
    const uint64_t b = (k >> 63) ? (k & 0x7fffffffffffffffull) : ~k;
    return __builtin_bit_cast(double, b);
}

// Adds 1 to hist[bin] for the lanes of `mine`: posteriors share their leading bytes (and the
// NaN ones all bytes), so the lanes with the first lane's bin count as one atomic, a few
// times, before the rest add theirs one by one.
__device__ __forceinline__ void r_hist_add(unsigned int *hist, int bin, bool mine) {
    uint64_t m = ballot(mine);
    for (int k = 0; k < 3 && m; k++) {
        const int lead = __builtin_ctzll(m), b = rl_i(bin, lead);
        const uint64_t same = ballot(mine && bin == b) & m;
        if (lane_id() == lead) atomicAdd(&hist[b], (unsigned int)__popcll(same));
        m &= ~same;
    }
    if ((m >> lane_id()) & 1) atomicAdd(&hist[bin], 1u);
}

// One workgroup per dataset: radix select (8 passes of 8 bits) of the element of rank
// floor(nchains * quantile) in the NaN-first order; cutoff[d] is its value.  Latency bounds
// the passes: the keys of up to R_SEL_KEYS chains per thread stay in registers between
// them, and one wave scans the 256 bins, four per lane, where a single thread walked them
// (1024 chains selected and re-drawn in 103 us with the
// call before, 29 us now).
#define R_SEL_WG 1024
#define R_SEL_KEYS 4
__global__ void __launch_bounds__(R_SEL_WG) k_rs_quantile_select(GprResampleArgs a) {
    const GprDataset d = a.ds[blockIdx.x];
    __shared__ unsigned int hist[256];
    __shared__ uint64_t s_prefix;
    __shared__ int s_rank;
    const int tid = threadIdx.x, l = lane_id();
    const auto key = [&](int i) { return r_key(a.prior[d.chain0 + i] + a.ll[d.chain0 + i]); };
    const bool held = d.nchains <= R_SEL_WG * R_SEL_KEYS;
    uint64_t kept[R_SEL_KEYS];
#pragma unroll
    for (int q = 0; q < R_SEL_KEYS; q++) kept[q] = held && tid + q * R_SEL_WG < d.nchains ? key(tid + q * R_SEL_WG) : 0;
    if (tid == 0) {
        s_prefix = 0;
        // the rank of the cutoff, cutoff = sorted[(int)(N * q)] (main.cu:1219); gpr_create
        // keeps q in [0, 1), and the clamp keeps the select inside the keys regardless
        s_rank = min(max((int)((float)d.nchains * a.quantile), 0), d.nchains - 1);
    }
    for (int pass = 7; pass >= 0; pass--) {
        if (tid < 256) hist[tid] = 0;
        __syncthreads();
        const uint64_t prefix = s_prefix;
        const uint64_t hmask = pass == 7 ? 0 : (~0ull << ((pass + 1) * 8));
        const auto add = [&](uint64_t k, bool in) {
            r_hist_add(hist, (int)(k >> (pass * 8)) & 255, in && (k & hmask) == prefix);
        };
        if (held) {
#pragma unroll
            for (int q = 0; q < R_SEL_KEYS; q++)
                if (q * R_SEL_WG < d.nchains) add(kept[q], tid + q * R_SEL_WG < d.nchains);
        } else {
            for (int i0 = 0; i0 < d.nchains; i0 += R_SEL_WG) {
                const bool in = i0 + tid < d.nchains;
                add(in ? key(i0 + tid) : 0, in);
            }
        }
        __syncthreads();
        if (tid < 64) {
            const int r = s_rank;
            int h[4], below = 0;
#pragma unroll
            for (int q = 0; q < 4; q++) below += h[q] = (int)hist[4 * l + q];
            below = wave_scan_i(below) - below;       // keys in the bins of the lanes before
            const int own = h[0] + h[1] + h[2] + h[3];
            if (r >= below && r < below + own) {      // one lane: the rank is below the sum of all
                int b = 0;
                int left = r - below;
                for (; b < 3 && left >= h[b]; b++) left -= h[b];
                s_rank = left;
                s_prefix = prefix | ((uint64_t)(4 * l + b) << (pass * 8));
            }
        }
        __syncthreads();
    }
    if (tid == 0) a.cutoff[blockIdx.x] = r_unkey(s_prefix);
}

template <int SET>
__global__ void __launch_bounds__(R_DRAW_WG) k_rs_quantile_redraw(GprResampleArgs a, int first) {
    const int c0 = (first + (int)blockIdx.x) * R_DRAW_CHAINS, c = c0 + (int)(threadIdx.x & 31);
    bool low = false;      // NaN posteriors never resampled
    if (c < a.nchains) low = a.prior[c] + a.ll[c] < a.cutoff[chain_dataset(a.ds, a.ndatasets, c)];
    const uint32_t who = (uint32_t)ballot(low);       // each half of each wave: the same 32 chains
    if (!who) return;
    r_draw_chains<SET>(a.seed, c0, who, a.clock ? a.clock[1] : a.block, GPR_P_RESAMPLE, a.ops, a.cs, a.nchains);
    if (threadIdx.x == 0) atomicAdd(a.nresampled, __popc(who));
}

hipError_t gpr_launch_resample_quantile(const GprResampleArgs &a, hipStream_t s) {
    hipLaunchKernelGGL(k_rs_quantile_select, dim3(a.ndatasets), dim3(R_SEL_WG), 0, s, a);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    GPR_DRAW_LAUNCH(k_rs_quantile_redraw, a.opset, s, a);
}

// ---------------------------------------------------------------- test hooks
// One wave per heap: run the wave decode and write the tape (ops, consts) and its
// length, count and description length, for comparison with the host decode.
__global__ void k_test_ref_decode(const uint8_t *hop, const float *hc, int nheaps, uint8_t *ops, float *cs,
                                  int32_t *meta) {
    const int h = uni((int)(blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)));
    if (h >= nheaps) return;
    const int l = lane_id();
    const int o = l < GPR_REF_SLOTS ? hop[(size_t)h * GPR_REF_SLOTS + l] : 0;
    const float c = l < GPR_REF_SLOTS ? hc[(size_t)h * GPR_REF_SLOTS + l] : 0.0f;
    const RefTape rt = r_decode_wave(o, c);
    ops[(size_t)h * 64 + l] = (uint8_t)rt.p.o0;
    cs[(size_t)h * 64 + l] = rt.p.c0;
    if (l == 0) {
        meta[h * 3 + 0] = rt.p.len;
        meta[h * 3 + 1] = rt.count;
        meta[h * 3 + 2] = rt.dl;
    }
}

hipError_t gpr_launch_test_ref_decode(const uint8_t *hop, const float *hc, int nheaps, uint8_t *ops, float *cs,
                                      int32_t *meta, hipStream_t s) {
    hipLaunchKernelGGL(k_test_ref_decode, dim3((nheaps + 3) / 4), dim3(256), 0, s, hop, hc, nheaps, ops, cs, meta);
    return hipGetLastError();
}

// The draw transforms on the device, one word per thread: u01, normal quantile, logf,
// expf, sin2pi of u, and the reference's random_float / random_normal /
// random_geometric / host random_normal of a Philox substream (seed, chain = i).
__global__ void k_test_draws(const uint32_t *words, int n, uint64_t seed, float *out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint32_t w = words[i];
    const float u = gpr_u01(w);
    float *o = out + (size_t)i * 10;
    o[0] = u;
    o[1] = gpr_normal(u);
    o[2] = gpr_logf(__builtin_bit_cast(float, w & 0x7fffffffu));
    o[3] = gpr_expf((float)((int32_t)w) * 0x1p-24f);
    o[4] = gpr_sin2pi(u);
    PhiloxSrc s;
    s.st.init(seed, (uint32_t)i, 0, 0, 0);
    o[5] = r_random_float(s);
    o[6] = r_random_normal(s);
    o[7] = r_random_geometric(s);
    o[8] = r_host_random_normal(s);
    o[9] = (float)r_random_int(27, s);
}

hipError_t gpr_launch_test_draws(const uint32_t *words, int n, uint64_t seed, float *out, hipStream_t s) {
    hipLaunchKernelGGL(k_test_draws, dim3((n + 255) / 256), dim3(256), 0, s, words, n, seed, out);
    return hipGetLastError();
}

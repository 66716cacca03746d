// Register-resident Lawson-Hanson NNLS (src/NNLS.jl:605-1061): the solves of the voxel kernel for trains whose live
// workspace rows fit a lane's registers. Included by dmi_kernels.hip inside its namespace.
//
// Lane j owns column j of the workspace: rows [p, mr) (p: the active set's size, mr: the rows appended so far) are in
// its registers a[], row r at a[r - base]. A row leaves the window when its pivot is taken: it then belongs to the
// triangular factor and goes to LDS. Both the window (p grows with mr in the Tikhonov solves) and the factor are small:
// the memory-resident solver (Wave) keeps (m + n) n doubles of workspace in LDS, this one n (n + 1) / 2. The registers
// allow two waves per SIMD (8 workgroups per CU; 1 to 4 memory-resident), and up to 60 bins so does the LDS: 20 KB a
// workgroup at 60 bins, 22 KB (7 workgroups) at 64. GCV's Gram matrix takes more than the factor where m and n are both
// large: 27 KB (6 workgroups) at 56 x 60, 35 KB (4, one wave per SIMD) at 64 x 64.
// The Householder apply, whose six 16-byte LDS operations per row pair bound the memory-resident solver, is three FMAs
// per row here: the reflector and the right-hand side are read once per step into registers with 16 rows in each
// 16-lane row (the same in all four), and every FMA takes its scalar from one of them with a DPP row broadcast (one wave
// per SIMD: 5.3 cycles, 4.2 for a plain FMA).
//
// Bound by the latency of a solve's chain (dependent FP64 operations, reductions over the wave, LDS round trips), of which
// two waves per SIMD hide a part: on the 240x240x113, 56-echo, 60-bin L-curve volume the VALU is busy 57% of the cycles (28%
// in the memory-resident kernel), a wave issues 52% of its time, waits 31% for results and 18% for its turn to issue. That
// volume takes 8.7 s (20.4 s memory-resident), the 240x240x48, 48-echo, 40-bin gcv volume 1.52 s (2.88 s).
//
// Every sum has the terms, the partial sums and the order of the memory-resident solver, so the two give the same bits.
#pragma once

struct RegSolve {
    double rnorm;
    int nsetp, idxl;  // idxl: the column at position L
    unsigned flops;
    int flags;        // kReg*
};
constexpr int kRegMaxIter = 1, kRegOverflow = 2;

__device__ __forceinline__ int tri(int j) { return (j * (j + 1)) >> 1; }
template <class P> __device__ __forceinline__ P *rflp(P *p) {
    const unsigned long long u = (unsigned long long)p;
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)u), hi = __builtin_amdgcn_readfirstlane((unsigned)(u >> 32));
    return (P *)(((unsigned long long)hi << 32) | lo);
}
__device__ __forceinline__ ldbl *rfll(ldbl *p) { return (ldbl *)(uintptr_t)(unsigned)__builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)p); }

// The lane's column, rows [0, S) of the window, in the registers v[256 - 2 S] .. v[255], addressed by name: the kernels
// that call nnls_reg are compiled for at most 512 / reg_cap_waves(S) compiler-allocated registers (the waves-per-SIMD
// attribute, which the called function inherits; the build reads the assembly for it), so nothing else lives there, and
// declare v255 so that all 256 are theirs. Left
// to the register allocator, the 72 values of a[] were copied and spilled wherever paths that shift the window meet
// paths that do not (60 to 140 scratch accesses per step). Every access is a volatile asm statement, so all of them stay
// in program order; none runs with lanes switched off except the dump of one lane's column.
template <int S> struct Bank {
    static constexpr int R0 = 256 - 2 * S;
    static constexpr int reg(int k) { return R0 + 2 * k; }
};
template <int N, class F, int... I>
__device__ __forceinline__ void each_impl(F &&f, std::integer_sequence<int, I...>) { (f(std::integral_constant<int, I>()), ...); }
// f(0), ..., f(N - 1) with the index as a constant
template <int N, class F> __device__ __forceinline__ void each(F &&f) { each_impl<N>(f, std::make_integer_sequence<int, N>()); }

template <int R> __device__ __forceinline__ double bank_get() {
    double v;
    asm volatile("v_mov_b64 %0, v[%1:%1+1]" : "=v"(v) : "i"(R));
    return v;
}
template <int R> __device__ __forceinline__ void bank_put(double v) { asm volatile("v_mov_b64 v[%1:%1+1], %0" : : "v"(v), "i"(R)); }
template <int R> __device__ __forceinline__ void bank_zero4() {
    asm volatile("v_mov_b64 v[%0:%0+1], 0\n\tv_mov_b64 v[%0+2:%0+3], 0\n\tv_mov_b64 v[%0+4:%0+5], 0\n\t"
                 "v_mov_b64 v[%0+6:%0+7], 0" : : "i"(R));
}
// registers R.. (four rows) take the rows at R + D
template <int R, int D> __device__ __forceinline__ void bank_move4() {
    asm volatile("v_mov_b64 v[%0:%0+1], v[%1:%1+1]\n\tv_mov_b64 v[%0+2:%0+3], v[%1+2:%1+3]\n\t"
                 "v_mov_b64 v[%0+4:%0+5], v[%1+4:%1+5]\n\tv_mov_b64 v[%0+6:%0+7], v[%1+6:%1+7]" : : "i"(R), "i"(R + D));
}
template <int R> __device__ __forceinline__ void bank_mul4(double f) {
    asm volatile("v_mul_f64 v[%1:%1+1], v[%1:%1+1], %0\n\tv_mul_f64 v[%1+2:%1+3], v[%1+2:%1+3], %0\n\t"
                 "v_mul_f64 v[%1+4:%1+5], v[%1+4:%1+5], %0\n\tv_mul_f64 v[%1+6:%1+7], v[%1+6:%1+7], %0" : : "v"(f), "i"(R));
}
// row o = 0..3 after the row at R, o uniform (a select of four: the indexed form, s_set_gpr_idx_on, took 74 cycles)
template <int R> __device__ __forceinline__ double bank_get_at(int o) {
    const double a0 = bank_get<R>(), a1 = bank_get<R + 2>(), a2 = bank_get<R + 4>(), a3 = bank_get<R + 6>();
    const double lo = (o & 1) ? a1 : a0, hi = (o & 1) ? a3 : a2;
    return (o & 2) ? hi : lo;
}
// two rows to LDS, 16-byte aligned
template <int R, int OFF> __device__ __forceinline__ void bank_store2(ldbl *p) {
    asm volatile("ds_write_b128 %0, v[%1:%1+3] offset:%2" : : "v"((unsigned)(uintptr_t)p), "i"(R), "i"(OFF) : "memory");
}

// c[k & 3] += v_k a[k] for the eight rows at R, v_k: lane 8 H + k of v's 16-lane row (v the same in all four rows). Every
// lane of the wave is active. The s_nop covers the two wait states between a VALU write and a DPP read of the same
// register, which the compiler does not see inside the block.
#define DMI_BC " row_mask:0xf bank_mask:0xf\n\t"
template <int H, int R> __device__ __forceinline__ void dot8(double &c0, double &c1, double &c2, double &c3, double v) {
    asm volatile("s_nop 1\n\t"
                 "v_fmac_f64_dpp %0, %4, v[%5:%5+1] row_newbcast:%6" DMI_BC
                 "v_fmac_f64_dpp %1, %4, v[%5+2:%5+3] row_newbcast:%6+1" DMI_BC
                 "v_fmac_f64_dpp %2, %4, v[%5+4:%5+5] row_newbcast:%6+2" DMI_BC
                 "v_fmac_f64_dpp %3, %4, v[%5+6:%5+7] row_newbcast:%6+3" DMI_BC
                 "v_fmac_f64_dpp %0, %4, v[%5+8:%5+9] row_newbcast:%6+4" DMI_BC
                 "v_fmac_f64_dpp %1, %4, v[%5+10:%5+11] row_newbcast:%6+5" DMI_BC
                 "v_fmac_f64_dpp %2, %4, v[%5+12:%5+13] row_newbcast:%6+6" DMI_BC
                 "v_fmac_f64_dpp %3, %4, v[%5+14:%5+15] row_newbcast:%6+7" DMI_BC
                 : "+v"(c0), "+v"(c1), "+v"(c2), "+v"(c3)
                 : "v"(v), "i"(R), "i"(8 * H));
}
// a[k] += sm u_k, then the dual sums over the updated rows: we += b_k a[k] (even k), wo += b_k a[k] (odd k)
template <int H, int R> __device__ __forceinline__ void upd8(double u, double sm, double b, double &we, double &wo) {
    asm volatile("s_nop 1\n\t"
                 "v_fmac_f64_dpp v[%5:%5+1], %2, %3 row_newbcast:%6" DMI_BC
                 "v_fmac_f64_dpp v[%5+2:%5+3], %2, %3 row_newbcast:%6+1" DMI_BC
                 "v_fmac_f64_dpp v[%5+4:%5+5], %2, %3 row_newbcast:%6+2" DMI_BC
                 "v_fmac_f64_dpp v[%5+6:%5+7], %2, %3 row_newbcast:%6+3" DMI_BC
                 "v_fmac_f64_dpp v[%5+8:%5+9], %2, %3 row_newbcast:%6+4" DMI_BC
                 "v_fmac_f64_dpp v[%5+10:%5+11], %2, %3 row_newbcast:%6+5" DMI_BC
                 "v_fmac_f64_dpp v[%5+12:%5+13], %2, %3 row_newbcast:%6+6" DMI_BC
                 "v_fmac_f64_dpp v[%5+14:%5+15], %2, %3 row_newbcast:%6+7" DMI_BC
                 "v_fmac_f64_dpp %0, %4, v[%5:%5+1] row_newbcast:%6" DMI_BC
                 "v_fmac_f64_dpp %1, %4, v[%5+2:%5+3] row_newbcast:%6+1" DMI_BC
                 "v_fmac_f64_dpp %0, %4, v[%5+4:%5+5] row_newbcast:%6+2" DMI_BC
                 "v_fmac_f64_dpp %1, %4, v[%5+6:%5+7] row_newbcast:%6+3" DMI_BC
                 "v_fmac_f64_dpp %0, %4, v[%5+8:%5+9] row_newbcast:%6+4" DMI_BC
                 "v_fmac_f64_dpp %1, %4, v[%5+10:%5+11] row_newbcast:%6+5" DMI_BC
                 "v_fmac_f64_dpp %0, %4, v[%5+12:%5+13] row_newbcast:%6+6" DMI_BC
                 "v_fmac_f64_dpp %1, %4, v[%5+14:%5+15] row_newbcast:%6+7" DMI_BC
                 : "+v"(we), "+v"(wo)
                 : "v"(u), "v"(sm), "v"(b), "i"(R), "i"(8 * H));
}
// w += v_k a[k] in the order of k, product and sum each rounded
template <int H, int R> __device__ __forceinline__ void mac8(double &w, double v) {
    double t0, t1;
    asm volatile("s_nop 1\n\t"
                 "v_mov_b64_dpp %1, %3 row_newbcast:%5" DMI_BC "v_mov_b64_dpp %2, %3 row_newbcast:%5+1" DMI_BC
                 "v_mul_f64 %1, %1, v[%4:%4+1]\n\tv_mul_f64 %2, %2, v[%4+2:%4+3]\n\t"
                 "v_add_f64 %0, %0, %1\n\tv_mov_b64_dpp %1, %3 row_newbcast:%5+2" DMI_BC
                 "v_add_f64 %0, %0, %2\n\tv_mov_b64_dpp %2, %3 row_newbcast:%5+3" DMI_BC
                 "v_mul_f64 %1, %1, v[%4+4:%4+5]\n\tv_mul_f64 %2, %2, v[%4+6:%4+7]\n\t"
                 "v_add_f64 %0, %0, %1\n\tv_mov_b64_dpp %1, %3 row_newbcast:%5+4" DMI_BC
                 "v_add_f64 %0, %0, %2\n\tv_mov_b64_dpp %2, %3 row_newbcast:%5+5" DMI_BC
                 "v_mul_f64 %1, %1, v[%4+8:%4+9]\n\tv_mul_f64 %2, %2, v[%4+10:%4+11]\n\t"
                 "v_add_f64 %0, %0, %1\n\tv_mov_b64_dpp %1, %3 row_newbcast:%5+6" DMI_BC
                 "v_add_f64 %0, %0, %2\n\tv_mov_b64_dpp %2, %3 row_newbcast:%5+7" DMI_BC
                 "v_mul_f64 %1, %1, v[%4+12:%4+13]\n\tv_mul_f64 %2, %2, v[%4+14:%4+15]\n\t"
                 "v_add_f64 %0, %0, %1\n\tv_add_f64 %0, %0, %2"
                 : "+v"(w), "=&v"(t0), "=&v"(t1)
                 : "v"(v), "i"(R), "i"(8 * H));
}
// One column of the triangular solve inside the 16-lane row RHO: z += q c in that row, q from its lane T, kept in x's bank
// (four lanes) of lane T. q was just computed: two wait states before the DPP reads.
template <int RHO, int T> __device__ __forceinline__ void tri_step(double &z, double &x, double q, double c) {
    asm volatile("s_nop 1\n\t"
                 "v_fmac_f64_dpp %0, %2, %3 row_newbcast:%4 row_mask:%5 bank_mask:0xf\n\t"
                 "v_mov_b64_dpp %1, %2 row_newbcast:%4 row_mask:%5 bank_mask:%6"
                 : "+v"(z), "+v"(x) : "v"(q), "v"(c), "i"(T), "i"(1 << RHO), "i"(1 << (T >> 2)));
}
// z += q_T c in the rows below RHO, q_T: lane T of q's 16-lane rows
template <int RHO, int T> __device__ __forceinline__ void tri_below(double &z, double q, double c) {
    asm volatile("v_fmac_f64_dpp %0, %1, %2 row_newbcast:%3 row_mask:%4 bank_mask:0xf"
                 : "+v"(z) : "v"(q), "v"(c), "i"(T), "i"((1 << RHO) - 1));
}
#undef DMI_BC

// The lanes holding the largest of v >= 0 (0 if every v is 0). Non-negative doubles order as their bits: the high words'
// maximum takes one DPP instruction per level (a maximum of doubles takes five), the low words' is needed only where
// two lanes share the high word.
__device__ __forceinline__ unsigned wave_umax(unsigned v) {
    auto mx = [](unsigned a, unsigned b) { return a > b ? a : b; };
    v = mx(v, (unsigned)dpp_i<kQuadSwap1>((int)v));
    v = mx(v, (unsigned)dpp_i<kQuadSwap2>((int)v));
    v = mx(v, (unsigned)dpp_i<kHalfMirror>((int)v));
    v = mx(v, (unsigned)dpp_i<kRowMirror>((int)v));
    v = mx(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, kRowBcast15, 0xA, 0xf, false));
    v = mx(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, kRowBcast31, 0xC, 0xf, false));
    return (unsigned)__builtin_amdgcn_readlane((int)v, 63);
}
__device__ __forceinline__ unsigned long long lanes_of_max(double v) {
    const unsigned long long u = (unsigned long long)__double_as_longlong(v);
    const unsigned hi = (unsigned)(u >> 32), lo = (unsigned)u, hm = wave_umax(hi);
    unsigned long long hit = ballot(hi == hm);
    if ((hit & (hit - 1)) || hm == 0) {
        const unsigned lm = wave_umax(hi == hm ? lo : 0u);
        hit = (hm | lm) ? ballot(hi == hm && lo == lm) : 0ull;
    }
    return hit;
}

// One solve: NNLSProblem solve! with the reference warm start (src/lsqnonneg.jl:30-84), or its Tikhonov form (:86-164)
// with tikh. A0: the m x n basis, row-major. b0: the right-hand side (each lane reads rows L, L + 64). dims: m, n and
// tikh packed as m | n << 8 | tikh << 16. On return x (LDS) holds the solution by column.
//
// A function of its own, called, so that its registers are allocated apart from the searches around it and its code
// (the row loops are unrolled over the S registers) exists once per kernel and stays in the instruction cache.
template <int S>
__device__ __attribute__((noinline)) RegSolve nnls_reg(cgdbl *A0_, cgdbl *b0_, ldbl *lds_, int dims_, double mu_) {
    constexpr int SP = (S + 15) & ~15, NV = SP / 16;
    constexpr int NB = 2;  // rows L and L + 64 of a vector held by row: m + n <= 128
    static_assert(S <= 80, "");
    // rows [0, R1) of the window always run, then a block of 16 and blocks of 8 as far as the window reaches (a
    // comparison and branch cost 16 cycles, as much as one row's three FMAs); the largest class serves shorter trains too
    constexpr int R1 = S == 80 ? 40 : S - 32;
    auto block = [](int k0) constexpr { return k0 < R1 ? 0 : k0 < R1 + 16 ? R1 : k0; };
    static_assert(S % 8 == 0 && R1 >= 8, "");
    const int L = lane_id();
    cgdbl *A0 = rflp(A0_);
    cgdbl *b0 = rflp(b0_);
    const int dims = rfl(dims_);
    const double mu = rfl(mu_);
    const int m = dims & 255, n = (dims >> 8) & 255;
    const bool tikh = (dims >> 16) != 0;
    const int M = tikh ? m + n : m;
    const RegLayout lay = reg_layout(m, n, false);
    ldbl *lds = rfll(lds_), *x = lds, *bl = lds + lay.b, *T = lds + lay.T, *tmp = lds + lay.tmp;
    constexpr int RS = kRegStage;  // rows of a staged vector: a window's last row is below base + SP <= 60 + SP
    static_assert(NB * kWave + 16 <= RS && 60 + SP < RS, "");
    ldbl *ud = lds + lay.stg, *uf = ud + RS, *bm = uf + RS;
    if (L < RS - NB * kWave) ud[NB * kWave + L] = uf[NB * kWave + L] = bm[NB * kWave + L] = 0.0;
    RegSolve out;
    out.flags = 0;
    unsigned flops = 2u * m * n + 6u * m;

    DMI_PT0();
    // ---- set-up: the last column and the right-hand side by row, then the lane's column ----
    const double g0 = (L < m) ? A0[L * n + n - 1] : 0.0, g1 = (L + kWave < m) ? A0[(L + kWave) * n + n - 1] : 0.0;
    double br[NB];
#pragma unroll
    for (int k = 0; k < NB; ++k) br[k] = (L + k * kWave < m) ? b0[L + k * kWave] : 0.0;
    using BK = Bank<S>;
    const int col = min(L, n - 1);
    each<S / 8>([&](auto g) __attribute__((always_inline)) {
        constexpr int k0 = 8 * decltype(g)::value;
        double t[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
        if (k0 + 8 <= m) {
#pragma unroll
            for (int k = 0; k < 8; ++k) t[k] = A0[(k0 + k) * n + col];
        } else if (k0 < m) {
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const double v = A0[min(k0 + k, m - 1) * n + col];
                t[k] = (k0 + k < m) ? v : 0.0;
            }
        }
        each<8>([&](auto k) __attribute__((always_inline)) { bank_put<BK::reg(k0 + decltype(k)::value)>(t[decltype(k)::value]); });
    });
    double alast = A0[(m - 1) * n + col];  // row mr - 1 of the lane's column, kept beside a[]
    double wl;                              // the lane's dual
    {
        double pd = 0.0;
        if (L < m) pd += g0 * g0;
        if (L + kWave < m) pd += g1 * g1;
        double den = wsum(pd);
        if (tikh) den += mu * mu;
        double px = 0.0;
        if (L < m) px += (g0 / den) * br[0];
        if (L + kWave < m) px += (g1 / den) * br[1];
        const double xj = wsum(px);
        const double z0 = (L < m) ? br[0] - g0 * xj : 0.0, z1 = (L + kWave < m) ? br[1] - g1 * xj : 0.0;
        // w_j = sum_i A_ij z_i over the rows in order, z_i from 16-lane rows that hold 16 of them each
        ud[L] = z0;
        ud[L + kWave] = z1;
        lds_order();
        double zb[NV];
#pragma unroll
        for (int v = 0; v < NV; ++v) zb[v] = ud[16 * v + (L & 15)];
        double wj = 0.0;
        each<S / 8>([&](auto g) __attribute__((always_inline)) {
            constexpr int gi = decltype(g)::value;
            if (8 * gi < m) mac8<gi & 1, BK::reg(8 * gi)>(wj, zb[gi >> 1]);
        });
        const bool ps = L < n - 1 && !(wj <= 0);
        const unsigned long long bal = ballot(ps);
        wl = (L < n - 1) ? wj : 0.0;
        if (L == n - 1) wl = (bal == 0) ? 1.0 : 0.0;
    }

    DMI_LAP(kPhInit);
    double ap = bank_get<BK::reg(0)>();  // row nsetp of the lane's column
    int pos = L, pidx = L;  // position of the lane's column; column at position L
    double xp = 0.0;        // coefficient at position L
    int mr = m, nsetp = 0, base = 0, iter = 0;
    const int max_iter = 3 * n;
    unsigned long long dmask = 0ull;  // columns whose Tikhonov row has been appended
    auto row2 = [&](const double *v, const double *w, int i, double &vi, double &wi) {  // row i of vectors held by row
        if (i >= kWave) {
            vi = readlane(v[1], i - kWave);
            wi = readlane(w[1], i - kWave);
        } else {
            vi = readlane(v[0], i);
            wi = readlane(w[0], i);
        }
    };
    // solve_triangular_system! on R = T[0:k], lane i holding z_i, its diagonal aL and minus the diagonal's reciprocal nL; see
    // Wave::tri_solve for the quotients (formed negated here). In blocks of 16 columns, one per 16-lane row: inside the
    // block's own row the quotient of lane T reaches the other lanes by a DPP broadcast (a column then costs 45 cycles;
    // through a lane read into scalar registers it cost 98), and the rows below take the whole block's quotients
    // afterwards, 16 FMAs without a chain between lanes. Lanes at and past a column take its update too, from whatever
    // lies past the column's end: their quotients have been taken by then. Columns past k - 1 in the first group of four
    // are read as zeros.
    double aL = 1.0, nL = 0.0;
    auto tri_solve = [&](int k, double z) __attribute__((always_inline)) -> double {
        double xq = 0.0;
        each<4>([&](auto ri) __attribute__((always_inline)) {
            constexpr int rho = 3 - decltype(ri)::value;
            if (k > 16 * rho) {
                double cc[8], x[4] = {0.0, 0.0, 0.0, 0.0};
                each<4>([&](auto gi) __attribute__((always_inline)) {
                    constexpr int g = 3 - decltype(gi)::value, j0 = 16 * rho + 4 * g;
                    if (k > j0) {
                        if (g == 3 || k <= j0 + 4)
                            each<4>([&](auto q) __attribute__((always_inline)) {
                                constexpr int j = j0 + 3 - decltype(q)::value;
                                const ldbl *pc = (j < k) ? T + tri(j) + L : ud + RS - 1;
                                cc[j & 7] = *(volatile const ldbl *)pc;
                            });
                        if constexpr (g > 0)
                            each<4>([&](auto q) __attribute__((always_inline)) {
                                constexpr int j = j0 - 1 - decltype(q)::value;
                                cc[j & 7] = *(volatile const ldbl *)(T + tri(j) + L);
                            });
                        each<4>([&](auto q) __attribute__((always_inline)) {
                            constexpr int t = 4 * g + 3 - decltype(q)::value;
                            const double q0 = z * nL, qn = fma(fma(q0, aL, z), nL, q0);
                            tri_step<rho, t>(z, x[t & 3], qn, cc[t & 7]);
                        });
                    }
                });
                const double xl = (L & 1) ? x[1] : x[0], xh = (L & 1) ? x[3] : x[2], xv = (L & 2) ? xh : xl;
                if ((L >> 4) == rho) xq = xv;
                if constexpr (rho > 0) {
                    if ((L >> 4) == rho) tmp[L & 15] = xv;
                    lds_order();
                    const double qr = tmp[L & 15];
                    each<4>([&](auto gi) __attribute__((always_inline)) {
                        constexpr int j0 = 16 * rho + 4 * (3 - decltype(gi)::value);
                        if (k > j0) {
                            double c[4];  // columns past k - 1 meet zero quotients here
#pragma unroll
                            for (int q = 0; q < 4; ++q) c[q] = *(volatile const ldbl *)((j0 + q < k ? T + tri(j0 + q) : T + tri(j0)) + L);
                            tri_below<rho, (j0 & 15) + 3>(z, qr, c[3]);
                            tri_below<rho, (j0 & 15) + 2>(z, qr, c[2]);
                            tri_below<rho, (j0 & 15) + 1>(z, qr, c[1]);
                            tri_below<rho, (j0 & 15)>(z, qr, c[0]);
                        }
                    });
                }
            }
        });
        flops += (unsigned)(k * k);
        return -xq;
    };
    for (;;) {
        if (tikh ? (nsetp >= n) : (nsetp >= n || nsetp >= mr)) break;
        const int ip = nsetp;
        // ---- select the pivot column and form its reflector (construct_apply_householder!) ----
        double wv = (pos >= ip && L < n) ? wl : 0.0;
        bool term = false, newdiag = false;
        int cl = 0, jmax = 0, mrh = mr;
        double tau = 0.0, diag = 0.0, nd = 0.0, tj = 0.0, ti = 0.0, u[NB];
        for (;;) {
            const unsigned long long hit = lanes_of_max((wv > 0) ? wv : 0.0);
            if (hit == 0) { term = true; break; }
            cl = __ffsll((long long)hit) - 1;
            if (hit & (hit - 1)) {  // equal duals: the lowest position
                int best = readlane(pos, cl);
                for (unsigned long long h = hit & (hit - 1); h; h &= h - 1) {
                    const int c = __ffsll((long long)h) - 1, q = readlane(pos, c);
                    if (q < best) { best = q; cl = c; }
                }
            }
            jmax = readlane(pos, cl);
            newdiag = tikh && !((dmask >> cl) & 1ull);
            mrh = tikh ? min(mr + 1, M) : mr;
            const int len = mr - base;
            if (newdiag && len >= S) { out.flags |= kRegOverflow; term = true; break; }
            // the factor's columns at its position and at ip, for the exchange below; the pivot column by row, through LDS
            tj = (L < ip) ? T[tri(jmax) + L] : 0.0;
            ti = (L < ip) ? T[tri(ip) + L] : 0.0;
            if (L == cl)
                each<S / 8>([&](auto g) __attribute__((always_inline)) {
                    constexpr int k0 = 8 * decltype(g)::value;
                    if (k0 < R1 || len > block(k0))
                        each<4>([&](auto i) __attribute__((always_inline)) {
                            constexpr int k = k0 + 2 * decltype(i)::value;
                            bank_store2<BK::reg(k), 8 * k>(ud + base);
                        });
                });
            lds_order();
            DMI_LAP(kPhSelect);
            double c[NB];
            const bool two = mrh > kWave;
            c[0] = (L >= ip && L < mr) ? ud[L] : 0.0;
            if (newdiag && L == mr) c[0] = mu;
            double part = c[0] * c[0];
            c[1] = 0.0;
            if (two) {
                c[1] = (L + kWave < mr) ? ud[L + kWave] : 0.0;
                if (newdiag && L + kWave == mr) c[1] = mu;
                part = fma(c[1], c[1], part);
            }
            const double cip = readlane(c[0], ip);
            const double xnorm = sqrt(wsum(part));
            flops += 2u * (mrh - ip) + 8u;
            tau = -1.0;
            if (xnorm != 0) {
                // quotients by reciprocals: x / a = q0 + (x - q0 a) y with y = 1 / a, q0 = x y, as in the triangular solve
                const double beta = copysign(xnorm, cip), alpha = cip + beta, yb = 1.0 / beta, ya = 1.0 / alpha;
                auto quot = [](double x, double a, double y) {
                    const double q0 = x * y;
                    return fma(fma(-q0, a, x), y, q0);
                };
                tau = quot(alpha, beta, yb);
                nd = yb;  // -1 / diag where diag = -beta
                const double bip = readlane(br[0], ip);
                u[0] = (L == ip) ? 0.0 : quot(c[0], alpha, ya);  // zero outside rows (ip, mrh)
                part = (L > ip && L < mrh) ? br[0] * u[0] : 0.0;
                u[1] = 0.0;
                if (two) {
                    u[1] = quot(c[1], alpha, ya);
                    if (L + kWave < mrh) part = fma(br[1], u[1], part);
                }
                double sm = bip + wsum(part);
                sm *= -tau;
                const double A1 = -beta, b1 = bip + sm;
                flops += 3u * (mrh - ip);
                const bool up = (b1 > 0 && A1 > 0) || (b1 < 0 && A1 < 0);
                if (!(fabs(b1) >= 1e-290 ? up : (b1 / A1 > 0))) {
                    tau = -1.0;
                } else if (ip < mrh - 1) {
                    diag = A1;
                    if (L >= ip && L < mrh) br[0] = (L == ip) ? b1 : fma(sm, u[0], br[0]);
                    if (two && L + kWave < mrh) br[1] = fma(sm, u[1], br[1]);
                    flops += 3u * (mrh - ip);
                } else {
                    tau = 0.0;
                    diag = cip;
                    nd = -1.0 / cip;
                }
            }
            if (tau >= 0) break;
            if (L == cl) { wv = 0.0; wl = 0.0; }
        }
        DMI_LAP(kPhConstruct);
        if (term) break;
        if (newdiag) {
            mr = min(mr + 1, M);
            dmask |= 1ull << cl;
            alast = 0.0;
        }
        nsetp += 1;
        {
            // column cl takes position ip, with its rows above the window; the column there takes position jmax
            if (L < ip) {
                T[tri(ip) + L] = tj;
                if (jmax != ip) T[tri(jmax) + L] = ti;
            }
            if (L == ip) T[tri(ip) + ip] = diag;
            const int pa = readlane(pidx, ip);
            if (L == ip) pidx = cl;
            else if (L == jmax) pidx = pa;
            if (L == pa) pos = jmax;
            if (L == cl) pos = ip;
        }
        DMI_LAP(kPhSwapApply);
        // ---- apply the reflector to the inactive columns, with their duals (apply_householder_dual!) ----
        const int o = ip - base;
        double anext = 0.0;  // row ip + 1, the next pivot's
        if (nsetp < n && ip < mr - 1) {
            const int lo = ip + 1, hi = mr, h = lo & 1, bs = lo + h, t = (hi - bs) & 1;
            // by row: the reflector for the update, and for the dot product and the dual without the single rows
#pragma unroll
            for (int k = 0; k < NB; ++k) {
                const int i = L + k * kWave;
                uf[i] = u[k];
                ud[i] = u[k];
                bm[i] = (k > 0 || i >= bs) ? br[k] : 0.0;  // rows from mr on hold zeros
            }
            const int r0 = h ? lo : RS - 1, r1 = t ? hi - 1 : RS - 1;  // RS - 1: a row past every window
            ud[r0] = 0.0;
            ud[r1] = 0.0;
            bm[r1] = 0.0;
            lds_order();
            double ub[NV], uu[NV], bb[NV];
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                ub[v] = ud[base + 16 * v + (L & 15)];
                uu[v] = uf[base + 16 * v + (L & 15)];
            }
            const double alo = bank_get_at<BK::reg(1)>(o);
            // row lo < n <= 64 and the last row of the two vectors
            const double ulo = readlane(u[0], lo), blo = readlane(br[0], lo);
            double ula, bla;
            row2(u, br, hi - 1, ula, bla);
            // four partial sums over the row pairs from bs: chain c takes the rows = c mod 4 (base is a multiple of 4)
            const double i1 = h ? alo * ulo : 0.0, i2 = t ? alast * ula : 0.0;
            const bool ph = (bs & 2) != 0;
            double c0 = ph ? i2 : ap, c1 = ph ? 0.0 : i1, c2 = ph ? ap : i2, c3 = ph ? i1 : 0.0;
            const int len = hi - base;
            each<S / 8>([&](auto gi) __attribute__((always_inline)) {
                constexpr int g = decltype(gi)::value;
                if (8 * g < R1 || len > block(8 * g)) dot8<g & 1, BK::reg(8 * g)>(c0, c1, c2, c3, ub[g >> 1]);
                if constexpr (g == 3)  // once the first registers of ub are free
#pragma unroll
                    for (int v = 0; v < NV; ++v) bb[v] = bm[base + 16 * v + (L & 15)];
            });
            const double sm = ((c0 + c1) + (c2 + c3)) * -tau;
            ap = ap + sm;
            alast = fma(sm, ula, alast);
            anext = fma(sm, ulo, alo);
            // the dual's two chains: a single first row starts the even one, a single last row ends the odd one
            double we = h ? anext * blo : 0.0, wo = 0.0;
            each<S / 8>([&](auto gi) __attribute__((always_inline)) {
                constexpr int g = decltype(gi)::value;
                if (8 * g < R1 || len > block(8 * g)) upd8<g & 1, BK::reg(8 * g)>(uu[g >> 1], sm, bb[g >> 1], we, wo);
            });
            if (t) wo = fma(alast, bla, wo);
            if (pos >= nsetp) wl = we + wo;
            flops += 6u * (mr - ip) * (n - ip - 1);
        }
        DMI_LAP(kPhApply);
        // row ip leaves the window
        if (pos >= nsetp && L < n) T[tri(pos) + ip] = ap;
        ap = anext;
        if (o == 3) {
            each<S / 4 - 1>([&](auto i) __attribute__((always_inline)) { bank_move4<BK::reg(4 * decltype(i)::value), 8>(); });
            bank_zero4<BK::reg(S - 4)>();
            base += 4;
        }
        lds_order();
        DMI_LAP(kPhPostApply);
        if (L == ip) { aL = diag; nL = nd; }
        double zr = tri_solve(nsetp, (L < nsetp) ? br[0] : 0.0);
        DMI_LAP(kPhTriSolve);
        // ---- feasibility: step to the first coefficient that reaches zero and remove it (:729-779) ----
        bool dual_flag = false, terminated = false;
        for (;;) {
            iter += 1;
            if (iter > max_iter) { out.flags |= kRegMaxIter; terminated = true; break; }
            if (ballot(L < nsetp && zr <= 0) == 0) break;
            double t = INFINITY;
            int ti = INT_MAX;
            if (L < nsetp && zr <= 0) {
                const double tt = -xp / (zr - xp);
                if (tt < 2.0) { t = tt; ti = L; }
            }
            wargmin(t, ti);
            if (ti == INT_MAX) break;
            dual_flag = true;
            int imv = ti;
            if (L < nsetp) xp = fma(t, zr - xp, xp);
            for (;;) {
                if (L == imv) xp = 0.0;
                if (imv != nsetp - 1) {
                    // the removed column, zero below its diagonal, moves through the rotations in tmp. Lane = position: p
                    // and q are rows i - 1 and i of its column; q becomes the next rotation's p in the register, and the
                    // pivot entries come from lane i's, so a rotation waits for no LDS read (row i + 1 is read ahead)
                    if (L < nsetp) tmp[L] = (L <= imv) ? T[tri(imv) + L] : 0.0;
                    lds_order();
                    ldbl *cj = (L == imv) ? tmp : T + tri(min(L, n - 1));
                    double p = cj[imv], q = cj[imv + 1];
                    for (int i = imv + 1; i <= nsetp - 1; ++i) {
                        const double qn = cj[min(i + 1, nsetp - 1)];
                        const double aa = readlane(p, i), bb = readlane(q, i);
                        const double sig = hypot(aa, bb), cs = aa / sig, ss = bb / sig;
                        const double pn = fma(cs, p, ss * q);
                        p = fma(-ss, p, cs * q);
                        q = qn;
                        if (L < n && (L >= i || L == imv)) cj[i - 1] = (L == i) ? sig : pn;
                        const double bp = readlane(br[0], i - 1), bq = readlane(br[0], i);
                        if (L == i - 1) br[0] = fma(cs, bp, ss * bq);
                        if (L == i) br[0] = fma(-ss, bp, cs * bq);
                        flops += 6u * (n + 1);
                    }
                    if (L < n && (L >= nsetp || L == imv)) cj[nsetp - 1] = p;
                    lds_order();
                    for (int j = imv; j < nsetp - 1; j += 4) {
                        double v[4];
#pragma unroll
                        for (int q = 0; q < 4; ++q) v[q] = T[tri(min(j + 1 + q, nsetp - 1)) + L];
                        lds_order();
#pragma unroll
                        for (int q = 0; q < 4; ++q)
                            if (L <= j + q && j + q < nsetp - 1) T[tri(j + q) + L] = v[q];
                        lds_order();
                    }
                    if (L < nsetp) T[tri(nsetp - 1) + L] = tmp[L];
                    lds_order();
                    const int pim = readlane(pidx, imv);
                    const double xim = readlane(xp, imv);
                    const int pdn = __shfl_down(pidx, 1);
                    const double xdn = __shfl_down(xp, 1);
                    if (L >= imv && L < nsetp - 1) { pidx = pdn; xp = xdn; }
                    else if (L == nsetp - 1) { pidx = pim; xp = xim; }
                    if (pos == imv) pos = nsetp - 1;
                    else if (pos > imv && pos < nsetp) pos -= 1;
                }
                nsetp -= 1;
                const int f = first_set(ballot(L < nsetp && xp <= 0));
                if (f < 0) break;
                imv = f;
            }
            // the rotations changed the diagonal
            aL = (L < nsetp) ? T[tri(L) + L] : 1.0;
            nL = (L < nsetp) ? -1.0 / aL : 0.0;
            zr = tri_solve(nsetp, (L < nsetp) ? br[0] : 0.0);
        }
        DMI_LAP(kPhDelete);
        if (terminated) break;
        if (dual_flag) {
            // rows [nsetp, ip] come back into the window: an inactive column's from T (a removed one has only its rows up
            // to its position there, and zeros below)
            if (mr - (base - ((max(base - nsetp, 0) + 3) & ~3)) > S) { out.flags |= kRegOverflow; break; }
            const double keep = (pos >= nsetp && pos <= ip) ? 0.0 : 1.0;
            each<S / 4>([&](auto i) __attribute__((always_inline)) { bank_mul4<BK::reg(4 * decltype(i)::value)>(keep); });
            alast *= keep;
            for (int r = ip; r >= nsetp; --r) {
                if (r < base) {
                    each<S / 4 - 1>([&](auto i) __attribute__((always_inline)) {
                        bank_move4<BK::reg(S - 4 - 4 * decltype(i)::value), -8>();
                    });
                    bank_zero4<BK::reg(0)>();
                    base -= 4;
                }
                const double back = (pos >= nsetp && pos >= r && L < n) ? T[tri(pos) + r] : 0.0;
                const int ob = r - base;
                if (ob == 0) bank_put<BK::reg(0)>(back);
                else if (ob == 1) bank_put<BK::reg(1)>(back);
                else if (ob == 2) bank_put<BK::reg(2)>(back);
                else bank_put<BK::reg(3)>(back);
                if (r == mr - 1) alast = back;
            }
            // compute_dual! over rows [nsetp, mr)
            double w = 0.0;
            if (nsetp < mr) {
                const int lo = nsetp, hi = mr, h = lo & 1, bs = lo + h, t = (hi - bs) & 1, ob = lo - base;
#pragma unroll
                for (int k = 0; k < NB; ++k) {
                    const int i = L + k * kWave;
                    bm[i] = (k > 0 || i >= bs) ? br[k] : 0.0;
                }
                bm[t ? hi - 1 : RS - 1] = 0.0;
                lds_order();
                double bb[NV];
#pragma unroll
                for (int v = 0; v < NV; ++v) bb[v] = bm[base + 16 * v + (L & 15)];
                const double alo = bank_get_at<BK::reg(0)>(ob);
                ap = alo;
                double bla, unused;
                row2(br, br, hi - 1, bla, unused);
                const double i0 = h ? alo * readlane(br[0], lo & 63) : 0.0, i1 = t ? alast * bla : 0.0;
                const bool ph = (bs & 2) != 0;
                double c0 = ph ? 0.0 : i0, c1 = ph ? 0.0 : i1, c2 = ph ? i0 : 0.0, c3 = ph ? i1 : 0.0;
                const int len = hi - base;
                each<S / 8>([&](auto gi) __attribute__((always_inline)) {
                    constexpr int g = decltype(gi)::value;
                    if (8 * g < R1 || len > block(8 * g)) dot8<g & 1, BK::reg(8 * g)>(c0, c1, c2, c3, bb[g >> 1]);
                });
                w = (c0 + c1) + (c2 + c3);
            }
            if (pos >= nsetp && L < n) wl = w;
            flops += 2u * (mr - nsetp) * (n - nsetp);
            lds_order();
        }
        if (L < nsetp) xp = zr;
        DMI_LAP(kPhDual);
    }
    if (L < n) x[pidx] = (L < nsetp) ? xp : 0.0;
#pragma unroll
    for (int k = 0; k < NB; ++k)
        if (L + k * kWave < M) bl[L + k * kWave] = br[k];
    lds_order();
    const int Mlim = tikh ? M : mr;
    double part = 0.0;
    for (int i = nsetp + L; i < Mlim; i += kWave) { const double bi = bl[i]; part = fma(bi, bi, part); }
    out.rnorm = sqrt(wsum(part));
    out.nsetp = nsetp;
    out.idxl = pidx;
    if (tikh) DMI_TIKH_ROWS(__popcll(dmask));
    out.flops = flops;
    return out;
}

// The voxel's basis at a constant flip angle, row-major: epg_const's recursion on two curves per LPC-lane group, with its
// operations in its order. A step is 10 FP operations, 4 selects that shift the phase states and 2 that push the echo
// into a shift register: v_cndmask takes its shifted operand through DPP, so a shift and its end condition are one
// instruction per word, and the echoes are scaled and stored once per LPC steps instead of one lane's store per step. A
// function of its own, since inside the voxel kernel the loop reloads spilled scalar registers. Per pair of curves and
// echo 590 cycles before, about 310 now; a 56 x 60 basis is 2% of a voxel's L-curve (4% before).

// One step's shifts: F takes Fr of the lane below, Fb the lane above's Fbr, R its own value of the lane below; the lanes in
// `first` take Fbr for F and R, those in `last` zero for Fb.
#define DMI_SHR " wave_shr:1 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
#define DMI_SHL " wave_shl:1 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
__device__ __forceinline__ void shift_states(int Fr, int Fbr, int &F, int &Fb, int &R, unsigned long long first,
                                             unsigned long long last) {
    asm("s_mov_b64 vcc, %5\n\ts_nop 1\n\tv_cndmask_b32_dpp %0, %3, %4, vcc" DMI_SHR "v_cndmask_b32_dpp %2, %2, %4, vcc" DMI_SHR
        "s_mov_b64 vcc, %6\n\tv_cndmask_b32_dpp %1, %4, %7, vcc" DMI_SHL
        : "=&v"(F), "=&v"(Fb), "+v"(R) : "v"(Fr), "v"(Fbr), "s"(first), "s"(last), "v"(0) : "vcc");
}
__device__ __forceinline__ void shift_states(float Fr, float Fbr, float &F, float &Fb, float &R, unsigned long long first,
                                             unsigned long long last) {
    int f, g, r = __float_as_int(R);
    shift_states(__float_as_int(Fr), __float_as_int(Fbr), f, g, r, first, last);
    F = __int_as_float(f);
    Fb = __int_as_float(g);
    R = __int_as_float(r);
}
__device__ __forceinline__ void shift_states(double Fr, double Fbr, double &F, double &Fb, double &R, unsigned long long first,
                                             unsigned long long last) {
    int f0, f1, g0, g1, r0 = __double2loint(R), r1 = __double2hiint(R);
    asm("s_mov_b64 vcc, %10\n\ts_nop 1\n\tv_cndmask_b32_dpp %0, %6, %8, vcc" DMI_SHR "v_cndmask_b32_dpp %1, %7, %9, vcc" DMI_SHR
        "v_cndmask_b32_dpp %4, %4, %8, vcc" DMI_SHR "v_cndmask_b32_dpp %5, %5, %9, vcc" DMI_SHR
        "s_mov_b64 vcc, %11\n\tv_cndmask_b32_dpp %2, %8, %12, vcc" DMI_SHL "v_cndmask_b32_dpp %3, %9, %12, vcc" DMI_SHL
        : "=&v"(f0), "=&v"(f1), "=&v"(g0), "=&v"(g1), "+v"(r0), "+v"(r1)
        : "v"(__double2loint(Fr)), "v"(__double2hiint(Fr)), "v"(__double2loint(Fbr)), "v"(__double2hiint(Fbr)), "s"(first),
          "s"(last), "v"(0)
        : "vcc");
    F = __hiloint2double(f1, f0);
    Fb = __hiloint2double(g1, g0);
    R = __hiloint2double(r1, r0);
}
#undef DMI_SHR
#undef DMI_SHL

template <typename T, int LPC>
__device__ __forceinline__ void basis_rows(double sn_, double cs_, double m0_, double E1, cgdbl *E2, int m, int n, gdbl *A0) {
    using N = Num<T>;
    constexpr int G = kWave / LPC;  // curves side by side; each lane runs two
    const int L = lane_id(), h = L / LPC, s = L % LPC;
    const unsigned long long first = LPC == 64 ? 1ull : 0x100000001ull, last = LPC == 64 ? 1ull << 63 : 0x8000000080000000ull;
    const T sn = N::c(sn_), cs = N::c(cs_), m0 = N::c(m0_);
    const double E1sq = E1 * E1;
    const T d = cs * E1sq, zero = N::c(0.0);
#pragma unroll 1
    for (int jp = 0; jp < n; jp += 2 * G) {
        int j[2];
        T a[2], b[2], c[2], cp[2], mc[2], F[2], Fb[2], Z[2], R[2];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            j[q] = jp + q * G + h;
            const double e2 = E2[min(j[q], n - 1)], E2h = (e2 * e2) / 2, E1E2 = E1 * e2;
            a[q] = N::c(E2h);
            b[q] = cs * E2h;
            c[q] = sn * E1E2;
            cp[q] = (-c[q]) / 2.0;
            mc[q] = -c[q];
            F[q] = N::c(s == 0 ? 1.0 : 0.0);
            Fb[q] = Z[q] = R[q] = zero;
        }
#pragma unroll 1
        for (int i0 = 0; i0 < m; i0 += LPC) {
            const int cnt = min(LPC, m - i0), full = (i0 + cnt == m) ? cnt - 1 : cnt;
#pragma unroll 1
            for (int i = 0; i < full; ++i) {
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    const T C = F[q] + Fb[q], S = F[q] - Fb[q], Cp = a[q] * C, Sp = b[q] * S;
                    const T Fr = tfma(c[q], Z[q], Cp + Sp), Fbr = tfma(mc[q], Z[q], Cp - Sp);
                    Z[q] = tfma(cp[q], S, d * Z[q]);
                    shift_states(Fr, Fbr, F[q], Fb[q], R[q], first, last);
                }
            }
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                if (full < cnt) {  // the train's last echo
                    const T C = F[q] + Fb[q], S = F[q] - Fb[q];
                    T f, g;
                    shift_states(zero, tfma(mc[q], Z[q], tfma(a[q], C, -(b[q] * S))), f, g, R[q], first, last);
                }
                // lane s holds echo i0 + cnt - 1 - s
                if (s < cnt && j[q] < n) A0[(i0 + cnt - 1 - s) * n + j[q]] = N::val(tabs(m0 * R[q]));
            }
        }
    }
}
__device__ __attribute__((noinline)) void basis_rows_call(int fp32, double alpha_, double E1_, cgdbl *E2_, int dims_, gdbl *A0_) {
    const double alpha = rfl(alpha_), E1 = rfl(E1_);
    cgdbl *E2 = rflp(E2_);
    gdbl *A0 = rflp(A0_);
    const int dims = rfl(dims_), m = dims & 255, n = dims >> 8;
    // the angle in radians rounded to the recursion's type, its sine and cosine rounded once more there (tsincos)
    const bool f32 = rfl(fp32) != 0;
    const double al = alpha * kDeg2Rad, m0 = dsind(alpha / 2);
    double sn, cs;
    sincos(f32 ? (double)(float)al : al, &sn, &cs);
    if (f32) {
        if (m / 2 + 2 <= 32) basis_rows<float, 32>(sn, cs, m0, E1, E2, m, n, A0);
        else basis_rows<float, 64>(sn, cs, m0, E1, E2, m, n, A0);
    } else {
        if (m / 2 + 2 <= 32) basis_rows<double, 32>(sn, cs, m0, E1, E2, m, n, A0);
        else basis_rows<double, 64>(sn, cs, m0, E1, E2, m, n, A0);
    }
}

// Wave state of the register-resident kernel, with the interface of Wave that the searches use.
template <int S> struct RegWave {
    ldbl *lds, *x, *b, *cmu, *crn, *csemi, *G;
    gdbl *xf, *b0, *cx, *A0s, *lc;
    cgdbl *A0;   // basis used by the regularization solves, row-major m x n
    ldbl *spt, *spc;  // the legacy path is memory-resident: unused
    int m, n, L, idxl, ccur;
    unsigned long long flops, flops32, solves, nfailed;
    int status;
    bool failed, over;  // over: a solve's window outgrew the registers, the voxel is left to the memory-resident kernel

    static constexpr bool kRowMajor = true;
    __device__ __forceinline__ double basis(int i, int j) const { return A0[i * n + j]; }
    __device__ __forceinline__ int basis_cs() const { return 1; }
    __device__ __forceinline__ int basis_rs() const { return n; }
    // GCV's Gram matrix: columns of odd stride over the factor's region, formed from the basis in global memory (L2)
    __device__ __forceinline__ void gram_begin() { lds_order(); }
    __device__ __forceinline__ double gram_basis(int i, int j) const { return A0[i * n + j]; }
    __device__ __forceinline__ ldbl &gram_at(int r, int c) { return G[c * (min(m, n) | 1) + r]; }
    __device__ __forceinline__ bool redo() const { return over; }
    __device__ __forceinline__ void begin_voxel() { over = false; }
    __device__ __forceinline__ bool basis_const(bool fp32, double alpha, double E1, cgdbl *E2, gdbl *A0out) {
        basis_rows_call(fp32, alpha, E1, E2, m | (n << 8), A0out);
        return true;
    }

    __device__ __forceinline__ void solve(cgdbl *A0g, bool tikh, double mu, int &nsetp, double &rnorm) {
        nsetp = 0;
        rnorm = 0.0;
        if (over) return;
        DMI_PT0();
        const RegSolve r = nnls_reg<S>(A0g, b0, lds, m | (n << 8) | ((int)tikh << 16), mu);
        DMI_PT1(kPhNnls);
        nsetp = rfl(r.nsetp);
        rnorm = rfl(r.rnorm);
        idxl = r.idxl;
        const int fl = rfl(r.flags);
        if (fl & kRegMaxIter) status |= kStatusNnlsMaxIter;
        over = (fl & kRegOverflow) != 0;
        flops += (unsigned)rfl((int)r.flops);
        solves += 1;
    }

    // the Tikhonov cache of Wave (src/lsqnonneg.jl:392-444)
    __device__ __forceinline__ void cache_reset() {
        if (L < kTikhCache) cmu[L] = NAN;
        lds_order();
    }
    __device__ __forceinline__ int cache_solve(double mu) {
        int hit = -1, emp = -1;
        for (int i = 0; i < kTikhCache; ++i) {
            const double c = rfl(cmu[i]);
            if (hit < 0 && !isnan(c) && c == mu) hit = i;
            if (emp < 0 && isnan(c)) emp = i;
        }
        if (hit >= 0) { ccur = hit; return hit; }
        const int slot = emp >= 0 ? emp : ((ccur + 1) % kTikhCache);
        ccur = slot;
        int ns;
        double rn;
        solve(A0, true, mu, ns, rn);
        const double v = (L < ns) ? x[idxl] : 0.0;
        const double semi = wsum(v * v);
        if (L < n) cx[slot * n + L] = x[L];
        if (L == 0) { cmu[slot] = mu; crn[slot] = rn; csemi[slot] = semi; }
        __syncthreads();
        return slot;
    }
    __device__ __forceinline__ double cur_mu() { return rfl(cmu[ccur]); }
    __device__ __forceinline__ double cur_semi() { return rfl(csemi[ccur]); }
    __device__ __forceinline__ double cur_resnorm_sq() {
        const double mu = cur_mu(), rn = rfl(crn[ccur]);
        return jl_max(rn * rn - (mu * mu) * cur_semi(), 0.0);
    }
    __device__ __forceinline__ void take_cur_solution() {
        if (L < n) xf[L] = cx[ccur * n + L];
        __syncthreads();
    }
    __device__ __forceinline__ double plain_solve_to_xf() {
        int ns;
        double rn;
        solve(A0, false, 0.0, ns, rn);
        if (L < n) xf[L] = x[L];
        __syncthreads();
        return rn;
    }
    __device__ __forceinline__ double plain_solve_res2(int &ns) {
        double rn;
        solve(A0, false, 0.0, ns, rn);
        return rn * rn;
    }
};

// Chunked forward of the KDA operator (the gated delta rule with a decay per key feature), 64-token chunks, K, V <= 128
// (zero-padded to 128 by the host).  Replaces chunk_kda_fwd (fla/ops/kda/chunk_fwd.py:20-134): the gate activation and
// chunk-local cumsum (fla/ops/kda/gate.py), the intra-chunk stage (fla/ops/kda/chunk_intra.py), recompute_w_u_fwd
// (fla/ops/kda/wy_fast.py), chunk_gated_delta_rule_fwd_h and chunk_gla_fwd_o_gk.  Two kernels:
//
//   prepare  per (chunk, v-head): Gam = cumsum of the log decays inside the chunk [64][K];
//            M_ij = sum_k k_ik k_jk e^(Gam_ik - Gam_jk) (i > j),  P_ij = scale sum_k q_ik k_jk e^(Gam_ik - Gam_jk) (i >= j);
//            A = (I + diag(beta) M)^-1,  w = A (beta k e^Gam),  u = A (beta v);
//            also qg = scale q e^Gam, kg = k e^(Gam_last - Gam), e^Gam_last: what the scan needs, so that it never sees a gate
//   scan     per (sequence, v-head, VBT value columns), chunks in order, state slice in registers:
//            v_new = u - w S;  o = qg S + P v_new;  S <- diag(e^Gam_last) S + kg^T v_new
//
// The exponent Gam_ik - Gam_jk is only ever non-positive for i >= j, but it cannot be split into a factor of row i and a
// factor of row j without overflow unless a reference row lies between them.  Blocks of 16 rows: for j in an earlier
// block than i the reference is the last row in front of i's block, e^(Gam_i - ref) e^(ref - Gam_j) with both exponents <= 0,
// and the products run on the matrix cores; inside a 16 x 16 diagonal block every pair gets its own exponentials
// (the reference does the same, fla/ops/kda/chunk_intra.py: sub-chunks of 16).
//
// The comba operator (one decay per token and head, a second key p for the prediction, which sees the state before the
// token's decay; fla/ops/comba/chunk.py:22-90) has a prepare kernel of its own that writes the same per-chunk operands,
// and shares the scan:  M_ij = (p_i . k_j) e^(Gam0_i - Gam_j) with Gam0 = Gam - g,  w = A (beta p e^Gam0).
#include "gdn_chunk_kda.h"

namespace gdn {

// ---------------------------------------------------------------------------------------------
// prepare
// ---------------------------------------------------------------------------------------------
// Two workgroups share a CU (80 KB of LDS each; a workgroup's phases are chains of dependent steps that leave most of a CU idle).
// Wave w owns the rows 16w .. of the chunk: q and k are matrix-core operand fragments (row 16w + c16, features 32s + 8g ..) from the load on,
// and every decay of a row is a product of two per element,
//     f = e^(Gam_i - R) (R: the row in front of the block)   and   h = e^(E - Gam_i) (E: the block's last row),
// with factors per feature between the ends of the blocks (seven rows of 128, once per unit): k f and q f meet k h of the earlier blocks,
// k / f of their own; e^Gam_i = f e^R, e^(Gam_last - Gam_i) = h e^(Gam_last - E).  The blocks 2 and 3 meet the rows 0 .. 31 with the
// decay to row 31 on them, which is block 2's reference; only block 3 needs k f and q f a second time.  All exponents but that of 1 / f are <= 0, so
// that a factor that underflows stands for a product that does.  What leaves does so as whole rows: through rows of LDS that only the
// wave itself uses by then.
// Bound by the rate at which two waves per SIMD issue vector instructions: with exponentials for every pair of blocks and every use, six to
// eight per element, 592 us at 8192 tokens, 96 heads; with these two 446 us (1.96 GB, 4.4 TB/s), in the backward pass, where A and Gam
// leave as well, 490 us (2.47 GB, 5.0 TB/s).
static_assert(64 * PL * 4 == 64 * P128 * 2, "the rows of v, and on their way out qg and kg, take the place of the matrix L, row by row");
static_assert(10 * BD * 4 <= 64 * P64 * 2, "the factors per feature lie where A will");
constexpr size_t KDA_PREP_SMEM = (2 * 64 * P128 + 64 * P64) * 2 + (64 * PG + 64) * 4;

template <typename T>
__global__ __launch_bounds__(256, 2) void gdn_kda_prepare_kernel(KdaParams p, int64_t units) {
    typedef typename Mma<T>::V8 V8;
    typedef typename Mma<T>::V4 V4;
    extern __shared__ __align__(16) char smem[];
    T* sK = (T*)smem; T* sV = sK + 64 * P128; T* sA = sV + 64 * P128;
    float* sL = (float*)sV;
    float* sF = (float*)sA;                                     // ones, e^R of blocks 1 .. 3, e^(Gam_last - E) of blocks 0 .. 2, the decays across blocks 1 and 2, zeros
    float* sG = (float*)(sA + 64 * P64); float* sBeta = sG + 64 * PG;      // (Gam / ln 2: every decay is one exp2)
    // (the later row blocks meet more of the earlier ones: of the two workgroups of a CU one takes the blocks in reverse, so that every
    // SIMD gets as much)
    const bool flip = blockIdx.x >= 256;

    // A workgroup walks over the units; the next unit's rows are fetched into registers meanwhile.
    TileRegs<BD> rV;
    V8 rK[4], rQ[4];                                            // row 16w + c16, features 32s + 8g .. + 7
    float rG[32];                                               // gates: a thread per key feature and half of the chunk's rows
    uint32_t rB = 0;                                            // (raw bits: converted when the unit's turn comes)
    // (the lane number is an argument: inside the loop over the units it is the opaque copy, see there)
    auto block_of = [&](int tid) { const int w = __builtin_amdgcn_readfirstlane(tid >> 6); return flip ? 3 - w : w; };
    auto fetch_v = [&](int64_t u, int tid) {
        const UnitAt at = unit_at(p, u);
        fetch_tile<BD>(rV, (const T*)p.v + (at.c.tok0 * p.HV + at.hv) * BD, (int64_t)p.HV * BD, at.c.valid, tid);
    };
    auto fetch = [&](int64_t u, int tid) {
        const int lane = tid & 63, row = 16 * block_of(tid) + (lane & 15), g = lane >> 4;
        const UnitAt at = unit_at(p, u);
        const int64_t off = ((at.c.tok0 + row) * p.H + at.hq) * BD + 8 * g;
        if (at.c.valid == CH) {
#pragma unroll
            for (int s = 0; s < 4; ++s) { rK[s] = *(const V8*)((const T*)p.k + off + 32 * s); rQ[s] = *(const V8*)((const T*)p.q + off + 32 * s); }
        } else {
#pragma unroll
            for (int s = 0; s < 4; ++s) {
#pragma unroll
                for (int e = 0; e < 8; ++e) rK[s][e] = rQ[s][e] = (T)0.f;
                if (row < at.c.valid) { rK[s] = *(const V8*)((const T*)p.k + off + 32 * s); rQ[s] = *(const V8*)((const T*)p.q + off + 32 * s); }
            }
        }
        rB = (tid < 64 && tid < at.c.valid) ? load_scalar_bits(p.beta, (at.c.tok0 + tid) * p.HV + at.hv, p.gb_dtype) : 0;
    };
    auto fetch_g = [&](int64_t u, int tid) {
        const UnitAt at = unit_at(p, u);
        const int col = tid & 127, half = tid >> 7;
        const float* gp = p.g + ((at.c.tok0 + 32 * half) * p.HV + at.hv) * BD + col;
#pragma unroll
        for (int r = 0; r < 32; ++r) rG[r] = 32 * half + r < at.c.valid ? gp[(int64_t)r * p.HV * BD] : 0.f;
    };
    fetch(blockIdx.x, threadIdx.x);
    for (int64_t u = blockIdx.x; u < units; u += gridDim.x) {
    // (everything derived from the lane number is derived again per unit from a copy the compiler cannot see through: hoisted out
    // of this loop, the addresses of its fully unrolled body would fill the register file before the loop starts, and spill)
    int tid_opaque = threadIdx.x;
    asm volatile("" : "+v"(tid_opaque));
    const int tid = tid_opaque, lane = tid & 63, c16 = lane & 15, g = lane >> 4;
    const int w = block_of(tid);
    const UnitAt at = unit_at(p, u);
    const int hv = at.hv;
    const ChunkAt c = at.c;
    const int i = 16 * w + c16;                                 // the row this lane's operand fragments belong to
    fetch_g(u, tid);                                            // (the gates are not fetched ahead: no 32 registers to carry them round the loop)
    V8 kx[4], qx[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) { kx[s] = rK[s]; qx[s] = rQ[s]; }
    if (tid < 64) {
        float b = scalar_of_bits(rB, p.gb_dtype);
        if ((p.flags & GDN_FLAG_BETA_SIGMOID) && tid < c.valid) b = sigmoid_f(b) * ((p.flags & GDN_FLAG_NEG_EIGVAL) ? 2.f : 1.f);
        sBeta[tid] = b;
    }
    if (p.flags & GDN_FLAG_QK_L2NORM) {
        // rows of q and k divided by sqrt(sum x^2 + 1e-6): the four lanes that share c16 hold a row
        float sk = 0.f, sq = 0.f;
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int e = 0; e < 8; ++e) { sk += (float)kx[s][e] * (float)kx[s][e]; sq += (float)qx[s][e] * (float)qx[s][e]; }
        const float rk = rsqrtf(sum_over_g(sk) + 1e-6f), rq = rsqrtf(sum_over_g(sq) + 1e-6f);
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int e = 0; e < 8; ++e) { kx[s][e] = (T)((float)kx[s][e] * rk); qx[s][e] = (T)((float)qx[s][e] * rq); }
    }
    {
        // running sums of the gates inside each half of the rows first
        const int col = tid & 127, half = tid >> 7;
        const float a_k = p.gk_act ? (p.A_log ? __expf(p.A_log[hv]) : (p.gk_act == 2 ? 1.f : __expf(1.f))) : 0.f;
        const float bias = (p.gk_act && p.gk_bias) ? p.gk_bias[hv * BD + col] : 0.f;
        if (p.gk_act) {
#pragma unroll
            for (int r = 0; r < 32; ++r) {
                if (32 * half + r >= c.valid) break;
                const float gt = rG[r] + bias;
                rG[r] = p.gk_act == 2 ? p.gk_lower * sigmoid_f(a_k * gt) : -a_k * softplus_f(gt);
                __builtin_amdgcn_sched_barrier(0);              // (one row at a time: 32 activations in flight at once cost 100 registers)
            }
        }
        // (after a mask of the type's lowest value the sums must stay numbers whose differences are numbers, also divided by ln 2: e to this is 0 as
        // well.  `maximum`, not fmaxf: a NaN stays one)
        constexpr float LOWEST = -1e36f;
        float run = 0.f;
#pragma unroll
        for (int r = 0; r < 32; ++r) {
            run = __builtin_elementwise_maximum(run + rG[r], LOWEST);
            sG[(32 * half + r) * PG + col] = run * RCP_LN2_F;
        }
    }
    lds_barrier();
    if (tid >> 7) {
        // second half of the rows: add the first half's total; and the factors between the ends of the blocks
        const int col = tid & 127;
        float* gc = sG + col;
        const float G15 = gc[15 * PG], G31 = gc[31 * PG];
#pragma unroll
        for (int r = 0; r < 32; ++r) gc[(32 + r) * PG] += G31;
        const float G47 = gc[47 * PG], G63 = gc[63 * PG];
        sF[0 * BD + col] = 1.f;
        sF[1 * BD + col] = fast_exp2(G15); sF[2 * BD + col] = fast_exp2(G31); sF[3 * BD + col] = fast_exp2(G47);
        sF[4 * BD + col] = fast_exp2(G63 - G15); sF[5 * BD + col] = fast_exp2(G63 - G31); sF[6 * BD + col] = fast_exp2(G63 - G47);
        sF[7 * BD + col] = fast_exp2(G31 - G15); sF[8 * BD + col] = fast_exp2(G47 - G31);
        sF[9 * BD + col] = 0.f;
        p.ws.EGL[u * BD + col] = fast_exp2(G63);
    }
    lds_barrier();

    // ---- every row's factors; qg and kg leave, k h goes to LDS for the later blocks ----
    const float bi = sBeta[i];
    float f[4][8];
    V8 kw[4];                                                   // beta k e^Gam, the factor of w
    V8 kd[4], qd[4];                                            // k f, q f
    // 16 rows of 128 through this wave's own rows of LDS
    auto rows_out = [&](T* rows) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        u32x4 x[4];
#pragma unroll
        for (int n = 0; n < 4; ++n) x[n] = *(const u32x4*)(sV + (16 * w + (lane >> 4) + 4 * n) * P128 + (lane & 15) * 8);
#pragma unroll
        for (int n = 0; n < 4; ++n) *(u32x4*)(rows + (16 * w + (lane >> 4) + 4 * n) * BD + (lane & 15) * 8) = x[n];
        asm volatile("" ::: "memory");
    };
    {
        const float* gi = sG + i * PG + 8 * g;
        const float* gr = (w > 0 ? sG + (16 * w - 1) * PG : sF + 9 * BD) + 8 * g;
        const float* ge = sG + (16 * w + 15) * PG + 8 * g;
        const float* t2 = sF + w * BD + 8 * g;                  // e^R
        const float* t1 = sF + (w < 3 ? 4 + w : 0) * BD + 8 * g;       // e^(Gam_last - E)
        const float* t0 = sF + (w == 0 ? 7 : 0) * BD + 8 * g;   // from the block's end to row 31, or to its end
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            __builtin_amdgcn_sched_barrier(0);
            V8 kn, kg, k1;
#pragma unroll
            for (int h4 = 0; h4 < 2; ++h4) {
                const int o = 32 * s + 4 * h4;
                const f32x4 G = *(const f32x4*)(gi + o), R = *(const f32x4*)(gr + o), E = *(const f32x4*)(ge + o);
                const f32x4 eR = *(const f32x4*)(t2 + o), eL = *(const f32x4*)(t1 + o), e1 = *(const f32x4*)(t0 + o);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int e = 4 * h4 + r;
                    f[s][e] = fast_exp2(G[r] - R[r]);
                    const float k = (float)kx[s][e], kh = k * fast_exp2(E[r] - G[r]), kf = k * f[s][e];
                    kd[s][e] = (T)kf;
                    qd[s][e] = (T)((float)qx[s][e] * f[s][e]);
                    kn[e] = (T)(kh * e1[r]);
                    k1[e] = (T)kh;
                    kg[e] = (T)(kh * eL[r]);
                    kw[s][e] = (T)(kf * (bi * eR[r]));
                }
            }
            // (with the decay to row 31 on block 0; to its own end, for block 1, in the rows of block 3, which no later block meets)
            if (w < 3) *(V8*)(sK + i * P128 + 32 * s + 8 * g) = kn;
            if (w == 0) *(V8*)(sK + (48 + i) * P128 + 32 * s + 8 * g) = k1;
            *(V8*)(sV + i * P128 + 32 * s + 8 * g) = kg;
        }
        rows_out((T*)p.ws.KG + u * 64 * BD);
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            V8 qg;
#pragma unroll
            for (int h4 = 0; h4 < 2; ++h4) {
                const f32x4 eR = *(const f32x4*)(t2 + 32 * s + 4 * h4);
#pragma unroll
                for (int r = 0; r < 4; ++r) { const int e = 4 * h4 + r; qg[e] = (T)((float)qx[s][e] * f[s][e] * (p.scale * eR[r])); }
            }
            *(V8*)(sV + i * P128 + 32 * s + 8 * g) = qg;
        }
        rows_out((T*)p.ws.QG + u * 64 * BD);
    }
    lds_barrier();

    // (the rows anew for every use that follows: converted once they would take 64 registers)
    auto anew = [&] {
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            u32x4 a = __builtin_bit_cast(u32x4, kx[s]), b = __builtin_bit_cast(u32x4, qx[s]);
            asm volatile("" : "+v"(a), "+v"(b));
            kx[s] = __builtin_bit_cast(V8, a); qx[s] = __builtin_bit_cast(V8, b);
        }
    };
    anew();
    // ---- M (as L = diag(beta) M, for the substitution) and P, this wave's 16 rows ----
    {
        T* Pu = (T*)p.ws.Pm + u * 64 * 64;
        // rows of this block against rows of an earlier block (at `at` in sK)
        auto pair = [&](int tj, int at) {
            __builtin_amdgcn_sched_barrier(0);
            f32x4 m = ZERO4, pt = ZERO4;
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const V8 kn = frag_rows(sK, P128, at, 32 * s, lane);
                m = Mma<T>::run(kd[s], kn, m);                 // lane: column j = 16tj + c16, rows i = 16w + 4g + r
                pt = Mma<T>::run(kn, qd[s], pt);               // lane: column i = 16w + c16, rows j = 16tj + 4g + r
            }
            const int j = 16 * tj + c16;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int ir = 16 * w + 4 * g + r;
                sL[ir * PL + (j & 3) * 16 + (j >> 2)] = sBeta[ir] * m[r];
            }
            *(V4*)(Pu + i * 64 + 16 * tj + 4 * g) = pack4<T>(pt * p.scale);
        };
        if (w == 1) pair(0, 48);
        else if (w == 2) { pair(0, 0); pair(1, 16); }
        else if (w == 3) pair(2, 32);
        // blocks to the right of the diagonal: zeros
#pragma unroll
        for (int tj = 1; tj < 4; ++tj)
            if (tj > w) *(V4*)(Pu + i * 64 + 16 * tj + 4 * g) = pack4<T>(ZERO4);
        // The diagonal block.  Where the decay across the block stays within what the operand type can hold as a factor
        // e^(R - Gam_j) >= 1 (the usual case), the same reference serves and the block is one more tile on the matrix
        // cores; otherwise every pair of rows gets its own exponentials.
        float span = 0.f;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int col = lane + 64 * h;
            span = fminf(span, sG[(16 * w + 15) * PG + col] - (w > 0 ? sG[(16 * w - 1) * PG + col] : 0.f));
        }
        anew();
        if (min_over_wave(span) >= SpanOk<T>::value) {
            f32x4 m = ZERO4, pt = ZERO4;
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                V8 kn;
#pragma unroll
                for (int e = 0; e < 8; ++e) kn[e] = (T)((float)kx[s][e] * __builtin_amdgcn_rcpf(f[s][e]));
                m = Mma<T>::run(kd[s], kn, m);                 // lane: column j = 16w + c16, rows i = 16w + 4g + r
                pt = Mma<T>::run(kn, qd[s], pt);               // lane: column i = 16w + c16, rows j = 16w + 4g + r
            }
            const int j = 16 * w + c16;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int ir = 16 * w + 4 * g + r;
                sL[ir * PL + (j & 3) * 16 + (j >> 2)] = ir > j ? sBeta[ir] * m[r] : 0.f;
                pt[r] = (16 * w + 4 * g + r) <= i ? pt[r] * p.scale : 0.f;
            }
            *(V4*)(Pu + i * 64 + 16 * w + 4 * g) = pack4<T>(pt);
        } else
        // (lane (c16, g) takes row i against every row j of the block over the features of its own fragments, row j's from the lane
        // that holds them; the four lanes that share a row add up)
        {
#pragma unroll 1
            for (int jl = 0; jl < 16; ++jl) {
                const int rj = 16 * w + jl;
                float mj = 0.f, pj = 0.f;
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    // (the rows and their place anew every time: converted once they would take the registers of the whole kernel)
                    u32x4 bits = __builtin_bit_cast(u32x4, kx[s]), qbits = __builtin_bit_cast(u32x4, qx[s]);
                    int row = i;
                    asm volatile("" : "+v"(bits), "+v"(qbits), "+v"(row));
                    const V8 ki = __builtin_bit_cast(V8, bits), qi = __builtin_bit_cast(V8, qbits);
#pragma unroll
                    for (int n = 0; n < 4; ++n) bits[n] = (uint32_t)__shfl((int)bits[n], (lane & 48) + jl, 64);
                    const V8 kj = __builtin_bit_cast(V8, bits);
                    const float* gi = sG + row * PG + 32 * s + 8 * g;
                    const float* gj = sG + rj * PG + 32 * s + 8 * g;
                    if (jl <= c16) {
#pragma unroll
                        for (int e = 0; e < 8; ++e) {
                            const float kk = (float)kj[e] * fast_exp2(gi[e] - gj[e]);
                            mj += (float)ki[e] * kk;
                            pj += (float)qi[e] * kk;
                        }
                    }
                }
                mj = sum_over_g(mj); pj = sum_over_g(pj);
                if (g == 0) {
                    sL[i * PL + (rj & 3) * 16 + (rj >> 2)] = jl < c16 ? sBeta[i] * mj : 0.f;
                    Pu[i * 64 + rj] = (T)(jl <= c16 ? p.scale * pj : 0.f);
                }
            }
        }
        if (w == 3) {
            // the rows 0 .. 31: the decay across block 2 lies between
            anew();
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int h4 = 0; h4 < 2; ++h4) {
                    __builtin_amdgcn_sched_barrier(0);
                    const f32x4 F = *(const f32x4*)(sF + 8 * BD + 32 * s + 8 * g + 4 * h4);
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int e = 4 * h4 + r;
                        const float x = f[s][e] * F[r];
                        kd[s][e] = (T)((float)kx[s][e] * x);
                        qd[s][e] = (T)((float)qx[s][e] * x);
                    }
                }
            pair(0, 0); pair(1, 16);
        }
    }
    lds_barrier();
    fetch_v(u, tid);
    solve_unit_lower_blocks<T>(sL, (float*)sA, sA, w, lane);
    lds_barrier();
    if (p.ws.Am) {                                              // (for the backward pass; A: this wave's own rows)
        T* Au = (T*)p.ws.Am + u * 64 * 64;
        float* Gu = p.ws.Gk + u * 64 * BD;
#pragma unroll
        for (int n = 0; n < 2; ++n) {
            const int row = 16 * w + 8 * n + (lane >> 3), pc = lane & 7;
            *(u32x4*)(Au + row * 64 + pc * 8) = *(const u32x4*)(sA + row * P64 + pc * 8);
        }
#pragma unroll
        for (int n = 0; n < 8; ++n) {
            const int idx = tid + 256 * n, row = idx >> 5, pc = idx & 31;
            *(f32x4*)(Gu + row * BD + pc * 4) = *(const f32x4*)(sG + row * PG + pc * 4);
        }
    }
    // the factors of w and u (that of u in the place of L: the substitution is over); beta goes onto them and not onto A, whose
    // rounded entries the backward pass takes as they are: with other ones the parts of dGk would not cancel
#pragma unroll
    for (int s = 0; s < 4; ++s) *(V8*)(sK + i * P128 + 32 * s + 8 * g) = kw[s];
#pragma unroll
    for (int n = 0; n < 4; ++n) {
        const float b = sBeta[(tid >> 4) + 16 * n];
        V8 vx = __builtin_bit_cast(V8, rV.x[n]);
#pragma unroll
        for (int e = 0; e < 8; ++e) vx[e] = (T)((float)vx[e] * b);
        rV.x[n] = __builtin_bit_cast(u32x4, vx);
    }
    put_tile<BD>(sV, P128, rV, tid);
    // (the next unit's rows: requested this late because the phases above have no registers to spare under the cap that lets two
    // workgroups share a CU; the other workgroup covers the wait)
    fetch(u + gridDim.x < units ? u + gridDim.x : u, tid);
    lds_barrier();
    {
        // w^T and u^T tiles: features on the rows, this wave's 16 tokens on the columns; 64 features at a time they leave through this
        // wave's own rows of A, which it has read
        V8 fa[2];
#pragma unroll
        for (int s = 0; s < 2; ++s) fa[s] = frag_rows(sA, P64, 16 * w, 32 * s, lane);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
        for (int q4 = 0; q4 < 4; ++q4) {
            const T* rows = q4 < 2 ? sK : sV;
            T* out = (T*)(q4 < 2 ? p.ws.Wm : p.ws.Um) + u * 64 * BD + 64 * (q4 & 1);
#pragma unroll
            for (int n = 0; n < 4; ++n) {
                f32x4 acc = ZERO4;
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    if (2 * s > w) continue;                    // A is lower triangular
                    acc = Mma<T>::run(frag_cols(rows, P128, 32 * s, 64 * (q4 & 1) + 16 * n, lane), fa[s], acc);
                }
                *(V4*)(sA + i * P64 + 16 * n + 4 * g) = pack4<T>(acc);
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
            for (int n = 0; n < 2; ++n) {
                const int row = 16 * w + 8 * n + (lane >> 3), pc = lane & 7;
                *(u32x4*)(out + row * BD + pc * 8) = *(const u32x4*)(sA + row * P64 + pc * 8);
            }
            asm volatile("" ::: "memory");
        }
    }
    lds_barrier();
    }
}

// ---------------------------------------------------------------------------------------------
// prepare, comba
// ---------------------------------------------------------------------------------------------
constexpr size_t COMBA_PREP_SMEM = (4 * 64 * P128 + 64 * P64) * 2 + 3 * 64 * 4;
static_assert(64 * PL * 4 <= 64 * P128 * 2, "the matrix L takes the place of the q tile");

template <typename T>
__global__ __launch_bounds__(256, 2) void gdn_comba_prepare_kernel(KdaParams p, int64_t units) {
    typedef typename Mma<T>::V8 V8;
    typedef typename Mma<T>::V4 V4;
    extern __shared__ __align__(16) char smem[];
    T* sK = (T*)smem; T* sQ = sK + 64 * P128; T* sP = sQ + 64 * P128; T* sV = sP + 64 * P128; T* sA = sV + 64 * P128;
    float* sGam = (float*)(sA + 64 * P64); float* sGam0 = sGam + 64; float* sBeta = sGam0 + 64;
    float* sL = (float*)sQ;                                     // once q has been used
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, c16 = lane & 15, g = lane >> 4;

    // Two workgroups per CU walk over the units; the next unit's rows and gates are fetched into registers meanwhile.
    TileRegs<BD> rK, rQ, rP, rV;
    uint32_t rG = 0, rB = 0;                                    // (raw bits: converted when the unit's turn comes)
    auto fetch_v = [&](int64_t u) {                             // (on its own, later than the rest: fewer registers live across the substitution)
        const int hv = (int)(u % p.HV);
        const ChunkAt c = chunk_at(p, u / p.HV);
        fetch_tile<BD>(rV, (const T*)p.v + (c.tok0 * p.HV + hv) * BD, (int64_t)p.HV * BD, c.valid, tid);
    };
    auto fetch = [&](int64_t u) {
        const int hv = (int)(u % p.HV), hq = hv / (p.HV / p.H);
        const ChunkAt c = chunk_at(p, u / p.HV);
        fetch_tile<BD>(rK, (const T*)p.k + (c.tok0 * p.H + hq) * BD, (int64_t)p.H * BD, c.valid, tid);
        fetch_tile<BD>(rQ, (const T*)p.q + (c.tok0 * p.H + hq) * BD, (int64_t)p.H * BD, c.valid, tid);
        fetch_tile<BD>(rP, (const T*)p.pk + (c.tok0 * p.H + hq) * BD, (int64_t)p.H * BD, c.valid, tid);
        const bool have = tid < 64 && tid < c.valid;
        rG = have ? load_scalar_bits(p.gs, (c.tok0 + tid) * p.HV + hv, p.gb_dtype) : 0;
        rB = have ? load_scalar_bits(p.beta, (c.tok0 + tid) * p.HV + hv, p.gb_dtype) : 0;
    };
    fetch(blockIdx.x);
    fetch_v(blockIdx.x);
    for (int64_t u = blockIdx.x; u < units; u += gridDim.x) {
    // (everything derived from the lane number is derived again per unit from a copy the compiler cannot see through: hoisted
    // out of this loop, the addresses of its unrolled body would fill the register file and spill)
    int tid_opaque = threadIdx.x;
    asm volatile("" : "+v"(tid_opaque));
    const int tid = tid_opaque, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), c16 = lane & 15, g = lane >> 4;
    put_tile<BD>(sK, P128, rK, tid);
    put_tile<BD>(sQ, P128, rQ, tid);
    put_tile<BD>(sP, P128, rP, tid);
    put_tile<BD>(sV, P128, rV, tid);
    if (w == 0) {
        const float g_own = scalar_of_bits(rG, p.gb_dtype);
        float run = g_own;                                      // running sum over the chunk's tokens (rows past the end add 0)
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const float t = __shfl_up(run, off, 64);
            if (lane >= off) run += t;
        }
        sGam[lane] = run;
        sGam0[lane] = run - g_own;
        sBeta[lane] = scalar_of_bits(rB, p.gb_dtype);
    }
    lds_barrier();
    if (u + gridDim.x < units) fetch(u + gridDim.x);
    if (p.flags & GDN_FLAG_QK_L2NORM) {
        // rows of q, k and p divided by sqrt(sum x^2 + 1e-6): 16 consecutive lanes hold the 16 pieces of a row
#pragma unroll 2
        for (int i = 0; i < 4; ++i) {
            const int row = (tid >> 4) + 16 * i, pc = tid & 15;
#pragma unroll
            for (int which = 0; which < 3; ++which) {
                T* at = (which == 0 ? sK : which == 1 ? sQ : sP) + row * P128 + pc * 8;
                V8 x = *(V8*)at;
                float ss = 0.f;
#pragma unroll
                for (int e = 0; e < 8; ++e) ss += (float)x[e] * (float)x[e];
                const float r = rsqrtf(sum_over_c16(ss) + 1e-6f);
#pragma unroll
                for (int e = 0; e < 8; ++e) x[e] = (T)((float)x[e] * r);
                *(V8*)at = x;
            }
        }
        lds_barrier();
    }
    const float gl = sGam[63];
    {
        // P, this wave's 16 rows; and what the scan needs of q and k
        T* Pu = (T*)p.ws.Pm + u * 64 * 64;
        const int i = 16 * w + c16;
        V8 qf[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) qf[s] = frag_rows(sQ, P128, 16 * w, 32 * s, lane);
        const float gam_i = sGam[i];
#pragma unroll
        for (int tj = 0; tj < 4; ++tj) {
            if (tj > w) { *(V4*)(Pu + i * 64 + 16 * tj + 4 * g) = pack4<T>(ZERO4); continue; }
            f32x4 pt = ZERO4;
#pragma unroll
            for (int s = 0; s < 4; ++s)
                pt = Mma<T>::run(frag_rows(sK, P128, 16 * tj, 32 * s, lane), qf[s], pt);     // lane: column i = 16w + c16, rows j = 16tj + 4g + r
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int jr = 16 * tj + 4 * g + r;
                pt[r] = jr <= i ? p.scale * pt[r] * __expf(gam_i - sGam[jr]) : 0.f;
            }
            *(V4*)(Pu + i * 64 + 16 * tj + 4 * g) = pack4<T>(pt);
        }
        T* QGu = (T*)p.ws.QG + u * 64 * BD;
        T* KGu = (T*)p.ws.KG + u * 64 * BD;
#pragma unroll 2                                        // (unrolled fully, the kernel spills registers)
        for (int it = 0; it < 4; ++it) {
            const int row = (tid >> 4) + 16 * it, pc = tid & 15;
            V8 kx = *(V8*)(sK + row * P128 + pc * 8), qx = *(V8*)(sQ + row * P128 + pc * 8);
            const float fk = __expf(gl - sGam[row]), fq = p.scale * __expf(sGam[row]);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                kx[e] = (T)((float)kx[e] * fk);
                qx[e] = (T)((float)qx[e] * fq);
            }
            *(V8*)(KGu + row * BD + pc * 8) = kx;
            *(V8*)(QGu + row * BD + pc * 8) = qx;
        }
        if (tid < BD) p.ws.EGL[u * BD + tid] = __expf(gl);
    }
    lds_barrier();                                              // q is done with: L takes its place
    {
        // L = diag(beta) M for the substitution, this wave's 16 rows
        V8 pf[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) pf[s] = frag_rows(sP, P128, 16 * w, 32 * s, lane);
#pragma unroll
        for (int tj = 0; tj < 4; ++tj) {
            if (tj > w) continue;
            f32x4 m = ZERO4;
#pragma unroll
            for (int s = 0; s < 4; ++s)
                m = Mma<T>::run(pf[s], frag_rows(sK, P128, 16 * tj, 32 * s, lane), m);       // lane: column j = 16tj + c16, rows i = 16w + 4g + r
            const int j = 16 * tj + c16;
            const float gam_j = sGam[j];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int ir = 16 * w + 4 * g + r;
                sL[ir * PL + (j & 3) * 16 + (j >> 2)] = ir > j ? sBeta[ir] * m[r] * __expf(sGam0[ir] - gam_j) : 0.f;
            }
        }
    }
    lds_barrier();
    solve_unit_lower_blocks<T>(sL, (float*)sA, sA, w, lane);
    {
        // p, v as the factors of w, u
#pragma unroll 2                                        // (unrolled fully, the kernel spills registers)
        for (int it = 0; it < 4; ++it) {
            const int row = (tid >> 4) + 16 * it, pc = tid & 15;
            V8 px = *(V8*)(sP + row * P128 + pc * 8), vx = *(V8*)(sV + row * P128 + pc * 8);
            const float b = sBeta[row], fp = b * __expf(sGam0[row]);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                px[e] = (T)((float)px[e] * fp);
                vx[e] = (T)((float)vx[e] * b);
            }
            *(V8*)(sP + row * P128 + pc * 8) = px;
            *(V8*)(sV + row * P128 + pc * 8) = vx;
        }
    }
    lds_barrier();
    if (u + gridDim.x < units) fetch_v(u + gridDim.x);
    {
        // w^T and u^T tiles: features on the rows, this wave's 16 tokens on the columns
        T* Wu = (T*)p.ws.Wm + u * 64 * BD;
        T* Uu = (T*)p.ws.Um + u * 64 * BD;
        const int i = 16 * w + c16;
        V8 fa[2];
#pragma unroll
        for (int s = 0; s < 2; ++s) fa[s] = frag_rows(sA, P64, 16 * w, 32 * s, lane);
#pragma unroll
        for (int n = 0; n < 8; ++n) {
            f32x4 aw = ZERO4, au = ZERO4;
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                if (2 * s > w) continue;                        // A is lower triangular
                aw = Mma<T>::run(frag_cols(sP, P128, 32 * s, 16 * n, lane), fa[s], aw);
                au = Mma<T>::run(frag_cols(sV, P128, 32 * s, 16 * n, lane), fa[s], au);
            }
            *(V4*)(Wu + i * BD + 16 * n + 4 * g) = pack4<T>(aw);
            *(V4*)(Uu + i * BD + 16 * n + 4 * g) = pack4<T>(au);
        }
    }
    lds_barrier();
    }
}

// ---------------------------------------------------------------------------------------------
// scan: the state slice [128][VBT] lives in registers as transposed tiles (wave w: key rows 32w .. 32w+31 as two tiles a2,
// lane (c16, g): key 16(2w+a2) + c16, value columns 16b + 4g .. +3); the next chunk's tiles are fetched into registers
// while the current chunk is computed.  64 and 128 columns: eight waves, two per SIMD, waves w and w + 4 the same rows of either
// half of the columns (with four, nothing covers a step's chains and barriers: 8192 tokens,
// 96 heads 345 -> 313 us; 4 x 2000 tokens, 64 heads, 128 columns 164 -> 153.  At 64 runs 32 columns stay the better ones: the step 1141 against 1158 us).
// ---------------------------------------------------------------------------------------------
// (u comes in, and o leaves, as whole rows through LDS tiles of their own: the lanes that hold them as matrix-instruction operands
// and results would move 8-byte pieces of 16 rows per instruction)
template <int VBT> constexpr size_t kda_scan_smem() { return (3 * 64 * P128 + 64 * P64 + BD * (VBT + 8) + 3 * 64 * (VBT + 8)) * 2 + (BD + 64) * 4; }

template <int VBT> constexpr int kda_scan_waves() { return VBT >= 64 ? 8 : 4; }

template <typename T, int VBT>
__global__ __launch_bounds__(64 * kda_scan_waves<VBT>()) void gdn_kda_scan_kernel(KdaParams p) {
    typedef typename Mma<T>::V8 V8;
    typedef typename Mma<T>::V4 V4;
    constexpr int NTH = 64 * kda_scan_waves<VBT>(), PV = VBT + 8, NVS = BD / VBT, NB = VBT / 16 / (NTH / 256);      // (16-column blocks of a wave)
    extern __shared__ __align__(16) char smem[];
    T* sW = (T*)smem; T* sKG = sW + 64 * P128; T* sQG = sKG + 64 * P128; T* sP = sQG + 64 * P128;
    T* sS = sP + 64 * P64; T* sVn = sS + BD * PV; T* sU = sVn + 64 * PV; T* sO = sU + 64 * PV;
    float* sE = (float*)(sO + 64 * PV);
    const int tid = threadIdx.x, lane = tid & 63, w = (tid >> 6) & 3, c16 = lane & 15, g = lane >> 4;
    const int wcol = 16 * NB * (tid >> 8);                       // first value column of this wave in the slice
    const int64_t run = (int64_t)(blockIdx.x / (8 * NVS)) * 8 + blockIdx.x % 8;       // (slices of one head on one XCD)
    if (run >= p.N * p.HV) return;
    const int vs = (blockIdx.x / 8) % NVS, hv = (int)(run % p.HV);
    const int64_t n = run / p.HV;
    const SeqAt sq = seq_at(p, n);
    const int vcol0 = vs * VBT;

    f32x4 S[2][NB];
#pragma unroll
    for (int a2 = 0; a2 < 2; ++a2)
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            const int kk = 16 * (2 * w + a2) + c16;
            S[a2][b] = p.h0 ? *(const f32x4*)(p.h0 + ((n * p.HV + hv) * BD + kk) * BD + vcol0 + wcol + 16 * b + 4 * g) : ZERO4;
        }
    TileRegs<BD, NTH> rW, rKG, rQG;
    TileRegs<CH, NTH> rP;
    TileRegs<VBT, NTH> rU;
    float rE = 0.f;
    auto fetch = [&](int64_t ic) {
        const int64_t u = (sq.cbase + ic) * p.HV + hv;
        fetch_tile<BD, NTH>(rW, (const T*)p.ws.Wm + u * 64 * BD, BD, 64, tid);
        fetch_tile<BD, NTH>(rKG, (const T*)p.ws.KG + u * 64 * BD, BD, 64, tid);
        fetch_tile<BD, NTH>(rQG, (const T*)p.ws.QG + u * 64 * BD, BD, 64, tid);
        fetch_tile<CH, NTH>(rP, (const T*)p.ws.Pm + u * 64 * 64, 64, 64, tid);
        if (tid < BD) rE = p.ws.EGL[u * BD + tid];
        fetch_tile<VBT, NTH>(rU, (const T*)p.ws.Um + u * 64 * BD + vcol0, BD, 64, tid);
    };
    if (sq.nc > 0) fetch(0);
    for (int64_t ic = 0; ic < sq.nc; ++ic) {
        const int64_t tok0 = sq.bos + ic * CH;
        const int valid = (int)min((int64_t)CH, sq.len - ic * CH);
        put_tile<BD, NTH>(sW, P128, rW, tid);
        put_tile<BD, NTH>(sKG, P128, rKG, tid);
        put_tile<BD, NTH>(sQG, P128, rQG, tid);
        put_tile<CH, NTH>(sP, P64, rP, tid);
        put_tile<VBT, NTH>(sU, PV, rU, tid);
        if (tid < BD) sE[tid] = rE;
#pragma unroll
        for (int a2 = 0; a2 < 2; ++a2)
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                const V4 s4 = pack4<T>(S[a2][b]);
                *(V4*)(sS + (16 * (2 * w + a2) + c16) * PV + wcol + 16 * b + 4 * g) = s4;
                if (p.hs) *(V4*)((T*)p.hs + (((sq.cbase + ic) * p.HV + hv) * BD + 16 * (2 * w + a2) + c16) * BD + vcol0 + wcol + 16 * b + 4 * g) = s4;
            }
        lds_barrier();
        if (ic + 1 < sq.nc) fetch(ic + 1);
        f32x4 oacc[NB];
        {
            // v_new^T and (qg S)^T tiles: value columns on the rows, this wave's 16 tokens on the columns
            const int i = 16 * w + c16;
            V8 wf[4], qf[4];
#pragma unroll
            for (int s = 0; s < 4; ++s) { wf[s] = frag_rows(sW, P128, 16 * w, 32 * s, lane); qf[s] = frag_rows(sQG, P128, 16 * w, 32 * s, lane); }
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                f32x4 acc = ZERO4;
                oacc[b] = ZERO4;
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    const V8 fs = frag_cols(sS, PV, 32 * s, wcol + 16 * b, lane);
                    acc = Mma<T>::run(fs, wf[s], acc);
                    oacc[b] = Mma<T>::run(fs, qf[s], oacc[b]);
                }
                const V4 u4 = *(const V4*)(sU + i * PV + wcol + 16 * b + 4 * g);
                f32x4 vn;
#pragma unroll
                for (int r = 0; r < 4; ++r) vn[r] = (float)u4[r] - acc[r];
                *(V4*)(sVn + i * PV + wcol + 16 * b + 4 * g) = pack4<T>(vn);
            }
        }
        lds_barrier();
        {
            // o += P v_new;  S <- diag(e^Gam_last) S + kg^T v_new
            const int i = 16 * w + c16;
            V8 pf[2], kf[2][2];
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                pf[s] = frag_rows(sP, P64, 16 * w, 32 * s, lane);
#pragma unroll
                for (int a2 = 0; a2 < 2; ++a2) kf[a2][s] = frag_cols(sKG, P128, 32 * s, 16 * (2 * w + a2), lane);
            }
#pragma unroll
            for (int a2 = 0; a2 < 2; ++a2) {
                const float e = sE[16 * (2 * w + a2) + c16];
#pragma unroll
                for (int b = 0; b < NB; ++b) S[a2][b] *= e;
            }
#pragma unroll
            for (int b = 0; b < NB; ++b) {
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    const V8 fv = frag_cols(sVn, PV, 32 * s, wcol + 16 * b, lane);
                    if (32 * s <= 16 * w + 15) oacc[b] = Mma<T>::run(fv, pf[s], oacc[b]);      // P[i][j] = 0 for j > i
#pragma unroll
                    for (int a2 = 0; a2 < 2; ++a2) S[a2][b] = Mma<T>::run(fv, kf[a2][s], S[a2][b]);
                }
                *(V4*)(sO + i * PV + wcol + 16 * b + 4 * g) = pack4<T>(oacc[b]);
            }
        }
        lds_barrier();
        copy_rows_out<64, VBT, NTH>((T*)p.o + (tok0 * p.HV + hv) * BD + vcol0, (int64_t)p.HV * BD, sO, PV, tid, valid);
    }
    if (p.ht) {
#pragma unroll
        for (int a2 = 0; a2 < 2; ++a2)
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                const int kk = 16 * (2 * w + a2) + c16;
                *(f32x4*)(p.ht + ((n * p.HV + hv) * BD + kk) * BD + vcol0 + wcol + 16 * b + 4 * g) = S[a2][b];
            }
    }
}

template <typename T>
static int launch_kda(const KdaParams& p, int64_t num_chunks, hipStream_t stream, bool comba = false) {
    const int64_t runs1 = p.N * p.HV;
    const int vbt = runs1 <= 64 ? 32 : runs1 <= 128 ? 64 : 128;
    const unsigned units = (unsigned)(num_chunks * p.HV), runs = (unsigned)((runs1 + 7) / 8 * 8 * (BD / vbt));
    struct K { const void* f; size_t smem; const char* name; unsigned grid, threads; };
    K scan;
    if (vbt == 32) scan = {(const void*)gdn_kda_scan_kernel<T, 32>, kda_scan_smem<32>(), "gdn_kda_scan_kernel", runs, 64u * kda_scan_waves<32>()};
    else if (vbt == 64) scan = {(const void*)gdn_kda_scan_kernel<T, 64>, kda_scan_smem<64>(), "gdn_kda_scan_kernel", runs, 64u * kda_scan_waves<64>()};
    else scan = {(const void*)gdn_kda_scan_kernel<T, 128>, kda_scan_smem<128>(), "gdn_kda_scan_kernel", runs, 64u * kda_scan_waves<128>()};
    const K prep = comba ? K{(const void*)gdn_comba_prepare_kernel<T>, COMBA_PREP_SMEM, "gdn_comba_prepare_kernel", units < 512u ? units : 512u, 256}
                         : K{(const void*)gdn_kda_prepare_kernel<T>, KDA_PREP_SMEM, "gdn_kda_prepare_kernel", units < 512u ? units : 512u, 256};
    const K ks[2] = {prep, scan};
    for (int i = 0; i < 2; ++i) {
        if (int rc = ensure_dynamic_smem_for(ks[i].f, ks[i].smem, ks[i].name)) return rc;
        int64_t nunits = units;
        void* args[] = {(void*)&p, (void*)&nunits};             // (the prepare kernel walks over the units and takes their number)
        if (hipLaunchKernel(ks[i].f, dim3(ks[i].grid), dim3(ks[i].threads), args, ks[i].smem, stream) != hipSuccess) return check_launch(ks[i].name);
        if (int rc = check_launch(ks[i].name)) return rc;
    }
    return GDN_OK;
}


int launch_kda_prepare(const KdaParams& p, int64_t num_chunks, int qkv_dtype, hipStream_t stream) {
    const unsigned units = (unsigned)(num_chunks * p.HV);
    const void* f = qkv_dtype == GDN_DTYPE_BF16 ? (const void*)gdn_kda_prepare_kernel<bf16_t> : (const void*)gdn_kda_prepare_kernel<f16_t>;
    if (int rc = ensure_dynamic_smem_for(f, KDA_PREP_SMEM, "gdn_kda_prepare_kernel")) return rc;
    int64_t nunits = units;
    void* args[] = {(void*)&p, (void*)&nunits};
    if (hipLaunchKernel(f, dim3(units < 512u ? units : 512u), dim3(256), args, KDA_PREP_SMEM, stream) != hipSuccess) return check_launch("gdn_kda_prepare_kernel");
    return check_launch("gdn_kda_prepare_kernel");
}

// checks shared by the two entry points
static int check_shapes(const char* who, int64_t B, int64_t T, int64_t H, int64_t HV, int64_t K, int64_t V, int64_t N, int64_t num_chunks,
                        const void* cu_seqlens, const void* chunk_table, const void* chunk_offsets, int qkv_dtype, uint32_t flags, uint32_t known) {
    GDN_CHECK_ARG(B >= 1 && T >= 0 && H >= 1 && HV >= 1 && N >= 1 && num_chunks >= 0, GDN_ERR_INVALID, "%s: bad dimension", who);
    GDN_CHECK_ARG(HV % H == 0, GDN_ERR_INVALID, "%s: HV=%lld not divisible by H=%lld", who, (long long)HV, (long long)H);
    GDN_CHECK_ARG(K == BD && V == BD, GDN_ERR_UNSUPPORTED, "%s: K = V = 128 only (got K=%lld V=%lld); pad smaller head dims with zeros",
                  who, (long long)K, (long long)V);
    GDN_CHECK_ARG(qkv_dtype == GDN_DTYPE_BF16 || qkv_dtype == GDN_DTYPE_F16, GDN_ERR_UNSUPPORTED, "%s: q/k/v must be bf16 or f16", who);
    GDN_CHECK_ARG((flags & ~known) == 0, GDN_ERR_UNSUPPORTED, "%s: unknown flag (the state layout is the caller's)", who);
    GDN_CHECK_ARG(HV <= 65535 && num_chunks * HV < (1ll << 31) && N * HV * 4 < (1ll << 31), GDN_ERR_UNSUPPORTED,
                  "%s: too many heads or chunks for one launch", who);
    if (cu_seqlens) {
        GDN_CHECK_ARG(B == 1, GDN_ERR_INVALID, "%s: with cu_seqlens B must be 1", who);
        GDN_CHECK_ARG((chunk_table || num_chunks == 0) && chunk_offsets, GDN_ERR_INVALID, "%s: packed input needs chunk_table and chunk_offsets", who);
    } else {
        GDN_CHECK_ARG(N == B, GDN_ERR_INVALID, "%s: without cu_seqlens N must equal B", who);
        GDN_CHECK_ARG(num_chunks == B * ((T + CH - 1) / CH), GDN_ERR_INVALID, "%s: num_chunks does not match B and T", who);
    }
    return GDN_OK;
}

}  // namespace gdn

extern "C" size_t gdn_chunk_kda_workspace_bytes(int64_t num_chunks, int64_t HV) {
    if (num_chunks < 0 || HV < 1) return 0;
    return gdn::kda_ws_layout(num_chunks * HV, nullptr, nullptr);
}

static int kda_fwd_entry(
    const char* who,
    const void* q, const void* k, const void* v, const float* g, const void* beta,
    const float* A_log, const float* dt_bias, float lower_bound, int gate_mode,
    const float* h0, float* ht, void* o, void* states,
    const void* cu_seqlens, const void* chunk_table, const void* chunk_offsets,
    void* workspace, size_t workspace_bytes,
    int64_t B, int64_t T, int64_t H, int64_t HV, int64_t K, int64_t V,
    int64_t N, int64_t num_chunks,
    float scale, int qkv_dtype, int gb_dtype, uint32_t flags, void* stream) {
    using namespace gdn;
    const uint32_t known = GDN_FLAG_CU_INT32 | GDN_FLAG_QK_L2NORM | GDN_FLAG_BETA_SIGMOID | GDN_FLAG_NEG_EIGVAL;
    if (int rc = check_shapes(who, B, T, H, HV, K, V, N, num_chunks, cu_seqlens, chunk_table, chunk_offsets, qkv_dtype, flags, known)) return rc;
    GDN_CHECK_ARG(gate_mode >= 0 && gate_mode <= 2, GDN_ERR_INVALID, "%s: gate_mode must be 0, 1 or 2", who);
    GDN_CHECK_ARG(gate_mode != 0 || (!A_log && !dt_bias), GDN_ERR_INVALID, "%s: A_log / dt_bias without a gate activation", who);
    GDN_CHECK_ARG(!(flags & GDN_FLAG_NEG_EIGVAL) || (flags & GDN_FLAG_BETA_SIGMOID), GDN_ERR_INVALID, "%s: GDN_FLAG_NEG_EIGVAL needs GDN_FLAG_BETA_SIGMOID", who);
    hipStream_t s = (hipStream_t)stream;
    if (T == 0 || num_chunks == 0) {
        if (ht) return launch_state_copy(h0, ht, N * HV * K * V, s);
        return GDN_OK;
    }
    GDN_CHECK_ARG(q && k && v && g && beta && o, GDN_ERR_INVALID, "%s: q, k, v, g, beta, o must not be NULL", who);
    for (const void* x : {q, k, v, (const void*)g, (const void*)h0, (const void*)ht, (const void*)o, (const void*)states})
        GDN_CHECK_ARG(((uintptr_t)x % 16) == 0, GDN_ERR_INVALID, "%s: tensors must be 16-byte aligned", who);
    GDN_CHECK_ARG(((uintptr_t)workspace % 256) == 0, GDN_ERR_INVALID, "%s: the workspace must be 256-byte aligned", who);
    KdaParams p;
    const size_t need = kda_ws_layout(num_chunks * HV, (char*)workspace, &p.ws);
    GDN_CHECK_ARG(workspace && workspace_bytes >= need, GDN_ERR_WORKSPACE, "%s: workspace of %zu bytes needed, %zu given", who,
                  need, workspace_bytes);
    p.q = q; p.k = k; p.v = v; p.g = g; p.beta = beta; p.pk = nullptr; p.gs = nullptr; p.A_log = A_log; p.gk_bias = dt_bias; p.gk_lower = lower_bound; p.gk_act = gate_mode;
    p.h0 = h0; p.ht = ht; p.o = o; p.hs = states;
    p.cu_seqlens = cu_seqlens; p.chunk_table = chunk_table; p.chunk_offsets = chunk_offsets;
    p.T = T; p.H = (int)H; p.HV = (int)HV; p.N = N; p.NT = (T + CH - 1) / CH;
    p.scale = scale; p.gb_dtype = gb_dtype; p.flags = flags;
    return qkv_dtype == GDN_DTYPE_BF16 ? launch_kda<bf16_t>(p, num_chunks, s) : launch_kda<f16_t>(p, num_chunks, s);
}

extern "C" int gdn_chunk_kda_fwd(
    const void* q, const void* k, const void* v, const float* g, const void* beta,
    const float* A_log, const float* dt_bias, float lower_bound, int gate_mode,
    const float* h0, float* ht, void* o,
    const void* cu_seqlens, const void* chunk_table, const void* chunk_offsets,
    void* workspace, size_t workspace_bytes,
    int64_t B, int64_t T, int64_t H, int64_t HV, int64_t K, int64_t V,
    int64_t N, int64_t num_chunks,
    float scale, int qkv_dtype, int gb_dtype, uint32_t flags, void* stream) {
    return kda_fwd_entry("gdn_chunk_kda_fwd", q, k, v, g, beta, A_log, dt_bias, lower_bound, gate_mode, h0, ht, o, nullptr, cu_seqlens, chunk_table,
                         chunk_offsets, workspace, workspace_bytes, B, T, H, HV, K, V, N, num_chunks, scale, qkv_dtype, gb_dtype, flags, stream);
}

// ... and the state in front of every chunk, states [num_chunks][HV][K][V] in qkv_dtype (the reference's h with return_intermediate_states)
extern "C" int gdn_chunk_kda_fwd_states(
    const void* q, const void* k, const void* v, const float* g, const void* beta,
    const float* A_log, const float* dt_bias, float lower_bound, int gate_mode,
    const float* h0, float* ht, void* o, void* states,
    const void* cu_seqlens, const void* chunk_table, const void* chunk_offsets,
    void* workspace, size_t workspace_bytes,
    int64_t B, int64_t T, int64_t H, int64_t HV, int64_t K, int64_t V,
    int64_t N, int64_t num_chunks,
    float scale, int qkv_dtype, int gb_dtype, uint32_t flags, void* stream) {
    GDN_CHECK_ARG(states || T == 0 || num_chunks == 0, GDN_ERR_INVALID, "gdn_chunk_kda_fwd_states: states must not be NULL");
    return kda_fwd_entry("gdn_chunk_kda_fwd_states", q, k, v, g, beta, A_log, dt_bias, lower_bound, gate_mode, h0, ht, o, states, cu_seqlens, chunk_table,
                         chunk_offsets, workspace, workspace_bytes, B, T, H, HV, K, V, N, num_chunks, scale, qkv_dtype, gb_dtype, flags, stream);
}

extern "C" int gdn_chunk_comba_fwd(
    const void* q, const void* k, const void* v, const void* p_key, const void* g, const void* beta,
    const float* h0, float* ht, void* o,
    const void* cu_seqlens, const void* chunk_table, const void* chunk_offsets,
    void* workspace, size_t workspace_bytes,
    int64_t B, int64_t T, int64_t H, int64_t HV, int64_t K, int64_t V,
    int64_t N, int64_t num_chunks,
    float scale, int qkv_dtype, int gb_dtype, uint32_t flags, void* stream) {
    using namespace gdn;
    const char* who = "gdn_chunk_comba_fwd";
    if (int rc = check_shapes(who, B, T, H, HV, K, V, N, num_chunks, cu_seqlens, chunk_table, chunk_offsets, qkv_dtype, flags,
                              GDN_FLAG_CU_INT32 | GDN_FLAG_QK_L2NORM)) return rc;
    GDN_CHECK_ARG(gb_dtype == GDN_DTYPE_F32 || gb_dtype == GDN_DTYPE_BF16 || gb_dtype == GDN_DTYPE_F16, GDN_ERR_UNSUPPORTED,
                  "%s: g and beta must be f32, bf16 or f16", who);
    hipStream_t s = (hipStream_t)stream;
    if (T == 0 || num_chunks == 0) {
        if (ht) return launch_state_copy(h0, ht, N * HV * K * V, s);
        return GDN_OK;
    }
    GDN_CHECK_ARG(q && k && v && p_key && g && beta && o, GDN_ERR_INVALID, "%s: q, k, v, p, g, beta, o must not be NULL", who);
    for (const void* x : {q, k, v, p_key, (const void*)h0, (const void*)ht, (const void*)o})
        GDN_CHECK_ARG(((uintptr_t)x % 16) == 0, GDN_ERR_INVALID, "%s: tensors must be 16-byte aligned", who);
    GDN_CHECK_ARG(((uintptr_t)workspace % 256) == 0, GDN_ERR_INVALID, "%s: the workspace must be 256-byte aligned", who);
    KdaParams p;
    const size_t need = kda_ws_layout(num_chunks * HV, (char*)workspace, &p.ws);
    GDN_CHECK_ARG(workspace && workspace_bytes >= need, GDN_ERR_WORKSPACE, "%s: workspace of %zu bytes needed, %zu given", who,
                  need, workspace_bytes);
    p.q = q; p.k = k; p.v = v; p.g = nullptr; p.beta = beta; p.pk = p_key; p.gs = g;
    p.A_log = nullptr; p.gk_bias = nullptr; p.gk_lower = 0.f; p.gk_act = 0;
    p.h0 = h0; p.ht = ht; p.o = o; p.hs = nullptr;
    p.cu_seqlens = cu_seqlens; p.chunk_table = chunk_table; p.chunk_offsets = chunk_offsets;
    p.T = T; p.H = (int)H; p.HV = (int)HV; p.N = N; p.NT = (T + CH - 1) / CH;
    p.scale = scale; p.gb_dtype = gb_dtype; p.flags = flags;
    return qkv_dtype == GDN_DTYPE_BF16 ? launch_kda<bf16_t>(p, num_chunks, s, true) : launch_kda<f16_t>(p, num_chunks, s, true);
}

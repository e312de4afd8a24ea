// Chunk-parallel stage of the chunked prefill: one WAVE per (chunk, value head) - four where there are few - computes what does not depend on the
// running state and is not a plain copy of the inputs:
//   G = cumsum(g)/ln2,  L = beta*(K K^T)*2^(G_i-G_j) (i>j),  X = (I+L)^-1 in fp32,  Xb = X diag(beta),
//   the per-token gate tables, a bound on the chunk's transition, and for the scan in halves or on request
//   P = scale*tril(q k^T * 2^(G_i-G_j)).
// Optional prologues of the reference are folded in: the gate and beta activations, and the l2 normalisation of k as
// per-row factors 1/|k_t| on L and the tables (so the sequential stage reads q and k exactly as the caller gave them;
// q is read here only for P and, where the scan does not apply them - it has q in LDS anyway -, for its row factors
// 1/|q_t|).  Xb and P are written in the exact register order ("fragments") in which the scan kernel feeds them to the
// matrix cores; the scan forms v_new = Xb (v - 2^G (k S)) itself from the raw k and v, so neither
// w = Xb 2^G k nor u = Xb v is ever materialised.
//
// A wave shares nothing with the other waves of its workgroup, so there is no workgroup barrier:
//   * The k rows are loaded straight into matrix-core operand registers (the operand layout of A and of B is the same:
//     lane (c16, g) holds 8 features of token row c16), so K K^T needs no LDS; the value heads of a q/k head sit in
//     neighbouring waves and read the same lines, which come from memory once (32768 tokens, 16 q/k and 32 value heads: 1.58 M requests of
//     128 bytes, 1.05 M of them k; the others are the gates, a token's line of which the workgroups of 4 value heads each read on all XCDs).
//   * Everything is kept TRANSPOSED: the raw tile (a, b), a <= b, holds (k_j . k_i) for rows j of t-tile a and columns i
//     of t-tile b, gated it is U = L^T, and T = X^T = (I + U)^-1 is upper triangular (gdn_chunk_inverse.h).  The transposed X in
//     accumulator layout is also exactly the order of the Xb operand fragments (row c16, columns 4g + e): results go from
//     registers to memory.
#include "gdn_chunk_inverse.h"

namespace gdn {

// The three gate tables lie where the transposed diagonal blocks of X go afterwards, |k|^2 and 1/|q| where the first products go
// afterwards: 8.75 KB per wave, four workgroups per CU.
constexpr int PW_WAVES = 4;                                  // waves per workgroup: small workgroups keep the CU's wave slots filled
constexpr size_t PREP_SMEM = (size_t)PW_WAVES * PW_FLOATS * 4;

// WANT_P: also the records' P (for the scan in halves, and for callers that look at the records; the other scan kernels form P
// themselves): keeps the q rows in registers beside the k rows, so half as many waves fit.
template <typename T, bool WANT_P>
__global__ __launch_bounds__(64 * PW_WAVES, (WANT_P ? 8 : 16) / PW_WAVES) void gdn_chunk_prepare_kernel(ChunkParams p, int64_t units) {
    typedef typename Mma<T>::V8 V8;
    extern __shared__ __align__(16) char smem[];
    const int tid = threadIdx.x, lane = tid & 63, c16 = lane & 15, g = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int64_t u = (int64_t)blockIdx.x * PW_WAVES + w;    // (chunk, value head), heads fastest
    if (u >= units) return;
    float* base = (float*)smem + w * PW_FLOATS;
    float* tiles = base;
    float* sLd = tiles;                                      // [4][16 i][16 j] diagonal blocks of L, by rows (until the T(g,g) are written)
    float* sG = tiles + 1024; float* sBN = sG + 64; float* sNK = sG + 128;      // gate tables (likewise)
    float* sK2 = tiles + 4 * 16 * TP; float* sNQ = sK2 + 64; // (until the gated tiles are written)
    auto lds_sync = [] { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); };   // (LDS operations of a wave execute in order)

    const int H = p.H, HV = p.HV, G = HV / H, K = p.K;
    const int64_t ci = u / HV;
    const int hv = (int)(u % HV), h = hv / G;
    const bool cu32 = p.flags & GDN_FLAG_CU_INT32;
    int64_t tok0;
    int valid;
    if (p.cu_seqlens) {
        const int64_t n = load_index(p.chunk_table, 2 * ci, cu32), it = load_index(p.chunk_table, 2 * ci + 1, cu32);
        const int64_t bos = load_index(p.cu_seqlens, n, cu32), eos = load_index(p.cu_seqlens, n + 1, cu32);
        tok0 = bos + it * CH;
        valid = (int)min((int64_t)CH, eos - tok0);
    } else {
        const int64_t b = ci / p.NT, it = ci % p.NT;
        tok0 = b * p.T + it * CH;
        valid = (int)min((int64_t)CH, p.T - it * CH);
    }
    const bool l2 = p.flags & GDN_FLAG_QK_L2NORM;      // k is l2-normalised here, as row factors (q: by the scan, or below for P)
    const bool q_norms_here = l2 && !(p.flags & FLAG_Q_NORM_IN_SCAN);       // 1/|q_t| into the tables (else the scan applies it)

    // ---- loads: the gate inputs of token `lane`, then the k rows as operand fragments ----
    // (as raw bits, converted where they are used: a 16-bit value converted on the spot would hold the k rows' requests back
    // until it has arrived)
    uint32_t rg = 0, rb = 0;
    if (lane < valid) {
        rg = p.g ? load_scalar_bits(p.g, (tok0 + lane) * HV + hv, p.gb_dtype) : 0;   // (no gate: the plain delta rule)
        rb = load_scalar_bits(p.beta, (tok0 + lane) * HV + hv, p.beta_dtype);
    }
    f32x4 U[4][4];
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = a; b < 4; ++b) U[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
    float sq[4] = {0.f, 0.f, 0.f, 0.f};
    f32x4 QK[4][4], QQ[4];                       // (WANT_P) raw k q^T tiles, like U; the diagonal tiles of q q^T
    if constexpr (WANT_P) {
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            QQ[a] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int b = a; b < 4; ++b) QK[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
    }
    {
        const T* kg = (const T*)p.k + (tok0 * H + h) * K;
        const T* qg = (const T*)p.q + (tok0 * H + h) * K;
        const u32x4 z = {0u, 0u, 0u, 0u};
        // one 32-bit offset per lane (its row of a t-tile, its 8 features of a 32-feature block); tile and block
        // select a wave-uniform base
        const uint32_t lane_off = ((uint32_t)c16 * (uint32_t)(H * K) + 8u * g) * (uint32_t)sizeof(T);
        // (a full chunk with the 32 features in range - the common case - loads without any per-lane condition)
        auto fragment = [&](const T* rows, int t, int col0) {
            const char* bp = (const char*)(rows + (int64_t)(16 * t) * H * K + col0);
            if (valid == CH && col0 + 32 <= K) return *(const u32x4*)(bp + lane_off);
            return (16 * t + c16 < valid && col0 + 8 * g < K) ? *(const u32x4*)(bp + lane_off) : z;
        };
        // 128 features at a time: all 16 fragments of a round are requested before the first product; the q rows (for
        // their norms only) follow into the same registers once the products have been issued
        for (int k0 = 0; k0 < K; k0 += 128) {
            u32x4 fk[4][4], fq[WANT_P ? 4 : 1][4];
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int s4 = 0; s4 < 4; ++s4) fk[t][s4] = fragment(kg, t, k0 + 32 * s4);
            if constexpr (WANT_P) {
#pragma unroll
                for (int t = 0; t < 4; ++t)
#pragma unroll
                    for (int s4 = 0; s4 < 4; ++s4) fq[t][s4] = fragment(qg, t, k0 + 32 * s4);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int a = 0; a < 4; ++a)
#pragma unroll
                for (int b = a; b < 4; ++b)
#pragma unroll
                    for (int s4 = 0; s4 < 4; ++s4)
                        U[a][b] = Mma<T>::run(__builtin_bit_cast(V8, fk[a][s4]), __builtin_bit_cast(V8, fk[b][s4]), U[a][b]);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (WANT_P) {
#pragma unroll
                for (int a = 0; a < 4; ++a)
#pragma unroll
                    for (int b = a; b < 4; ++b)
#pragma unroll
                        for (int s4 = 0; s4 < 4; ++s4)      // rows: key tokens of tile a, column: query token 16b + c16
                            QK[a][b] = Mma<T>::run(__builtin_bit_cast(V8, fk[a][s4]), __builtin_bit_cast(V8, fq[b][s4]), QK[a][b]);
#pragma unroll
                for (int t = 0; t < 4; ++t)
#pragma unroll
                    for (int s4 = 0; s4 < 4; ++s4) {
                        const V8 q8 = __builtin_bit_cast(V8, fq[t][s4]);
                        QQ[t] = Mma<T>::run(q8, q8, QQ[t]);
                    }
            } else if (q_norms_here) {                       // the q rows into the registers that held k
#pragma unroll
                for (int t = 0; t < 4; ++t)
#pragma unroll
                    for (int s4 = 0; s4 < 4; ++s4) fk[t][s4] = fragment(qg, t, k0 + 32 * s4);
#pragma unroll
                for (int t = 0; t < 4; ++t)
#pragma unroll
                    for (int s4 = 0; s4 < 4; ++s4) {
                        const V8 q8 = __builtin_bit_cast(V8, fk[t][s4]);
#pragma unroll
                        for (int e = 0; e < 8; ++e) { const float x = to_f32(q8[e]); sq[t] += x * x; }
                    }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
    // |k_t|^2 is the diagonal of K K^T; |q_t|^2 that of q q^T, or summed over the four lanes that share a row
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        float d = 0.f, dq = 0.f;
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (r == (c16 & 3)) { d = U[t][t][r]; if constexpr (WANT_P) dq = QQ[t][r]; }
        if ((c16 >> 2) == g) {
            sK2[16 * t + c16] = d;
            if constexpr (WANT_P) sNQ[16 * t + c16] = l2 ? rsqrtf(dq + 1e-6f) : 1.f;
        }
        if (!WANT_P && q_norms_here) {
            float a = sq[t];
            a += __shfl_xor(a, 16, 64);
            a += __shfl_xor(a, 32, 64);
            if (g == t) sNQ[16 * t + c16] = l2 ? rsqrtf(a + 1e-6f) : 1.f;
        }
    }
    lds_sync();
    // ---- gates: inclusive scan over the chunk, one token per lane; the tables; the bound on the chunk's transition ----
    float beta_tok;
    {
        float x = scalar_of_bits(rg, p.gb_dtype), b = scalar_of_bits(rb, p.beta_dtype);
        if (lane < valid) {                      // optional activations of the raw gate / beta inputs
            if (p.A_log && p.g) x = -__expf(p.A_log[hv]) * softplus_f(x + (p.dt_bias ? p.dt_bias[hv] : 0.f));
            if (p.flags & GDN_FLAG_BETA_SIGMOID) b = sigmoid_f(b) * ((p.flags & GDN_FLAG_NEG_EIGVAL) ? 2.f : 1.f);
        }
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const float y = __shfl_up(x, off, 64);
            if (lane >= off) x += y;
        }
        x *= RCP_LN2_F;
        const float xl = __shfl(x, 63, 64);      // rows past the end carry the last valid sum
        const float ex = fast_exp2(x);
        const float k2 = sK2[lane];
        const float nk = l2 ? rsqrtf(k2 + 1e-6f) : 1.f, nq = q_norms_here ? sNQ[lane] : 1.f;
        beta_tok = b;
        sG[lane] = x;
        sBN[lane] = b * nk;
        sNK[lane] = nk;
        float* tab = (float*)(p.ws.Rec + (ci * HV + hv) * REC_BYTES + REC_TAB);
        tab[TAB_DEC + lane] = fast_exp2(xl - x) * nk;        // multiplies v_new rows on their way into k^T v_new
        tab[TAB_SG + lane] = p.scale * ex * nq;              // multiplies (q S) rows (nq = 1: the scan adds 1/|q_t|)
        tab[TAB_EG + lane] = ex * nk;                        // multiplies (k S) rows
        if (lane == 63) tab[TAB_GLAST] = x;
        float* tab2 = (float*)(p.ws.Rec + (ci * HV + hv) * REC_BYTES + REC_TAB2);
        tab2[TAB2_G + lane] = x;
        tab2[TAB2_NQS + lane] = p.scale * nq;
        tab2[TAB2_NK + lane] = nk;
        // every token contributes gamma_t max(1, |1 - beta_t |k~_t|^2|) (rows past the end have beta = 0 and g = 0)
        float lb = fabsf(1.f - b * k2 * nk * nk);
        lb = lb > 1.f ? __log2f(lb) : 0.f;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) lb += __shfl_xor(lb, off, 64);
        if (lane == 63) p.ws.Bound[ci * HV + hv] = x + lb;
    }
    lds_sync();
    if constexpr (WANT_P) {
        // ---- P^T tiles (rows: key tokens j, column: query token t; lower triangle incl. the diagonal), gated, as fragments ----
        char* rec = p.ws.Rec + (ci * HV + hv) * REC_BYTES;
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            const float gt = sG[16 * b + c16], st = p.scale * sNQ[16 * b + c16];
#pragma unroll
            for (int sp = 0; sp < 2; ++sp) {
                if (b < 2 && sp == 1) continue;         // identically zero, not stored
                V8 frag;
#pragma unroll
                for (int half = 0; half < 2; ++half) {
                    const int a = 2 * sp + half;
                    if (a > b) {                        // a key tile after the query tile: zero
#pragma unroll
                        for (int r = 0; r < 4; ++r) frag[half * 4 + r] = from_f32<T>(0.f);
                        continue;
                    }
                    const f32x4 gj = *(const f32x4*)(sG + 16 * a + 4 * g), nj = *(const f32x4*)(sNK + 16 * a + 4 * g);
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const bool below = a < b || c16 >= 4 * g + r;
                        frag[half * 4 + r] = from_f32<T>(below ? st * nj[r] * QK[a][b][r] * fast_exp2(gt - gj[r]) : 0.f);
                    }
                }
                store_frag<T>(rec + REC_P, b, sp, lane, frag);
            }
        }
    }
    // ---- U = L^T: gated, beta-scaled, strictly upper; diagonal blocks to LDS as L by rows, the others as left factors ----
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = a; b < 4; ++b) {
            const float gi = sG[16 * b + c16], bni = sBN[16 * b + c16];               // column: token i
            const f32x4 gj = *(const f32x4*)(sG + 16 * a + 4 * g), nj = *(const f32x4*)(sNK + 16 * a + 4 * g);   // rows: tokens j
            f32x4 val;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                // select, never multiply by a mask: 2^(G_i-G_j) may overflow for i < j
                const bool below = a < b || c16 > 4 * g + r;
                val[r] = below ? bni * nj[r] * U[a][b][r] * fast_exp2(gi - gj[r]) : 0.f;
            }
            if (a == b) *(f32x4*)(sLd + a * 256 + c16 * 16 + 4 * g) = val;             // L[i = c16][j = 4g + r]
            else U[a][b] = val;                                                        // stays in registers: a right factor
        }
    lds_sync();
    f32x4 X[4][4];
    inverse_transposed(tiles, U, X, c16, g);
    // ---- Xb = X diag(beta) as operand fragments: rows of t-tile tt, columns {32sp + 4g + e} and {32sp + 16 + 4g + e} ----
    {
        const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
        char* rec = p.ws.Rec + (ci * HV + hv) * REC_BYTES;
        auto emit = [&](int tt, int sp, f32x4 lo, f32x4 hi, bool has_hi) {
            V8 frag;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                frag[e] = from_f32<T>(lo[e] * __shfl(beta_tok, 32 * sp + 4 * g + e, 64));
                frag[4 + e] = from_f32<T>(has_hi ? hi[e] * __shfl(beta_tok, 32 * sp + 16 + 4 * g + e, 64) : 0.f);
            }
            store_frag<T>(rec + REC_X, tt, sp, lane, frag);
        };
        emit(0, 0, X[0][0], zero, false);
        emit(1, 0, X[0][1], X[1][1], true);
        emit(2, 0, X[0][2], X[1][2], true);
        emit(2, 1, X[2][2], zero, false);
        emit(3, 0, X[0][3], X[1][3], true);
        emit(3, 1, X[2][3], X[3][3], true);
    }
}

// The same with four waves to a unit, for calls of so few units that the waves of a CU have nobody to wait for but themselves (launch_prepare):
// what bounds them is one unit's chain of steps.  Wave w takes the tiles (a, w), a <= w, of K K^T and of k q^T - loads, products, gates,
// P and X of token tile w are its own -, the diagonal block w of the inverse, and after that the block column w of T from the bottom up,
//     T_aw = -T_aa sum_{a < m <= w} U_am T_mw,
// left factors U_am and T_aa from LDS, right factors the blocks it has just computed.  Two barriers: one for the gates and the norms, which wave 0
// and the diagonal tiles' owners supply, one for the left factors.
// A call with four waves to a unit instead of one, on inputs in the caches and out of them: 333 tokens, 32 heads (192 units) 27.0 -> 22.0 us and
// 28.1 -> 23.0; 1000 tokens, 16 heads 42.3 -> 37.1 and 43.3 -> 38.9; 1000 tokens, 8 heads of 256 77.5 -> 69.9 and 84.3 -> 76.3.
// Up to three workgroups a CU, one round of the chip: 32 heads, at 704 and 768 units still 54.6 -> 52.8 and 57.7 -> 56.0 us, at 800 already 59.1 -> 61.2.
// The results are not those of the other kernel bit by bit (sums in another order), so a sequence's last bits depend on how many units its call has.
constexpr int TEAM_TILE = 16 * TP;
constexpr int64_t TEAM_UNITS = 3 * 256;
template <typename T, bool WANT_P>
__global__ __launch_bounds__(256, 2) void gdn_chunk_prepare_team_kernel(ChunkParams p, uint32_t units, uint32_t share_log2, uint32_t G) {
    typedef typename Mma<T>::V8 V8;
    __shared__ __align__(16) float smem[10 * TEAM_TILE + 4 * 256 + 4 * 64];
    auto tile = [&](int n) { return smem + n * TEAM_TILE; };
    auto pair = [](int a, int m) { return 4 + m * (m - 1) / 2 + a; };        // U_am, a < m, behind the four T_aa
    float* sG = smem + 10 * TEAM_TILE + 4 * 256; float* sBeta = sG + 64; float* sK2 = sBeta + 64; float* sNQ = sK2 + 64;
    const int tid = threadIdx.x, lane = tid & 63, c16 = lane & 15, g = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    float* sLd = smem + 10 * TEAM_TILE + w * 256;                            // the diagonal block of L, by rows
    // (chunk, value head), heads fastest; 2^share_log2 in a row on one XCD (see launch_prepare_as)
    const uint32_t slot = blockIdx.x >> 3, run = (slot >> share_log2) * 8 + (blockIdx.x & 7);
    const uint32_t u = (run << share_log2) + (slot & ((1u << share_log2) - 1));
    if (u >= units) return;
    const int H = p.H, HV = p.HV, K = p.K;
    const int64_t ci = u / (uint32_t)HV;
    const int hv = (int)(u % (uint32_t)HV), h = (int)((uint32_t)hv / G);
    const bool cu32 = p.flags & GDN_FLAG_CU_INT32;
    int64_t tok0;
    int valid;
    if (p.cu_seqlens) {
        const int64_t n = load_index(p.chunk_table, 2 * ci, cu32), it = load_index(p.chunk_table, 2 * ci + 1, cu32);
        const int64_t bos = load_index(p.cu_seqlens, n, cu32), eos = load_index(p.cu_seqlens, n + 1, cu32);
        tok0 = bos + it * CH;
        valid = (int)min((int64_t)CH, eos - tok0);
    } else {
        const int64_t b = ci / p.NT, it = ci % p.NT;
        tok0 = b * p.T + it * CH;
        valid = (int)min((int64_t)CH, p.T - it * CH);
    }
    const bool l2 = p.flags & GDN_FLAG_QK_L2NORM, q_norms_here = l2 && !(p.flags & FLAG_Q_NORM_IN_SCAN), want_q = WANT_P || q_norms_here;
    char* rec = p.ws.Rec + (ci * HV + hv) * REC_BYTES;

    uint32_t rg = 0, rb = 0;
    if (w == 0 && lane < valid) {
        rg = p.g ? load_scalar_bits(p.g, (tok0 + lane) * HV + hv, p.gb_dtype) : 0;
        rb = load_scalar_bits(p.beta, (tok0 + lane) * HV + hv, p.beta_dtype);
    }
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    f32x4 U[4], QK[4], QQ = zero;                            // tiles (a, w): rows keys of tile a, columns tokens of tile w
#pragma unroll
    for (int a = 0; a < 4; ++a) U[a] = QK[a] = zero;
    {
        const T* kg = (const T*)p.k + (tok0 * H + h) * K;
        const T* qg = (const T*)p.q + (tok0 * H + h) * K;
        const u32x4 z = {0u, 0u, 0u, 0u};
        const uint32_t lane_off = ((uint32_t)c16 * (uint32_t)(H * K) + 8u * g) * (uint32_t)sizeof(T);
        auto fragment = [&](const T* rows, int t, int col0) {
            const char* bp = (const char*)(rows + (int64_t)(16 * t) * H * K + col0);
            if (valid == CH && col0 + 32 <= K) return *(const u32x4*)(bp + lane_off);
            return (16 * t + c16 < valid && col0 + 8 * g < K) ? *(const u32x4*)(bp + lane_off) : z;
        };
        for (int k0 = 0; k0 < K; k0 += 128) {
            u32x4 fo[4], fk[4][4], fq[4];                    // (fo: the wave's own tile)
#pragma unroll
            for (int s4 = 0; s4 < 4; ++s4) fo[s4] = fragment(kg, w, k0 + 32 * s4);
#pragma unroll
            for (int s4 = 0; s4 < 4; ++s4) fq[s4] = want_q ? fragment(qg, w, k0 + 32 * s4) : z;
#pragma unroll
            for (int a = 0; a < 3; ++a)
                if (a < w) {
#pragma unroll
                    for (int s4 = 0; s4 < 4; ++s4) fk[a][s4] = fragment(kg, a, k0 + 32 * s4);
                }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int s4 = 0; s4 < 4; ++s4) {
                const V8 o8 = __builtin_bit_cast(V8, fo[s4]), q8 = __builtin_bit_cast(V8, fq[s4]);
                U[3] = Mma<T>::run(o8, o8, U[3]);            // (the diagonal tile lies at 3 until it is moved to its place below)
                if constexpr (WANT_P) QK[3] = Mma<T>::run(o8, q8, QK[3]);
                if (want_q) QQ = Mma<T>::run(q8, q8, QQ);
            }
#pragma unroll
            for (int a = 0; a < 3; ++a)
                if (a < w) {
#pragma unroll
                    for (int s4 = 0; s4 < 4; ++s4) {
                        const V8 k8 = __builtin_bit_cast(V8, fk[a][s4]);
                        U[a] = Mma<T>::run(k8, __builtin_bit_cast(V8, fo[s4]), U[a]);
                        if constexpr (WANT_P) QK[a] = Mma<T>::run(k8, __builtin_bit_cast(V8, fq[s4]), QK[a]);
                    }
                }
        }
    }
    const f32x4 Ud = U[3], QKd = QK[3];
    // |k_t|^2 and |q_t|^2 are the diagonals of the diagonal tiles
    {
        float dk = 0.f, dq = 0.f;
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (r == (c16 & 3)) { dk = Ud[r]; dq = QQ[r]; }
        if ((c16 >> 2) == g) { sK2[16 * w + c16] = dk; sNQ[16 * w + c16] = l2 && want_q ? rsqrtf(dq + 1e-6f) : 1.f; }
    }
    float x = 0.f, b = 0.f;                                  // (wave 0: the running sum of the gates and beta of token `lane`)
    if (w == 0) {
        x = scalar_of_bits(rg, p.gb_dtype); b = scalar_of_bits(rb, p.beta_dtype);
        if (lane < valid) {
            if (p.A_log && p.g) x = -__expf(p.A_log[hv]) * softplus_f(x + (p.dt_bias ? p.dt_bias[hv] : 0.f));
            if (p.flags & GDN_FLAG_BETA_SIGMOID) b = sigmoid_f(b) * ((p.flags & GDN_FLAG_NEG_EIGVAL) ? 2.f : 1.f);
        }
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const float y = __shfl_up(x, off, 64);
            if (lane >= off) x += y;
        }
        x *= RCP_LN2_F;
        sG[lane] = x;
        sBeta[lane] = b;
    }
    __syncthreads();

    auto norm_of = [&](float k2) { return l2 ? rsqrtf(k2 + 1e-6f) : 1.f; };
    const int i = 16 * w + c16;                              // this lane's column: token i
    const float gi = sG[i], nki = norm_of(sK2[i]), bni = sBeta[i] * nki, st = p.scale * sNQ[i];
    V8 pf[2];
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int e = 0; e < 8; ++e) pf[s][e] = from_f32<T>(0.f);
#pragma unroll
    for (int a = 0; a < 4; ++a) {
        if (a > w) continue;
        const f32x4 gj = *(const f32x4*)(sG + 16 * a + 4 * g), kj = *(const f32x4*)(sK2 + 16 * a + 4 * g);
        const f32x4 Ua = a == w ? Ud : U[a < 3 ? a : 0], Qa = a == w ? QKd : QK[a < 3 ? a : 0];
        f32x4 val;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            // select, never multiply by a mask: 2^(G_i-G_j) may overflow for i < j
            const float d = a < w || c16 >= 4 * g + r ? fast_exp2(gi - gj[r]) * norm_of(kj[r]) : 0.f;
            val[r] = a < w || c16 > 4 * g + r ? bni * Ua[r] * d : 0.f;
            if constexpr (WANT_P) pf[a >> 1][4 * (a & 1) + r] = from_f32<T>(st * Qa[r] * d);
        }
        if (a == w) *(f32x4*)(sLd + c16 * 16 + 4 * g) = val;           // L[i = c16][j = 4g + r]
        else {
            float* t = tile(pair(a, w));
#pragma unroll
            for (int r = 0; r < 4; ++r) t[(4 * g + r) * TP + c16] = val[r];
        }
    }
    if constexpr (WANT_P) {
        store_frag<T>(rec + REC_P, w, 0, lane, pf[0]);
        if (w >= 2) store_frag<T>(rec + REC_P, w, 1, lane, pf[1]);     // (identically zero for the first two tiles, not stored)
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");       // (LDS operations of a wave execute in order)
    // ---- the diagonal block: X (I + L) = I by rows, from the right; lane c16 owns row c16 (every lane group the same) ----
    {
        float xr[16], acc[16];
#pragma unroll
        for (int n = 0; n < 16; ++n) acc[n] = 0.f;
#pragma unroll
        for (int n = 15; n >= 0; --n) {
            xr[n] = ((n == c16) ? 1.f : 0.f) - acc[n];
            float row[16];
#pragma unroll
            for (int q4 = 0; q4 < (n + 3) / 4; ++q4) *(f32x4*)(row + 4 * q4) = *(const f32x4*)(sLd + n * 16 + 4 * q4);
#pragma unroll
            for (int j = 0; j < n; ++j) acc[j] += row[j] * xr[n];
        }
        if (g == 0) {                                        // T(w,w) = X^T as a left factor: [row j][column c16]
            float* t = tile(w);
#pragma unroll
            for (int j = 0; j < 16; ++j) t[j * TP + c16] = xr[j];
        }
    }
    if (w == 0) {
        // the tables and the bound on the chunk's transition (as in gdn_chunk_prepare_kernel)
        const float xl = __shfl(x, 63, 64), ex = fast_exp2(x);
        const float k2 = sK2[lane], nk = norm_of(k2), nq = q_norms_here ? sNQ[lane] : 1.f;
        float* tab = (float*)(rec + REC_TAB);
        tab[TAB_DEC + lane] = fast_exp2(xl - x) * nk;
        tab[TAB_SG + lane] = p.scale * ex * nq;
        tab[TAB_EG + lane] = ex * nk;
        if (lane == 63) tab[TAB_GLAST] = x;
        float* tab2 = (float*)(rec + REC_TAB2);
        tab2[TAB2_G + lane] = x;
        tab2[TAB2_NQS + lane] = p.scale * nq;
        tab2[TAB2_NK + lane] = nk;
        float lb = fabsf(1.f - b * k2 * nk * nk);
        lb = lb > 1.f ? __log2f(lb) : 0.f;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) lb += __shfl_xor(lb, off, 64);
        if (lane == 63) p.ws.Bound[ci * HV + hv] = x + lb;
    }
    __syncthreads();

    // ---- block column w of T ----
    auto mul = [&](int n, f32x4 B, f32x4 acc) {              // acc + A B: A a tile of LDS by rows, B in accumulator layout
        const f32x4 A = *(const f32x4*)(tile(n) + c16 * TP + 4 * g);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(A[e], B[e], acc, 0, 0, 0);
        return acc;
    };
    f32x4 X[4];
#pragma unroll
    for (int a = 3; a >= 0; --a) {
        X[a] = zero;
        if (a > w) continue;
        if (a == w) {
            const float* t = tile(a);
            X[a] = f32x4{t[(4 * g) * TP + c16], t[(4 * g + 1) * TP + c16], t[(4 * g + 2) * TP + c16], t[(4 * g + 3) * TP + c16]};
            continue;
        }
        f32x4 t = zero;
#pragma unroll
        for (int m = a + 1; m < 4; ++m)
            if (m <= w) t = mul(pair(a, m), X[m], t);
        X[a] = -mul(a, t, zero);
    }
    // ---- Xb = X diag(beta) of token tile w as operand fragments: columns {32sp + 4g + e} and {32sp + 16 + 4g + e} ----
#pragma unroll
    for (int sp = 0; sp < 2; ++sp) {
        if (2 * sp > w) continue;
        const f32x4 blo = *(const f32x4*)(sBeta + 32 * sp + 4 * g), bhi = *(const f32x4*)(sBeta + 32 * sp + 16 + 4 * g);
        V8 frag;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            frag[e] = from_f32<T>(X[2 * sp][e] * blo[e]);
            frag[4 + e] = from_f32<T>(X[2 * sp + 1][e] * bhi[e]);
        }
        store_frag<T>(rec + REC_X, w, sp, lane, frag);
    }
}

template <typename T, bool WANT_P>
static int launch_prepare_as(const ChunkParams& p, int64_t units, hipStream_t stream) {
    if (units <= TEAM_UNITS) {
        // The value heads of a q/k head read the same rows: they go to one XCD (workgroups are dealt to the 8 of them in turn), and where the
        // q/k heads are a multiple of 8 to that of the scan's workgroups, so that the rows come from memory once: 333 tokens, 16 q/k and 32 value
        // heads 6.4 -> 3.7 MB read, the call 22.5 -> 22.0 us, on inputs out of the caches 23.4 -> 23.0; 700 tokens 33.2 -> 31.9 and 34.2 -> 33.2.
        // As many of a group as a power of two counts, and no more than an XCD's 32 CUs: 32 value heads to a q/k head 31.1 -> 29.8 us (190 tokens,
        // 3 q/k heads), 64 to one 32.0 -> 33.1, 128 to one 52.3 -> 59.5 (64 tokens).
        const uint32_t G = (uint32_t)(p.HV / p.H), share = G <= 32 ? G & (0u - G) : 1, n = (uint32_t)units;
        hipLaunchKernelGGL((gdn_chunk_prepare_team_kernel<T, WANT_P>), dim3((n / share + 7) / 8 * 8 * share), dim3(256), 0, stream, p, n,
                           (uint32_t)__builtin_ctz(share), G);
        return check_launch("gdn_chunk_prepare_team_kernel");
    }
    auto kern = gdn_chunk_prepare_kernel<T, WANT_P>;
    static SmemAttrDone attr_done;       // per instantiation
    if (int rc = ensure_dynamic_smem((const void*)kern, PREP_SMEM, attr_done, "hipFuncSetAttribute(prepare)")) return rc;
    hipLaunchKernelGGL(kern, dim3((unsigned)((units + PW_WAVES - 1) / PW_WAVES)), dim3(64 * PW_WAVES), PREP_SMEM, stream, p, units);
    return check_launch("gdn_chunk_prepare_kernel");
}

template <typename T>
int launch_prepare(const ChunkParams& p, int64_t num_chunks, hipStream_t stream) {
    const int64_t units = num_chunks * p.HV;
    if (units <= 0) return GDN_OK;
    return p.want_P ? launch_prepare_as<T, true>(p, units, stream) : launch_prepare_as<T, false>(p, units, stream);
}
template int launch_prepare<bf16_t>(const ChunkParams&, int64_t, hipStream_t);
template int launch_prepare<f16_t>(const ChunkParams&, int64_t, hipStream_t);

}  // namespace gdn

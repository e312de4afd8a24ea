// Backward pass of the chunked gated delta rule (gfx950, 64-token chunks; 64 key features and value columns, or 128 or 256 key features
// and blocks of 128 value columns; the host pads other head dims).
// Replaces the reference's backward pipeline fla/ops/gated_delta_rule/chunk.py:125-257 (recompute_w_u_fwd,
// chunk_gated_delta_rule_fwd_h, chunk_bwd_dv_local, chunk_gated_delta_rule_bwd_dhu, chunk_bwd_dqkwg, prepare_wy_repr_bwd,
// reverse chunk_local_cumsum) by three stages:
//
//   prepare   per (chunk, v-head)      gam = cumsum(g), A = (I + diag(beta) stril(k k^T o D))^-1, P = scale tril(q k^T o D);
//                                      D_ij = e^(gam_i - gam_j)
//   scans     per (sequence, v-head, slice of value columns), with w = A (beta e^gam k), u = A (beta v):
//             chunks in order          S_c (state in front of chunk c), v_new = u - w S_c
//             and in reverse order     dS_c (gradient of the state behind chunk c), dv_new = P^T do + (k e^(gam_last - gam)) dS_c,
//                                      dS <- e^gam_last dS + scale (q e^gam)^T do - w^T dv_new
//   unit      per (chunk, q/k head)    from S, dS, v_new, dv_new to dq, dk, dv, dbeta, dg
//
// The comba operator (fla/ops/comba/chunk.py:92-178) predicts with a second key p and the state BEFORE the token's decay:
// with gam0 = gam - g its chunk form has A = (I + diag(beta) stril(p k^T o D0))^-1, D0_ij = e^(gam0_i - gam_j), and
// w = A (beta e^gam0 p); everything between w, u and the state is the gated delta rule's.  Its prepare kernel writes w and u, the two
// scans read them, and two kernels take the place of the last one (dqkw: dq, the parts of dk and dgam from the output and the state
// update, dw = -dv_new S^T; wy: through w, u, A back to k, p, v, beta, gam - with a second gradient, dgam0, whose reverse cumulative
// sum enters dg without its own token).
//
// All matrix products run on the matrix cores from row-major LDS tiles.  A product's two operands have the same register
// layout (lane (c16, g) holds index c16 and the 8 contraction indices 8g .. 8g+7 of a 32-wide step), so there are just two
// ways to fetch an operand fragment from a row-major tile: `frag_rows` (the contraction runs along a row: one 16-byte read)
// and `frag_cols` (the contraction runs down a column: two transposing LDS reads).  The result of run(a, b) holds, in lane
// (c16, g), column c16 (b's index) and rows 4g .. 4g+3 (a's index): whichever side carries the features gets them four in a
// row per lane, which is what an 8-byte store into a row-major [token][feature] array wants.
#include "gdn_chunk_inverse.h"
#include "gdn_chunk_kda.h"

namespace gdn {

// In separate arrays, per (chunk, v-head): gam, beta [64] fp32, A, P [64][64], Bound (one float, see gdn_chunk_common.h, WARM_LOG2); and per
// (chunk, v-head, block of VD value columns): v_new, dv_new [64][VD], S, dS [KD][VD] as operand fragments (state_frag), all in the operand type.
// Comba adds gam0 and dgam [64] fp32 (dgam partial, between the last two kernels), P^T in P's place, w, dw [64][128], u [64][128].
// The KDA operator (a decay per key feature) has instead: Gk, the running sums of the log decays, divided by ln 2, [64][128] fp32; QG = scale q e^Gk,
// KG = k e^(Gk_last - Gk) [64][128] and P [64][64] in the operand type, EGL = e^Gk_last [128] fp32 (all four as the forward's
// chunk-parallel kernel writes them); w, u; u and v_new share their place.
struct BwdWs {
    float* Gam; float* Bet; float* Dgam; float* Gam0;
    void* Am; void* PT; void* Wm; void* Vn; void* Hs; void* dHs; void* dVn; void* dWm;
    float* Gk; void* QG; void* KG; void* Pm; float* EGL;
    void* Um; float* Bound;
};
struct WsTake {
    char* base; size_t off = 0;
    void* operator()(size_t bytes) { const size_t o = off; off += ws_align(bytes); return base ? (void*)(base + o) : nullptr; }
};
inline size_t bwd_ws_layout(int64_t num_chunks, int64_t HV, int64_t nb, int64_t KD, int64_t VD, char* base, BwdWs* ws) {
    WsTake take{base};
    const size_t ug = (size_t)(num_chunks * HV), u = ug * nb;
    BwdWs x{};
    x.Gam = (float*)take(ug * 64 * 4); x.Bet = (float*)take(ug * 64 * 4);
    x.Am = take(ug * 64 * 64 * 2); x.Pm = take(ug * 64 * 64 * 2);
    x.Vn = take(u * 64 * VD * 2); x.dVn = take(u * 64 * VD * 2);
    x.Hs = take(u * KD * VD * 2); x.dHs = take(u * KD * VD * 2);
    x.Bound = (float*)take(ug * 4);
    if (ws) *ws = x;
    return take.off;
}
inline size_t comba_bwd_ws_layout(int64_t units, char* base, BwdWs* ws) {
    WsTake take{base};
    const size_t u = (size_t)units;
    BwdWs x{};
    x.Gam = (float*)take(u * 64 * 4); x.Dgam = (float*)take(u * 64 * 4); x.Gam0 = (float*)take(u * 64 * 4);
    x.Am = take(u * 64 * 64 * 2); x.PT = take(u * 64 * 64 * 2);
    x.Wm = take(u * 64 * BD * 2); x.Vn = take(u * 64 * BD * 2); x.Um = take(u * 64 * BD * 2);
    x.Hs = take(u * BD * BD * 2); x.dHs = take(u * BD * BD * 2);
    x.dVn = take(u * 64 * BD * 2); x.dWm = take(u * 64 * BD * 2);
    if (ws) *ws = x;
    return take.off;
}
inline size_t kda_bwd_ws_layout(int64_t units, char* base, BwdWs* ws) {
    WsTake take{base};
    const size_t u = (size_t)units;
    BwdWs x{};
    x.Am = take(u * 64 * 64 * 2); x.Pm = take(u * 64 * 64 * 2);
    x.Wm = take(u * 64 * BD * 2); x.Um = x.Vn = take(u * 64 * BD * 2);
    x.QG = take(u * 64 * BD * 2); x.KG = take(u * 64 * BD * 2);
    x.Hs = take(u * BD * BD * 2); x.dHs = take(u * BD * BD * 2);
    x.dVn = take(u * 64 * BD * 2);
    x.Gk = (float*)take(u * 64 * BD * 4); x.EGL = (float*)take(u * BD * 4);
    if (ws) *ws = x;
    return take.off;
}

struct BwdParams {
    const void* q; const void* k; const void* v; const void* g; const void* beta;
    const float* A_log; const float* dt_bias;     // optional gate activation (per value head)
    const float* h0; const void* dout; const float* dht;
    void* dq; void* dk; void* dv; float* dg; float* dbeta; float* dh0;
    const void* pk; void* dp;            // (comba) the second key, the one the prediction is made with, and its gradient
    float* dgk;                          // (KDA) gradient of the log decays [B,T,HV,128] fp32
    // The l2 normalisation of q and k taken in here: the rows as the caller has them; q and k
    // above are then places in the workspace that the prepare kernel fills with the normalised rows, and these with the factors
    // [tokens,H] (fla/modules/l2norm.py:222-262); dq and dk come back as the gradients of the rows before the normalisation,
    // dx = (dy - y (y . dy)) rstd (fla/modules/l2norm.py:265-298).  NULL: q and k are what the recurrence uses.
    const void* q_raw; const void* k_raw; const void* pk_raw;    // (pk_raw, p_rstd: comba's second key, the same way)
    const float* q_rstd; const float* k_rstd; const float* p_rstd;
    const void* cu_seqlens; const void* chunk_table; const void* chunk_offsets;
    BwdWs ws;
    int64_t T; int H, HV; int64_t N; int64_t NT;
    int nb;                              // HV counts blocks of value columns: nb of them share a value head's gate and beta
    float scale; int gb_dtype, beta_dtype; uint32_t flags;
    // The two scans cut into `nseg` time segments of `seg_chunks` chunks (1: whole sequences): a segment starts from a zero state up
    // to `warm_cap` chunks outside its range where the chunks' transition bounds say that this is forgotten by the time its own
    // range begins (gdn_chunk_common.h, WARM_LOG2); a head with a segment that cannot is walked whole by the workgroups of segment 0.
    int nseg, seg_chunks, warm_cap;
    int parts;                           // dq and dk leave as this many partial rows per token and q/k head (a divisor of HV / H)
    // Partial rows that are added up here (BwdParts) leave in fp32 to these places instead of dq and dk (NULL: they do not), and where
    // the parts cut a value head's blocks of columns, `split` > 1 parts to a head, so do the partial sums of dg and dbeta.
    float* dq_part; float* dk_part; float* dg_part; float* db_part;
    int split;
};

// How a q/k head's value heads (their blocks of columns, `nb` each) are dealt out to the workgroups of the unit kernels: all to one
// where (chunk, q/k head) pairs fill the chip, in equal parts where they do not.  In units of what a block takes (7 us at 64 and 128 key
// features, 14 us at 256), a workgroup spends 0.3 on its rows of q and k, and the pass over the parts costs a half, at 64 and 128 features as much
// again where the parts fill the chip: there memory bounds them, and fp32 rows are twice as long.  It is a launch more
// too, which a call waits for on the host where its sequences are short (fewer than 8 chunks on average, of `num_seqs`): not for one
// block saved.  (The workspace is sized as for one sequence: never smaller.)  Training step with one part, with the number chosen, with others:
//   1024 tokens, 2 q/k and 16 value heads of 128   163, 125 us (8 parts; 4: 127)    2 and 8 heads of 256           275, 194 us (8; 4: 200)
//   2048 tokens, 4 and 32 heads of 128             233, 218 us (2; 4: 225)          2 and 16 heads of 64           168, 129 us (8; 4: 132)
//   2048 tokens, 8 and 32 heads of 128 (256 pairs) 211 us (2: 228)                  1000 tokens, 6 heads of 256 x 512   225, 207 us (2; 4: 218)
//   4096 tokens, 2 and 4 heads of 128              169 us (2: 171)                  768 tokens, 10 and 30 heads of 128  117 us (3: 124)
//   1024 tokens, 16 and 32 heads of 64             99.5 us (2: 101.5)               256 tokens, 16 and 32 heads of 128  89 us (2: 92)
struct BwdParts {
    int parts = 1, split = 1;
    size_t row_bytes = 0, head_bytes = 0;        // of dq_part (dk_part), of dg_part (db_part); 0: none
    size_t bytes() const { return 2 * ws_align(row_bytes) + 2 * ws_align(head_bytes); }
};
inline BwdParts bwd_parts(int64_t num_chunks, int64_t num_seqs, int64_t tokens, int64_t H, int64_t HV, int64_t nb, int64_t KD) {
    const int64_t slots = KD == 64 ? 512 : 256, items = num_chunks * H, heads = HV / H * nb;
    BwdParts x;
    if (items >= slots) return x;
    double best = 1e30;
    for (int64_t n = 1; n <= heads && items * n <= 2 * slots; ++n) {
        // whole value heads, or an equal share of one's blocks
        if (heads % n || !((heads / n) % nb == 0 || nb % (heads / n) == 0)) continue;
        const double pass = (num_chunks < 8 * num_seqs ? 1.2 : 0.5) + (KD <= BD ? 0.5 * (double)(items * n) / (double)slots : 0.0);
        const double cost = (double)((items * n + slots - 1) / slots) * ((double)(heads / n) + 0.3) + (n == 1 ? 0.0 : pass);
        if (cost < best) { best = cost; x.parts = (int)n; }
    }
    if (x.parts > 1) {
        x.split = (int)std::max<int64_t>(1, nb / (heads / x.parts));
        x.row_bytes = (size_t)(tokens * H * x.parts) * KD * 4;
        if (x.split > 1) x.head_bytes = (size_t)(tokens * HV * x.split) * 4;
    }
    return x;
}

// The mirror image of warm_chunks() for the scan that runs backwards: how many chunks AFTER chunk it1 - 1 a run must start from a
// zero state so that at it1 - 1 it has forgotten the difference to the true state.  When the end of the sequence comes first the
// answer is nc - it1 (the run starts from the true gradient of the final state and is exact).  -1: not within `cap` chunks.
__device__ __forceinline__ int warm_chunks_rev(const float* bound, int HV, int64_t it1, int64_t nc, int cap, int lane) {
    const bool in = lane < cap && it1 + lane < nc;
    float x = in ? bound[(it1 + lane) * HV] : 0.f;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const float y = __shfl_up(x, off, 64);
        if (lane >= off) x += y;
    }
    const uint64_t hit = __builtin_amdgcn_ballot_w64(in && x <= WARM_LOG2);
    if (hit) return __builtin_ctzll(hit) + 1;
    return nc - it1 <= cap ? (int)(nc - it1) : -1;
}

// What a workgroup of the two scans does with time segments: `whole`: segment 0 walks the sequence, the others leave;
// otherwise the forward scan walks chunks [f0 - fw, f1) and keeps its results from f0 on, the reverse scan walks [f0, f1 + rw)
// downwards and keeps its results below f1.  The same in every wave of a workgroup (both scans need both answers: side by side
// in one workgroup they must take the same number of barriers).
struct ScanPlan { bool whole; int64_t f0, f1; int fw, rw; };
__device__ __forceinline__ ScanPlan scan_plan(const BwdParams& p, const SeqAt& sq, int hg, int seg, int lane) {
    ScanPlan sp{false, 0, sq.nc, 0, 0};
    if (p.nseg <= 1) return sp;
    const int HVg = p.HV / p.nb;
    const float* bound = p.ws.Bound + sq.cbase * HVg + hg;
    sp.f0 = (int64_t)seg * p.seg_chunks;
    sp.f1 = seg == p.nseg - 1 ? sq.nc : (int64_t)(seg + 1) * p.seg_chunks;
    for (int s = 1; s < p.nseg; ++s) {
        const int64_t at = (int64_t)s * p.seg_chunks;           // the boundary between segments s - 1 and s
        const int fw = warm_chunks(bound, HVg, at, p.warm_cap, lane), rw = warm_chunks_rev(bound, HVg, at, sq.nc, p.warm_cap, lane);
        sp.whole |= fw < 0 || rw < 0;
        if (s == seg) sp.fw = fw;
        if (s == seg + 1) sp.rw = rw;
    }
    if (sp.whole) { sp.f0 = 0; sp.f1 = sq.nc; sp.fw = sp.rw = 0; }
    return sp;
}

// The i-th sequence in the order the scans take them: the longest first where the caller has sorted them (GDN_FLAG_SEQ_ORDER).
__device__ __forceinline__ int64_t seq_in_order(const BwdParams& p, int64_t i) {
    return p.cu_seqlens && (p.flags & GDN_FLAG_SEQ_ORDER) ? load_index_uniform(p.chunk_offsets, p.N + 1 + i, p.flags & GDN_FLAG_CU_INT32) : i;
}

// steps of the longer of the two scans of a workgroup
__device__ __forceinline__ int64_t pad_steps_of(const ScanPlan& sp) { return (sp.f1 - sp.f0) + (sp.fw > sp.rw ? sp.fw : sp.rw); }

// ---------------------------------------------------------------------------------------------
// prepare
// ---------------------------------------------------------------------------------------------
// (comba; a third tile of rows, those of p; the matrix L takes the place of the q tile once q has been used, which keeps a
// workgroup at 80 KB: two per CU)
constexpr size_t BWD_PREP_COMBA_SMEM = (4 * 64 * P128 + 64 * P64) * 2 + 192 * 4;

// Rows of a tile on their way from memory to LDS (a row: 16 lanes next to each other, 8 features each) divided by their
// length, as gdn_l2norm_fwd does it; the normalised rows and the factors are left for the kernels that follow.
template <typename T>
__device__ __forceinline__ void l2norm_tile_rows(TileRegs<BD>& r, T* out, float* rstd_out, int H, int valid, int tid) {
    typedef typename Mma<T>::V8 V8;
    const int row0 = tid >> 4, pc = tid & 15;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        V8 x = __builtin_bit_cast(V8, r.x[i]);
        float f[8], ss = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) { f[e] = (float)x[e]; ss += f[e] * f[e]; }
        const float rs = rsqrtf(sum_over_c16(ss) + 1e-6f);
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = (T)(f[e] * rs);
        r.x[i] = __builtin_bit_cast(u32x4, x);
        const int row = row0 + 16 * i;
        if (row < valid) {
            *(u32x4*)(out + (int64_t)row * H * BD + pc * 8) = r.x[i];
            if (pc == 0) rstd_out[(int64_t)row * H] = rs;
        }
    }
}

template <typename T, bool L2>
__global__ __launch_bounds__(256, 2) void gdn_bwd_prepare_comba_kernel(BwdParams p, int64_t units) {
    typedef typename Mma<T>::V8 V8;
    typedef typename Mma<T>::V4 V4;
    constexpr int KD = BD, PK = KD + 8;
    extern __shared__ __align__(16) char smem[];
    T* sK = (T*)smem; T* sQ = sK + 64 * PK; T* sV = sQ + 64 * PK; T* sA = sV + 64 * P128;
    T* sP = sA + 64 * P64;                                       // (comba) rows of the second key
    static_assert(64 * PL * 4 <= 64 * PK * 2, "the matrix L fits the q tile");
    float* sL = (float*)sQ;
    float* sGam = (float*)(sP + 64 * PK); float* sBeta = sGam + 64; float* sGam0 = sBeta + 64;
    T* sRows = sP;                                  // the rows that enter L from the left and w
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, c16 = lane & 15, g = lane >> 4;

    // Units in turn; the next unit's rows are fetched into registers while this one is worked on.
    TileRegs<KD> rK, rQ, rP;
    TileRegs<BD> rV;
    uint32_t rG = 0, rB = 0;                                     // (raw bits: converted when the unit's turn comes)
    auto fetch = [&](int64_t u) {
        const UnitAt at = unit_at(p, u);
        const int hv = at.hv, hq = at.hq;
        const ChunkAt c = at.c;
        fetch_tile<KD>(rK, (const T*)(L2 ? p.k_raw : p.k) + (c.tok0 * p.H + hq) * KD, (int64_t)p.H * KD, c.valid, tid);
        fetch_tile<KD>(rQ, (const T*)(L2 ? p.q_raw : p.q) + (c.tok0 * p.H + hq) * KD, (int64_t)p.H * KD, c.valid, tid);
        fetch_tile<KD>(rP, (const T*)(L2 ? p.pk_raw : p.pk) + (c.tok0 * p.H + hq) * KD, (int64_t)p.H * KD, c.valid, tid);
        fetch_tile<BD>(rV, (const T*)p.v + (c.tok0 * p.HV + hv) * BD, (int64_t)p.HV * BD, c.valid, tid);
        rG = rB = 0;
        if (w == 0 && lane < c.valid) {
            rG = p.g ? load_scalar_bits(p.g, (c.tok0 + lane) * p.HV + hv, p.gb_dtype) : 0;
            rB = load_scalar_bits(p.beta, (c.tok0 + lane) * p.HV + hv, p.gb_dtype);
        }
    };
    fetch(blockIdx.x);
    for (int64_t u = blockIdx.x; u < units; u += gridDim.x) {
        // (everything derived from the lane number is derived again per unit from a copy the compiler cannot see through:
        // hoisted out of this loop, the addresses of its unrolled body would sit in registers, or spill, for its whole length)
        int tid_opaque = threadIdx.x;
        asm volatile("" : "+v"(tid_opaque));
        const int tid = tid_opaque, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), c16 = lane & 15, g = lane >> 4;
        if constexpr (L2) {
            const UnitAt at = unit_at(p, u);
            const ChunkAt c = at.c;
            const int64_t row0 = c.tok0 * p.H + at.hq;
            const int keep = at.hq * (p.HV / p.H) == at.hv ? c.valid : 0;      // (the first of the value heads that share the rows leaves them)
            l2norm_tile_rows<T>(rK, (T*)p.k + row0 * KD, (float*)p.k_rstd + row0, p.H, keep, tid);
            l2norm_tile_rows<T>(rQ, (T*)p.q + row0 * KD, (float*)p.q_rstd + row0, p.H, keep, tid);
            l2norm_tile_rows<T>(rP, (T*)p.pk + row0 * KD, (float*)p.p_rstd + row0, p.H, keep, tid);
        }
        put_tile<KD>(sK, PK, rK, tid);
        put_tile<KD>(sQ, PK, rQ, tid);
        put_tile<BD>(sV, P128, rV, tid);
        put_tile<KD>(sP, PK, rP, tid);
        if (w == 0) {
            const float g_own = scalar_of_bits(rG, p.gb_dtype);
            float x = g_own;
#pragma unroll
            for (int off = 1; off < 64; off <<= 1) {
                const float y = __shfl_up(x, off, 64);
                if (lane >= off) x += y;
            }
            sGam[lane] = x; sBeta[lane] = scalar_of_bits(rB, p.gb_dtype);
            sGam0[lane] = x - g_own;                 // (comba) the sum in front of this token: the prediction sees the state before its decay
            p.ws.Gam[u * 64 + lane] = x;
            p.ws.Gam0[u * 64 + lane] = x - g_own;
        }
        lds_barrier();
        if (u + gridDim.x < units) fetch(u + gridDim.x);

        // strip of 16 token rows per wave: L (fp32, for the substitution; entry (i, j) at [i][j % 4][j / 4]) and P^T
        {
            T* PTu = (T*)p.ws.PT + u * 64 * 64;
            f32x4 lrow[4];                          // (comba) this wave's entries of L, until q's tile is free for them
#pragma unroll
            for (int tj = 0; tj < 4; ++tj) {
                f32x4 kk = ZERO4, qk = ZERO4;
                if (tj <= w) {
#pragma unroll
                    for (int s = 0; s < 4; ++s) {
                        const V8 b = frag_rows(sK, PK, 16 * tj, 32 * s, lane);
                        kk = Mma<T>::run(frag_rows(sRows, PK, 16 * w, 32 * s, lane), b, kk);
                        qk = Mma<T>::run(frag_rows(sQ, PK, 16 * w, 32 * s, lane), b, qk);
                    }
                }
                const int j = 16 * tj + c16;
                const float gj = sGam[j];
                f32x4 pt;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int i = 16 * w + 4 * g + r;
                    const float d = i >= j ? __expf(sGam[i] - gj) : 0.f;
                    const float d0 = i > j ? __expf(sGam0[i] - gj) : 0.f;
                    const float l = i > j ? sBeta[i] * kk[r] * d0 : 0.f;
                    lrow[tj][r] = l;
                    pt[r] = p.scale * qk[r] * d;
                }
                *(V4*)(PTu + j * 64 + 16 * w + 4 * g) = pack4<T>(pt);
            }
            {
                lds_barrier();                                  // (every wave has read its rows of q)
#pragma unroll
                for (int tj = 0; tj < 4; ++tj) {
                    const int j = 16 * tj + c16;
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (tj <= w) sL[(16 * w + 4 * g + r) * PL + (j & 3) * 16 + (j >> 2)] = lrow[tj][r];
                }
            }
        }
        lds_barrier();
        // k -> beta e^gam k (comba: p -> beta e^gam0 p) and v -> beta v, in place
        for (int idx = tid; idx < 64 * 16 * 2; idx += 256) {
            const int row = idx / (16 * 2), pc = idx % (16 * 2);      // the row's pieces of k, then those of v
            T* at = pc < 16 ? sRows + row * PK + pc * 8 : sV + row * P128 + (pc - 16) * 8;
            const float f = pc < 16 ? sBeta[row] * __expf(sGam0[row]) : sBeta[row];
            V8 x = *(V8*)at;
#pragma unroll
            for (int e = 0; e < 8; ++e) x[e] = (T)((float)x[e] * f);
            *(V8*)at = x;
        }
        solve_unit_lower_blocks<T>(sL, (float*)sA, sA, w, lane);
        lds_barrier();
        {
            T* Au = (T*)p.ws.Am + u * 64 * 64;
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int idx = tid + 256 * i, row = idx >> 3, pc = idx & 7;
                *(u32x4*)(Au + row * 64 + pc * 8) = *(const u32x4*)(sA + row * P64 + pc * 8);
            }
        }
        // w^T and u^T tiles: features on the rows, this wave's 16 tokens on the columns
        {
            T* Wu = (T*)p.ws.Wm + u * 64 * KD;
            T* Uu = (T*)p.ws.Um + u * 64 * BD;
            const int i = 16 * w + c16;
            V8 fa[2];
#pragma unroll
            for (int s = 0; s < 2; ++s) fa[s] = frag_rows(sA, P64, 16 * w, 32 * s, lane);
#pragma unroll
            for (int n = 0; n < 8; ++n) {
                f32x4 aw = ZERO4;
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    if (2 * s > w) continue;                    // A is lower triangular
                    aw = Mma<T>::run(frag_cols(sRows, PK, 32 * s, 16 * n, lane), fa[s], aw);
                }
                *(V4*)(Wu + i * KD + 16 * n + 4 * g) = pack4<T>(aw);
            }
#pragma unroll
            for (int n = 0; n < 8; ++n) {
                f32x4 au = ZERO4;
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    if (2 * s > w) continue;
                    au = Mma<T>::run(frag_cols(sV, P128, 32 * s, 16 * n, lane), fa[s], au);
                }
                *(V4*)(Uu + i * BD + 16 * n + 4 * g) = pack4<T>(au);
            }
        }
        lds_barrier();
    }
}

#include "gdn_chunk_bwd_prepare.h"

#include "gdn_chunk_bwd_scans.h"

// ---------------------------------------------------------------------------------------------
// (comba) dq, dw and the first parts of dk and dgam.  Wave w owns key features 32w .. + 31 (two tiles a2) of all 64 tokens (four
// tiles t): lane (c16, g) holds token 16t + c16 and features 16(2w+a2) + 4g .. +3.
// ---------------------------------------------------------------------------------------------
// One workgroup per CU walks over the units and fetches everything the next unit needs (five tiles and its
// fragments of S and dS) into registers while it works on the current one.
// L2: dq goes back through the l2 normalisation of q before it is written (its rows wait in registers for the row sums of q . dq).
constexpr size_t BWD_DQKW_SMEM = (5 * 64 * P128 + 64 * P64) * 2 + 640 * 4;

template <typename T, bool L2 = false>
__global__ __launch_bounds__(256, 1) void gdn_bwd_dqkw_kernel(BwdParams p, int64_t units) {
    typedef typename Mma<T>::V8 V8;
    typedef typename Mma<T>::V4 V4;
    constexpr int KD = BD, PK = KD + 8;
    extern __shared__ __align__(16) char smem[];
    T* sDO = (T*)smem; T* sVn = sDO + 64 * P128; T* sDvn = sVn + 64 * P128; T* sK = sDvn + 64 * P128; T* sQ = sK + 64 * PK;
    T* sDP = sQ + 64 * PK;
    float* sGam = (float*)(sDP + 64 * P64); float* sDg = sGam + 64;    // sDg [4][64]: a row per wave, added up in a fixed order (same bits every run)
    float* sQd = sDg + 256; float* sRq = sQd + 256;                    // (L2) q . dq per wave and token; the tokens' factors
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, c16 = lane & 15, g = lane >> 4;

    TileRegs<BD> rDO, rVn, rDvn;
    TileRegs<KD> rK, rQ;
    V8 rS[2][4], rdS[2][4];
    float rGam = 0.f, rRq = 0.f;
    auto fetch = [&](int64_t u) {
        const UnitAt at = unit_at(p, u);
        const int hv = at.hv, hq = at.hq;
        const ChunkAt c = at.c;
        fetch_tile<BD>(rDO, (const T*)p.dout + (c.tok0 * p.HV + hv) * BD, (int64_t)p.HV * BD, c.valid, tid);
        fetch_tile<BD>(rVn, (const T*)p.ws.Vn + u * 64 * BD, BD, 64, tid);
        fetch_tile<BD>(rDvn, (const T*)p.ws.dVn + u * 64 * BD, BD, 64, tid);
        {
            const T* Hu = (const T*)p.ws.Hs + u * KD * BD;
            const T* dHu = (const T*)p.ws.dHs + u * KD * BD;
#pragma unroll
            for (int a2 = 0; a2 < 2; ++a2)
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    rS[a2][s] = *(const V8*)(Hu + state_frag<BD>(2 * w + a2, s, lane));
                    rdS[a2][s] = *(const V8*)(dHu + state_frag<BD>(2 * w + a2, s, lane));
                }
        }
        fetch_tile<KD>(rK, (const T*)p.k + (c.tok0 * p.H + hq) * KD, (int64_t)p.H * KD, c.valid, tid);
        fetch_tile<KD>(rQ, (const T*)p.q + (c.tok0 * p.H + hq) * KD, (int64_t)p.H * KD, c.valid, tid);
        if (tid < 64) rGam = p.ws.Gam[u * 64 + tid];
        if constexpr (L2) rRq = tid < c.valid ? p.q_rstd[(c.tok0 + tid) * p.H + hq] : 0.f;
    };
    fetch(blockIdx.x);
    for (int64_t u = blockIdx.x; u < units; u += gridDim.x) {
        const UnitAt at = unit_at(p, u);
        const int hv = at.hv;
        const ChunkAt c = at.c;
        put_tile<BD>(sDO, P128, rDO, tid);
        put_tile<BD>(sVn, P128, rVn, tid);
        put_tile<BD>(sDvn, P128, rDvn, tid);
        put_tile<KD>(sK, PK, rK, tid);
        put_tile<KD>(sQ, PK, rQ, tid);
        if (tid < 64) sGam[tid] = rGam;
        if constexpr (L2) { if (tid < 64) sRq[tid] = rRq; }
        sDg[tid] = 0.f;
        V8 sf[2][4], df[2][4];
        {
#pragma unroll
            for (int a2 = 0; a2 < 2; ++a2)
#pragma unroll
                for (int s = 0; s < 4; ++s) { sf[a2][s] = rS[a2][s]; df[a2][s] = rdS[a2][s]; }
        }
        lds_barrier();
        if (u + gridDim.x < units) fetch(u + gridDim.x);

        float sdot = 0.f, dglast = 0.f;
        f32x4 dq_rows[L2 ? 2 : 1][4];
        {
            // Operand fragments are fetched from LDS once per use across the two feature tiles of this wave.
            f32x4 G1[2][4], dKS[2][4], dWt[2][4], dPt[4];
#pragma unroll
            for (int a2 = 0; a2 < 2; ++a2)
#pragma unroll
                for (int t = 0; t < 4; ++t) G1[a2][t] = dWt[a2][t] = dKS[a2][t] = ZERO4;
#pragma unroll
            for (int t = 0; t < 4; ++t) dPt[t] = ZERO4;
#pragma unroll
            for (int s = 0; s < 4; ++s) {
#pragma unroll
                for (int a2 = 0; a2 < 2; ++a2)
#pragma unroll
                    for (int e = 0; e < 8; ++e) sdot += (float)sf[a2][s][e] * (float)df[a2][s][e];
                const V8 own = frag_rows(sDO, P128, 16 * w, 32 * s, lane);      // this wave's 16 token rows of do, for dP
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    const V8 bdo = frag_rows(sDO, P128, 16 * t, 32 * s, lane), bdv = frag_rows(sDvn, P128, 16 * t, 32 * s, lane),
                             bvn = frag_rows(sVn, P128, 16 * t, 32 * s, lane);
#pragma unroll
                    for (int a2 = 0; a2 < 2; ++a2) {
                        G1[a2][t] = Mma<T>::run(sf[a2][s], bdo, G1[a2][t]);
                        dWt[a2][t] = Mma<T>::run(sf[a2][s], bdv, dWt[a2][t]);
                        dKS[a2][t] = Mma<T>::run(df[a2][s], bvn, dKS[a2][t]);
                    }
                    if (t <= w) dPt[t] = Mma<T>::run(own, bvn, dPt[t]);
                }
            }
            {
                T* dWu = (T*)p.ws.dWm + u * 64 * KD;
#pragma unroll
                for (int a2 = 0; a2 < 2; ++a2)
#pragma unroll
                    for (int t = 0; t < 4; ++t)
                        *(V4*)(dWu + (16 * t + c16) * KD + 16 * (2 * w + a2) + 4 * g) = pack4<T>(-dWt[a2][t]);
            }
            {
                // dP o D for this wave's 16 token rows, as an operand tile
                float gi[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) gi[r] = sGam[16 * w + 4 * g + r];
#pragma unroll
                for (int tj = 0; tj < 4; ++tj) {
                    const int j = 16 * tj + c16;
                    const float gj = sGam[j];
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int i = 16 * w + 4 * g + r;
                        sDP[i * P64 + j] = (T)(i >= j ? p.scale * dPt[tj][r] * __expf(gi[r] - gj) : 0.f);
                    }
                }
                lds_barrier();
            }

            const float glast = sGam[63];
            V8 fk[2][2], fq[2][2];
#pragma unroll
            for (int a2 = 0; a2 < 2; ++a2)
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    fk[a2][s] = frag_cols(sK, PK, 32 * s, 16 * (2 * w + a2), lane);
                    fq[a2][s] = frag_cols(sQ, PK, 32 * s, 16 * (2 * w + a2), lane);
                }
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const int x = 16 * t + c16;
                const float gx = sGam[x];
                const float fqs = p.scale * __expf(gx), fks = __expf(glast - gx);
                f32x4 dq[2], dk[2];
                V4 q4[2], k4[2];
#pragma unroll
                for (int a2 = 0; a2 < 2; ++a2) {
                    const int n16 = 16 * (2 * w + a2);
                    dq[a2] = G1[a2][t] * fqs;
                    dk[a2] = dKS[a2][t] * fks;
                    q4[a2] = *(const V4*)(sQ + x * PK + n16 + 4 * g);
                    k4[a2] = *(const V4*)(sK + x * PK + n16 + 4 * g);
#pragma unroll
                    for (int r = 0; r < 4; ++r) dglast += (float)k4[a2][r] * dk[a2][r];
                }
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    if (32 * s <= 16 * t + 15) {                // dP[i][j] = 0 for j > i
                        const V8 e = frag_rows(sDP, P64, 16 * t, 32 * s, lane);
#pragma unroll
                        for (int a2 = 0; a2 < 2; ++a2) dq[a2] = Mma<T>::run(fk[a2][s], e, dq[a2]);
                    }
                    if (32 * s + 31 >= 16 * t) {                // ... and for i < j
                        const V8 e = frag_cols(sDP, P64, 32 * s, 16 * t, lane);
#pragma unroll
                        for (int a2 = 0; a2 < 2; ++a2) dk[a2] = Mma<T>::run(fq[a2][s], e, dk[a2]);
                    }
                }
                float qdq = 0.f, kdk = 0.f;
#pragma unroll
                for (int a2 = 0; a2 < 2; ++a2)
#pragma unroll
                    for (int r = 0; r < 4; ++r) { qdq += (float)q4[a2][r] * dq[a2][r]; kdk += (float)k4[a2][r] * dk[a2][r]; }
                const float dgx = sum_over_g(qdq - kdk);
                if (g == 0) atomicAdd(&sDg[64 * w + x], dgx);
                if constexpr (L2) {
                    qdq = sum_over_g(qdq);
                    if (g == 0) sQd[64 * w + x] = qdq;
                    dq_rows[0][t] = dq[0]; dq_rows[1][t] = dq[1];
                }
                if (x < c.valid) {
#pragma unroll
                    for (int a2 = 0; a2 < 2; ++a2) {
                        const int n16 = 16 * (2 * w + a2);
                        if constexpr (!L2) *(V4*)((T*)p.dq + ((c.tok0 + x) * p.HV + hv) * KD + n16 + 4 * g) = pack4<T>(dq[a2]);
                        *(V4*)((T*)p.dk + ((c.tok0 + x) * p.HV + hv) * KD + n16 + 4 * g) = pack4<T>(dk[a2]);
                    }
                }
            }
        }
        dglast += __expf(sGam[63]) * sdot;
        dglast = sum_over_c16(sum_over_g(dglast));
        if (lane == 0) atomicAdd(&sDg[64 * w + 63], dglast);
        lds_barrier();
        if constexpr (L2) {
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const int x = 16 * t + c16;
                const float dot = (sQd[x] + sQd[64 + x]) + (sQd[128 + x] + sQd[192 + x]), rs = sRq[x];
                if (x < c.valid) {
#pragma unroll
                    for (int a2 = 0; a2 < 2; ++a2) {
                        const int n16 = 16 * (2 * w + a2);
                        const V4 q4 = *(const V4*)(sQ + x * PK + n16 + 4 * g);
                        f32x4 out;
#pragma unroll
                        for (int r = 0; r < 4; ++r) out[r] = (dq_rows[a2][t][r] - (float)q4[r] * dot) * rs;
                        *(V4*)((T*)p.dq + ((c.tok0 + x) * p.HV + hv) * KD + n16 + 4 * g) = pack4<T>(out);
                    }
                }
            }
        }
        if (tid < 64) p.ws.Dgam[u * 64 + tid] = (sDg[tid] + sDg[64 + tid]) + (sDg[128 + tid] + sDg[192 + tid]);
        lds_barrier();
    }
}

// ---------------------------------------------------------------------------------------------
// (comba) back through w = X (e^gam0 p), u = X v, X = A diag(beta), A = (I + diag(beta) stril(k k^T o D))^-1
// ---------------------------------------------------------------------------------------------
// Workgroups walk over the units (chunk, v-head), the next unit's tiles on their way into registers meanwhile: dX = tril(dw (e^gam k)^T
// + du v^T), dA = stril(dX diag(beta)); dv = beta (A^T du); d(e^gam k) = beta (A^T dw), into dk, dbeta, dgam; Y = dA A^T,
// dL = -stril(A^T Y), E = diag(beta) dL o D; dk += E k + E^T k; dbeta, dgam from L = diag(beta) stril(k k^T o D); dg = the reverse
// cumulative sum of dgam inside the chunk.  sDg, sDb [4][64]: a row per wave, added up in a fixed order at the end - the same
// bits every run.
// One block of key features in at most 76 KB of LDS, so that two workgroups share a CU: the unit is walked
// in two halves over the same two tile places - first dv_new and v (dX's first term, dv and its share of dbeta), then dw and k
// (dX's second term, k k^T, the first part of dk; comba: with the rows of p in a third place) - with the second set on its way
// into registers during the first half and the next unit's first pair during the second; Y = dA A^T takes dw's place once dw is done with.
// L2: dk goes back through the l2 normalisation of k before it is written.
constexpr size_t BWD_WY2_SMEM = (3 * 64 * P128 + 2 * 64 * P64) * 2 + (960 + 640) * 4;

template <typename T, bool L2 = false>
__global__ __launch_bounds__(256, 2) void gdn_bwd_wy2_kernel(BwdParams p, int64_t units) {
    static_assert(2 * BWD_WY2_SMEM <= 160 * 1024, "two workgroups per CU");
    typedef typename Mma<T>::V8 V8;
    typedef typename Mma<T>::V4 V4;
    constexpr int KD = BD, PK = P128, NA = 2;
    extern __shared__ __align__(16) char smem[];
    T* sX0 = (T*)smem; T* sX1 = sX0 + 64 * P128;               // dv_new | v, then dw | k
    T* sA = sX1 + 64 * P128; T* sM1 = sA + 64 * P64; T* sP = sM1 + 64 * P64;     // (comba) rows of the second key
    float* sGam = (float*)(sP + 64 * P128); float* sBeta = sGam + 64; float* sDg = sBeta + 64; float* sDb = sDg + 256;
    float* sKd = sDb + 256; float* sRk = sKd + 256;              // (L2) k . dk per wave and token; the tokens' factors
    float* sDg0 = sRk + 64; float* sGam0 = sDg0 + 256;           // (comba)
    float* sPd = sGam0 + 64; float* sRp = sPd + 256;             // (comba, L2) p . dp per wave and token; the tokens' factors
    T* sDvn = sX0; T* sV = sX1; T* sDW = sX0; T* sK = sX1; T* sM2 = sX0;
    T* sRows = sP;
    float* sGamRow = sGam0; float* sDgRow = sDg0;

    TileRegs<BD> rDvn, rV, rDW, rK, rP;
    TileRegs<CH> rA;
    float rGam = 0.f, rDg = 0.f, rRk = 0.f, rGam0 = 0.f, rRp = 0.f;
    uint32_t rBeta = 0;                                          // (raw bits: converted when the unit's turn comes)
    auto fetch_first = [&](int64_t u, int tid) {
        const UnitAt at = unit_at(p, u);
        const int hv = at.hv;
        const ChunkAt c = at.c;
        fetch_tile<BD>(rDvn, (const T*)p.ws.dVn + u * 64 * BD, BD, 64, tid);
        fetch_tile<BD>(rV, (const T*)p.v + (c.tok0 * p.HV + hv) * BD, (int64_t)p.HV * BD, c.valid, tid);
        fetch_tile<CH>(rA, (const T*)p.ws.Am + u * 64 * 64, 64, 64, tid);
        if (tid < 64) {
            rGam = p.ws.Gam[u * 64 + tid];
            rBeta = tid < c.valid ? load_scalar_bits(p.beta, (c.tok0 + tid) * p.HV + hv, p.gb_dtype) : 0;
            rDg = p.ws.Dgam[u * 64 + tid];
            rGam0 = p.ws.Gam0[u * 64 + tid];
            if constexpr (L2) rRk = tid < c.valid ? p.k_rstd[(c.tok0 + tid) * p.H + hv] : 0.f;
            if constexpr (L2) rRp = tid < c.valid ? p.p_rstd[(c.tok0 + tid) * p.H + hv] : 0.f;
        }
    };
    fetch_first(blockIdx.x, threadIdx.x);
    for (int64_t u = blockIdx.x; u < units; u += gridDim.x) {
        // (everything derived from the lane number is derived again per unit from a copy the compiler cannot see through:
        // hoisted out of this loop, the addresses of its unrolled body would sit in registers, or spill, for its whole length)
        int tid_opaque = threadIdx.x;
        asm volatile("" : "+v"(tid_opaque));
        const int tid = tid_opaque, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), c16 = lane & 15, g = lane >> 4;
        auto feat = [&](int a) { return 16 * (2 * w + a); };    // first key feature of this wave's tile a
        const UnitAt at = unit_at(p, u);
        const int hv = at.hv, hq = at.hq;
        const ChunkAt c = at.c;
        put_tile<BD>(sDvn, P128, rDvn, tid);
        put_tile<BD>(sV, P128, rV, tid);
        put_tile<CH>(sA, P64, rA, tid);
        if (tid < 64) { sGam[tid] = rGam; sBeta[tid] = scalar_of_bits(rBeta, p.gb_dtype); if constexpr (L2) sRk[tid] = rRk; sGam0[tid] = rGam0; if constexpr (L2) sRp[tid] = rRp; }
        sDg[tid] = tid < 64 ? rDg : 0.f;
        sDb[tid] = 0.f;
        sDg0[tid] = 0.f;
        // the second pair of this unit, and what the previous kernel left in dk at this lane's places
        fetch_tile<KD>(rDW, (const T*)p.ws.dWm + u * 64 * KD, KD, 64, tid);
        fetch_tile<KD>(rK, (const T*)p.k + (c.tok0 * p.H + hq) * KD, (int64_t)p.H * KD, c.valid, tid);
        fetch_tile<KD>(rP, (const T*)p.pk + (c.tok0 * p.H + hq) * KD, (int64_t)p.H * KD, c.valid, tid);
        V4 dk_old[NA][4];
#pragma unroll
        for (int a2 = 0; a2 < NA; ++a2)
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const int x = 16 * t + c16;
                dk_old[a2][t] = V4{(T)0.f, (T)0.f, (T)0.f, (T)0.f};
                if (x < c.valid) dk_old[a2][t] = *(const V4*)((const T*)p.dk + ((c.tok0 + x) * p.HV + hv) * KD + feat(a2) + 4 * g);
            }
        lds_barrier();

        // ---- first half: dX's first term du v^T (this wave's 16 rows i; lane: column j, rows 4g + r), and dv = beta (A^T du) ----
        f32x4 dXv[4];
        {
            V8 fa[4];
#pragma unroll
            for (int s = 0; s < 4; ++s) fa[s] = frag_rows(sDvn, P128, 16 * w, 32 * s, lane);
#pragma unroll
            for (int tj = 0; tj < 4; ++tj) {
                dXv[tj] = ZERO4;
                if (tj <= w) {
#pragma unroll
                    for (int s = 0; s < 4; ++s) dXv[tj] = Mma<T>::run(fa[s], frag_rows(sV, P128, 16 * tj, 32 * s, lane), dXv[tj]);
                }
            }
        }
        {
            V8 fA[4][2];                                        // A^T operand of token tile t, step s (zero where A is)
            float bj[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) {
#pragma unroll
                for (int s = 0; s < 2; ++s)
                    if (32 * s + 31 >= 16 * t) fA[t][s] = frag_cols(sA, P64, 32 * s, 16 * t, lane);
                bj[t] = sBeta[16 * t + c16];
            }
#pragma unroll
            for (int a2 = 0; a2 < 2; ++a2) {                    // value columns 16(2w+a2) ..
                const int n16 = 16 * (2 * w + a2);
                V8 fdv[2];
#pragma unroll
                for (int s = 0; s < 2; ++s) fdv[s] = frag_cols(sDvn, P128, 32 * s, n16, lane);
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    f32x4 av = ZERO4;
#pragma unroll
                    for (int s = 0; s < 2; ++s) {
                        if (32 * s + 31 < 16 * t) continue;     // A[i][j] = 0 for i < j
                        av = Mma<T>::run(fdv[s], fA[t][s], av);
                    }
                    const int j = 16 * t + c16;
                    const V4 v4 = *(const V4*)(sV + j * P128 + n16 + 4 * g);
                    float dbv = 0.f;
#pragma unroll
                    for (int r = 0; r < 4; ++r) dbv += av[r] * (float)v4[r];
                    dbv = sum_over_g(dbv);
                    if (g == 0) atomicAdd(&sDb[64 * w + j], dbv);
                    if (j < c.valid) *(V4*)((T*)p.dv + ((c.tok0 + j) * p.HV + hv) * BD + n16 + 4 * g) = pack4<T>(av * bj[t]);
                }
            }
        }
        lds_barrier();                                          // (dv_new and v are done with)
        put_tile<KD>(sDW, PK, rDW, tid);
        put_tile<KD>(sK, PK, rK, tid);
        put_tile<KD>(sP, PK, rP, tid);
        lds_barrier();
        if (u + gridDim.x < units) fetch_first(u + gridDim.x, tid);

        // ---- second half: dX's second term dw (e^gam k)^T, dA = stril(dX diag(beta)), k k^T of the same rows and columns ----
        // (comba: e^gam0 p in k's place wherever k stood on the left of k k^T or under e^gam)
        f32x4 kkT[4];
        {
            V8 fw[4], fk[4];
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                fw[s] = frag_rows(sDW, PK, 16 * w, 32 * s, lane);
                fk[s] = frag_rows(sRows, PK, 16 * w, 32 * s, lane);
            }
#pragma unroll
            for (int tj = 0; tj < 4; ++tj) {
                f32x4 dXw = ZERO4;
                kkT[tj] = ZERO4;
                if (tj <= w) {
#pragma unroll
                    for (int s = 0; s < 4; ++s) {
                        const V8 bk = frag_rows(sK, PK, 16 * tj, 32 * s, lane);
                        dXw = Mma<T>::run(fw[s], frag_rows(sP, PK, 16 * tj, 32 * s, lane), dXw);
                        kkT[tj] = Mma<T>::run(fk[s], bk, kkT[tj]);
                    }
                }
                const int j = 16 * tj + c16;
                const float ej = __expf(sGamRow[j]), bj = sBeta[j];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int i = 16 * w + 4 * g + r;
                    sM1[i * P64 + j] = (T)(i > j ? (dXv[tj][r] + ej * dXw[r]) * bj : 0.f);
                }
            }
        }
        // d(e^gam k) = beta (A^T dw): into dk, dbeta, dgam  (comba: d(e^gam0 p), into dp, dbeta, dgam0)
        f32x4 dk[NA][4], dpk[NA][4];
        {
            V8 fA[4][2];
            float ej[4], bj[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) {
#pragma unroll
                for (int s = 0; s < 2; ++s)
                    if (32 * s + 31 >= 16 * t) fA[t][s] = frag_cols(sA, P64, 32 * s, 16 * t, lane);
                ej[t] = __expf(sGamRow[16 * t + c16]);
                bj[t] = sBeta[16 * t + c16];
            }
#pragma unroll
            for (int a2 = 0; a2 < NA; ++a2) {                   // key features feat(a2) ..
                const int n16 = feat(a2);
                V8 fdw[2];
#pragma unroll
                for (int s = 0; s < 2; ++s) fdw[s] = frag_cols(sDW, PK, 32 * s, n16, lane);
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    f32x4 ak = ZERO4;
#pragma unroll
                    for (int s = 0; s < 2; ++s) {
                        if (32 * s + 31 < 16 * t) continue;
                        ak = Mma<T>::run(fdw[s], fA[t][s], ak);
                    }
                    const int j = 16 * t + c16;
                    const V4 k4 = *(const V4*)(sRows + j * PK + n16 + 4 * g);
                    float dot = 0.f;
#pragma unroll
                    for (int r = 0; r < 4; ++r) dot += ak[r] * (float)k4[r];
                    dot = sum_over_g(dot);
                    if (g == 0) { atomicAdd(&sDb[64 * w + j], ej[t] * dot); atomicAdd(&sDgRow[64 * w + j], bj[t] * ej[t] * dot); }
                    { dpk[a2][t] = ak * (bj[t] * ej[t]); dk[a2][t] = ZERO4; }
                }
            }
        }
        lds_barrier();
        // Y = dA A^T
        {
            V8 fd[2];
#pragma unroll
            for (int s = 0; s < 2; ++s) fd[s] = frag_rows(sM1, P64, 16 * w, 32 * s, lane);
#pragma unroll
            for (int tl = 0; tl < 4; ++tl) {
                f32x4 acc = ZERO4;
#pragma unroll
                for (int s = 0; s < 2; ++s) acc = Mma<T>::run(fd[s], frag_rows(sA, P64, 16 * tl, 32 * s, lane), acc);
                const int l = 16 * tl + c16;
#pragma unroll
                for (int r = 0; r < 4; ++r) sM2[(16 * w + 4 * g + r) * P64 + l] = (T)acc[r];
            }
        }
        lds_barrier();
        // dL = -stril(A^T Y);  E = diag(beta) dL o D as an operand tile;  dbeta, dgam from L = diag(beta) stril(k k^T o D)
        {
            float dbi[4] = {0.f, 0.f, 0.f, 0.f}, rowF[4] = {0.f, 0.f, 0.f, 0.f}, gi[4], bi[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) { gi[r] = sGamRow[16 * w + 4 * g + r]; bi[r] = sBeta[16 * w + 4 * g + r]; }
            V8 fAt[2];
#pragma unroll
            for (int s = 0; s < 2; ++s) fAt[s] = frag_cols(sA, P64, 32 * s, 16 * w, lane);
#pragma unroll
            for (int tl = 0; tl < 4; ++tl) {
                f32x4 acc = ZERO4;
                if (tl <= w) {
#pragma unroll
                    for (int s = 0; s < 2; ++s) acc = Mma<T>::run(fAt[s], frag_cols(sM2, P64, 32 * s, 16 * tl, lane), acc);
                }
                const f32x4 kk = kkT[tl];
                const int l = 16 * tl + c16;
                const float gl = sGam[l];
                float colF = 0.f;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int i = 16 * w + 4 * g + r;
                    float E = 0.f;
                    if (i > l) {
                        const float d = __expf(gi[r] - gl), dL = -acc[r];
                        dbi[r] += dL * kk[r] * d;
                        E = dL * bi[r] * d;
                        const float F = E * kk[r];
                        rowF[r] += F;
                        colF += F;
                    }
                    sM1[i * P64 + l] = (T)E;
                }
                colF = sum_over_g(colF);
                if (g == 0 && tl <= w) atomicAdd(&sDg[64 * w + l], -colF);
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float a = sum_over_c16(dbi[r]), b = sum_over_c16(rowF[r]);
                if (c16 == 0) { atomicAdd(&sDb[64 * w + 16 * w + 4 * g + r], a); atomicAdd(&sDgRow[64 * w + 16 * w + 4 * g + r], b); }
            }
        }
        lds_barrier();
        // dk += E k + E^T k, on top of what the previous kernel left  (comba: dp += E k, dk += E^T p)
        {
            V8 fk[NA][2], fp[NA][2];
#pragma unroll
            for (int a2 = 0; a2 < NA; ++a2)
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    fk[a2][s] = frag_cols(sK, PK, 32 * s, feat(a2), lane);
                    fp[a2][s] = frag_cols(sP, PK, 32 * s, feat(a2), lane);
                }
#pragma unroll
            for (int t = 0; t < 4; ++t) {
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    if (32 * s <= 16 * t + 15) {                // E[i][l], l < i
                        const V8 e = frag_rows(sM1, P64, 16 * t, 32 * s, lane);
#pragma unroll
                        for (int a2 = 0; a2 < NA; ++a2) {
                            dpk[a2][t] = Mma<T>::run(fk[a2][s], e, dpk[a2][t]);
                        }
                    }
                    if (32 * s + 31 >= 16 * t) {                // E[i][l], i > l
                        const V8 e = frag_cols(sM1, P64, 32 * s, 16 * t, lane);
#pragma unroll
                        for (int a2 = 0; a2 < NA; ++a2) {
                            dk[a2][t] = Mma<T>::run(fp[a2][s], e, dk[a2][t]);
                        }
                    }
                }
                const int x = 16 * t + c16;
                if constexpr (L2) {
                    float kdk = 0.f;
#pragma unroll
                    for (int a2 = 0; a2 < NA; ++a2) {
                        const V4 k4 = *(const V4*)(sK + x * PK + feat(a2) + 4 * g);
#pragma unroll
                        for (int r = 0; r < 4; ++r) { dk[a2][t][r] += (float)dk_old[a2][t][r]; kdk += (float)k4[r] * dk[a2][t][r]; }
                    }
                    kdk = sum_over_g(kdk);
                    if (g == 0) sKd[64 * w + x] = kdk;
                    {
                        float pdp = 0.f;
#pragma unroll
                        for (int a2 = 0; a2 < NA; ++a2) {
                            const V4 p4 = *(const V4*)(sP + x * PK + feat(a2) + 4 * g);
#pragma unroll
                            for (int r = 0; r < 4; ++r) pdp += (float)p4[r] * dpk[a2][t][r];
                        }
                        pdp = sum_over_g(pdp);
                        if (g == 0) sPd[64 * w + x] = pdp;
                    }
                } else if (x < c.valid) {
#pragma unroll
                    for (int a2 = 0; a2 < NA; ++a2) {
                        f32x4 acc = dk[a2][t];
#pragma unroll
                        for (int r = 0; r < 4; ++r) acc[r] += (float)dk_old[a2][t][r];
                        *(V4*)((T*)p.dk + ((c.tok0 + x) * p.HV + hv) * KD + feat(a2) + 4 * g) = pack4<T>(acc);
                        *(V4*)((T*)p.dp + ((c.tok0 + x) * p.HV + hv) * KD + feat(a2) + 4 * g) = pack4<T>(dpk[a2][t]);
                    }
                }
            }
        }
        if constexpr (L2) {
            lds_barrier();
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const int x = 16 * t + c16;
                const float dot = (sKd[x] + sKd[64 + x]) + (sKd[128 + x] + sKd[192 + x]), rs = sRk[x];
                if (x < c.valid) {
#pragma unroll
                    for (int a2 = 0; a2 < NA; ++a2) {
                        const V4 k4 = *(const V4*)(sK + x * PK + feat(a2) + 4 * g);
                        f32x4 out;
#pragma unroll
                        for (int r = 0; r < 4; ++r) out[r] = (dk[a2][t][r] - (float)k4[r] * dot) * rs;
                        *(V4*)((T*)p.dk + ((c.tok0 + x) * p.HV + hv) * KD + feat(a2) + 4 * g) = pack4<T>(out);
                    }
                }
                {
                    const float dotp = (sPd[x] + sPd[64 + x]) + (sPd[128 + x] + sPd[192 + x]), rp = sRp[x];
                    if (x < c.valid) {
#pragma unroll
                        for (int a2 = 0; a2 < NA; ++a2) {
                            const V4 p4 = *(const V4*)(sP + x * PK + feat(a2) + 4 * g);
                            f32x4 out;
#pragma unroll
                            for (int r = 0; r < 4; ++r) out[r] = (dpk[a2][t][r] - (float)p4[r] * dotp) * rp;
                            *(V4*)((T*)p.dp + ((c.tok0 + x) * p.HV + hv) * KD + feat(a2) + 4 * g) = pack4<T>(out);
                        }
                    }
                }
            }
        }
        if (w == 0) {
            float x = (sDg[lane] + sDg[64 + lane]) + (sDg[128 + lane] + sDg[192 + lane]);
            // (comba) dg_t = sum_{s >= t} dgam_s + sum_{s > t} dgam0_s: one reverse cumulative sum of both, less the token's own dgam0
            float own0 = 0.f;
            { own0 = (sDg0[lane] + sDg0[64 + lane]) + (sDg0[128 + lane] + sDg0[192 + lane]); x += own0; }
#pragma unroll
            for (int off = 1; off < 64; off <<= 1) {
                const float y = __shfl_down(x, off, 64);
                if (lane + off < 64) x += y;
            }
            x -= own0;
            if (lane < c.valid) {
                p.dg[(c.tok0 + lane) * p.HV + hv] = x;
                p.dbeta[(c.tok0 + lane) * p.HV + hv] = (sDb[lane] + sDb[64 + lane]) + (sDb[128 + lane] + sDb[192 + lane]);
            }
        }
        lds_barrier();
    }
}

#include "gdn_chunk_bwd_unit.h"
#include "gdn_chunk_bwd_unit256.h"

// The partial rows of dq and dk (and, where parts cut a value head, the partial sums of dg and dbeta) added up in fp32, in a fixed order:
// eight rows of a chunk and q/k head per workgroup.
template <typename T, int KD>
__global__ __launch_bounds__(256) void gdn_bwd_add_parts_kernel(BwdParams p, int64_t) {
    typedef typename Mma<T>::V4 V4;
    const uint32_t unit = blockIdx.x >> 3, ch = unit / (uint32_t)p.H, hq = unit - ch * p.H;
    const ChunkAt c = chunk_at(p, ch);
    const int row0 = 8 * (blockIdx.x & 7), rows = min(8, c.valid - row0);        // (none: the loops below have nothing to do)
    constexpr int PIECES = KD / 4;
    for (int i = threadIdx.x; i < 2 * PIECES * rows; i += 256) {
        const int piece = i % PIECES, r = i / PIECES, isk = r >= rows;
        const int64_t row = (c.tok0 + row0 + (isk ? r - rows : r)) * p.H + hq;
        const f32x4* part = (const f32x4*)(isk ? p.dk_part : p.dq_part) + row * p.parts * PIECES + piece;
        f32x4 sum = part[0];
        for (int n = 1; n < p.parts; ++n) sum += part[(int64_t)n * PIECES];
        *(V4*)((T*)(isk ? p.dk : p.dq) + row * KD + 4 * piece) = pack4<T>(sum);
    }
    if (p.split > 1) {
        const int HVg = p.HV / p.nb, group = HVg / p.H;
        for (int i = threadIdx.x; i < group * rows; i += 256) {
            const int64_t at = (c.tok0 + row0 + i / group) * HVg + hq * group + i % group;
            float dg = 0.f, db = 0.f;
            for (int n = 0; n < p.split; ++n) { dg += p.dg_part[at * p.split + n]; db += p.db_part[at * p.split + n]; }
            p.dg[at] = dg; p.dbeta[at] = db;
        }
    }
}

struct BwdLaunch { const void* f; size_t smem; const char* name; unsigned grid, threads; int64_t arg; };
static int launch_all(const BwdParams& p, const BwdLaunch* ks, int n, hipStream_t stream) {
    for (int i = 0; i < n; ++i) {
        if (ks[i].grid == 0) continue;
        if (int rc = ensure_dynamic_smem_for(ks[i].f, ks[i].smem, ks[i].name)) return rc;
        void* args[] = {(void*)&p, (void*)&ks[i].arg};
        if (hipLaunchKernel(ks[i].f, dim3(ks[i].grid), dim3(ks[i].threads), args, ks[i].smem, stream) != hipSuccess) return check_launch(ks[i].name);
        if (int rc = check_launch(ks[i].name)) return rc;
    }
    return GDN_OK;
}

// workgroups of a scan with slices of v value columns: the runs in eighths (XCDs), each with its slices
static unsigned scan_grid(const BwdParams& p, int VD, int v) { return (unsigned)((p.N * p.HV + 7) / 8 * 8 * (VD / v)); }

// Both scans of whole sequences in one launch, up to 128 runs every workgroup with a CU to itself, as many value columns each as that
// allows.  What a CU moves per step bounds the step (some 22 GB/s per CU, loads and stores together, whatever shares the CU).
template <typename T, int FORM, bool EXACT>
static BwdLaunch scans_128_of(const BwdParams& p) {
    const int64_t runs = p.N * p.HV;
    auto apart = [&](const void* f, size_t smem, int v, int vr) {         // columns forwards, backwards
        const unsigned nrev = scan_grid(p, BD, vr);
        return BwdLaunch{f, smem, "gdn_bwd_scans_apart_kernel", nrev + scan_grid(p, BD, v), v >= 64 ? 512u : 256u, (int64_t)nrev};
    };
    if (runs <= 32) return apart((const void*)gdn_bwd_scans_apart_kernel<T, 32, 32, BD, BD, FORM, EXACT>, bwd_scans_apart_smem<32, 32, BD, FORM>(), 32, 32);
    if (runs <= 64) return apart((const void*)gdn_bwd_scans_apart_kernel<T, 64, 64, BD, BD, FORM, EXACT>, bwd_scans_apart_smem<64, 64, BD, FORM>(), 64, 64);
    // (65 to 80 runs: the longer, backward scan halves its columns where a workgroup each still has a CU to itself: the launch with 64 / 128 and 64 / 128 columns, 72 runs of
    // 500 tokens 36.0 / 29.7 / 37.6 us, 80 of 1500 101.3 / 84.6 / 118.9, of 5000 342 / 277 / 388; 96 of 2000 175.9 / 207.9 / 164.3, 128 of 1000 92.5 / 107.1 / 89.5)
    if (scan_grid(p, BD, 128) + scan_grid(p, BD, 64) <= 256)
        return apart((const void*)gdn_bwd_scans_apart_kernel<T, 128, 64, BD, BD, FORM, EXACT>, bwd_scans_apart_smem<128, 64, BD, FORM>(), 128, 64);
    return apart((const void*)gdn_bwd_scans_apart_kernel<T, 128, 128, BD, BD, FORM, EXACT>, bwd_scans_apart_smem<128, 128, BD, FORM>(), 128, 128);
}
// (EXACT requests pay once the sequences have some chunks: figures at fetch_scan)
template <typename T, int FORM>
static BwdLaunch scans_128(const BwdParams& p, int64_t num_chunks) {
    const int64_t least = FORM == FORM_GATED && p.N * p.HV > 64 ? 16 : 8;
    return num_chunks >= least * p.N ? scans_128_of<T, FORM, true>(p) : scans_128_of<T, FORM, false>(p);
}

template <typename T, int KD, int VD>
static int launch_bwd(const BwdParams& p_in, int64_t num_chunks, hipStream_t stream) {
    BwdParams p = p_in;
    const int64_t runs = p.N * p.HV;
    const unsigned units = (unsigned)(num_chunks * (p.HV / p.nb));
    const bool l2 = p.q_raw != nullptr;
    // Time segments for the two scans (up to 128 key features, dense input): long sequences on few heads leave CUs without a
    // workgroup; never more workgroups than CUs, segments of 8 chunks or more, and at least 24 steps saved per workgroup
    // (a warm-up of typical length must pay).  GDN_FLAG_SCAN_WIDE asks for whole sequences, GDN_FLAG_SCAN_SEGMENTS for segments of 4.
    p.nseg = 1; p.seg_chunks = (int)p.NT; p.warm_cap = 0;
    if (KD <= BD && !p.cu_seqlens && runs <= 64 && !(p.flags & GDN_FLAG_SCAN_WIDE)) {
        const bool force = p.flags & GDN_FLAG_SCAN_SEGMENTS;
        const int nseg = (int)std::min<int64_t>(256 / scan_grid(p, VD, 32), p.NT / (force ? 4 : 8));
        if (nseg >= 2 && (force || p.NT - p.NT / nseg >= 24)) {
            p.nseg = nseg;
            p.seg_chunks = (int)((p.NT + nseg - 1) / nseg);
            p.warm_cap = std::min(WARM_CAP_MAX, p.seg_chunks + p.seg_chunks / 4 + 6);
        }
    }
    BwdLaunch ks[5] = {};
    const unsigned pgrid = (units + BP_WAVES - 1) / BP_WAVES;
    ks[0] = {l2 ? (const void*)gdn_bwd_prepare_kernel<T, KD, true> : (const void*)gdn_bwd_prepare_kernel<T, KD, false>, 0, "gdn_bwd_prepare_kernel", pgrid, 64 * BP_WAVES, units};
    if constexpr (KD <= BD) {
        if (p.nseg > 1)                                         // both scans side by side in a workgroup: every CU has one already
            ks[1] = {(const void*)gdn_bwd_scans_kernel<T, 32, KD, VD>, bwd_scans_smem<32, KD>(), "gdn_bwd_scans_kernel", scan_grid(p, VD, 32) * p.nseg, 512, 0};
        else if constexpr (VD == BD) ks[1] = scans_128<T, FORM_GATED>(p, num_chunks);
        // (64 x 64: two workgroups fit a CU, so that 32-column slices pay up to twice as many runs.  They read every tile twice, which
        // costs once the tiles outgrow the caches, from some 2200 (chunk, head) pairs on, the step from 2600: the launch with 32 / 64 columns, 72 heads of 1500 tokens 50.1 / 53.2 us,
        // of 2000 68.0 / 68.7, of 2500 90.8 / 87.1; 80 heads of 1800 tokens 64.2 / 63.7, of 2200 86.3 / 80.0; 96 heads of 1300 tokens 44.6 / 46.2, of 1500 56.2 / 53.8, of
        // 2000 86.2 / 77.7; 112 heads of 1200 tokens 43.8 / 43.9, of 1300 51.9 / 49.1; 128 heads of 1000 tokens 37.6 / 37.5, of 2000 96.6 / 78.6; the step, 112 heads of 1300 tokens 211.8 / 213.1, 80 of 2200 276.6 / 272.8, 96 of 2000 286 / 276)
        else if (runs <= 64 || (runs < 128 && units <= 2600)) ks[1] = {(const void*)gdn_bwd_scans_apart_kernel<T, 32, 32, KD, VD, FORM_GATED, false>, bwd_scans_apart_smem<32, 32, KD, FORM_GATED>(), "gdn_bwd_scans_apart_kernel", 2 * scan_grid(p, VD, 32), 256, (int64_t)scan_grid(p, VD, 32)};
        else ks[1] = {(const void*)gdn_bwd_scans_apart_kernel<T, 64, 64, KD, VD, FORM_GATED, false>, bwd_scans_apart_smem<64, 64, KD, FORM_GATED>(), "gdn_bwd_scans_apart_kernel", 2 * scan_grid(p, VD, 64), 512, (int64_t)scan_grid(p, VD, 64)};
    } else {
        // 256 key features: the reverse scan's tiles leave room for 64 columns at most, the forward scan can take 128: fewer workgroups, each 1.2 times as long.
        // Up to 256 runs what counts are the rounds of 256 workgroups (one to a CU) that the launch takes: with 64 / 128 columns forwards, 80 runs of 500 tokens 53.2 / 44.2
        // us, 96 64.2 / 77.7, 128 68.6 / 79.4, 144 91.7 / 84.9, 176 111.3 / 125.6, 192 112.7 / 126.0, 192 of 2000 449 / 508, 224 of 1000 277 / 270, 256 289 / 271.  With
        // more runs rounds of sequences of different lengths fill one another up and 128 pays on the whole: 320 of 1500 560 / 545, 384 of 700 303 / 311, the step of 384
        // packed runs 1638 / 1620, 512 of 1000 575 / 543.
        const unsigned half = scan_grid(p, VD, 64), whole = scan_grid(p, VD, 128);
        // (EXACT requests: up to 32 runs four chunks or more on average, where 64 columns go round more than once 32; figures at fetch_scan)
        if (runs <= 32)
            ks[1] = {num_chunks >= 4 * p.N ? (const void*)gdn_bwd_scans_apart_kernel<T, 32, 32, KD, VD, FORM_GATED, true> : (const void*)gdn_bwd_scans_apart_kernel<T, 32, 32, KD, VD, FORM_GATED, false>,
                     bwd_scans_apart_smem<32, 32, KD, FORM_GATED>(), "gdn_bwd_scans_apart_kernel", 2 * scan_grid(p, VD, 32), 256, (int64_t)scan_grid(p, VD, 32)};
        else if (runs > 256 || (runs > 64 && 6 * ((half + whole + 255) / 256) < 5 * ((2 * half + 255) / 256))) ks[1] = {(const void*)gdn_bwd_scans_apart_kernel<T, 128, 64, KD, VD, FORM_GATED, false>, bwd_scans_apart_smem<128, 64, KD, FORM_GATED>(), "gdn_bwd_scans_apart_kernel", half + whole, 512, (int64_t)half};
        else
            ks[1] = {runs > 64 && num_chunks >= 32 * p.N ? (const void*)gdn_bwd_scans_apart_kernel<T, 64, 64, KD, VD, FORM_GATED, true> : (const void*)gdn_bwd_scans_apart_kernel<T, 64, 64, KD, VD, FORM_GATED, false>,
                     bwd_scans_apart_smem<64, 64, KD, FORM_GATED>(), "gdn_bwd_scans_apart_kernel", 2 * half, 512, (int64_t)half};
    }
    const int64_t items = num_chunks * p.H * p.parts;
    if constexpr (KD <= BD) {
        const void* unit = p.dq_part ? (l2 ? (const void*)gdn_bwd_unit_kernel<T, KD, true, true> : (const void*)gdn_bwd_unit_kernel<T, KD, false, true>)
                                     : (l2 ? (const void*)gdn_bwd_unit_kernel<T, KD, true, false> : (const void*)gdn_bwd_unit_kernel<T, KD, false, false>);
        ks[3] = {unit, bwd_unit_smem<KD>(), "gdn_bwd_unit_kernel", (unsigned)std::min<int64_t>(items, KD == 64 ? 512 : 256), 64 * bwd_unit_waves<KD>(), items};
    } else {
        const void* unit = l2 ? (const void*)gdn_bwd_unit256_kernel<T, true> : (const void*)gdn_bwd_unit256_kernel<T, false>;
        ks[3] = {unit, BWD_UNIT256_SMEM, "gdn_bwd_unit256_kernel", (unsigned)std::min<int64_t>(items, 256), 64 * UNIT256_NW, items};
    }
    if (p.dq_part) ks[4] = {(const void*)gdn_bwd_add_parts_kernel<T, KD>, 0, "gdn_bwd_add_parts_kernel", (unsigned)(num_chunks * p.H * 8), 256, 0};
    return launch_all(p, ks, 5, stream);
}

template <typename T>
static int launch_bwd_comba(const BwdParams& p, int64_t num_chunks, hipStream_t stream) {
    const unsigned units = (unsigned)(num_chunks * p.HV);
    const bool l2 = p.q_raw != nullptr;                         // (the entry has checked H == HV)
    const BwdLaunch ks[4] = {
        {l2 ? (const void*)gdn_bwd_prepare_comba_kernel<T, true> : (const void*)gdn_bwd_prepare_comba_kernel<T, false>, BWD_PREP_COMBA_SMEM, "gdn_bwd_prepare_comba_kernel", units < 512u ? units : 512u, 256, units},
        scans_128<T, FORM_COMBA>(p, num_chunks),
        {l2 ? (const void*)gdn_bwd_dqkw_kernel<T, true> : (const void*)gdn_bwd_dqkw_kernel<T, false>, BWD_DQKW_SMEM, "gdn_bwd_dqkw_kernel", units < 256u ? units : 256u, 256, units},
        {l2 ? (const void*)gdn_bwd_wy2_kernel<T, true> : (const void*)gdn_bwd_wy2_kernel<T, false>, BWD_WY2_SMEM, "gdn_bwd_wy2_kernel", units < 512u ? units : 512u, 256, units},
    };
    return launch_all(p, ks, 4, stream);
}

#include "gdn_chunk_kda_bwd.h"      // (inside the namespace: it builds on the types and the two scans above)

}  // namespace gdn

// All entries of the two operators.  dq and dk per q/k head when `per_head`, else per value head; `pk` (and `dp`): comba.
static int chunk_bwd_entry(
    const char* who, bool comba, bool per_head,
    const void* q, const void* k, const void* pk, const void* v, const void* g, const void* beta,
    const float* A_log, const float* dt_bias,
    const float* h0, const void* dout, const float* dht,
    void* dq, void* dk, void* dp, void* dv, float* dg, float* dbeta, float* dh0,
    const void* cu_seqlens, const void* chunk_table, const void* chunk_offsets,
    void* workspace, size_t workspace_bytes,
    int64_t B, int64_t T, int64_t H, int64_t HV, int64_t K, int64_t V,
    int64_t N, int64_t num_chunks,
    float scale, int qkv_dtype, int gb_dtype, uint32_t flags, void* stream) {
    using namespace gdn;
    const bool l2 = flags & GDN_FLAG_QK_L2NORM;
    const int64_t VD = K == 64 ? 64 : BD, nb = V / VD;
    GDN_CHECK_ARG(B >= 1 && T >= 0 && H >= 1 && HV >= 1 && N >= 1 && num_chunks >= 0 && V >= 1, GDN_ERR_INVALID, "%s: bad dimension", who);
    GDN_CHECK_ARG(HV % H == 0, GDN_ERR_INVALID, "%s: HV=%lld not divisible by H=%lld", who, (long long)HV, (long long)H);
    GDN_CHECK_ARG(qkv_dtype == GDN_DTYPE_BF16 || qkv_dtype == GDN_DTYPE_F16, GDN_ERR_UNSUPPORTED, "%s: q/k/v/do must be bf16 or f16", who);
    GDN_CHECK_ARG(HV * nb <= 65535 && num_chunks * HV * nb < (1ll << 31) && N * HV * nb * 4 < (1ll << 31), GDN_ERR_UNSUPPORTED,
                  "%s: too many heads or chunks for one launch", who);
    if (cu_seqlens) {
        GDN_CHECK_ARG(B == 1, GDN_ERR_INVALID, "%s: with cu_seqlens B must be 1", who);
        GDN_CHECK_ARG((chunk_table || num_chunks == 0) && chunk_offsets, GDN_ERR_INVALID, "%s: packed input needs chunk_table and chunk_offsets", who);
    } else {
        GDN_CHECK_ARG(N == B, GDN_ERR_INVALID, "%s: without cu_seqlens N must equal B", who);
        GDN_CHECK_ARG(num_chunks == B * ((T + CH - 1) / CH), GDN_ERR_INVALID, "%s: num_chunks does not match B and T", who);
    }
    hipStream_t s = (hipStream_t)stream;
    if (T == 0 || num_chunks == 0) {
        if (dh0) return launch_state_copy(dht, dh0, N * HV * K * V, s);
        return GDN_OK;
    }
    GDN_CHECK_ARG(q && k && v && beta && dout && dq && dk && dv && dg && dbeta, GDN_ERR_INVALID,
                  "%s: q, k, v, beta, do, dq, dk, dv, dg, dbeta must not be NULL", who);
    GDN_CHECK_ARG(!comba || (pk && dp && g), GDN_ERR_INVALID, "%s: p, g and dp must not be NULL", who);
    GDN_CHECK_ARG(!l2 || !comba || H == HV, GDN_ERR_UNSUPPORTED, "%s: the l2 normalisation is taken in here for H == HV only", who);
    for (const void* x : {q, k, pk, v, dout, (const void*)h0, (const void*)dht, (const void*)dq, (const void*)dk, (const void*)dp, (const void*)dv, (const void*)dh0})
        GDN_CHECK_ARG(((uintptr_t)x % 16) == 0, GDN_ERR_INVALID, "%s: tensors must be 16-byte aligned", who);
    GDN_CHECK_ARG(((uintptr_t)workspace % 256) == 0, GDN_ERR_INVALID, "%s: the workspace must be 256-byte aligned", who);
    BwdParams p{};
    size_t need = comba ? comba_bwd_ws_layout(num_chunks * HV, (char*)workspace, &p.ws) : bwd_ws_layout(num_chunks, HV, nb, K, VD, (char*)workspace, &p.ws);
    const size_t rows_bytes = ws_align((size_t)(B * T * H) * K * 2), factors_bytes = ws_align((size_t)(B * T * H) * 4);
    const size_t l2_at = need;
    if (l2) need += (comba ? 3 : 2) * (rows_bytes + factors_bytes);
    const size_t parts_at = need;
    BwdParts parts;
    if (per_head && !comba) parts = bwd_parts(num_chunks, N, B * T, H, HV, nb, K);
    if (workspace_bytes < need + parts.bytes()) parts = BwdParts();      // (a caller's workspace without room for them: one part)
    need += parts.bytes();
    GDN_CHECK_ARG(workspace && workspace_bytes >= need, GDN_ERR_WORKSPACE, "%s: workspace of %zu bytes needed, %zu given", who,
                  need, workspace_bytes);
    if (l2) {
        char* at = (char*)workspace + l2_at;
        p.q_raw = q; p.k_raw = k;
        q = at; k = at + rows_bytes;
        p.q_rstd = (const float*)(at + 2 * rows_bytes); p.k_rstd = (const float*)(at + 2 * rows_bytes + factors_bytes);
        if (comba) {
            at += 2 * (rows_bytes + factors_bytes);
            p.pk_raw = pk;
            pk = at;
            p.p_rstd = (const float*)(at + rows_bytes);
        }
    }
    p.q = q; p.k = k; p.v = v; p.g = g; p.beta = beta; p.A_log = A_log; p.dt_bias = dt_bias; p.h0 = h0; p.dout = dout; p.dht = dht;
    p.dq = dq; p.dk = dk; p.dv = dv; p.dg = dg; p.dbeta = dbeta; p.dh0 = dh0; p.pk = pk; p.dp = dp;
    p.cu_seqlens = cu_seqlens; p.chunk_table = chunk_table; p.chunk_offsets = chunk_offsets;
    p.T = T; p.H = (int)H; p.HV = (int)(HV * nb); p.nb = (int)nb; p.N = N; p.NT = (T + CH - 1) / CH;
    p.scale = scale; p.gb_dtype = gb_dtype & 255; p.beta_dtype = beta_dtype_of(gb_dtype); p.flags = flags;
    p.nseg = 1; p.seg_chunks = (int)p.NT; p.warm_cap = 0;
    p.parts = per_head ? parts.parts : (int)(HV / H);
    p.split = parts.split;
    if (parts.row_bytes) {
        WsTake take{(char*)workspace + parts_at};
        p.dq_part = (float*)take(parts.row_bytes); p.dk_part = (float*)take(parts.row_bytes);
        if (parts.split > 1) { p.dg_part = (float*)take(parts.head_bytes); p.db_part = (float*)take(parts.head_bytes); }
    }
    const bool b16 = qkv_dtype == GDN_DTYPE_BF16;
    if (comba) return b16 ? launch_bwd_comba<bf16_t>(p, num_chunks, s) : launch_bwd_comba<f16_t>(p, num_chunks, s);
    if (K == 64) return b16 ? launch_bwd<bf16_t, 64, 64>(p, num_chunks, s) : launch_bwd<f16_t, 64, 64>(p, num_chunks, s);
    if (K == BD) return b16 ? launch_bwd<bf16_t, BD, BD>(p, num_chunks, s) : launch_bwd<f16_t, BD, BD>(p, num_chunks, s);
    return b16 ? launch_bwd<bf16_t, 2 * BD, BD>(p, num_chunks, s) : launch_bwd<f16_t, 2 * BD, BD>(p, num_chunks, s);
}

constexpr uint32_t BWD_PLAIN_FLAGS = GDN_FLAG_CU_INT32 | GDN_FLAG_SEQ_ORDER | GDN_FLAG_SCAN_WIDE | GDN_FLAG_SCAN_SEGMENTS;
static int bwd_plain_args(const char* who, int64_t K, int64_t V, bool wide, uint32_t flags) {
    using namespace gdn;
    GDN_CHECK_ARG((K == BD || (K == 2 * BD && wide)) && V == BD, GDN_ERR_UNSUPPORTED,
                  "%s: K = 128%s and V = 128 only (got K=%lld V=%lld); pad smaller head dims with zeros", who, wide ? " or 256" : "",
                  (long long)K, (long long)V);
    GDN_CHECK_ARG((flags & ~BWD_PLAIN_FLAGS) == 0, GDN_ERR_UNSUPPORTED,
                  "%s: only the flags on the tables and on the form of the scans are understood here (activations and the state layout are the caller's)", who);
    return GDN_OK;
}

extern "C" size_t gdn_chunk_bwd_heads_workspace_bytes(int64_t num_chunks, int64_t H, int64_t HV, int64_t K, int64_t V, int64_t tokens, uint32_t flags) {
    using namespace gdn;
    if (num_chunks < 0 || H < 1 || HV < 1 || tokens < 0) return 0;
    if (!(K == 64 && V == 64) && !((K == BD || K == 2 * BD) && V >= BD && V % BD == 0)) return 0;
    const int64_t VD = K == 64 ? 64 : BD;
    size_t need = bwd_ws_layout(num_chunks, HV, V / VD, K, VD, nullptr, nullptr);
    if (flags & GDN_FLAG_QK_L2NORM) need += 2 * ws_align((size_t)(tokens * H) * K * 2) + 2 * ws_align((size_t)(tokens * H) * 4);
    return need + (HV % H == 0 ? bwd_parts(num_chunks, 1, tokens, H, HV, V / VD, K).bytes() : 0);
}

extern "C" int gdn_chunk_bwd_heads(
    const void* q, const void* k, const void* v, const void* g, const void* beta,
    const float* A_log, const float* dt_bias,
    const float* h0, const void* dout, const float* dht,
    void* dq, void* dk, void* dv, float* dg, float* dbeta, float* dh0,
    const void* cu_seqlens, const void* chunk_table, const void* chunk_offsets,
    void* workspace, size_t workspace_bytes,
    int64_t B, int64_t T, int64_t H, int64_t HV, int64_t K, int64_t V,
    int64_t N, int64_t num_chunks,
    float scale, int qkv_dtype, int gb_dtype, uint32_t flags, void* stream) {
    using namespace gdn;
    const char* who = "gdn_chunk_bwd_heads";
    GDN_CHECK_ARG((K == 64 && V == 64) || ((K == BD || K == 2 * BD) && V >= BD && V % BD == 0), GDN_ERR_UNSUPPORTED,
                  "%s: K = V = 64, or K = 128 or 256 with V a multiple of 128 (got K=%lld V=%lld); pad other head dims with zeros", who, (long long)K, (long long)V);
    GDN_CHECK_ARG((flags & ~(BWD_PLAIN_FLAGS | GDN_FLAG_QK_L2NORM | GDN_FLAG_BETA_SIGMOID | GDN_FLAG_NEG_EIGVAL)) == 0, GDN_ERR_UNSUPPORTED,
                  "%s: unknown flag", who);
    return chunk_bwd_entry(who, false, true, q, k, nullptr, v, g, beta, A_log, dt_bias, h0, dout, dht, dq, dk, nullptr, dv, dg, dbeta, dh0,
                           cu_seqlens, chunk_table, chunk_offsets, workspace, workspace_bytes, B, T, H, HV, K, V, N, num_chunks,
                           scale, qkv_dtype, gb_dtype, flags, stream);
}

extern "C" size_t gdn_chunk_bwd_workspace_bytes(int64_t num_chunks, int64_t HV, int64_t K) {
    const size_t own = gdn_chunk_bwd_heads_workspace_bytes(num_chunks, 1, HV, K, gdn::BD, 0, 0);
    return K == gdn::BD && own ? std::max(own, gdn::comba_bwd_ws_layout(num_chunks * HV, nullptr, nullptr)) : own;      // (gdn_chunk_comba_bwd's too)
}

extern "C" int gdn_chunk_bwd(
    const void* q, const void* k, const void* v, const void* g, const void* beta,
    const float* h0, const void* dout, const float* dht,
    void* dq, void* dk, void* dv, float* dg, float* dbeta, float* dh0,
    const void* cu_seqlens, const void* chunk_table, const void* chunk_offsets,
    void* workspace, size_t workspace_bytes,
    int64_t B, int64_t T, int64_t H, int64_t HV, int64_t K, int64_t V,
    int64_t N, int64_t num_chunks,
    float scale, int qkv_dtype, int gb_dtype, uint32_t flags, void* stream) {
    if (int rc = bwd_plain_args("gdn_chunk_bwd", K, V, true, flags)) return rc;
    return chunk_bwd_entry("gdn_chunk_bwd", false, false, q, k, nullptr, v, g, beta, nullptr, nullptr, h0, dout, dht, dq, dk, nullptr, dv, dg, dbeta, dh0,
                           cu_seqlens, chunk_table, chunk_offsets, workspace, workspace_bytes, B, T, H, HV, K, V, N, num_chunks,
                           scale, qkv_dtype, gb_dtype, flags, stream);
}

extern "C" size_t gdn_chunk_bwd_qk_l2norm_workspace_bytes(int64_t num_chunks, int64_t HV, int64_t K, int64_t tokens) {
    if (K != 128 || tokens < 0) return 0;
    const size_t rows = gdn_chunk_bwd_heads_workspace_bytes(0, HV, HV, K, gdn::BD, tokens, GDN_FLAG_QK_L2NORM);
    return rows ? gdn_chunk_bwd_workspace_bytes(num_chunks, HV, K) + rows : 0;
}

extern "C" int gdn_chunk_bwd_qk_l2norm(
    const void* q, const void* k, const void* v, const void* g, const void* beta,
    const float* h0, const void* dout, const float* dht,
    void* dq, void* dk, void* dv, float* dg, float* dbeta, float* dh0,
    const void* cu_seqlens, const void* chunk_table, const void* chunk_offsets,
    void* workspace, size_t workspace_bytes,
    int64_t B, int64_t T, int64_t H, int64_t HV, int64_t K, int64_t V,
    int64_t N, int64_t num_chunks,
    float scale, int qkv_dtype, int gb_dtype, uint32_t flags, void* stream) {
    using namespace gdn;
    const char* who = "gdn_chunk_bwd_qk_l2norm";
    if (int rc = bwd_plain_args(who, K, V, true, flags)) return rc;
    GDN_CHECK_ARG(H == HV && K == BD, GDN_ERR_UNSUPPORTED, "%s: H == HV and K = 128 only (gdn_chunk_bwd_heads takes the others)", who);
    const size_t need = gdn_chunk_bwd_qk_l2norm_workspace_bytes(num_chunks, HV, K, B * T);
    GDN_CHECK_ARG(num_chunks <= 0 || T <= 0 || workspace_bytes >= need, GDN_ERR_WORKSPACE, "%s: workspace of %zu bytes needed, %zu given", who, need, workspace_bytes);
    return chunk_bwd_entry(who, false, true, q, k, nullptr, v, g, beta, nullptr, nullptr, h0, dout, dht, dq, dk, nullptr, dv, dg, dbeta, dh0,
                           cu_seqlens, chunk_table, chunk_offsets, workspace, workspace_bytes, B, T, H, HV, K, V, N, num_chunks,
                           scale, qkv_dtype, gb_dtype, flags | GDN_FLAG_QK_L2NORM, stream);
}

extern "C" int gdn_chunk_comba_bwd(
    const void* q, const void* k, const void* p, const void* v, const void* g, const void* beta,
    const float* h0, const void* dout, const float* dht,
    void* dq, void* dk, void* dp, void* dv, float* dg, float* dbeta, float* dh0,
    const void* cu_seqlens, const void* chunk_table, const void* chunk_offsets,
    void* workspace, size_t workspace_bytes,
    int64_t B, int64_t T, int64_t H, int64_t HV, int64_t K, int64_t V,
    int64_t N, int64_t num_chunks,
    float scale, int qkv_dtype, int gb_dtype, uint32_t flags, void* stream) {
    if (int rc = bwd_plain_args("gdn_chunk_comba_bwd", K, V, false, flags)) return rc;
    return chunk_bwd_entry("gdn_chunk_comba_bwd", true, false, q, k, p, v, g, beta, nullptr, nullptr, h0, dout, dht, dq, dk, dp, dv, dg, dbeta, dh0,
                           cu_seqlens, chunk_table, chunk_offsets, workspace, workspace_bytes, B, T, H, HV, K, V, N, num_chunks,
                           scale, qkv_dtype, gb_dtype, flags, stream);
}

extern "C" size_t gdn_chunk_comba_bwd_qk_l2norm_workspace_bytes(int64_t num_chunks, int64_t HV, int64_t tokens) {
    if (num_chunks < 0 || HV < 1 || tokens < 0) return 0;
    return gdn::comba_bwd_ws_layout(num_chunks * HV, nullptr, nullptr) + 3 * gdn::ws_align((size_t)(tokens * HV) * gdn::BD * 2) +
           3 * gdn::ws_align((size_t)(tokens * HV) * 4);
}

extern "C" int gdn_chunk_comba_bwd_qk_l2norm(
    const void* q, const void* k, const void* p, const void* v, const void* g, const void* beta,
    const float* h0, const void* dout, const float* dht,
    void* dq, void* dk, void* dp, void* dv, float* dg, float* dbeta, float* dh0,
    const void* cu_seqlens, const void* chunk_table, const void* chunk_offsets,
    void* workspace, size_t workspace_bytes,
    int64_t B, int64_t T, int64_t H, int64_t HV, int64_t K, int64_t V,
    int64_t N, int64_t num_chunks,
    float scale, int qkv_dtype, int gb_dtype, uint32_t flags, void* stream) {
    if (int rc = bwd_plain_args("gdn_chunk_comba_bwd_qk_l2norm", K, V, false, flags)) return rc;
    return chunk_bwd_entry("gdn_chunk_comba_bwd_qk_l2norm", true, true, q, k, p, v, g, beta, nullptr, nullptr, h0, dout, dht, dq, dk, dp, dv, dg, dbeta, dh0,
                           cu_seqlens, chunk_table, chunk_offsets, workspace, workspace_bytes, B, T, H, HV, K, V, N, num_chunks,
                           scale, qkv_dtype, gb_dtype, flags | GDN_FLAG_QK_L2NORM, stream);
}

extern "C" size_t gdn_chunk_kda_bwd_workspace_bytes(int64_t num_chunks, int64_t HV) {
    if (num_chunks < 0 || HV < 1) return 0;
    return gdn::kda_bwd_ws_layout(num_chunks * HV, nullptr, nullptr);
}

static int kda_bwd_entry(
    const char* who, bool l2,
    const void* q, const void* k, const void* v, const float* g, const void* beta,
    const float* h0, const void* dout, const float* dht,
    void* dq, void* dk, void* dv, float* dg, float* dbeta, float* dh0,
    const void* cu_seqlens, const void* chunk_table, const void* chunk_offsets,
    void* workspace, size_t workspace_bytes,
    int64_t B, int64_t T, int64_t H, int64_t HV, int64_t K, int64_t V,
    int64_t N, int64_t num_chunks,
    float scale, int qkv_dtype, int gb_dtype, uint32_t flags, void* stream) {
    using namespace gdn;
    GDN_CHECK_ARG(B >= 1 && T >= 0 && H >= 1 && HV >= 1 && N >= 1 && num_chunks >= 0, GDN_ERR_INVALID, "%s: bad dimension", who);
    GDN_CHECK_ARG(HV % H == 0, GDN_ERR_INVALID, "%s: HV=%lld not divisible by H=%lld", who, (long long)HV, (long long)H);
    GDN_CHECK_ARG(!l2 || H == HV, GDN_ERR_UNSUPPORTED, "%s: the l2 normalisation is taken in here for H == HV only", who);
    GDN_CHECK_ARG(K == BD && V == BD, GDN_ERR_UNSUPPORTED, "%s: K = V = 128 only (got K=%lld V=%lld); pad smaller head dims with zeros",
                  who, (long long)K, (long long)V);
    GDN_CHECK_ARG(qkv_dtype == GDN_DTYPE_BF16 || qkv_dtype == GDN_DTYPE_F16, GDN_ERR_UNSUPPORTED, "%s: q/k/v/do must be bf16 or f16", who);
    GDN_CHECK_ARG((flags & ~(uint32_t)(GDN_FLAG_CU_INT32 | GDN_FLAG_SEQ_ORDER)) == 0, GDN_ERR_UNSUPPORTED,
                  "%s: only GDN_FLAG_CU_INT32 is understood here (activations and the state layout are the caller's)", who);
    GDN_CHECK_ARG(HV <= 65535 && num_chunks * HV < (1ll << 31) && N * HV * 4 < (1ll << 31), GDN_ERR_UNSUPPORTED,
                  "%s: too many heads or chunks for one launch", who);
    if (cu_seqlens) {
        GDN_CHECK_ARG(B == 1, GDN_ERR_INVALID, "%s: with cu_seqlens B must be 1", who);
        GDN_CHECK_ARG((chunk_table || num_chunks == 0) && chunk_offsets, GDN_ERR_INVALID, "%s: packed input needs chunk_table and chunk_offsets", who);
    } else {
        GDN_CHECK_ARG(N == B, GDN_ERR_INVALID, "%s: without cu_seqlens N must equal B", who);
        GDN_CHECK_ARG(num_chunks == B * ((T + CH - 1) / CH), GDN_ERR_INVALID, "%s: num_chunks does not match B and T", who);
    }
    hipStream_t s = (hipStream_t)stream;
    if (T == 0 || num_chunks == 0) {
        if (dh0) return launch_state_copy(dht, dh0, N * HV * K * V, s);
        return GDN_OK;
    }
    GDN_CHECK_ARG(q && k && v && g && beta && dout && dq && dk && dv && dg && dbeta, GDN_ERR_INVALID,
                  "%s: q, k, v, g, beta, do, dq, dk, dv, dg, dbeta must not be NULL", who);
    for (const void* x : {q, k, v, dout, (const void*)g, (const void*)h0, (const void*)dht, (const void*)dq, (const void*)dk, (const void*)dv,
                          (const void*)dg, (const void*)dh0})
        GDN_CHECK_ARG(((uintptr_t)x % 16) == 0, GDN_ERR_INVALID, "%s: tensors must be 16-byte aligned", who);
    GDN_CHECK_ARG(((uintptr_t)workspace % 256) == 0, GDN_ERR_INVALID, "%s: the workspace must be 256-byte aligned", who);
    BwdParams p{};
    const size_t need = kda_bwd_ws_layout(num_chunks * HV, (char*)workspace, &p.ws);
    GDN_CHECK_ARG(workspace && workspace_bytes >= need, GDN_ERR_WORKSPACE, "%s: workspace of %zu bytes needed, %zu given", who,
                  need, workspace_bytes);
    p.q = q; p.k = k; p.v = v; p.g = nullptr; p.beta = beta; p.h0 = h0; p.dout = dout; p.dht = dht;
    p.dq = dq; p.dk = dk; p.dv = dv; p.dg = nullptr; p.dbeta = dbeta; p.dh0 = dh0; p.dgk = dg;
    p.cu_seqlens = cu_seqlens; p.chunk_table = chunk_table; p.chunk_offsets = chunk_offsets;
    p.T = T; p.H = (int)H; p.HV = (int)HV; p.N = N; p.NT = (T + CH - 1) / CH; p.nb = 1;
    p.scale = scale; p.gb_dtype = p.beta_dtype = gb_dtype; p.flags = flags;
    p.nseg = 1; p.seg_chunks = (int)p.NT; p.warm_cap = 0;
    // the forward's chunk-parallel kernel again, writing into this workspace (u where the scan will put v_new)
    KdaParams kp;
    kp.q = q; kp.k = k; kp.v = v; kp.g = g; kp.beta = beta; kp.pk = nullptr; kp.gs = nullptr;
    kp.A_log = nullptr; kp.gk_bias = nullptr; kp.gk_lower = 0.f; kp.gk_act = 0;
    kp.h0 = nullptr; kp.ht = nullptr; kp.o = nullptr; kp.hs = nullptr;
    kp.cu_seqlens = cu_seqlens; kp.chunk_table = chunk_table; kp.chunk_offsets = chunk_offsets;
    kp.ws = KdaWs{p.ws.Wm, p.ws.Vn, p.ws.QG, p.ws.KG, p.ws.Pm, p.ws.EGL, p.ws.Am, p.ws.Gk};
    kp.T = T; kp.H = (int)H; kp.HV = (int)HV; kp.N = N; kp.NT = p.NT;
    kp.scale = scale; kp.gb_dtype = gb_dtype; kp.flags = flags | (l2 ? GDN_FLAG_QK_L2NORM : 0);
    return qkv_dtype == GDN_DTYPE_BF16 ? launch_bwd_kda<bf16_t>(p, kp, num_chunks, qkv_dtype, s) : launch_bwd_kda<f16_t>(p, kp, num_chunks, qkv_dtype, s);
}

extern "C" int gdn_chunk_kda_bwd(
    const void* q, const void* k, const void* v, const float* g, const void* beta,
    const float* h0, const void* dout, const float* dht,
    void* dq, void* dk, void* dv, float* dg, float* dbeta, float* dh0,
    const void* cu_seqlens, const void* chunk_table, const void* chunk_offsets,
    void* workspace, size_t workspace_bytes,
    int64_t B, int64_t T, int64_t H, int64_t HV, int64_t K, int64_t V,
    int64_t N, int64_t num_chunks,
    float scale, int qkv_dtype, int gb_dtype, uint32_t flags, void* stream) {
    return kda_bwd_entry("gdn_chunk_kda_bwd", false, q, k, v, g, beta, h0, dout, dht, dq, dk, dv, dg, dbeta, dh0, cu_seqlens, chunk_table, chunk_offsets,
                         workspace, workspace_bytes, B, T, H, HV, K, V, N, num_chunks, scale, qkv_dtype, gb_dtype, flags, stream);
}

extern "C" int gdn_chunk_kda_bwd_qk_l2norm(
    const void* q, const void* k, const void* v, const float* g, const void* beta,
    const float* h0, const void* dout, const float* dht,
    void* dq, void* dk, void* dv, float* dg, float* dbeta, float* dh0,
    const void* cu_seqlens, const void* chunk_table, const void* chunk_offsets,
    void* workspace, size_t workspace_bytes,
    int64_t B, int64_t T, int64_t H, int64_t HV, int64_t K, int64_t V,
    int64_t N, int64_t num_chunks,
    float scale, int qkv_dtype, int gb_dtype, uint32_t flags, void* stream) {
    return kda_bwd_entry("gdn_chunk_kda_bwd_qk_l2norm", true, q, k, v, g, beta, h0, dout, dht, dq, dk, dv, dg, dbeta, dh0, cu_seqlens, chunk_table, chunk_offsets,
                         workspace, workspace_bytes, B, T, H, HV, K, V, N, num_chunks, scale, qkv_dtype, gb_dtype, flags, stream);
}

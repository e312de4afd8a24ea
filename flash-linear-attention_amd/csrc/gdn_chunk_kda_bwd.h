// Backward pass of the chunked KDA operator (the gated delta rule with a decay per key feature; K, V <= 128, zero-padded
// to 128 by the host).  Included by gdn_chunk_bwd.hip inside namespace gdn, after its types and its two scans, which serve this
// pass in their KDA form.  Replaces
// chunk_kda_bwd (fla/ops/kda/chunk_bwd.py): the forward's chunk-parallel kernel runs again (A, w, u, qg, kg, P and the
// running sums Gk of the log decays, in log2 units), then
//
//   state, dstate   as for the gated delta rule, with kg / qg in place of k / q and a decay per key feature
//   unit            per (chunk, v-head), from S, dS, v_new, dv_new to dq, dk, dv, dg, dbeta:
//                   dw = -dv_new S^T, dPs = scale tril(do v_new^T), the parts of dq, dk, dGk that come through qg, kg and e^Gk_last;
//                   back through w = A (beta k e^Gk), u = A (beta v), A = (I + diag(beta) M)^-1; and through the two matrices
//                   with a decay per pair and feature,
//                       M_ij = sum_d k_id k_jd e^(Gk_id - Gk_jd) (i > j),   P_ij = scale sum_d q_id k_jd e^(Gk_id - Gk_jd) (i >= j);
//                   dg = reverse cumulative sum of dGk over the chunk's tokens
//
// Pairs and features: with dL the gradient of diag(beta)^-1 L and dPs that of P / scale o mask,
//   row side   dq_i  += sum_j dPs_ij k_j e^(Gk_i - Gk_j),     rk_i = sum_j dL_ij k_j e^(Gk_i - Gk_j)  (dbeta_i += k_i . rk_i,  dk_i += beta_i rk_i)
//   col side   dk_j  += sum_i (dPs_ij q_i + dL_ij beta_i k_i) e^(Gk_i - Gk_j)
//   dGk_i += q_i dq_i + k_i (beta_i rk_i),   dGk_j -= k_j (col side)_j        (elementwise in the feature)
// The exponent splits into a factor of row i and one of row j around a reference row R that lies between them: blocks of 16
// rows, R = the row in front of i's block, e^(Gk_i - R) <= 1.  For j in an earlier block t, whose last row is E_t, e^(R - Gk_j) is
// e^(E_t - Gk_j) <= 1 times the decays across the blocks between, a factor per feature that goes onto the sums; inside the diagonal block
// it is >= 1, which the operand type holds as long as the block's total decay stays above a bound - otherwise every pair of the
// diagonal block gets its own exponentials, as in the forward kernel and in the reference's sub-chunks of 16,
// fla/ops/kda/chunk_intra.py.  All of it runs on the matrix cores: per block of rows k e^(E - Gk) and k e^(R - Gk) for the row side, and
// for the column side one 32-deep step whose contraction index runs over the block's 16 rows twice (dPs^T against q e^(Gk - R),
// dL^T against beta k e^(Gk - R)).

// x + the y of the first lane of its row of sixteen (row_newbcast)
__device__ __forceinline__ float add_first_c16(float x, float y) {
    return x + __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, y), 0x150, 0xF, 0xF, true));
}
// x of this lane and of the lanes behind it in its row of sixteen, added up
template <int N> __device__ __forceinline__ float add_behind(float x) {
    return x + __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x100 + N, 0xF, 0xF, true));     // row_shl: N lanes on, zero past the row
}
__device__ __forceinline__ float suffix_sum_c16(float x) { return add_behind<8>(add_behind<4>(add_behind<2>(add_behind<1>(x)))); }

// Eight waves, one workgroup per CU walking over the units; wave w owns the key features 16w .. of all 64 tokens, so that dq, dk and
// dGk stay in registers from the first part to the last, and so do the operands of the pair matrices: each wave scales the 16 features of
// k and q that it needs itself, straight from the tiles into matrix-core registers, and that phase needs no barrier.
// L2: q and k are the rows before their l2 normalisation and dq, dk the gradients of those.
// As two kernels of four waves this moved 530 KB per unit (dw, dPs, the first parts of dq, dk and dGk through memory, k, q and Gk twice) where
// it now moves 280 KB, and the l2 normalisation was four passes over q and k around it.  8192 tokens, 96 heads: 1834 us + 320 us of passes ->
// 1006 us, the step 4250 -> 3093 us.  Bound by the vector instructions of two waves per SIMD: with k e^(R - Gk) anew for every block of rows and
// e^(R - Gk) for every tile of the column side (ten exponentials an element) 3100 of them a unit and wave; with three for operands and three for results,
// block factors on the sums, e^Gk kept between the two phases that use it and the unit's place carried over from the request for its tiles 2600:
// 1006 -> 885 us (3.63 GB, 4.1 TB/s), the step 2815 -> 2693.  The next unit's tiles are requested in the order of their use, the state's
// fragments last.  (`pin`: the compiler moves sums down to their next use, here two phases on, and keeps their factors: 100 registers.)
constexpr size_t BWD_UNIT_KDA_SMEM = (6 * 64 * P128 + 2 * 64 * P64) * 2 + (64 * PG + 3 * 64 + 8 * 64 + 4) * 4;

template <typename T, bool L2>
__global__ __launch_bounds__(512, 2) void gdn_bwd_unit_kda_kernel(BwdParams p, int64_t units) {
    typedef typename Mma<T>::V8 V8;
    typedef typename Mma<T>::V4 V4;
    constexpr int NW = 8, NTH = 64 * NW, NTRI = 2;
    extern __shared__ __align__(16) char smem[];
    T* sDO = (T*)smem; T* sVn = sDO + 64 * P128; T* sDvn = sVn + 64 * P128; T* sV = sDvn + 64 * P128; T* sK = sV + 64 * P128; T* sQ = sK + 64 * P128;
    T* sA = sQ + 64 * P128; T* sPs = sA + 64 * P64;
    float* sG = (float*)(sPs + 64 * P64);                        // Gk / ln 2: every decay is one exp2
    float* sBeta = sG + 64 * PG; float* sRq = sBeta + 64; float* sRk = sRq + 64; float* sDb = sRk + 64;      // (sDb: a row per wave)
    float* sSpan = sDb + NW * 64;
    T* sDW = sDO; T* sDL = sVn; T* sY = sDvn; T* sKp = sV;       // dw, dA and then dL, Y, k e^Gk take the places of what is done with
    T* sDq = sDO; T* sDk = sV; float* sDot = (float*)sA;         // ... and so do dq, dk on their way out, and the rows' products with them

    TileRegs<BD, NTH> rDO, rVn, rDvn, rV, rK, rQ;
    TileRegs<CH, NTH> rA;
    V8 sf[4], df[4];
    f32x4 rG[4];
    uint32_t rBeta = 0;                                          // (raw bits: converted when the unit's turn comes)
    auto fetch_out = [&](const UnitAt& at, int64_t u, int tid) {
        fetch_tile<BD, NTH>(rDO, (const T*)p.dout + (at.c.tok0 * p.HV + at.hv) * BD, (int64_t)p.HV * BD, at.c.valid, tid);
        fetch_tile<BD, NTH>(rVn, (const T*)p.ws.Vn + u * 64 * BD, BD, 64, tid);
    };
    auto fetch_in = [&](const UnitAt& at, int64_t u, int tid) {
        fetch_tile<BD, NTH>(rDvn, (const T*)p.ws.dVn + u * 64 * BD, BD, 64, tid);
        fetch_tile<BD, NTH>(rV, (const T*)p.v + (at.c.tok0 * p.HV + at.hv) * BD, (int64_t)p.HV * BD, at.c.valid, tid);
    };
    auto fetch_state = [&](const UnitAt& at, int64_t u, int tid) {
        const int64_t off = u * BD * BD + state_frag<BD>(tid >> 6, 0, tid & 63);
#pragma unroll
        for (int s = 0; s < 4; ++s) { sf[s] = *(const V8*)((const T*)p.ws.Hs + off + 512 * s); df[s] = *(const V8*)((const T*)p.ws.dHs + off + 512 * s); }
        fetch_tile<CH, NTH>(rA, (const T*)p.ws.Am + u * 64 * 64, 64, 64, tid);
        if (tid < 64) rBeta = tid < at.c.valid ? load_scalar_bits(p.beta, (at.c.tok0 + tid) * p.HV + at.hv, p.gb_dtype) : 0;
    };
    auto fetch_qk = [&](const UnitAt& at, int64_t u, int tid) {
        fetch_tile<BD, NTH>(rK, (const T*)p.k + (at.c.tok0 * p.H + at.hq) * BD, (int64_t)p.H * BD, at.c.valid, tid);
        fetch_tile<BD, NTH>(rQ, (const T*)p.q + (at.c.tok0 * p.H + at.hq) * BD, (int64_t)p.H * BD, at.c.valid, tid);
#pragma unroll
        for (int i = 0; i < 4; ++i) rG[i] = *(const f32x4*)(p.ws.Gk + u * 64 * BD + (tid + NTH * i) * 4);
    };
    // the rows of a tile on their way into LDS, divided by their lengths (16 lanes hold a row); the factors to `r`
    auto put_unit_rows = [&](T* s, TileRegs<BD, NTH>& x, float* r, int tid) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            V8 v = __builtin_bit_cast(V8, x.x[i]);
            float ss = 0.f;
#pragma unroll
            for (int e = 0; e < 8; ++e) ss += (float)v[e] * (float)v[e];
            const float f = rsqrtf(sum_over_c16(ss) + 1e-6f);
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = (T)((float)v[e] * f);
            x.x[i] = __builtin_bit_cast(u32x4, v);
            if ((tid & 15) == 0) r[(tid >> 4) + 32 * i] = f;
        }
        put_tile<BD, NTH>(s, P128, x, tid);
    };
    UnitAt nx = unit_at(p, blockIdx.x);
    {
        const int tid = threadIdx.x;
        const UnitAt& at = nx;
        fetch_qk(at, blockIdx.x, tid); fetch_out(at, blockIdx.x, tid); fetch_in(at, blockIdx.x, tid); fetch_state(at, blockIdx.x, tid);
    }
    for (int64_t u = blockIdx.x; u < units; u += gridDim.x) {
        // (everything derived from the lane number is derived again per unit from a copy the compiler cannot see through:
        // hoisted out of this loop, the addresses of its unrolled body would fill the register file and spill)
        int tid_opaque = threadIdx.x;
        asm volatile("" : "+v"(tid_opaque));
        const int tid = tid_opaque, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), c16 = lane & 15, g = lane >> 4;
        const UnitAt at = nx;
        const int hv = at.hv;
        const ChunkAt c = at.c;
        // (what comes next is requested in any case, the last time for nothing: behind a condition the registers of the last request
        // stay alive through the whole unit)
        const int64_t un = u + gridDim.x < units ? u + gridDim.x : u;
        nx = unit_at(p, un);
        const int n16 = 16 * w, f4 = n16 + 4 * g;                // this wave's features, this lane's four of them in a result
        put_tile<BD, NTH>(sDO, P128, rDO, tid);
        put_tile<BD, NTH>(sVn, P128, rVn, tid);
        put_tile<BD, NTH>(sDvn, P128, rDvn, tid);
        put_tile<BD, NTH>(sV, P128, rV, tid);
        put_tile<CH, NTH>(sA, P64, rA, tid);
        if constexpr (L2) { put_unit_rows(sK, rK, sRk, tid); put_unit_rows(sQ, rQ, sRq, tid); }
        else { put_tile<BD, NTH>(sK, P128, rK, tid); put_tile<BD, NTH>(sQ, P128, rQ, tid); }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int idx = tid + NTH * i;
            *(f32x4*)(sG + (idx >> 5) * PG + (idx & 31) * 4) = rG[i];
        }
        if (tid < 64) sBeta[tid] = scalar_of_bits(rBeta, p.gb_dtype);
        lds_barrier();
        fetch_out(nx, un, tid);

        // dPs = scale tril(do v_new^T), tile by tile
#pragma unroll
        for (int n = 0; n < NTRI; ++n) {
            __builtin_amdgcn_sched_barrier(0);
            const int idx = w + NW * n;
            if (idx < 10) {
                const int ti = tri_row(idx), tj = tri_col(idx);
                f32x4 acc = ZERO4;
#pragma unroll
                for (int s = 0; s < 4; ++s) acc = Mma<T>::run(frag_rows(sDO, P128, 16 * ti, 32 * s, lane), frag_rows(sVn, P128, 16 * tj, 32 * s, lane), acc);
                const int j = 16 * tj + c16;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int i = 16 * ti + 4 * g + r;
                    sPs[i * P64 + j] = (T)(i >= j ? p.scale * acc[r] : 0.f);
                }
            }
        }
        // dq, dk, dGk of the output and the state update, dw (kept until do is done with)
        f32x4 dq[4], dk[4], dG[4], eG[4];                       // (eG: e^Gk)
        float dbx[4] = {0.f, 0.f, 0.f, 0.f};                     // this lane's share of dbeta of token 16t + c16
        V4 dw[4];
        {
            f32x4 G1[4], dKS[4], dWt[4], sd = ZERO4;             // (sd: <S, dS> of this wave's features on its diagonal)
#pragma unroll
            for (int t = 0; t < 4; ++t) G1[t] = dKS[t] = dWt[t] = ZERO4;
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                __builtin_amdgcn_sched_barrier(0);
                sd = Mma<T>::run(sf[s], df[s], sd);
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    G1[t] = Mma<T>::run(sf[s], frag_rows(sDO, P128, 16 * t, 32 * s, lane), G1[t]);
                    dWt[t] = Mma<T>::run(sf[s], frag_rows(sDvn, P128, 16 * t, 32 * s, lane), dWt[t]);
                    dKS[t] = Mma<T>::run(df[s], frag_rows(sVn, P128, 16 * t, 32 * s, lane), dKS[t]);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            const f32x4 Gl = *(const f32x4*)(sG + 63 * PG + f4);
            f32x4 last = ZERO4;
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                __builtin_amdgcn_sched_barrier(0);
                dw[t] = pack4<T>(-dWt[t]);
                const int x = 16 * t + c16;
                const f32x4 Gx = *(const f32x4*)(sG + x * PG + f4);
                const V4 q4 = *(const V4*)(sQ + x * P128 + f4), k4 = *(const V4*)(sK + x * P128 + f4);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    eG[t][r] = fast_exp2(Gx[r]);
                    dq[t][r] = G1[t][r] * (p.scale * eG[t][r]);
                    dk[t][r] = dKS[t][r] * fast_exp2(Gl[r] - Gx[r]);
                    const float kdk = (float)k4[r] * dk[t][r];
                    last[r] += kdk;
                    dG[t][r] = (float)q4[r] * dq[t][r] - kdk;
                }
                pin(dq[t]); pin(dk[t]); pin(dG[t]); pin(eG[t]); // (sunk to their uses the sums would keep their factors alive)
            }
            // the chunk's last row also takes what goes through e^Gk_last
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float x = sum_over_c16(last[r] + (c16 == 4 * g + r ? fast_exp2(Gl[r]) * sd[r] : 0.f));
                dG[3][r] += c16 == 15 ? x : 0.f;
            }
            pin(dG[3]);
        }

        // dX's first term dv_new v^T (the same tiles as above), and dv = beta (A^T dv_new)
        f32x4 dX[NTRI];
#pragma unroll
        for (int n = 0; n < NTRI; ++n) {
            __builtin_amdgcn_sched_barrier(0);
            const int idx = w + NW * n;
            dX[n] = ZERO4;
            if (idx < 10) {
#pragma unroll
                for (int s = 0; s < 4; ++s)
                    dX[n] = Mma<T>::run(frag_rows(sDvn, P128, 16 * tri_row(idx), 32 * s, lane), frag_rows(sV, P128, 16 * tri_col(idx), 32 * s, lane), dX[n]);
            }
        }
        {
            V8 fdv[2];
#pragma unroll
            for (int s = 0; s < 2; ++s) fdv[s] = frag_cols(sDvn, P128, 32 * s, n16, lane);
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                __builtin_amdgcn_sched_barrier(0);
                f32x4 av = ZERO4;
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    if (32 * s + 31 < 16 * t) continue;         // A[i][j] = 0 for i < j
                    av = Mma<T>::run(fdv[s], frag_cols(sA, P64, 32 * s, 16 * t, lane), av);
                }
                const int j = 16 * t + c16;
                const V4 v4 = *(const V4*)(sV + j * P128 + f4);
#pragma unroll
                for (int r = 0; r < 4; ++r) dbx[t] += av[r] * (float)v4[r];
                pin(dbx[t]);
                if (j < c.valid) *(V4*)((T*)p.dv + ((c.tok0 + j) * p.HV + hv) * BD + f4) = pack4<T>(av * sBeta[j]);
            }
        }
        lds_barrier();                                          // (do, v_new, dv_new and v are done with)
#pragma unroll
        for (int t = 0; t < 4; ++t) *(V4*)(sDW + (16 * t + c16) * P128 + f4) = dw[t];
        // k e^Gk, the factor of w
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int row = (tid >> 4) + 32 * i, pc = tid & 15;
            V8 kx = *(const V8*)(sK + row * P128 + pc * 8);
            const float* gi = sG + row * PG + pc * 8;
#pragma unroll
            for (int e = 0; e < 8; ++e) kx[e] = (T)((float)kx[e] * fast_exp2(gi[e]));
            *(V8*)(sKp + row * P128 + pc * 8) = kx;
        }
        if (w < 4) {
            // the decay across the block of rows 16w .., the strongest over the features: decides how its diagonal block is treated
            float span = 0.f;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const float* col = sG + lane + 64 * h;
                span = fminf(span, col[(16 * w + 15) * PG] - (w > 0 ? col[(16 * w - 1) * PG] : 0.f));
            }
            span = min_over_wave(span);
            if (lane == 0) sSpan[w] = span;
        }
        {                                                       // (the zero tiles of dA and dL, in v_new's place)
            const int t = tid >> 8, r = (tid >> 4) & 15, cc = tid & 15;
            sDL[(32 * t + r) * P64 + 32 * t + 16 + cc] = (T)0.f;
        }
        lds_barrier();
        fetch_in(nx, un, tid);
        // dX's second term dw (k e^Gk)^T, dA = stril(dX diag(beta))
#pragma unroll
        for (int n = 0; n < NTRI; ++n) {
            __builtin_amdgcn_sched_barrier(0);
            const int idx = w + NW * n;
            if (idx < 10) {
                const int ti = tri_row(idx), tj = tri_col(idx);
#pragma unroll
                for (int s = 0; s < 4; ++s)
                    dX[n] = Mma<T>::run(frag_rows(sDW, P128, 16 * ti, 32 * s, lane), frag_rows(sKp, P128, 16 * tj, 32 * s, lane), dX[n]);
                const int j = 16 * tj + c16;
                const float bj = sBeta[j];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int i = 16 * ti + 4 * g + r;
                    sDL[i * P64 + j] = (T)(i > j ? dX[n][r] * bj : 0.f);
                }
            }
        }
        // d(k e^Gk) = beta (A^T dw): into dk, dbeta, dGk
        {
            V8 fdw[2];
#pragma unroll
            for (int s = 0; s < 2; ++s) fdw[s] = frag_cols(sDW, P128, 32 * s, n16, lane);
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                __builtin_amdgcn_sched_barrier(0);
                f32x4 ak = ZERO4;
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    if (32 * s + 31 < 16 * t) continue;
                    ak = Mma<T>::run(fdw[s], frag_cols(sA, P64, 32 * s, 16 * t, lane), ak);
                }
                const int j = 16 * t + c16;
                const float bj = sBeta[j];
                const V4 kp4 = *(const V4*)(sKp + j * P128 + f4);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float x = ak[r] * (float)kp4[r];
                    dbx[t] += x;
                    dG[t][r] += bj * x;
                    dk[t][r] += ak[r] * (bj * eG[t][r]);
                }
                pin(dbx[t]); pin(dk[t]); pin(dG[t]);
            }
        }
        lds_barrier();
        // Y = dA A^T
#pragma unroll
        for (int n = 0; n < 2; ++n) {
            __builtin_amdgcn_sched_barrier(0);
            const int ti = (w + NW * n) >> 2, tl = (w + NW * n) & 3;
            f32x4 acc = ZERO4;
#pragma unroll
            for (int s = 0; s < 2; ++s)
                if (32 * s <= 16 * ti + 15) acc = Mma<T>::run(frag_rows(sDL, P64, 16 * ti, 32 * s, lane), frag_rows(sA, P64, 16 * tl, 32 * s, lane), acc);
#pragma unroll
            for (int r = 0; r < 4; ++r) sY[(16 * ti + 4 * g + r) * P64 + 16 * tl + c16] = (T)acc[r];
        }
        lds_barrier();
        // dL = -stril(A^T Y): the gradient of stril(M) once its rows are scaled by beta
#pragma unroll
        for (int n = 0; n < NTRI; ++n) {
            __builtin_amdgcn_sched_barrier(0);
            const int idx = w + NW * n;
            if (idx < 10) {
                const int ti = tri_row(idx), tl = tri_col(idx);
                f32x4 acc = ZERO4;
#pragma unroll
                for (int s = 0; s < 2; ++s)
                    if (32 * s + 31 >= 16 * ti) acc = Mma<T>::run(frag_cols(sA, P64, 32 * s, 16 * ti, lane), frag_cols(sY, P64, 32 * s, 16 * tl, lane), acc);
                const int l = 16 * tl + c16;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int i = 16 * ti + 4 * g + r;
                    sDL[i * P64 + l] = (T)(i > l ? -acc[r] : 0.f);
                }
            }
        }
        lds_barrier();

        // The two matrices with a decay per pair and feature, a block of 16 rows at a time from the last; a wave on its own from here on.
        // E_t: the last row of block t, the reference row R of block t + 1.  Every element has three exponentials for its operands and three for
        // results: f = e^(Gk - R) as a row, e^(E - Gk) as a column (or 1 / f in its own block); between blocks lies a factor per feature, D_t = e^(E_t - E_(t-1)),
        // on the sums so far.  Operand layout: feature n16 + c16, tokens 4g + e of a block, two blocks or two matrices to a product.
        V4 kn[3];                                                // k e^(E - Gk) of blocks 0 .. 2
        f32x4 D[3], cs[3];                                       // (cs: what the later blocks' rows leave to the columns of block t, before e^(E_t - Gk))
        {
            int lane_opaque = tid & 63;
            asm volatile("" : "+v"(lane_opaque));
            const int lane = lane_opaque, c16 = lane & 15, g = lane >> 4, f4 = n16 + 4 * g;
#pragma unroll
            for (int t = 0; t < 3; ++t) {
                __builtin_amdgcn_sched_barrier(0);
                const float* gt = sG + 16 * t * PG + n16 + c16;
                const float E = gt[15 * PG];
                kn[t] = tile_cols(sK, P128, 16 * t, n16, lane);
#pragma unroll
                for (int e = 0; e < 4; ++e) kn[t][e] = (T)((float)kn[t][e] * fast_exp2(E - gt[(4 * g + e) * PG]));
                if (t > 0) {
                    const f32x4 E4 = *(const f32x4*)(sG + (16 * t + 15) * PG + f4), R4 = *(const f32x4*)(sG + (16 * t - 1) * PG + f4);
#pragma unroll
                    for (int r = 0; r < 4; ++r) D[t][r] = fast_exp2(E4[r] - R4[r]);
                }
                cs[t] = ZERO4;
            }
        }
#pragma unroll
        for (int a = 3; a >= 0; --a) {
            __builtin_amdgcn_sched_barrier(0);
            // (the lane number anew: what the four blocks read alike would stay in registers from the first to the last)
            int lane_opaque = tid & 63;
            asm volatile("" : "+v"(lane_opaque));
            const int lane = lane_opaque, c16 = lane & 15, g = lane >> 4, f4 = n16 + 4 * g;
            const bool ok = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, sSpan[a]))) >= SpanOk<T>::value;
            const int x = 16 * a + c16;
            const float bx = sBeta[x];
            V4 qf = tile_cols(sQ, P128, 16 * a, n16, lane), kf = tile_cols(sK, P128, 16 * a, n16, lane), kd;      // q f, beta k f, k / f
            {
                const float* ga = sG + (16 * a + 4 * g) * PG + n16 + c16;
                const float R = a > 0 ? sG[(16 * a - 1) * PG + n16 + c16] : 0.f;
                const f32x4 b4 = *(const f32x4*)(sBeta + 16 * a + 4 * g);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float d = ga[e * PG] - R, f = fast_exp2(d), k = (float)kf[e];
                    kd[e] = ok ? (T)(k * fast_exp2(-d)) : (T)0.f;
                    qf[e] = (T)((float)qf[e] * f);
                    kf[e] = (T)(k * (b4[e] * f));
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            // row side: against k of the earlier blocks and of this one
            f32x4 rq = ZERO4, rk = ZERO4;                       // (rk: before the row's beta)
            const T* prow = sPs + x * P64 + 4 * g; const T* lrow = sDL + x * P64 + 4 * g;
#pragma unroll
            for (int t = 0; t < a - 1; ++t) {
                rq = Mma<T>::run16(kn[t], *(const V4*)(prow + 16 * t), rq);
                rk = Mma<T>::run16(kn[t], *(const V4*)(lrow + 16 * t), rk);
                rq *= D[t + 1]; rk *= D[t + 1];
            }
            if (a > 0) {
                const V8 kk = join<V8>(kn[a > 0 ? a - 1 : 0], kd);
                rq = Mma<T>::run(kk, join<V8>(*(const V4*)(prow + 16 * a - 16), *(const V4*)(prow + 16 * a)), rq);
                rk = Mma<T>::run(kk, join<V8>(*(const V4*)(lrow + 16 * a - 16), *(const V4*)(lrow + 16 * a)), rk);
            } else {
                rq = Mma<T>::run16(kd, *(const V4*)prow, rq);
                rk = Mma<T>::run16(kd, *(const V4*)lrow, rk);
            }
            __builtin_amdgcn_sched_barrier(0);
            const f32x4 Gx = *(const f32x4*)(sG + x * PG + f4), R4 = a > 0 ? *(const f32x4*)(sG + (16 * a - 1) * PG + f4) : ZERO4;
            const V4 qx = *(const V4*)(sQ + x * P128 + f4), kx = *(const V4*)(sK + x * P128 + f4);
            // dGk takes every product dPs_ij (q_i f_i) (k_j e^(R - Gk_j)) twice, once with each sign (row i, column j), and
            // the sums down the columns leave the difference: both sides form it from the same rounded operands
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float f = fast_exp2(Gx[r] - R4[r]);
                dG[a][r] += (float)(T)((float)qx[r] * f) * rq[r] + (float)(T)((float)kx[r] * (bx * f)) * rk[r];
                rq[r] *= f; rk[r] *= f;
            }
            if (!ok) {
                // the diagonal block pair by pair: row side for this lane's token x
#pragma unroll 1
                for (int jl = 0; jl < 16; ++jl) {
                    const int j = 16 * a + jl;
                    if (j > x) continue;
                    const float av = (float)sPs[x * P64 + j], bv = (float)sDL[x * P64 + j];
                    const V4 k4 = *(const V4*)(sK + j * P128 + f4);
                    const f32x4 Gj = *(const f32x4*)(sG + j * PG + f4);
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const float kd = (float)k4[r] * fast_exp2(Gx[r] - Gj[r]);
                        rq[r] += av * kd; rk[r] += bv * kd;
                        dG[a][r] += ((float)qx[r] * av + (float)kx[r] * (bx * bv)) * kd;
                    }
                }
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                dbx[a] += (float)kx[r] * rk[r];
                dk[a][r] += bx * rk[r];
                dq[a][r] += rq[r];
            }
            __builtin_amdgcn_sched_barrier(0);
            // column side: the block's rows (q f against dPs, beta k f against dL) for the columns of the earlier blocks and of this one
            const V8 op = join<V8>(qf, kf);
            auto columns = [&](int t, const f32x4& acc) {
                return Mma<T>::run(op, join<V8>(tile_cols(sPs, P64, 16 * a, 16 * t, lane), tile_cols(sDL, P64, 16 * a, 16 * t, lane)), acc);
            };
            auto into = [&](const f32x4& sum, int r, float e) {
                dk[a][r] += sum[r] * e;
                dG[a][r] -= (float)(T)((float)kx[r] * e) * sum[r];
            };
#pragma unroll
            for (int t = 0; t < a; ++t) {
                __builtin_amdgcn_sched_barrier(0);
                if (a < 3) cs[t] *= D[a];
                cs[t] = columns(t, cs[t]);
            }
            __builtin_amdgcn_sched_barrier(0);
            if (a < 3) {
                const f32x4 E4 = *(const f32x4*)(sG + (16 * a + 15) * PG + f4);
#pragma unroll
                for (int r = 0; r < 4; ++r) into(cs[a < 3 ? a : 0], r, fast_exp2(E4[r] - Gx[r]));
            }
            if (ok) {
                const f32x4 own = columns(a, ZERO4);
#pragma unroll
                for (int r = 0; r < 4; ++r) into(own, r, fast_exp2(R4[r] - Gx[r]));
            } else {
                // ... and the column side for this lane's token x
#pragma unroll 1
                for (int il = 0; il < 16; ++il) {
                    const int i = 16 * a + il;
                    if (i < x) continue;
                    const float av = (float)sPs[i * P64 + x], bv = (float)sDL[i * P64 + x] * sBeta[i];
                    const V4 q4 = *(const V4*)(sQ + i * P128 + f4), k4 = *(const V4*)(sK + i * P128 + f4);
                    const f32x4 Gi = *(const f32x4*)(sG + i * PG + f4);
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const float cv = (av * (float)q4[r] + bv * (float)k4[r]) * fast_exp2(Gi[r] - Gx[r]);
                        dk[a][r] += cv;
                        dG[a][r] -= (float)kx[r] * cv;
                    }
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        fetch_qk(nx, un, tid);
        fetch_state(nx, un, tid);
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const float dbt = sum_over_g(dbx[t]);
            if (g == 0) sDb[64 * w + 16 * t + c16] = dbt;
        }
        // dg = the reverse cumulative sum of dGk, in this wave's columns of the gates
        {
            f32x4 behind = ZERO4;
#pragma unroll
            for (int t = 3; t >= 0; --t) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float x = dG[t][r];
                    const float sum = suffix_sum_c16(x);
                    dG[t][r] = sum + behind[r];
                    behind[r] = add_first_c16(behind[r], sum);
                }
                *(f32x4*)(sG + (16 * t + c16) * PG + f4) = dG[t];
            }
        }
        if constexpr (L2) {
            // back through the l2 normalisation: dx = (dy - y <y, dy>) / |x|
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const int x = 16 * t + c16;
                const V4 q4 = *(const V4*)(sQ + x * P128 + f4), k4 = *(const V4*)(sK + x * P128 + f4);
                float qd = 0.f, kd = 0.f;
#pragma unroll
                for (int r = 0; r < 4; ++r) { qd += (float)q4[r] * dq[t][r]; kd += (float)k4[r] * dk[t][r]; }
                qd = sum_over_g(qd); kd = sum_over_g(kd);
                if (g == 0) { sDot[64 * w + x] = qd; sDot[64 * (NW + w) + x] = kd; }
            }
            lds_barrier();
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const int x = 16 * t + c16;
                const V4 q4 = *(const V4*)(sQ + x * P128 + f4), k4 = *(const V4*)(sK + x * P128 + f4);
                float qd = 0.f, kd = 0.f;
#pragma unroll
                for (int i = 0; i < NW; ++i) { qd += sDot[64 * i + x]; kd += sDot[64 * (NW + i) + x]; }
                const float rq = sRq[x], rk = sRk[x];
#pragma unroll
                for (int r = 0; r < 4; ++r) { dq[t][r] = (dq[t][r] - (float)q4[r] * qd) * rq; dk[t][r] = (dk[t][r] - (float)k4[r] * kd) * rk; }
            }
        }
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            *(V4*)(sDq + (16 * t + c16) * P128 + f4) = pack4<T>(dq[t]);
            *(V4*)(sDk + (16 * t + c16) * P128 + f4) = pack4<T>(dk[t]);
        }
        lds_barrier();
        copy_rows_out<64, BD, NTH>((T*)p.dq + (c.tok0 * p.HV + hv) * BD, (int64_t)p.HV * BD, sDq, P128, tid, c.valid);
        copy_rows_out<64, BD, NTH>((T*)p.dk + (c.tok0 * p.HV + hv) * BD, (int64_t)p.HV * BD, sDk, P128, tid, c.valid);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int idx = tid + NTH * i, row = idx >> 5, pc = idx & 31;
            if (row < c.valid) *(f32x4*)(p.dgk + ((c.tok0 + row) * p.HV + hv) * BD + pc * 4) = *(const f32x4*)(sG + row * PG + pc * 4);
        }
        if (tid < c.valid) {
            float b = 0.f;
#pragma unroll
            for (int i = 0; i < NW; ++i) b += sDb[64 * i + tid];
            p.dbeta[(c.tok0 + tid) * p.HV + hv] = b;
        }
        lds_barrier();
    }
}

template <typename T>
static int launch_bwd_kda(const BwdParams& p, const KdaParams& kp, int64_t num_chunks, int qkv_dtype, hipStream_t stream) {
    if (int rc = launch_kda_prepare(kp, num_chunks, qkv_dtype, stream)) return rc;
    const unsigned units = (unsigned)(num_chunks * p.HV), grid = units < 256u ? units : 256u;
    const bool l2 = kp.flags & GDN_FLAG_QK_L2NORM;
    const BwdLaunch ks[2] = {
        scans_128<T, FORM_KDA>(p, num_chunks),
        {l2 ? (const void*)gdn_bwd_unit_kda_kernel<T, true> : (const void*)gdn_bwd_unit_kda_kernel<T, false>, BWD_UNIT_KDA_SMEM, "gdn_bwd_unit_kda_kernel", grid, 512, units},
    };
    return launch_all(p, ks, 2, stream);
}

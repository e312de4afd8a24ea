// The chunk-parallel end of the backward pass at 256 key features (included by gdn_chunk_bwd.hip, inside the namespace, after gdn_chunk_bwd_unit.h, which has the
// mathematics).  Eight waves of 256 registers, one workgroup per CU: wave w owns the key features 32w .. of all 64 tokens, the tiles of the 64 x 64 lower triangles are
// dealt out one by one; k and q of all features and one copy of every other tile fill the LDS, what comes next waits in registers.
// 8 x 2048 tokens, 32 heads of 256 x 256: 1205 us (4.8 GB at 4.0 TB/s).  The sixteen waves of 128 registers that serve 64 and 128 features took 1440 us here: dq, dk and
// both states' rows are 64 of a wave's registers before its first product, 30 more spill, and every spilled register that is read again waits for all that is under
// way.  What it took at eight: the first feature tile's fragments requested in front of the dP phase and the products with the state one after the other (1642 us
// with the three of them side by side, whose accumulators spilled); no sum's terms kept in registers (1570 us with those of dglast kept to the end of the products, 1250 with those of dq and dk kept to the end of the head); the next
// head's tiles requested in three places, the last of them late (all at once behind the products 1400 us); the states as operand fragments (state_frag; 1330 us as rows).
// The registers that are left over do not pay as a place for the next head's first state fragments: the step 3114 -> 3121 us.
constexpr int UNIT256_NW = 8;
constexpr size_t BWD_UNIT256_SMEM = (4 * 64 * P128 + 2 * 64 * (256 + 8) + 2 * 64 * P64) * 2 + (6 * 64 + 2 * UNIT256_NW * 64) * 4;

template <typename T, bool L2>
__global__ __launch_bounds__(64 * UNIT256_NW, 2) void gdn_bwd_unit256_kernel(BwdParams p, int64_t items) {
    typedef typename Mma<T>::V8 V8;
    typedef typename Mma<T>::V4 V4;
    constexpr int KD = 256, VD = BD, NW = UNIT256_NW, NTH = 64 * NW, PK = KD + 8, PV = VD + 8, NA = KD / 16 / NW, NV = VD / 16 / NW, SV = VD / 32, SK = KD / 32, NTRI = (10 + NW - 1) / NW;
    static_assert(NA >= 1 && NV >= 1 && 64 * PK <= 2 * 64 * PV && 64 * P64 <= 64 * PV, "dw fits the tiles of do and v_new, Y that of dv_new");
    extern __shared__ __align__(16) char smem[];
    T* sDO = (T*)smem; T* sVn = sDO + 64 * PV; T* sDvn = sVn + 64 * PV; T* sV = sDvn + 64 * PV; T* sK = sV + 64 * PV; T* sQ = sK + 64 * PK;
    T* sA = sQ + 64 * PK; T* sM1 = sA + 64 * P64;
    T* sDW = sDO; T* sM2 = sDvn;
    float* sGam = (float*)(sM1 + 64 * P64); float* sBeta = sGam + 64; float* sRq = sBeta + 64; float* sRk = sRq + 64;
    float* sEg = sRk + 64; float* sEl = sEg + 64;                // e^gam and e^(gam_last - gam)
    float* sDg = sEl + 64; float* sDb = sDg + NW * 64;           // a row per wave, added up in a fixed order: the same bits every run

    const int parts = p.parts, heads = p.HV / p.H / parts;       // value heads an item takes
    // item = (chunk * H + q/k head) * parts + part
    struct Item { int hq, hv0, part; int64_t ch; ChunkAt c; };
    auto item_at = [&](int64_t it) {
        const uint32_t grp = (uint32_t)it / (uint32_t)parts, part = (uint32_t)it - grp * parts, ch = grp / (uint32_t)p.H, hq = grp - ch * p.H;
        return Item{(int)hq, (int)(hq * (p.HV / p.H) + part * heads), (int)part, (int64_t)ch, chunk_at(p, ch)};
    };
    TileRegs<VD, NTH> rDO, rVn, rDvn, rV;
    TileRegs<CH, NTH> rA;
    TileRegs<KD, NTH> rK, rQ;
    V8 sf[SV], df[SV];
    float rGam = 0.f, rBeta = 0.f, rRq = 0.f, rRk = 0.f;
    const int HVg = p.HV / p.nb;
    const bool parts_out = p.dq_part != nullptr;
    auto fetch_state = [&](const Item& at, int hv, int a, int w, int lane, bool S = true, bool dS = true) {     // feature tile a of this wave
        const int64_t u = at.ch * p.HV + hv;
        const int64_t off = u * KD * VD + state_frag<VD>(NA * w + a, 0, lane);
#pragma unroll
        for (int s = 0; s < SV; ++s) {
            if (S) sf[s] = *(const V8*)((const T*)p.ws.Hs + off + 512 * s);
            if (dS) df[s] = *(const V8*)((const T*)p.ws.dHs + off + 512 * s);
        }
    };
    auto fetch_out = [&](const Item& at, int hv, int tid) {
        const int64_t u = at.ch * p.HV + hv;
        fetch_tile<VD, NTH>(rDO, (const T*)p.dout + (at.c.tok0 * p.HV + hv) * VD, (int64_t)p.HV * VD, at.c.valid, tid);
        fetch_tile<VD, NTH>(rVn, (const T*)p.ws.Vn + u * 64 * VD, VD, 64, tid);
    };
    auto fetch_in = [&](const Item& at, int hv, int tid) {
        const int64_t u = at.ch * p.HV + hv;
        fetch_tile<VD, NTH>(rDvn, (const T*)p.ws.dVn + u * 64 * VD, VD, 64, tid);
        fetch_tile<VD, NTH>(rV, (const T*)p.v + (at.c.tok0 * p.HV + hv) * VD, (int64_t)p.HV * VD, at.c.valid, tid);
    };
    auto fetch_rest = [&](const Item& at, int hv, int tid) {
        const int64_t ug = at.ch * HVg + hv / p.nb;
        fetch_tile<CH, NTH>(rA, (const T*)p.ws.Am + ug * 64 * 64, 64, 64, tid);
        if (tid < 64) { rGam = p.ws.Gam[ug * 64 + tid]; rBeta = p.ws.Bet[ug * 64 + tid]; }
    };
    auto fetch_qk = [&](const Item& at, int tid) {
        fetch_tile<KD, NTH>(rK, (const T*)p.k + (at.c.tok0 * p.H + at.hq) * KD, (int64_t)p.H * KD, at.c.valid, tid);
        fetch_tile<KD, NTH>(rQ, (const T*)p.q + (at.c.tok0 * p.H + at.hq) * KD, (int64_t)p.H * KD, at.c.valid, tid);
        if constexpr (L2) {
            if (tid < 64) {
                rRq = tid < at.c.valid ? p.q_rstd[(at.c.tok0 + tid) * p.H + at.hq] : 0.f;
                rRk = tid < at.c.valid ? p.k_rstd[(at.c.tok0 + tid) * p.H + at.hq] : 0.f;
            }
        }
    };
    {
        const int tid = threadIdx.x;
        const Item at = item_at(blockIdx.x);
        fetch_qk(at, tid);
        fetch_out(at, at.hv0, tid); fetch_in(at, at.hv0, tid); fetch_rest(at, at.hv0, tid);
        // (the two tiles above the diagonal that a 32-wide step over the lower triangle reads stay zero)
        for (int i = tid; i < 512; i += NTH) {
            const int t = i >> 8, r = (i >> 4) & 15, c = i & 15;
            sM1[(32 * t + r) * P64 + 32 * t + 16 + c] = (T)0.f;
        }
    }
    for (int64_t it = blockIdx.x; it < items; it += gridDim.x) {
        const Item at = item_at(it);
        const bool more = it + gridDim.x < items;
        const Item nx = item_at(more ? it + gridDim.x : it);
        {
            int tid = threadIdx.x;
            asm volatile("" : "+v"(tid));
            put_tile<KD, NTH>(sK, PK, rK, tid);
            put_tile<KD, NTH>(sQ, PK, rQ, tid);
            if constexpr (L2) { if (tid < 64) { sRq[tid] = rRq; sRk[tid] = rRk; } }
        }
        float gb_sum = 0.f;                                          // wave 0: of dg, wave 1: of dbeta
        f32x4 dq[NA][4], dk[NA][4];
#pragma unroll
        for (int a = 0; a < NA; ++a)
#pragma unroll
            for (int t = 0; t < 4; ++t) dq[a][t] = dk[a][t] = ZERO4;
#pragma unroll 1
        for (int hi = 0; hi < heads; ++hi) {
            // (everything derived from the lane number is derived again per head from a copy the compiler cannot see through:
            // hoisted out of this loop, the addresses of its unrolled body would sit in registers, or spill, for its whole length)
            int tid_opaque = threadIdx.x;
            asm volatile("" : "+v"(tid_opaque));
            const int tid = tid_opaque, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), c16 = lane & 15, g = lane >> 4;
            const int hv = at.hv0 + hi;
            auto feat = [&](int a) { return 16 * (NA * w + a); };
            put_tile<VD, NTH>(sDO, PV, rDO, tid);
            put_tile<VD, NTH>(sVn, PV, rVn, tid);
            put_tile<VD, NTH>(sDvn, PV, rDvn, tid);
            put_tile<VD, NTH>(sV, PV, rV, tid);
            put_tile<CH, NTH>(sA, P64, rA, tid);
            if (tid < 64) {
                sGam[tid] = rGam; sBeta[tid] = rBeta;
                sEg[tid] = __expf(rGam);
                sEl[tid] = __expf(__builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, rGam), 63)) - rGam);
            }
            // what comes next is requested a few tiles at a time over the phases of this head: a wave stands at a load for which
            // the CU's path to the L2 (some 25 bytes per clock) has no room yet
            const bool last = hi + 1 == heads;
            const Item& to = last ? nx : at;
            const int to_hv = last ? nx.hv0 : hv + 1;
            fetch_state(at, hv, 0, w, lane);
            lds_barrier();
            // dP o D, tile by tile
#pragma unroll
            for (int n = 0; n < NTRI; ++n) {
                __builtin_amdgcn_sched_barrier(0);
                const int idx = w + NW * n;
                if (idx < 10) {
                    const int ti = tri_row(idx), tj = tri_col(idx);
                    f32x4 acc = ZERO4;
#pragma unroll
                    for (int s = 0; s < SV; ++s) acc = Mma<T>::run(frag_rows(sDO, PV, 16 * ti, 32 * s, lane), frag_rows(sVn, PV, 16 * tj, 32 * s, lane), acc);
                    const int j = 16 * tj + c16;
                    const float gj = sGam[j];
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int i = 16 * ti + 4 * g + r;
                        sM1[i * P64 + j] = (T)(i >= j ? p.scale * acc[r] * __expf(sGam[i] - gj) : 0.f);
                    }
                }
            }
            lds_barrier();

            // dq, dk of the output and the state update, dw (kept until do and v_new are done with)
            float dglast = 0.f, dgx[4] = {0.f, 0.f, 0.f, 0.f}, dbx[4] = {0.f, 0.f, 0.f, 0.f};    // this lane's share of dgam, dbeta of token 16t + c16
            f32x4 sd = ZERO4;                                    // diagonal: <S, dS> of this wave's rows
            V4 dw[NA][4];
#pragma unroll
            for (int a = 0; a < NA; ++a) {
                const int n16 = feat(a);
                // one product with the state at a time: sixteen accumulator registers instead of forty-eight, and the next tile's fragments
                // on their way from where this tile has used its own for the last time
                f32x4 acc[4];
                auto product = [&](const V8 (&f)[SV], const T* rows) {
#pragma unroll
                    for (int t = 0; t < 4; ++t) acc[t] = ZERO4;
#pragma unroll
                    for (int s = 0; s < SV; ++s) {
                        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                        for (int t = 0; t < 4; ++t) acc[t] = Mma<T>::run(f[s], frag_rows(rows, PV, 16 * t, 32 * s, lane), acc[t]);
                    }
                };
                product(sf, sDO);
                {
                    V8 fk[2];
#pragma unroll
                    for (int s = 0; s < 2; ++s) fk[s] = frag_cols(sK, PK, 32 * s, n16, lane);
#pragma unroll
                    for (int t = 0; t < 4; ++t) {
                        __builtin_amdgcn_sched_barrier(0);
                        const int x = 16 * t + c16;
                        f32x4 q_ = acc[t] * (p.scale * sEg[x]);
                        const V4 q4 = *(const V4*)(sQ + x * PK + n16 + 4 * g);
#pragma unroll
                        for (int s = 0; s < 2; ++s)
                            if (32 * s <= 16 * t + 15) q_ = Mma<T>::run(fk[s], frag_rows(sM1, P64, 16 * t, 32 * s, lane), q_);     // dP[i][j] = 0 for j > i
#pragma unroll
                        for (int r = 0; r < 4; ++r) dgx[t] += (float)q4[r] * q_[r];
                        pin(dgx[t]);
                        dq[a][t] += q_; pin(dq[a][t]);   // (added here: the compiler moves the sums to the end of the head and keeps both terms, 96 registers)
                    }
                }
                product(sf, sDvn);
#pragma unroll
                for (int t = 0; t < 4; ++t) dw[a][t] = pack4<T>(-acc[t]);
#pragma unroll
                for (int s = 0; s < SV; ++s) sd = Mma<T>::run(sf[s], df[s], sd);
                __builtin_amdgcn_sched_barrier(0);
                if (a + 1 < NA) fetch_state(at, hv, a + 1, w, lane, true, false);
                product(df, sVn);
                __builtin_amdgcn_sched_barrier(0);
                if (a + 1 < NA) fetch_state(at, hv, a + 1, w, lane, false, true);
                {
                    V8 fq[2];
#pragma unroll
                    for (int s = 0; s < 2; ++s) fq[s] = frag_cols(sQ, PK, 32 * s, n16, lane);
#pragma unroll
                    for (int t = 0; t < 4; ++t) {
                        __builtin_amdgcn_sched_barrier(0);
                        const int x = 16 * t + c16;
                        f32x4 k_ = acc[t] * sEl[x];
                        const V4 k4 = *(const V4*)(sK + x * PK + n16 + 4 * g);
#pragma unroll
                        for (int r = 0; r < 4; ++r) dglast += (float)k4[r] * k_[r];
                        pin(dglast);
#pragma unroll
                        for (int s = 0; s < 2; ++s)
                            if (32 * s + 31 >= 16 * t) k_ = Mma<T>::run(fq[s], frag_cols(sM1, P64, 32 * s, 16 * t, lane), k_);     // ... and for i < j
#pragma unroll
                        for (int r = 0; r < 4; ++r) dgx[t] -= (float)k4[r] * k_[r];
                        pin(dgx[t]);
                        dk[a][t] += k_; pin(dk[a][t]);
                    }
                }
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) dglast += c16 == 4 * g + r ? sEg[63] * sd[r] : 0.f;
            dglast = sum_over_c16(sum_over_g(dglast));

            // dX's first term dv_new v^T (the same tiles as above), and dv = beta (A^T dv_new)
            f32x4 dX[NTRI];
#pragma unroll
            for (int n = 0; n < NTRI; ++n) {
                __builtin_amdgcn_sched_barrier(0);
                const int idx = w + NW * n;
                dX[n] = ZERO4;
                if (idx < 10) {
#pragma unroll
                    for (int s = 0; s < SV; ++s)
                        dX[n] = Mma<T>::run(frag_rows(sDvn, PV, 16 * tri_row(idx), 32 * s, lane), frag_rows(sV, PV, 16 * tri_col(idx), 32 * s, lane), dX[n]);
                }
            }
#pragma unroll
            for (int a = 0; a < NV; ++a) {                      // value columns 16 (NV w + a) ..
                const int n16 = 16 * (NV * w + a);
                V8 fdv[2];
#pragma unroll
                for (int s = 0; s < 2; ++s) fdv[s] = frag_cols(sDvn, PV, 32 * s, n16, lane);
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    __builtin_amdgcn_sched_barrier(0);
                    f32x4 av = ZERO4;
#pragma unroll
                    for (int s = 0; s < 2; ++s) {
                        if (32 * s + 31 < 16 * t) continue;     // A[i][j] = 0 for i < j
                        av = Mma<T>::run(fdv[s], frag_cols(sA, P64, 32 * s, 16 * t, lane), av);
                    }
                    const int j = 16 * t + c16;
                    const V4 v4 = *(const V4*)(sV + j * PV + n16 + 4 * g);
#pragma unroll
                    for (int r = 0; r < 4; ++r) dbx[t] += av[r] * (float)v4[r];
                    pin(dbx[t]);
                    if (j < at.c.valid) *(V4*)((T*)p.dv + ((at.c.tok0 + j) * p.HV + hv) * VD + n16 + 4 * g) = pack4<T>(av * sBeta[j]);
                }
            }
            lds_barrier();                                      // (do, v_new, dv_new and v are done with)
#pragma unroll
            for (int a = 0; a < NA; ++a)
#pragma unroll
                for (int t = 0; t < 4; ++t) *(V4*)(sDW + (16 * t + c16) * PK + feat(a) + 4 * g) = dw[a][t];
            lds_barrier();
            fetch_out(to, to_hv, tid);
            // dX's second term dw (e^gam k)^T, dA = stril(dX diag(beta)), k k^T of the same tiles
            f32x4 kk[NTRI];
#pragma unroll
            for (int n = 0; n < NTRI; ++n) {
                __builtin_amdgcn_sched_barrier(0);
                const int idx = w + NW * n;
                kk[n] = ZERO4;
                if (idx < 10) {
                    const int ti = tri_row(idx), tj = tri_col(idx);
                    f32x4 dXw = ZERO4;
#pragma unroll
                    for (int s = 0; s < SK; ++s) {
                        if (s % 2 == 0) __builtin_amdgcn_sched_barrier(0);
                        const V8 bk = frag_rows(sK, PK, 16 * tj, 32 * s, lane);
                        dXw = Mma<T>::run(frag_rows(sDW, PK, 16 * ti, 32 * s, lane), bk, dXw);
                        kk[n] = Mma<T>::run(frag_rows(sK, PK, 16 * ti, 32 * s, lane), bk, kk[n]);
                    }
                    const int j = 16 * tj + c16;
                    const float ej = sEg[j], bj = sBeta[j];
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int i = 16 * ti + 4 * g + r;
                        sM1[i * P64 + j] = (T)(i > j ? (dX[n][r] + ej * dXw[r]) * bj : 0.f);
                    }
                }
            }
            // d(e^gam k) = beta (A^T dw): into dk, dbeta, dgam
#pragma unroll
            for (int a = 0; a < NA; ++a) {
                const int n16 = feat(a);
                V8 fdw[2];
#pragma unroll
                for (int s = 0; s < 2; ++s) fdw[s] = frag_cols(sDW, PK, 32 * s, n16, lane);
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
                    const V4 k4 = *(const V4*)(sK + j * PK + n16 + 4 * g);
                    float dot = 0.f;
#pragma unroll
                    for (int r = 0; r < 4; ++r) dot += ak[r] * (float)k4[r];
                    const float ej = sEg[j], bj = sBeta[j];
                    dbx[t] += ej * dot;
                    dgx[t] += bj * ej * dot;
                    pin(dbx[t]); pin(dgx[t]);
                    dk[a][t] += ak * (bj * ej); pin(dk[a][t]);
                }
            }
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const float dgt = sum_over_g(dgx[t]), dbt = sum_over_g(dbx[t]);
                if (g == 0) { sDg[64 * w + 16 * t + c16] = dgt + (t == 3 && c16 == 15 ? dglast : 0.f); sDb[64 * w + 16 * t + c16] = dbt; }
            }
            lds_barrier();
            fetch_in(to, to_hv, tid);
            // Y = dA A^T (in dv_new's place)
#pragma unroll
            for (int n = 0; n < 16 / NW; ++n) {
                __builtin_amdgcn_sched_barrier(0);
                const int ti = (w + NW * n) >> 2, tl = (w + NW * n) & 3;
                f32x4 acc = ZERO4;
#pragma unroll
                for (int s = 0; s < 2; ++s)
                    if (32 * s <= 16 * ti + 15) acc = Mma<T>::run(frag_rows(sM1, P64, 16 * ti, 32 * s, lane), frag_rows(sA, P64, 16 * tl, 32 * s, lane), acc);
#pragma unroll
                for (int r = 0; r < 4; ++r) sM2[(16 * ti + 4 * g + r) * P64 + 16 * tl + c16] = (T)acc[r];
            }
            lds_barrier();
            // dL = -stril(A^T Y);  E = diag(beta) dL o D as an operand tile;  dbeta, dgam from L = diag(beta) stril(k k^T o D)
#pragma unroll
            for (int n = 0; n < NTRI; ++n) {
                __builtin_amdgcn_sched_barrier(0);
                const int idx = w + NW * n;
                if (idx < 10) {
                    const int ti = tri_row(idx), tl = tri_col(idx);
                    f32x4 acc = ZERO4;
#pragma unroll
                    for (int s = 0; s < 2; ++s)
                        if (32 * s + 31 >= 16 * ti) acc = Mma<T>::run(frag_cols(sA, P64, 32 * s, 16 * ti, lane), frag_cols(sM2, P64, 32 * s, 16 * tl, lane), acc);
                    const int l = 16 * tl + c16;
                    const float gl = sGam[l];
                    float colF = 0.f;
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int i = 16 * ti + 4 * g + r;
                        float E = 0.f, F = 0.f, db = 0.f;
                        if (i > l) {
                            const float d = __expf(sGam[i] - gl), dL = -acc[r], bi = sBeta[i];
                            db = dL * kk[n][r] * d;
                            E = dL * bi * d;
                            F = E * kk[n][r];
                            colF += F;
                        }
                        sM1[i * P64 + l] = (T)E;
                        db = sum_over_c16(db);
                        F = sum_over_c16(F);
                        if (c16 == 0) { atomicAdd(&sDb[64 * w + i], db); atomicAdd(&sDg[64 * w + i], F); }
                    }
                    colF = sum_over_g(colF);
                    if (g == 0) atomicAdd(&sDg[64 * w + l], -colF);
                }
            }
            lds_barrier();
            // dk += E k + E^T k
            fetch_rest(to, to_hv, tid);
#pragma unroll
            for (int a = 0; a < NA; ++a) {
                V8 fk[2];
#pragma unroll
                for (int s = 0; s < 2; ++s) fk[s] = frag_cols(sK, PK, 32 * s, feat(a), lane);
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int s = 0; s < 2; ++s) {
                        if (32 * s <= 16 * t + 15) dk[a][t] = Mma<T>::run(fk[s], frag_rows(sM1, P64, 16 * t, 32 * s, lane), dk[a][t]);      // E[i][l], l < i
                        if (32 * s + 31 >= 16 * t) dk[a][t] = Mma<T>::run(fk[s], frag_cols(sM1, P64, 32 * s, 16 * t, lane), dk[a][t]);      // E[i][l], i > l
                    }
                }
            }
            // (a wave each for dg and dbeta, while the others wait at the barrier)
            if (w < 2) {
                const float* rows = w == 0 ? sDg : sDb;
                float x = 0.f;
#pragma unroll
                for (int i = 0; i < NW; ++i) x += rows[64 * i + lane];
                if (w == 0) x = sum_of_lanes_from(x);
                // (the blocks of a value head one after the other: their sums leave together)
                const int nbp = parts_out ? min(p.nb, heads) : p.nb;     // (blocks of a value head that this item takes)
                const int blk = hv % nbp;
                gb_sum = blk ? gb_sum + x : x;
                if (blk == nbp - 1 && lane < at.c.valid) {
                    const int64_t to = (at.c.tok0 + lane) * (parts_out ? p.HV / nbp : HVg) + hv / nbp;
                    float* out = parts_out && p.split > 1 ? (w == 0 ? p.dg_part : p.db_part) : (w == 0 ? p.dg : p.dbeta);
                    out[to] = gb_sum;
                }
            }
            lds_barrier();
        }
        // the rows of dq and dk, back through the l2 normalisation of q and k where that is taken in here
        {
            int tid_opaque = threadIdx.x;
            asm volatile("" : "+v"(tid_opaque));
            const int tid = tid_opaque, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), c16 = lane & 15, g = lane >> 4;
            fetch_qk(nx, tid);
            if constexpr (L2) {
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    const int x = 16 * t + c16;
                    float qd = 0.f, kd = 0.f;
#pragma unroll
                    for (int a = 0; a < NA; ++a) {
                        const int n16 = 16 * (NA * w + a);
                        const V4 q4 = *(const V4*)(sQ + x * PK + n16 + 4 * g), k4 = *(const V4*)(sK + x * PK + n16 + 4 * g);
#pragma unroll
                        for (int r = 0; r < 4; ++r) { qd += (float)q4[r] * dq[a][t][r]; kd += (float)k4[r] * dk[a][t][r]; }
                    }
                    qd = sum_over_g(qd); kd = sum_over_g(kd);
                    if (g == 0) { sDg[64 * w + x] = qd; sDb[64 * w + x] = kd; }
                }
                lds_barrier();
            }
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const int x = 16 * t + c16;
                float qd = 0.f, kd = 0.f, rq = 1.f, rk = 1.f;
                if constexpr (L2) {
#pragma unroll
                    for (int i = 0; i < NW; ++i) { qd += sDg[64 * i + x]; kd += sDb[64 * i + x]; }
                    rq = sRq[x]; rk = sRk[x];
                }
                if (x < at.c.valid) {
                    const int64_t row = ((at.c.tok0 + x) * p.H + at.hq) * parts + at.part;
#pragma unroll
                    for (int a = 0; a < NA; ++a) {
                        const int n16 = 16 * (NA * w + a) + 4 * g;
                        f32x4 q_ = dq[a][t], k_ = dk[a][t];
                        if constexpr (L2) {
                            const V4 q4 = *(const V4*)(sQ + x * PK + n16), k4 = *(const V4*)(sK + x * PK + n16);
#pragma unroll
                            for (int r = 0; r < 4; ++r) { q_[r] = (q_[r] - (float)q4[r] * qd) * rq; k_[r] = (k_[r] - (float)k4[r] * kd) * rk; }
                        }
                        if (parts_out) {                  // (one of several parts of this row: gdn_bwd_add_parts_kernel)
                            *(f32x4*)(p.dq_part + row * KD + n16) = q_;
                            *(f32x4*)(p.dk_part + row * KD + n16) = k_;
                        } else {
                            *(V4*)((T*)p.dq + row * KD + n16) = pack4<T>(q_);
                            *(V4*)((T*)p.dk + row * KD + n16) = pack4<T>(k_);
                        }
                    }
                }
            }
            if constexpr (L2) lds_barrier();
        }
    }
}

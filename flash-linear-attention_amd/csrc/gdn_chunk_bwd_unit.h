// The chunk-parallel end of the backward pass in one kernel (included by gdn_chunk_bwd.hip, inside the namespace): from a chunk's
// state S, the gradient dS of the state behind it, v_new and dv_new to dq, dk, dv, dbeta and dg.  Per value head
//
//   dP = scale tril(do v_new^T) o D;   dq += scale e^gam (do S^T) + dP k;   dk += e^(gam_last - gam) (v_new dS^T) + dP^T q;   dw = -dv_new S^T
//   dX = tril(dw (e^gam k)^T + dv_new v^T), dA = stril(dX diag(beta));   dv = beta (A^T dv_new);   dk += d(e^gam k) = beta e^gam (A^T dw)
//   Y = dA A^T, dL = -stril(A^T Y), E = diag(beta) dL o D;   dk += E k + E^T k;   dbeta, dgam from every factor, dg = the reverse
//   cumulative sum of dgam inside the chunk.
//
// One workgroup takes the value heads of a q/k head (or an equal share of them, BwdParts; with more value columns than key features their blocks
// count as heads) of one chunk in turn, with k and q in LDS and dq, dk in fp32 registers over all of them; at 128 x 128 it moves
// 152 KB per chunk and value head (S, dS, v_new, dv_new, do, v, dv, A) and 64 KB per chunk and q/k head (k, q, dq, dk; of several parts 96: fp32 rows).
// 64 and 128 key features (256: gdn_chunk_bwd_unit256.h).
//
// What bounds it are chains - load, product, sum over lanes, barrier - and the rate at which a SIMD issues, so as many waves as there are registers for: sixteen of 128
// registers (64 features: two workgroups of eight), half of them q's side (do S^T, dw, dq, dv), half k's (v_new dS^T, dk), a wave a tile of sixteen features; the tiles of the
// lower triangles one by one.  A head is four phases (64 features: five) between barriers.  Before, eight waves of 256 registers took eight phases.
//   - dq's and dk's parts in dgam cancel in the tiles of dP (dP_ij (q_i . k_j) to i and from j: a number each, nothing on the diagonal); what dv and d(e^gam k) leave to dbeta
//     and dgam are column sums of A o dX.  So no element of q, k or v is multiplied again outside the products with the state.
//   - Y's column that a tile of dL needs is formed by that tile's wave, in the layout of a right factor: no tile of Y and no barrier.
//   - Tiles of the next head come straight into the LDS where this head is done with their places, in the order v_new and do, v; dv_new has two places.  The state's
//     fragments are requested one by one behind their last use, in the longest phase.  Registers that are spilled here cost a wait for everything under way.
//   - Everything scalar runs sixteen times (a SIMD issues one scalar instruction in four cycles): where an item lies is a few additions, not divisions.
// 16000 packed tokens, 16 q/k and 32 value heads of 128: the step 1074 -> 1006 us (the kernel 480 -> 412 us, 4.0 TB/s), 8 x 1024 tokens, 8 heads of 64 119.5 -> 116.9.

// lower triangle of 4 x 4 tiles, row by row
__device__ __forceinline__ int tri_row(int idx) { return idx < 1 ? 0 : idx < 3 ? 1 : idx < 6 ? 2 : 3; }
__device__ __forceinline__ int tri_col(int idx) { const int r = tri_row(idx); return idx - r * (r + 1) / 2; }

template <int KD> constexpr int bwd_unit_waves() { return KD / 8; }
// Room in the LDS beside one copy of every tile (160 KB a CU; 64 key features: 80 KB, two workgroups): for the next head's dv_new, and at 128 features for dw and dA
// in places of their own, which saves a barrier.
template <int KD> constexpr int bwd_unit_room() { return KD == 128 ? 64 * (2 * KD + CH) : 64 * KD; }
template <int KD> constexpr size_t bwd_unit_smem() { return (6 * 64 * KD + 2 * 64 * CH + bwd_unit_room<KD>()) * 2 + (6 * 64 + bwd_unit_waves<KD>() * 64 + 10 * 64) * 4; }

// The sum of this lane's number and those of the lanes behind it: inside rows of 16 lanes by shifts, then the rows behind.
__device__ __forceinline__ float sum_of_lanes_from(float x) {
    x = add_dpp<0x101>(x);                                       // row_shl:1, 2, 4, 8: zeros come in at the end of a row
    x = add_dpp<0x102>(x);
    x = add_dpp<0x104>(x);
    x = add_dpp<0x108>(x);
    auto row = [&](int r) { return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), 16 * r)); };
    const float r3 = row(3), r2 = row(2) + r3, r1 = row(1) + r2;
    const int r = (threadIdx.x & 63) >> 4;
    return x + (r == 0 ? r1 : r == 1 ? r2 : r == 2 ? r3 : 0.f);
}

// Computed here and not where it is used (the compiler would sink a sum to its use and keep all its terms in registers until then).
__device__ __forceinline__ void pin(float& x) { asm volatile("" : "+v"(x)); }
__device__ __forceinline__ void pin(f32x4& x) { asm volatile("" : "+v"(x)); }

// PARTS: rows and sums leave in fp32 to be added up (BwdParts); a choice inside one kernel cost 3 % (the step 1084 -> 1097 us at 16000 packed tokens, 32 heads).
template <typename T, int KD, bool L2, bool PARTS>
__global__ __launch_bounds__(64 * bwd_unit_waves<KD>(), 4) void gdn_bwd_unit_kernel(BwdParams p, int64_t items) {
    typedef typename Mma<T>::V8 V8;
    typedef typename Mma<T>::V4 V4;
    constexpr int NW = bwd_unit_waves<KD>(), NR = KD / 16, NTH = 64 * NW;
    constexpr int VD = KD, SV = VD / 32, SK = KD / 32, NTRI = (10 + NW - 1) / NW;      // (value columns: as many as key features)
    // (the tiles of the next head that have no place of their own wait in registers: A, at 64 features do, whose place dw and E take)
    constexpr bool ROOMY = KD == 128;
    static_assert(2 * NR == NW, "a wave a feature tile of a side, or a value tile");
    extern __shared__ __align__(16) char smem[];
    T* sDO = (T*)smem; T* sVn = sDO + 64 * VD; T* sDvn0 = sVn + 64 * VD; T* sV = sDvn0 + 64 * VD; T* sK = sV + 64 * VD; T* sQ = sK + 64 * KD;
    T* sA = sQ + 64 * KD; T* sM1 = sA + 64 * CH; T* sRoom = sM1 + 64 * CH;
    constexpr int DVN_STEP = 2 * 64 * VD + 2 * 64 * KD + 2 * 64 * CH;      // ... to the other place of dv_new, sRoom
    T* sDW = ROOMY ? sRoom + 64 * VD : sDO; T* sDA = ROOMY ? sDW + 64 * KD : sM1; T* sE = sDW;
    float* sGam = (float*)(sRoom + bwd_unit_room<KD>()); float* sBeta = sGam + 64; float* sRq = sBeta + 64; float* sRk = sRq + 64;
    float* sEg = sRk + 64; float* sEl = sEg + 64;                // e^gam and e^(gam_last - gam)
    float* sDg = sEl + 64;                                       // dgam through the state: a row per wave, added up in a fixed order (the same bits every run)
    // What the tiles of the triangles leave to dbeta and to dgam: a token of block t of sixteen is a row of tiles (t, 0 .. t) and a column of tiles (t .. 3, t), five
    // numbers; tile (ti, tj) leaves its rows' in line tj, its columns' in line ti + 1.
    float* sTb = sDg + NW * 64; float* sTg = sTb + 5 * 64;

    const int parts = p.parts, heads = p.HV / p.H / parts;       // value heads an item takes
    // item = (chunk * H + q/k head) * parts + part.  Sixteen waves walk over the items alike, so that every scalar instruction on the way counts sixteen times: steps of
    // gridDim.x by addition with carries, and where a chunk lies in two loads (its entry of the chunk table, its sequence's bounds) an item apart.
    struct Item { int hq, part, u0; int64_t row0; ChunkAt c; };      // u0, row0: of the item's first value head, its (chunk, head) unit and its first row in [tokens, HV]
    struct Pos { int ch, hq, part, n, it; };                       // n, it: sequence and chunk in it (packed: looked up)
    const bool packed = p.cu_seqlens != nullptr, cu32 = p.flags & GDN_FLAG_CU_INT32;
    const int NT = packed ? INT32_MAX : (int)p.NT;
    auto split = [&](uint32_t it) {
        const uint32_t grp = it / (uint32_t)parts, ch = grp / (uint32_t)p.H, n = packed ? 0u : ch / (uint32_t)NT;
        return Pos{(int)ch, (int)(grp - ch * p.H), (int)(it - grp * parts), (int)n, (int)(ch - n * (packed ? 0u : (uint32_t)NT))};
    };
    const Pos step = split(gridDim.x);
    auto on = [&](Pos a) {
        a.part += step.part;
        const int c0 = a.part >= parts ? 1 : 0;
        a.part -= c0 ? parts : 0;
        a.hq += step.hq + c0;
        const int c1 = a.hq >= p.H ? 1 : 0;
        a.hq -= c1 ? p.H : 0;
        a.ch += step.ch + c1;
        if (!packed) {
            a.it += step.it + c1;
            const int c2 = a.it >= NT ? 1 : 0;
            a.it -= c2 ? NT : 0;
            a.n += step.n + c2;
        }
        return a;
    };
    auto look_up = [&](Pos& a) {
        if (packed) { a.n = (int)load_index_uniform(p.chunk_table, 2 * (int64_t)a.ch, cu32); a.it = (int)load_index_uniform(p.chunk_table, 2 * (int64_t)a.ch + 1, cu32); }
    };
    auto item_at = [&](const Pos& a) {                             // (a: looked up)
        int64_t bos = (int64_t)a.n * p.T, eos = bos + p.T;         // (no 64-bit comparison: the scalar unit has none for less and greater)
        if (packed) { bos = load_index_uniform(p.cu_seqlens, a.n, cu32); eos = load_index_uniform(p.cu_seqlens, a.n + 1, cu32); }
        const int64_t tok0 = bos + (int64_t)a.it * CH, left = eos - tok0;
        const int hv0 = a.hq * (heads * parts) + a.part * heads;
        return Item{a.hq, a.part, a.ch * p.HV + hv0, tok0 * p.HV + hv0, ChunkAt{tok0, (left >> 6) != 0 ? CH : (int)left}};
    };
    // A role's whole walk over the items, in code of its own: what a wave keeps in registers never meets the other role's.
    auto walk = [&](auto role) __attribute__((always_inline)) {
    constexpr bool kside = decltype(role)::value, qside = !kside;
    TileRegs<VD, NTH> rDO;                                       // (64 key features)
    TileRegs<CH, 512> rA;                                        // (the first 512 threads)
    TileRegs<KD, NTH> rK, rQ;
    V8 sf[SV], df[SV];                                           // rows of S and (k's side) of dS
    float rGam = 0.f, rBeta = 0.f, rRq = 0.f, rRk = 0.f;
    const int HVg = p.HV / p.nb;
    constexpr bool parts_out = PARTS;
    // (hi: value head hv0 + hi of an item)
    auto state_at = [&](const void* x, const Item& at, int hi, int wf, int lane) { return (const T*)x + (int64_t)(at.u0 + hi) * (KD * VD) + state_frag<VD>(wf, 0, lane); };
    auto fetch_S = [&](const Item& at, int hi, int wf, int s, int lane) { sf[s] = *(const V8*)(state_at(p.ws.Hs, at, hi, wf, lane) + 512 * s); };
    auto fetch_dS = [&](const Item& at, int hi, int wf, int s, int lane) { df[s] = *(const V8*)(state_at(p.ws.dHs, at, hi, wf, lane) + 512 * s); };
    auto value_rows = [&](const void* x, const Item& at, int hi) { return (const T*)x + (at.row0 + hi) * VD; };
    auto unit_rows = [&](const void* x, const Item& at, int hi) { return (const T*)x + (int64_t)(at.u0 + hi) * (64 * VD); };
    auto fetch_rest = [&](const Item& at, int hi, int tid) {
        const int64_t ug = p.nb == 1 ? at.u0 + hi : (at.u0 + hi) / p.nb;
        if constexpr (!ROOMY) fetch_blocks<VD, NTH>(rDO, value_rows(p.dout, at, hi), (int64_t)p.HV * VD, at.c.valid, tid);
        if constexpr (qside || NTH == 512) fetch_blocks<CH, 512>(rA, (const T*)p.ws.Am + ug * 64 * 64, 64, 64, tid);
        if constexpr (qside) { if (tid < 64) { rGam = p.ws.Gam[ug * 64 + tid]; rBeta = p.ws.Bet[ug * 64 + tid]; } }
    };
    auto fetch_qk = [&](const Item& at, int tid) {
        fetch_blocks<KD, NTH>(rK, (const T*)p.k + (at.c.tok0 * p.H + at.hq) * KD, (int64_t)p.H * KD, at.c.valid, tid);
        fetch_blocks<KD, NTH>(rQ, (const T*)p.q + (at.c.tok0 * p.H + at.hq) * KD, (int64_t)p.H * KD, at.c.valid, tid);
        if constexpr (L2 && qside) {
            if (tid < 64) {
                rRq = tid < at.c.valid ? p.q_rstd[(at.c.tok0 + tid) * p.H + at.hq] : 0.f;
                rRk = tid < at.c.valid ? p.k_rstd[(at.c.tok0 + tid) * p.H + at.hq] : 0.f;
            }
        }
    };
    // The copies have landed, and what came into registers is waited for where nothing younger is under way.
    auto arrived = [&]() {
        wait_vm_at_most<0>();
#pragma unroll
        for (int s = 0; s < SV; ++s) asm volatile("" : "+v"(sf[s]));
        if constexpr (kside) {
#pragma unroll
            for (int s = 0; s < SV; ++s) asm volatile("" : "+v"(df[s]));
        }
        if constexpr (!ROOMY) asm volatile("" : "+v"(rDO.x[0]));
        if constexpr (qside || NTH == 512) asm volatile("" : "+v"(rA.x[0]));
#pragma unroll
        for (int i = 0; i < (int)(sizeof(rK.x) / 16); ++i) asm volatile("" : "+v"(rK.x[i]), "+v"(rQ.x[i]));
        if constexpr (qside) asm volatile("" : "+v"(rRq), "+v"(rRk), "+v"(rGam), "+v"(rBeta));
    };
    // (past the last item: that one again)
    Pos pos = split(blockIdx.x);                                   // of the item after `nx`
    look_up(pos);
    uint32_t to_come = (uint32_t)items - blockIdx.x;               // items from there on
    auto advance = [&]() {
        if (to_come > gridDim.x) { to_come -= gridDim.x; pos = on(pos); }
        look_up(pos);
    };
    Item at = item_at(pos);
    advance();
    Item nx = item_at(pos);
    advance();
    {
        const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
        fetch_qk(at, tid);
        fetch_rest(at, 0, tid);
#pragma unroll
        for (int s = 0; s < SV; ++s) { fetch_S(at, 0, w % NR, s, lane); if constexpr (kside) fetch_dS(at, 0, w % NR, s, lane); }
        if constexpr (ROOMY) copy_blocks<VD, NW>(sDO, value_rows(p.dout, at, 0), (int64_t)p.HV * VD, at.c.valid, w, lane);
        copy_blocks<VD, NW>(sVn, unit_rows(p.ws.Vn, at, 0), VD, 64, w, lane);
        copy_blocks<VD, NW>(sDvn0, unit_rows(p.ws.dVn, at, 0), VD, 64, w, lane);
        copy_blocks<VD, NW>(sV, value_rows(p.v, at, 0), (int64_t)p.HV * VD, at.c.valid, w, lane);
        arrived();
        // (the two tiles above the diagonal that a 32-wide step over the lower triangle reads stay zero)
        for (int i = tid; i < 512; i += NTH) {
            const int t = i >> 8, r = (i >> 4) & 15, c = i & 15;
            *(T*)((char*)sM1 + block_off<CH>(32 * t, 32 * t + 16) + (block_lane<CH>(r, c) ^ 32)) = (T)0.f;
            if constexpr (ROOMY) *(T*)((char*)sDA + block_off<CH>(32 * t, 32 * t + 16) + (block_lane<CH>(r, c) ^ 32)) = (T)0.f;
        }
    }
    int odd = 0;                                                 // which of dv_new's two places
    for (uint32_t left = ((uint32_t)items - blockIdx.x + gridDim.x - 1) / gridDim.x; left > 0; --left) {
        // (what comes next is requested in any case, the last time for nothing: behind a condition the registers of the last request would stay alive through the whole head)
        const Item nx2 = item_at(pos);
        advance();
        {
            int tid = threadIdx.x;
            asm volatile("" : "+v"(tid));
            put_blocks<KD, NTH>(sK, rK, at.c.valid, tid);
            put_blocks<KD, NTH>(sQ, rQ, at.c.valid, tid);
            if constexpr (L2 && qside) { if (tid < 64) { sRq[tid] = rRq; sRk[tid] = rRk; } }
        }
        float gb_sum = 0.f;                                          // wave 0: of dg, wave 1: of dbeta
        f32x4 dq[4], dk[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) dq[t] = dk[t] = ZERO4;
#pragma unroll 1
        for (int hi = 0; hi < heads; ++hi) {
            // (everything derived from the lane number is derived again per head from a copy the compiler cannot see through:
            // hoisted out of this loop, the addresses of its unrolled body would sit in registers, or spill, for its whole length)
            int tid_opaque = threadIdx.x;
            asm volatile("" : "+v"(tid_opaque));
            const int tid = tid_opaque, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), c16 = lane & 15, g = lane >> 4;
            const int wf = !qside ? w - NR : w, n16 = 16 * wf;            // this wave's features
            // this lane's shares of the addresses of operands by rows, by columns, of a result's four elements in a row, of a triangle tile's elements
            const int ro = opaque(block_rows_lane<KD>(lane)), ro_c = KD == CH ? ro : opaque(block_rows_lane<CH>(lane));
            auto cols_lane = [&](ColsLane x) { return ColsLane{opaque(x.a), opaque(x.b)}; };
            const ColsLane co_c = cols_lane(block_cols_lane<CH>(lane)), co_c1 = cols_lane(odd_tile(co_c));
            const int eo = opaque(block_lane<KD>(c16, 4 * g) ^ (32 * (wf & 1)));
            const ColsLane fk = block_cols_lane<KD>(lane), fo = cols_lane(wf & 1 ? odd_tile(fk) : fk);
            auto elem = [&](const T* x, int t) { return (V4*)((char*)x + block_off<KD>(16 * t, n16) + eo); };
            auto feat_cols = [&](const T* x, int r0) { return block_cols<KD>(x, r0, n16, fo); };
            const int to_ = opaque(block_lane<CH>(4 * g, c16));
            auto tri_at = [&](const T* x, int ti, int tj, int r) { return (T*)((char*)x + block_off<CH>(16 * ti, 16 * tj) + (to_ ^ (32 * (tj & 1))) + 64 * r); };
            T* sDvn = sDvn0 + odd;
            if constexpr (!ROOMY) put_blocks<VD, NTH>(sDO, rDO, at.c.valid, tid);
            if constexpr (qside || NTH == 512) put_blocks<CH, 512>(sA, rA, 64, tid);
            if constexpr (qside) {
                if (tid < 64) {
                    sGam[tid] = rGam; sBeta[tid] = rBeta;
                    sEg[tid] = __expf(rGam);
                    sEl[tid] = __expf(__builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, rGam), 63)) - rGam);
                }
            }
            const bool last = hi + 1 == heads;
            const Item& to = last ? nx : at;
            const int to_hi = last ? 0 : hi + 1;
            lds_barrier();
            // dv = beta (A^T dv_new), value columns 16 wf ..
            auto leave_dv = [&]() {
                V8 f[2];
#pragma unroll
                for (int s = 0; s < 2; ++s) f[s] = block_cols<VD>(sDvn, 32 * s, 16 * wf, fo);
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    __builtin_amdgcn_sched_barrier(0);
                    f32x4 av = ZERO4;
#pragma unroll
                    for (int s = 0; s < 2; ++s)
                        if (32 * s + 31 >= 16 * t) av = Mma<T>::run(f[s], block_cols<CH>(sA, 32 * s, 16 * t, t % 2 ? co_c1 : co_c), av);     // A[i][j] = 0 for i < j
                    const int j = 16 * t + c16;
                    if (j < at.c.valid) *(V4*)((T*)p.dv + (at.row0 + hi + (int64_t)j * p.HV) * VD + n16 + 4 * g) = pack4<T>(av * sBeta[j]);
                }
            };
            copy_blocks<VD, NW>(sDvn0 + (DVN_STEP - odd), unit_rows(p.ws.dVn, to, to_hi), VD, 64, w, lane);

            // products with the state, into dq and dk at once: q's side do S^T and dw = -dv_new S^T, k's side v_new dS^T; and the tiles of dP o D
            V4 dw[4];
            {
                float dgx[4] = {0.f, 0.f, 0.f, 0.f}, dglast = 0.f;    // this lane's share of dgam of token 16t + c16
                // (a step's rows of the state give their place to the next head's as soon as they are used for the last time: requests spread over the
                // longest phase, where the CU's path to the L2 has room for them)
                auto product = [&](f32x4 (&x)[4], const V8 (&f)[SV], const T* rows, auto behind) {
#pragma unroll
                    for (int t = 0; t < 4; ++t) x[t] = ZERO4;
#pragma unroll
                    for (int s = 0; s < SV; ++s) {
                        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                        for (int t = 0; t < 4; ++t) x[t] = Mma<T>::run(f[s], block_rows<VD>(rows, 16 * t, 32 * s, ro), x[t]);
                        behind(s);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                };
                f32x4 x[4];
                if constexpr (kside) {
                    f32x4 sd = ZERO4;                                // diagonal: <S, dS> of this wave's rows
                    product(x, df, sVn, [&](int s) { sd = Mma<T>::run(sf[s], df[s], sd); pin(sd); fetch_S(to, to_hi, wf, s, lane); fetch_dS(to, to_hi, wf, s, lane); });
#pragma unroll
                    for (int t = 0; t < 4; ++t) {
                        const V4 k4 = *elem(sK, t);
                        x[t] *= sEl[16 * t + c16];
                        float d = 0.f;
#pragma unroll
                        for (int r = 0; r < 4; ++r) d += (float)k4[r] * x[t][r];
                        dgx[t] -= d; dglast += d;
                        pin(dgx[t]); pin(dglast);
                        dk[t] += x[t];
                        pin(dk[t]);
                    }
#pragma unroll
                    for (int r = 0; r < 4; ++r) dglast += c16 == 4 * g + r ? sEg[63] * sd[r] : 0.f;
                    dglast = sum_over_c16(sum_over_g(dglast));
                }
                if constexpr (qside) {
                    product(x, sf, sDO, [](int) {});
#pragma unroll
                    for (int t = 0; t < 4; ++t) {
                        const V4 q4 = *elem(sQ, t);
                        x[t] *= p.scale * sEg[16 * t + c16];
#pragma unroll
                        for (int r = 0; r < 4; ++r) dgx[t] += (float)q4[r] * x[t][r];
                        pin(dgx[t]);
                        dq[t] += x[t];
                        pin(dq[t]);
                    }
                    product(x, sf, sDvn, [&](int s) { fetch_S(to, to_hi, wf, s, lane); });
#pragma unroll
                    for (int t = 0; t < 4; ++t) {
                        dw[t] = pack4<T>(-x[t]);
                        if constexpr (ROOMY) *elem(sDW, t) = dw[t];
                        else {
                            u32x2 b = __builtin_bit_cast(u32x2, dw[t]);
                            asm volatile("" : "+v"(b));
                            dw[t] = __builtin_bit_cast(V4, b);
                        }
                    }
                }
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    const float dgt = sum_over_g(dgx[t]);
                    if (g == 0) sDg[64 * w + 16 * t + c16] = dgt + (t == 3 && c16 == 15 ? dglast : 0.f);
                }
            }
#pragma unroll
            for (int n = 0; n < NTRI; ++n) {
                __builtin_amdgcn_sched_barrier(0);
                const int idx = w + NW * n;
                if (idx >= 10) continue;
                const int ti = tri_row(idx), tj = tri_col(idx);
                f32x4 d = ZERO4, qk = ZERO4;
#pragma unroll
                for (int s = 0; s < SV; ++s) {
                    if (s % 2 == 0) __builtin_amdgcn_sched_barrier(0);
                    d = Mma<T>::run(block_rows<VD>(sDO, 16 * ti, 32 * s, ro), block_rows<VD>(sVn, 16 * tj, 32 * s, ro), d);
                }
                pin(d);
#pragma unroll
                for (int s = 0; s < SK; ++s) {
                    if (s % 2 == 0) __builtin_amdgcn_sched_barrier(0);
                    qk = Mma<T>::run(block_rows<KD>(sQ, 16 * ti, 32 * s, ro), block_rows<KD>(sK, 16 * tj, 32 * s, ro), qk);
                }
                const int j = 16 * tj + c16;
                const float gj = sGam[j];
                float col = 0.f;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int i = 16 * ti + 4 * g + r;
                    const float dP = i >= j ? p.scale * d[r] * __expf(sGam[i] - gj) : 0.f;
                    *tri_at(sM1, ti, tj, r) = (T)dP;
                    float x = i > j ? dP * qk[r] : 0.f;              // (to dgam_i and from dgam_j: nothing on the diagonal)
                    col += x;
                    x = sum_over_c16(x);
                    if (c16 == 0) sTg[64 * tj + i] = x;
                }
                col = sum_over_g(col);
                if (g == 0) sTg[64 * (ti + 1) + j] = -col;
            }
            lds_barrier();                                          // (do and v_new are done with)
            // The next head: what waits in registers first (the compiler's waits for it do not know of the copies behind it), all of it done with in the
            // last phase of this head
            fetch_rest(to, to_hi, tid);
            if constexpr (ROOMY) copy_blocks<VD, NW>(sDO, value_rows(p.dout, to, to_hi), (int64_t)p.HV * VD, to.c.valid, w, lane);
            copy_blocks<VD, NW>(sVn, unit_rows(p.ws.Vn, to, to_hi), VD, 64, w, lane);

            // dq += dP k, dk += dP^T q
            if constexpr (qside) {
                V8 f[2];
                if constexpr (!ROOMY) {                              // (dw into the tiles of do and v_new)
#pragma unroll
                    for (int t = 0; t < 4; ++t) *elem(sDW, t) = dw[t];
                }
#pragma unroll
                for (int s = 0; s < 2; ++s) f[s] = feat_cols(sK, 32 * s);
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int s = 0; s < 2; ++s)
                        if (32 * s <= 16 * t + 15) dq[t] = Mma<T>::run(f[s], block_rows<CH>(sM1, 16 * t, 32 * s, ro_c), dq[t]);     // dP[i][j] = 0 for j > i
                    pin(dq[t]);
                }
            }
            if constexpr (kside) {
                V8 f[2];
#pragma unroll
                for (int s = 0; s < 2; ++s) f[s] = feat_cols(sQ, 32 * s);
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int s = 0; s < 2; ++s)
                        if (32 * s + 31 >= 16 * t) dk[t] = Mma<T>::run(f[s], block_cols<CH>(sM1, 32 * s, 16 * t, t % 2 ? co_c1 : co_c), dk[t]);     // ... and for i < j
                    pin(dk[t]);
                }
            }
            if constexpr (!ROOMY) lds_barrier();
            // dX = tril(dw (e^gam k)^T + dv_new v^T) tile by tile, dA = stril(dX diag(beta)), k k^T of the same tiles.  What dv and d(e^gam k) leave to dbeta
            // and dgam, sum_d (A^T dv_new)_jd v_jd and the like, is sum_i A_ij dX_ij: column sums here instead of products with every element there
            f32x4 kk[NTRI];
#pragma unroll
            for (int n = 0; n < NTRI; ++n) {
                __builtin_amdgcn_sched_barrier(0);
                const int idx = w + NW * n;
                kk[n] = ZERO4;
                if (idx < 10) {
                    const int ti = tri_row(idx), tj = tri_col(idx);
                    f32x4 dXv = ZERO4, dXw = ZERO4;
#pragma unroll
                    for (int s = 0; s < SV; ++s) {
                        if (s % 2 == 0) __builtin_amdgcn_sched_barrier(0);
                        dXv = Mma<T>::run(block_rows<VD>(sDvn, 16 * ti, 32 * s, ro), block_rows<VD>(sV, 16 * tj, 32 * s, ro), dXv);
                    }
#pragma unroll
                    for (int s = 0; s < SK; ++s) {
                        __builtin_amdgcn_sched_barrier(0);
                        const V8 bk = block_rows<KD>(sK, 16 * tj, 32 * s, ro);
                        dXw = Mma<T>::run(block_rows<KD>(sDW, 16 * ti, 32 * s, ro), bk, dXw);
                        kk[n] = Mma<T>::run(block_rows<KD>(sK, 16 * ti, 32 * s, ro), bk, kk[n]);
                    }
                    const int j = 16 * tj + c16;
                    pin(kk[n]);
                    const float ej = sEg[j], bj = sBeta[j];
                    float db = 0.f, dg = 0.f;
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int i = 16 * ti + 4 * g + r;
                        const float a = (float)*tri_at(sA, ti, tj, r), xw = ej * dXw[r], x = dXv[r] + xw;
                        db += a * x;
                        dg += a * xw;
                        *tri_at(sDA, ti, tj, r) = (T)(i > j ? x * bj : 0.f);
                    }
                    db = sum_over_g(db); dg = bj * sum_over_g(dg);
                    if (g == 0) { sTb[64 * (ti + 1) + j] = db; sTg[64 * (ti + 1) + j] += dg; }
                }
            }
            // k's side: d(e^gam k) = beta (A^T dw) into dk
            if constexpr (kside) {
                V8 f[2];
#pragma unroll
                for (int s = 0; s < 2; ++s) f[s] = feat_cols(sDW, 32 * s);
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    __builtin_amdgcn_sched_barrier(0);
                    f32x4 ak = ZERO4;
#pragma unroll
                    for (int s = 0; s < 2; ++s)
                        if (32 * s + 31 >= 16 * t) ak = Mma<T>::run(f[s], block_cols<CH>(sA, 32 * s, 16 * t, t % 2 ? co_c1 : co_c), ak);     // A[i][j] = 0 for i < j
                    const int j = 16 * t + c16;
                    dk[t] += ak * (sBeta[j] * sEg[j]);
                    pin(dk[t]);
                }
            }
            lds_barrier();                                          // (dw and v are done with)
            if (last) fetch_qk(nx, tid);
            copy_blocks<VD, NW>(sV, value_rows(p.v, to, to_hi), (int64_t)p.HV * VD, to.c.valid, w, lane);
            // Y = dA A^T, dL = -stril(A^T Y): a wave forms the column of Y that its tile of dL needs, whose tiles are right factors as they lie in its
            // registers.  E = diag(beta) dL o D as an operand tile;  dbeta, dgam from L = diag(beta) stril(k k^T o D)
#pragma unroll
            for (int n = 0; n < NTRI; ++n) {
                __builtin_amdgcn_sched_barrier(0);
                const int idx = w + NW * n;
                if (idx < 10) {
                    const int ti = tri_row(idx), tl = tri_col(idx);
                    V8 y[2], fa[2];
#pragma unroll
                    for (int ib = 0; ib < 4; ++ib) {
                        __builtin_amdgcn_sched_barrier(0);
                        f32x4 yt = ZERO4;
                        V4 at4 = pack4<T>(ZERO4);
                        if (ib >= ti) {
                            yt = Mma<T>::run(block_rows<CH>(sDA, 16 * ib, 0, ro_c), block_rows<CH>(sA, 16 * tl, 0, ro_c), yt);
                            if (tl >= 2) yt = Mma<T>::run(block_rows<CH>(sDA, 16 * ib, 32, ro_c), block_rows<CH>(sA, 16 * tl, 32, ro_c), yt);
                            at4 = Mma<T>::tr_read((const T*)((const char*)sA + block_off<CH>(16 * ib, 16 * ti) + (block_lane<CH>(4 * g + (c16 >> 2), 4 * (c16 & 3)) ^ (32 * (ti & 1)))));     // rows 16 ib + 4g .., column 16 ti + c16
                        }
                        const V4 y4 = pack4<T>(yt);
#pragma unroll
                        for (int r = 0; r < 4; ++r) { y[ib >> 1][4 * (ib & 1) + r] = y4[r]; fa[ib >> 1][4 * (ib & 1) + r] = at4[r]; }
                    }
                    const f32x4 acc_ = Mma<T>::run(fa[1], y[1], Mma<T>::run(fa[0], y[0], ZERO4));
                    const int l = 16 * tl + c16;
                    const float gl = sGam[l];
                    float colF = 0.f;
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int i = 16 * ti + 4 * g + r;
                        float E = 0.f, F = 0.f, db = 0.f;
                        if (i > l) {
                            const float d = __expf(sGam[i] - gl), dL = -acc_[r], bi = sBeta[i];
                            db = dL * kk[n][r] * d;
                            E = dL * bi * d;
                            F = E * kk[n][r];
                            colF += F;
                        }
                        *tri_at(sE, ti, tl, r) = (T)E;
                        db = sum_over_c16(db);
                        F = sum_over_c16(F);
                        if (c16 == 0) { sTb[64 * tl + i] = db; sTg[64 * tl + i] += F; }
                    }
                    colF = sum_over_g(colF);
                    if (g == 0) sTg[64 * (ti + 1) + l] -= colF;
                }
            }
            if (w >= NW - 2) {                              // (the two tiles above E's diagonal that 32-wide steps read)
                const int t = w - (NW - 2);
                *(V4*)((char*)sE + block_off<CH>(32 * t, 32 * t + 16) + (block_lane<CH>(lane >> 2, 4 * (lane & 3)) ^ 32)) = pack4<T>(ZERO4);
            }
            lds_barrier();
            arrived();
            if constexpr (kside) {
                // dk += E k + E^T k
                V8 f[2];
#pragma unroll
                for (int s = 0; s < 2; ++s) f[s] = feat_cols(sK, 32 * s);
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int s = 0; s < 2; ++s) {
                        if (32 * s <= 16 * t + 15) dk[t] = Mma<T>::run(f[s], block_rows<CH>(sE, 16 * t, 32 * s, ro_c), dk[t]);      // E[i][l], l < i
                        if (32 * s + 31 >= 16 * t) dk[t] = Mma<T>::run(f[s], block_cols<CH>(sE, 32 * s, 16 * t, t % 2 ? co_c1 : co_c), dk[t]);      // E[i][l], i > l
                    }
                }
            }
            if constexpr (qside) {
                leave_dv();
                // (a wave each for dg and dbeta)
                if (w < 2) {
                    float x = 0.f;
                    const float* lines = w == 0 ? sTg : sTb;
#pragma unroll
                    for (int o = 0; o < 5; ++o) x += lines[64 * o + lane];
                    if (w == 0) {
#pragma unroll
                        for (int i = 0; i < NW; ++i) x += sDg[64 * i + lane];
                    }
                    if (w == 0) x = sum_of_lanes_from(x);
                    // (the blocks of a value head one after the other: their sums leave together)
                    const int nbp = parts_out ? min(p.nb, heads) : p.nb;     // (blocks of a value head that this item takes)
                    const int hv = (at.hq * parts + at.part) * heads + hi, head = nbp == 1 ? hv : hv / nbp, blk = hv - head * nbp;
                    gb_sum = blk ? gb_sum + x : x;
                    if (blk == nbp - 1 && lane < at.c.valid) {
                        const int64_t to = (at.c.tok0 + lane) * (!parts_out ? HVg : nbp == 1 ? p.HV : p.HV / nbp) + head;
                        float* out = parts_out && p.split > 1 ? (w == 0 ? p.dg_part : p.db_part) : (w == 0 ? p.dg : p.dbeta);
                        out[to] = gb_sum;
                    }
                }
            }
            lds_barrier();
            odd = DVN_STEP - odd;
        }
        // the rows of dq and dk, back through the l2 normalisation of q and k where that is taken in here
        {
            int tid_opaque = threadIdx.x;
            asm volatile("" : "+v"(tid_opaque));
            const int tid = tid_opaque, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), c16 = lane & 15, g = lane >> 4;
            const int wf = !qside ? w - NR : w, n16 = 16 * wf, eo = block_lane<KD>(c16, 4 * g) ^ (32 * (wf & 1));
            auto elem = [&](const T* x, int t) { return *(const V4*)((const char*)x + block_off<KD>(16 * t, n16) + eo); };
            float* sDk = sDg + 64 * NR;                                  // (a row per wave again)
            if constexpr (L2) {
                auto dots = [&](const f32x4 (&dx)[4], const T* rows, float* to) {
#pragma unroll
                    for (int t = 0; t < 4; ++t) {
                        const V4 y4 = elem(rows, t);
                        float d = 0.f;
#pragma unroll
                        for (int r = 0; r < 4; ++r) d += (float)y4[r] * dx[t][r];
                        d = sum_over_g(d);
                        if (g == 0) to[64 * wf + 16 * t + c16] = d;
                    }
                };
                if constexpr (qside) dots(dq, sQ, sDg);
                if constexpr (kside) dots(dk, sK, sDk);
                lds_barrier();
            }
            auto leave = [&](const f32x4 (&dx)[4], const T* rows, const float* sum, const float* factor, void* out, float* out_part) {
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    const int x = 16 * t + c16;
                    f32x4 y = dx[t];
                    if constexpr (L2) {
                        float d = 0.f;
#pragma unroll
                        for (int i = 0; i < NR; ++i) d += sum[64 * i + x];
                        const float rs = factor[x];
                        const V4 y4 = elem(rows, t);
#pragma unroll
                        for (int r = 0; r < 4; ++r) y[r] = (y[r] - (float)y4[r] * d) * rs;
                    }
                    if (x < at.c.valid) {
                        const int64_t to = (((at.c.tok0 + x) * p.H + at.hq) * parts + at.part) * KD + n16 + 4 * g;
                        if (parts_out) *(f32x4*)(out_part + to) = y;     // (one of several parts of this row: gdn_bwd_add_parts_kernel)
                        else *(V4*)((T*)out + to) = pack4<T>(y);
                    }
                }
            };
            if constexpr (qside) leave(dq, sQ, sDg, sRq, p.dq, p.dq_part);
            if constexpr (kside) leave(dk, sK, sDk, sRk, p.dk, p.dk_part);
            if constexpr (L2) lds_barrier();
        }
        at = nx; nx = nx2;
    }
    };
    if (threadIdx.x >= 64 * NR) walk(std::true_type{}); else walk(std::false_type{});
}

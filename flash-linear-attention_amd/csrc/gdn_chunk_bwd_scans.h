// (included by gdn_chunk_bwd.hip, inside the namespace)
// ---------------------------------------------------------------------------------------------
// The two scans.  A workgroup owns VBT value columns of one (sequence, v-head): the state slice [KD][VBT] lives in
// registers as transposed tiles - wave w holds key rows KD/4 w .. as NA = KD/64 tiles (a2), lane (c16, g) key
// 16(NA w + a2) + c16 and value columns 16b + 4g .. +3.  The next chunk's tiles are fetched into registers while the
// current chunk is computed, and the barriers wait for LDS traffic only, so those loads stay in flight across them.
//
// Three forms.  GATED (the gated delta rule) never forms w = A (beta e^gam k) and u = A (beta v): the forward scan takes
// v_new = A (beta (v - e^gam (k S))), the reverse one -w^T dv_new = -k^T (beta e^gam (A^T dv_new)) - one product of 64 x 64 x VBT more per
// step against two tiles of KD and VBT features less to write and to read per unit (and the prepare kernel a sixth of its time).
// COMBA and KDA read w and u (their w is made from other rows than k); KDA's rows of k and q arrive as KG and QG (decays and the
// scale on them), its state decays per key feature (EGL), its P is row-major like GATED's; COMBA's arrives transposed.
// ---------------------------------------------------------------------------------------------
constexpr int FORM_GATED = 0, FORM_COMBA = 1, FORM_KDA = 2;
// (64 or 128 value columns: eight waves, two per SIMD, share one set of tiles.  64 columns with four waves: 8 x 2048 tokens, 32 heads of 256 features, the
// step 3765 us, with eight 3588; 8000 tokens in 4 sequences, 16 heads of 128: 486 and 458 us)
template <int VBT> constexpr int scan_waves() { return VBT >= 64 ? 8 : 4; }

// (the forward scan keeps v_new twice where a CU's LDS has the room: as the operand of the state update, with the decay to the end
// of the chunk on it, and as it is stored, so that it can leave as whole rows)
template <int VBT, int KD, int FORM> constexpr size_t bwd_state_tiles() {
    return (64 * (KD + 8) + (FORM == FORM_GATED ? 64 * P64 + 64 * (VBT + 8) : 64 * (KD + 8)) + KD * (VBT + 8) + 64 * (VBT + 8)) * 2 + 128 * 4;
}
template <int VBT, int KD, int FORM> constexpr bool state_out_tile() { return bwd_state_tiles<VBT, KD, FORM>() + 64 * (VBT + 8) * 2 <= 160 * 1024; }
template <int VBT, int KD, int FORM> constexpr size_t bwd_state_smem() {
    return bwd_state_tiles<VBT, KD, FORM>() + (state_out_tile<VBT, KD, FORM>() ? 64 * (VBT + 8) * 2 : 0);
}
template <int VBT, int KD, int FORM> constexpr size_t bwd_dstate_smem() {
    return (2 * 64 * (KD + 8) + (FORM == FORM_GATED ? 64 * P64 + 64 * (VBT + 8) : 64 * (KD + 8)) + 64 * P64 + 2 * 64 * (VBT + 8) + KD * (VBT + 8)) * 2 + 128 * 4;
}

// How a step requests the next one's tiles.  EXACT: with the same loads whatever the chunk and the step (fetch_rows; the last step its own tiles once more, for
// nothing), so that the compiler knows how many stores are younger and the wait for the loads leaves them in flight; and behind the state's stores, not before
// them (which makes every step 5 % longer).
// At 128 key features for sequences of eight chunks or more on average, the gated form beyond 64 runs sixteen (scans_128): 16000 packed tokens in 12 sequences, 32 heads the step
// 1003 -> 997 us; the launch, 30 heads of 1400 tokens 57.4 -> 55.9; KDA and comba, 64 heads of 4000 tokens 206 -> 188 and 210 -> 201, 96 heads 287 -> 275 and 299 -> 295.
// Short sequences lose by what the last step requests and by the rows past their end: gated, one chunk of 32 tokens 735 -> 836 us, of 64 tokens 422 -> 444, four
// chunks 327 -> 355, eight (992 runs) 319 -> 349; KDA and comba, one chunk of 32 tokens 365 -> 390 and 188 -> 209, of 64 tokens 196 -> 207 and 109 -> 115, two to four up to 1 and 6 %.
// At 256 features where a workgroup has a CU to itself, up to 32 runs, four chunks or more on average: 4 heads of 1024 tokens 61.0 -> 59.1 us, of 1400 tokens 83.5 -> 79.8; one
// chunk 13.7 and 14.0; and in the 64-column form beyond 64 runs 32 chunks or more: 48 heads of 3000 tokens 397 -> 390, 4 x 4096 tokens, 6 heads of 256 x 512 545 -> 528 (1500
// tokens equal, 700 86.3 and 89.4; up to 64 runs 0.5 to 1.5 % longer).  Elsewhere nothing gains: 8 x 2048 tokens, 32 heads the step 3103 -> 3111 us, 250 sequences of 32 tokens, 16
// heads the launch 612 -> 691.  Nor where a step has little to store and its instructions count (64 features: 116.5 -> 118.8 us), or where warm-up steps store nothing.
template <bool EXACT, int NCOLS, int NTH, typename T>
__device__ __forceinline__ void fetch_scan(TileRegs<NCOLS, NTH>& r, const T* g, int64_t stride, int valid, int tid) {
    if constexpr (EXACT) fetch_rows<NCOLS, NTH>(r, g, stride, valid, tid);
    else fetch_tile<NCOLS, NTH>(r, g, stride, valid, tid);
}

// Workgroups go to the 8 XCDs in turn: the slices of one (sequence, head) take the same residue, so that they share
// an L2 for the rows of k, q, w and A that all of them read.  With time segments (nwg workgroups each) a segment's come in a row.
struct ScanAt { bool out; int hv, hq, hg, vcol0; int64_t n; SeqAt sq; ScanPlan plan; };
template <bool SEG, int VBT, int VD>
__device__ __forceinline__ ScanAt scan_at(const BwdParams& p, unsigned bid_all, unsigned nwg, int lane, int& seg) {
    constexpr int NVS = VD / VBT;
    seg = SEG ? (int)(bid_all / (nwg / p.nseg)) : 0;
    const unsigned bid = SEG ? bid_all % (nwg / p.nseg) : bid_all;
    const int64_t run = (int64_t)(bid / (8 * NVS)) * 8 + bid % 8;
    ScanAt at{};
    at.out = run >= p.N * p.HV;
    if (at.out) return at;
    at.hv = (int)(run % p.HV); at.hg = at.hv / p.nb; at.hq = at.hv / (p.HV / p.H);
    at.n = seq_in_order(p, run / p.HV);
    at.sq = seq_at(p, at.n);
    at.vcol0 = ((bid / 8) % NVS) * VBT;
    at.plan = SEG ? scan_plan(p, at.sq, at.hg, seg, lane) : ScanPlan{false, 0, at.sq.nc, 0, 0};
    return at;
}
// entry (key row kk, value column 0 of the workgroup's slice) of the caller's states [N, HV / nb, KD, nb VD]
template <int KD, int VD>
__device__ __forceinline__ int64_t state_entry(const BwdParams& p, const ScanAt& at, int kk) {
    return ((at.n * (p.HV / p.nb) + at.hg) * KD + kk) * (int64_t)(VD * p.nb) + (at.hv % p.nb) * VD + at.vcol0;
}

template <typename T, bool SEG, bool EXACT, int VBT, int KD, int VD, int FORM, int NW>
__device__ __forceinline__ void bwd_state_body(const BwdParams& p, char* smem, const int tid, const unsigned bid_all, const unsigned nwg) {
    typedef typename Mma<T>::V8 V8;
    typedef typename Mma<T>::V4 V4;
    // NW waves in groups of four: a group takes VBQ of the workgroup's value columns (NB tiles per wave), every wave NA key tiles
    constexpr int PV = VBT + 8, VBQ = VBT / (NW / 4), NB = VBQ / 16, PK = KD + 8, NA = KD / 64, NS = KD / 32, NTH = 64 * NW;
    constexpr bool KDA = FORM == FORM_KDA, GATED = FORM == FORM_GATED, OUT_TILE = state_out_tile<VBT, KD, FORM>();
    T* sK = (T*)smem; T* sW = sK + 64 * PK;                      // (GATED: A in w's place)
    T* sR = sW + (GATED ? 64 * P64 : 64 * PK);                   // (GATED) beta (v - e^gam (k S))
    T* sS = sR + (GATED ? 64 * PV : 0); T* sVn = sS + KD * PV;
    T* sOut = sVn + 64 * PV;                                     // v_new as it is stored (sVn: with the decay to the end of the chunk on it)
    float* sGam = (float*)(sOut + (OUT_TILE ? 64 * PV : 0)); float* sBet = sGam + 64;
    const int lane = tid & 63, w = (tid >> 6) & 3, vq0 = (tid >> 8) * VBQ, c16 = lane & 15, g = lane >> 4;
    int seg;
    const ScanAt at = scan_at<SEG, VBT, VD>(p, bid_all, nwg, lane, seg);
    if (at.out || (at.plan.whole && seg != 0)) return;
    const SeqAt& sq = at.sq;
    const int hv = at.hv, vcol0 = at.vcol0, HVg = p.HV / p.nb;
    const int64_t c_first = at.plan.f0 - at.plan.fw, c_keep = at.plan.f0, c_end = at.plan.f1;     // walks [c_first, c_end), results kept from c_keep on

    f32x4 S[NA][NB];
#pragma unroll
    for (int a2 = 0; a2 < NA; ++a2)
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            const int kk = 16 * (NA * w + a2) + c16;
            S[a2][b] = (p.h0 && c_first == 0) ? *(const f32x4*)(p.h0 + state_entry<KD, VD>(p, at, kk) + vq0 + 16 * b + 4 * g) : ZERO4;
        }
    TileRegs<KD, NTH> rK, rW;
    TileRegs<CH, NTH> rA;
    V4 rU[NB];                                                   // u (GATED: v) of this lane's token
    float rGam = 0.f, rBet = 0.f, rE[NA];
    int rvalid = CH;                                             // the chunk's tokens
    auto fetch = [&](int64_t ic) __attribute__((always_inline)) {
        const int64_t u = (sq.cbase + ic) * p.HV + hv, ug = (sq.cbase + ic) * HVg + at.hg, tok0 = sq.bos + ic * CH;
        const int64_t left = sq.len - ic * CH;
        const int valid = (left >> 6) != 0 ? CH : (int)left, i = 16 * w + c16;
        rvalid = valid;
        if constexpr (KDA) {
            fetch_scan<EXACT, KD, NTH>(rK, (const T*)p.ws.KG + u * 64 * KD, KD, 64, tid);
#pragma unroll
            for (int a2 = 0; a2 < NA; ++a2) rE[a2] = p.ws.EGL[u * KD + 16 * (NA * w + a2) + c16];
        } else {
            fetch_scan<EXACT, KD, NTH>(rK, (const T*)p.k + (tok0 * p.H + at.hq) * KD, (int64_t)p.H * KD, valid, tid);
            if (EXACT || tid < 64) rGam = p.ws.Gam[ug * 64 + lane];
        }
        if constexpr (GATED) {
            fetch_scan<EXACT, CH, NTH>(rA, (const T*)p.ws.Am + ug * 64 * 64, 64, 64, tid);
            if (EXACT || tid < 64) rBet = p.ws.Bet[ug * 64 + lane];
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                if constexpr (!EXACT) rU[b] = V4{(T)0.f, (T)0.f, (T)0.f, (T)0.f};
                if (EXACT || i < valid) rU[b] = *(const V4*)((const T*)p.v + ((tok0 + (EXACT ? min(i, valid - 1) : i)) * p.HV + hv) * VD + vcol0 + vq0 + 16 * b + 4 * g);
            }
        } else {
            fetch_scan<EXACT, KD, NTH>(rW, (const T*)p.ws.Wm + u * 64 * KD, KD, 64, tid);
#pragma unroll
            for (int b = 0; b < NB; ++b) rU[b] = *(const V4*)((const T*)p.ws.Um + (u * 64 + i) * VD + vcol0 + vq0 + 16 * b + 4 * g);
        }
    };
    auto step = [&](int64_t ic) __attribute__((always_inline)) {
        const int64_t u = (sq.cbase + ic) * p.HV + hv;
        const bool keep = !SEG || ic >= c_keep;                 // (chunks of the warm-up belong to another segment: nothing of them is stored)
        const int valid = rvalid;
        if constexpr (EXACT && !KDA) clear_rows<KD, NTH>(rK, valid, tid);
        put_tile<KD, NTH>(sK, PK, rK, tid);
        if constexpr (GATED) put_tile<CH, NTH>(sW, P64, rA, tid);
        else put_tile<KD, NTH>(sW, PK, rW, tid);
        if (tid < 64) { sGam[tid] = rGam; if constexpr (GATED) sBet[tid] = rBet; }
        V4 u4[NB];
#pragma unroll
        for (int b = 0; b < NB; ++b) u4[b] = !EXACT || !GATED || 16 * w + c16 < valid ? rU[b] : V4{(T)0.f, (T)0.f, (T)0.f, (T)0.f};
        float egk[NA];
#pragma unroll
        for (int a2 = 0; a2 < NA; ++a2) egk[a2] = rE[a2];
        T* Hu = (T*)p.ws.Hs + u * KD * VD;
#pragma unroll
        for (int a2 = 0; a2 < NA; ++a2)
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                const int kk = 16 * (NA * w + a2) + c16;
                *(V4*)(sS + kk * PV + vq0 + 16 * b + 4 * g) = pack4<T>(S[a2][b]);
            }
        lds_barrier();
        if (keep) copy_state_out<KD, VBT, VD, NTH>(Hu, vcol0 / 32, sS, PV, tid);
        if (EXACT || ic + 1 < c_end) fetch(ic + 1 < c_end ? ic + 1 : ic);
        const float glast = sGam[63];
        // transposed tiles: value columns on the rows, this wave's 16 tokens on the columns
        const int i = 16 * w + c16;
        const float dec = KDA ? 1.f : __expf(glast - sGam[i]);
        auto leave = [&](int b, f32x4 vn) {
            const V4 vn4 = pack4<T>(vn);
            if constexpr (OUT_TILE) *(V4*)(sOut + i * PV + vq0 + 16 * b + 4 * g) = vn4;
            else if (keep) *(V4*)((T*)p.ws.Vn + (u * 64 + i) * VD + vcol0 + vq0 + 16 * b + 4 * g) = vn4;
#pragma unroll
            for (int r = 0; r < 4; ++r) vn[r] = (float)vn4[r] * dec;
            *(V4*)(sVn + i * PV + vq0 + 16 * b + 4 * g) = pack4<T>(vn);
        };
        {
            const T* rows = GATED ? sK : sW;
            V8 wf[NS];
#pragma unroll
            for (int s = 0; s < NS; ++s) wf[s] = frag_rows(rows, PK, 16 * w, 32 * s, lane);
            const float eg = GATED ? __expf(sGam[i]) : 1.f, bt = GATED ? sBet[i] : 1.f;
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                f32x4 acc = ZERO4;
#pragma unroll
                for (int s = 0; s < NS; ++s) acc = Mma<T>::run(frag_cols(sS, PV, 32 * s, vq0 + 16 * b, lane), wf[s], acc);
                f32x4 x;
#pragma unroll
                for (int r = 0; r < 4; ++r) x[r] = bt * ((float)u4[b][r] - eg * acc[r]);
                if constexpr (GATED) *(V4*)(sR + i * PV + vq0 + 16 * b + 4 * g) = pack4<T>(x);
                else leave(b, x);
            }
        }
        lds_barrier();
        if constexpr (GATED) {
            V8 fa[2];
#pragma unroll
            for (int s = 0; s < 2; ++s) fa[s] = frag_rows(sW, P64, 16 * w, 32 * s, lane);
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                f32x4 acc = ZERO4;
#pragma unroll
                for (int s = 0; s < 2; ++s)
                    if (32 * s <= 16 * w + 15) acc = Mma<T>::run(frag_cols(sR, PV, 32 * s, vq0 + 16 * b, lane), fa[s], acc);     // A[i][j] = 0 for j > i
                leave(b, acc);
            }
            lds_barrier();
        }
        if constexpr (OUT_TILE) { if (keep) copy_rows_out<64, VBT, NTH>((T*)p.ws.Vn + u * 64 * VD + vcol0, VD, sOut, PV, tid); }
        {
            const float eg = __expf(glast);
            V8 kf[NA][2];
#pragma unroll
            for (int a2 = 0; a2 < NA; ++a2)
#pragma unroll
                for (int s = 0; s < 2; ++s) kf[a2][s] = frag_cols(sK, PK, 32 * s, 16 * (NA * w + a2), lane);
#pragma unroll
            for (int a2 = 0; a2 < NA; ++a2)
#pragma unroll
                for (int b = 0; b < NB; ++b) S[a2][b] *= KDA ? egk[a2] : eg;
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    const V8 fv = frag_cols(sVn, PV, 32 * s, vq0 + 16 * b, lane);
#pragma unroll
                    for (int a2 = 0; a2 < NA; ++a2) S[a2][b] = Mma<T>::run(fv, kf[a2][s], S[a2][b]);
                }
        }
        lds_barrier();
    };
    if (c_end > c_first) fetch(c_first);
    if constexpr (EXACT) __builtin_amdgcn_s_waitcnt(0x0f70);    // vmcnt(0): here no stores are younger, and the waits in the loop would allow for that
    for (int64_t ic = c_first; ic < c_end; ++ic) step(ic);
    // (side by side with the reverse scan in one workgroup: as many barriers as the longer of the two takes)
    if constexpr (SEG) for (int64_t i = (c_end - c_first); i < pad_steps_of(at.plan); ++i)
        for (int n = 0; n < (GATED ? 4 : 3); ++n) lds_barrier();
}

template <typename T, bool SEG, bool EXACT, int VBT, int KD, int VD, int FORM, int NW>
__device__ __forceinline__ void bwd_dstate_body(const BwdParams& p, char* smem, const int tid, const unsigned bid_all, const unsigned nwg) {
    typedef typename Mma<T>::V8 V8;
    typedef typename Mma<T>::V4 V4;
    constexpr int PV = VBT + 8, VBQ = VBT / (NW / 4), NB = VBQ / 16, PK = KD + 8, NA = KD / 64, NS = KD / 32, NTH = 64 * NW;
    constexpr bool KDA = FORM == FORM_KDA, GATED = FORM == FORM_GATED;
    T* sK = (T*)smem; T* sQ = sK + 64 * PK; T* sW = sQ + 64 * PK;       // (GATED: A in w's place)
    T* sY = sW + (GATED ? 64 * P64 : 64 * PK);                          // (GATED) -beta e^gam (A^T dv_new)
    T* sP = sY + (GATED ? 64 * PV : 0); T* sDO = sP + 64 * P64; T* sDvn = sDO + 64 * PV; T* sDS = sDvn + 64 * PV;
    float* sGam = (float*)(sDS + KD * PV); float* sBet = sGam + 64;
    const int lane = tid & 63, w = (tid >> 6) & 3, vq0 = (tid >> 8) * VBQ, c16 = lane & 15, g = lane >> 4;
    int seg;
    const ScanAt at = scan_at<SEG, VBT, VD>(p, bid_all, nwg, lane, seg);
    if (at.out || (at.plan.whole && seg != 0)) return;
    const SeqAt& sq = at.sq;
    const int hv = at.hv, vcol0 = at.vcol0, HVg = p.HV / p.nb;
    const int64_t c_lo = at.plan.f0, c_keep = at.plan.f1, c_top = at.plan.f1 + at.plan.rw;       // walks [c_lo, c_top) downwards, results kept below c_keep

    f32x4 dS[NA][NB];
#pragma unroll
    for (int a2 = 0; a2 < NA; ++a2)
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            const int kk = 16 * (NA * w + a2) + c16;
            dS[a2][b] = (p.dht && c_top == sq.nc) ? *(const f32x4*)(p.dht + state_entry<KD, VD>(p, at, kk) + vq0 + 16 * b + 4 * g) : ZERO4;
        }
    // (the rows of q meet the state's gradient as scale e^gam_i q_i: a thread scales its pieces of the tile on their way into LDS, with
    // the gam of their rows fetched beside them)
    constexpr int QN = 64 * (KD / 8) / NTH, QPPR = KD / 8, QRPI = NTH / QPPR;
    TileRegs<KD, NTH> rK, rQ, rW;
    TileRegs<CH, NTH> rA, rP;
    TileRegs<VBT, NTH> rDO;
    float rGam = 0.f, rBet = 0.f, rE[NA], rGq[QN];
    int rvalid = CH;
    auto fetch = [&](int64_t ic) __attribute__((always_inline)) {
        const int64_t u = (sq.cbase + ic) * p.HV + hv, ug = (sq.cbase + ic) * HVg + at.hg, tok0 = sq.bos + ic * CH;
        const int64_t left = sq.len - ic * CH;
        const int valid = (left >> 6) != 0 ? CH : (int)left;
        rvalid = valid;
        if constexpr (KDA) {
            fetch_scan<EXACT, KD, NTH>(rK, (const T*)p.ws.KG + u * 64 * KD, KD, 64, tid);
            fetch_scan<EXACT, KD, NTH>(rQ, (const T*)p.ws.QG + u * 64 * KD, KD, 64, tid);
#pragma unroll
            for (int a2 = 0; a2 < NA; ++a2) rE[a2] = p.ws.EGL[u * KD + 16 * (NA * w + a2) + c16];
        } else {
            fetch_scan<EXACT, KD, NTH>(rK, (const T*)p.k + (tok0 * p.H + at.hq) * KD, (int64_t)p.H * KD, valid, tid);
            fetch_scan<EXACT, KD, NTH>(rQ, (const T*)p.q + (tok0 * p.H + at.hq) * KD, (int64_t)p.H * KD, valid, tid);
            if (EXACT || tid < 64) rGam = p.ws.Gam[ug * 64 + lane];
#pragma unroll
            for (int i = 0; i < QN; ++i) rGq[i] = p.ws.Gam[ug * 64 + tid / QPPR + QRPI * i];
        }
        fetch_scan<EXACT, CH, NTH>(rP, (const T*)(FORM == FORM_COMBA ? p.ws.PT : p.ws.Pm) + ug * 64 * 64, 64, 64, tid);
        if constexpr (GATED) {
            fetch_scan<EXACT, CH, NTH>(rA, (const T*)p.ws.Am + ug * 64 * 64, 64, 64, tid);
            if (EXACT || tid < 64) rBet = p.ws.Bet[ug * 64 + lane];
        } else fetch_scan<EXACT, KD, NTH>(rW, (const T*)p.ws.Wm + u * 64 * KD, KD, 64, tid);
        fetch_scan<EXACT, VBT, NTH>(rDO, (const T*)p.dout + (tok0 * p.HV + hv) * VD + vcol0, (int64_t)p.HV * VD, valid, tid);
    };
    auto step = [&](int64_t ic) __attribute__((always_inline)) {
        const int64_t u = (sq.cbase + ic) * p.HV + hv;
        const bool keep = !SEG || ic < c_keep;                  // (chunks of the warm-up belong to another segment: nothing of them is stored)
        const int valid = rvalid;
        if constexpr (EXACT && !KDA) { clear_rows<KD, NTH>(rK, valid, tid); clear_rows<KD, NTH>(rQ, valid, tid); }
        if constexpr (EXACT) clear_rows<VBT, NTH>(rDO, valid, tid);
        put_tile<KD, NTH>(sK, PK, rK, tid);
        if constexpr (!KDA) {                                   // (KDA: the factors are on the rows of q already)
#pragma unroll
            for (int i = 0; i < QN; ++i) {
                const float f = p.scale * __expf(rGq[i]);
                V8 x = __builtin_bit_cast(V8, rQ.x[i]);
#pragma unroll
                for (int e = 0; e < 8; ++e) x[e] = (T)((float)x[e] * f);
                rQ.x[i] = __builtin_bit_cast(u32x4, x);
            }
        }
        put_tile<KD, NTH>(sQ, PK, rQ, tid);
        if constexpr (GATED) put_tile<CH, NTH>(sW, P64, rA, tid);
        else {
            // (the rows of w change their sign on the way in - one bit per element - so that dv_new can stay in LDS as it is stored)
#pragma unroll
            for (int i = 0; i < (int)(sizeof(rW.x) / sizeof(rW.x[0])); ++i) rW.x[i] ^= u32x4{0x80008000u, 0x80008000u, 0x80008000u, 0x80008000u};
            put_tile<KD, NTH>(sW, PK, rW, tid);
        }
        put_tile<CH, NTH>(sP, P64, rP, tid);
        put_tile<VBT, NTH>(sDO, PV, rDO, tid);
        if (tid < 64) { sGam[tid] = rGam; if constexpr (GATED) sBet[tid] = rBet; }
        float egk[NA];
#pragma unroll
        for (int a2 = 0; a2 < NA; ++a2) egk[a2] = rE[a2];
        T* dHu = (T*)p.ws.dHs + u * KD * VD;
#pragma unroll
        for (int a2 = 0; a2 < NA; ++a2)
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                const int kk = 16 * (NA * w + a2) + c16;
                *(V4*)(sDS + kk * PV + vq0 + 16 * b + 4 * g) = pack4<T>(dS[a2][b]);
            }
        lds_barrier();
        if (keep) copy_state_out<KD, VBT, VD, NTH>(dHu, at.vcol0 / 32, sDS, PV, tid);
        if (EXACT || ic > c_lo) fetch(ic > c_lo ? ic - 1 : ic);
        const float glast = sGam[63];
        const int j = 16 * w + c16;
        {
            // dv_new^T tiles: value columns on the rows, this wave's 16 tokens on the columns
            const float dec = KDA ? 1.f : __expf(glast - sGam[j]);
            V8 kf[NS], pf[2];
#pragma unroll
            for (int s = 0; s < NS; ++s) kf[s] = frag_rows(sK, PK, 16 * w, 32 * s, lane);
#pragma unroll
            for (int s = 0; s < 2; ++s) pf[s] = FORM == FORM_COMBA ? frag_rows(sP, P64, 16 * w, 32 * s, lane) : frag_cols(sP, P64, 32 * s, 16 * w, lane);
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                f32x4 a1 = ZERO4, a2v = ZERO4;
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    if (32 * s + 31 < 16 * w) continue;         // P^T[j][i] = 0 for i < j
                    a1 = Mma<T>::run(frag_cols(sDO, PV, 32 * s, vq0 + 16 * b, lane), pf[s], a1);
                }
#pragma unroll
                for (int s = 0; s < NS; ++s) a2v = Mma<T>::run(frag_cols(sDS, PV, 32 * s, vq0 + 16 * b, lane), kf[s], a2v);
                f32x4 dvn = a1 + a2v * dec;
                *(V4*)(sDvn + j * PV + vq0 + 16 * b + 4 * g) = pack4<T>(dvn);
            }
        }
        lds_barrier();
        if (keep) copy_rows_out<64, VBT, NTH>((T*)p.ws.dVn + u * 64 * VD + vcol0, VD, sDvn, PV, tid);
        if constexpr (GATED) {
            V8 fa[2];
#pragma unroll
            for (int s = 0; s < 2; ++s) fa[s] = frag_cols(sW, P64, 32 * s, 16 * w, lane);
            const float f = -sBet[j] * __expf(sGam[j]);
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                f32x4 acc = ZERO4;
#pragma unroll
                for (int s = 0; s < 2; ++s)
                    if (32 * s + 31 >= 16 * w) acc = Mma<T>::run(frag_cols(sDvn, PV, 32 * s, vq0 + 16 * b, lane), fa[s], acc);     // A[i][j] = 0 for i < j
                *(V4*)(sY + j * PV + vq0 + 16 * b + 4 * g) = pack4<T>(acc * f);
            }
            lds_barrier();
        }
        {
            const float eg = __expf(glast);
            const T* rows = GATED ? sK : sW; const T* cols = GATED ? sY : sDvn;
            V8 qf[NA][2], wf[NA][2];
#pragma unroll
            for (int a2 = 0; a2 < NA; ++a2)
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    qf[a2][s] = frag_cols(sQ, PK, 32 * s, 16 * (NA * w + a2), lane);
                    wf[a2][s] = frag_cols(rows, PK, 32 * s, 16 * (NA * w + a2), lane);
                }
#pragma unroll
            for (int a2 = 0; a2 < NA; ++a2)
#pragma unroll
                for (int b = 0; b < NB; ++b) dS[a2][b] *= KDA ? egk[a2] : eg;
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    const V8 fo = frag_cols(sDO, PV, 32 * s, vq0 + 16 * b, lane), fv = frag_cols(cols, PV, 32 * s, vq0 + 16 * b, lane);
#pragma unroll
                    for (int a2 = 0; a2 < NA; ++a2) {
                        dS[a2][b] = Mma<T>::run(fo, qf[a2][s], dS[a2][b]);
                        dS[a2][b] = Mma<T>::run(fv, wf[a2][s], dS[a2][b]);
                    }
                }
        }
        lds_barrier();
    };
    if (c_top > c_lo) fetch(c_top - 1);
    if constexpr (EXACT) __builtin_amdgcn_s_waitcnt(0x0f70);
    for (int64_t ic = c_top - 1; ic >= c_lo; --ic) step(ic);
    if constexpr (SEG) for (int64_t i = (c_top - c_lo); i < pad_steps_of(at.plan); ++i)
        for (int n = 0; n < (GATED ? 4 : 3); ++n) lds_barrier();
    if (p.dh0 && c_lo == 0) {
#pragma unroll
        for (int a2 = 0; a2 < NA; ++a2)
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                const int kk = 16 * (NA * w + a2) + c16;
                *(f32x4*)(p.dh0 + state_entry<KD, VD>(p, at, kk) + vq0 + 16 * b + 4 * g) = dS[a2][b];
            }
    }
}

// Both scans in one workgroup of eight waves: waves 0-3 walk the chunks forwards (S, v_new), waves 4-7 backwards (dS, dv_new).
// Neither needs anything from the other and both take the same number of barriers per chunk.  What a CU can move per step bounds both,
// so side by side they take little less than one after the other: this form serves time segments, whose workgroups already fill
// every CU (32 value columns per workgroup, up to 128 key features: both sets of LDS tiles fit a CU); whole sequences take
// gdn_bwd_scans_apart_kernel below.
template <int VBT, int KD> constexpr size_t bwd_scans_smem() { return bwd_state_smem<VBT, KD, FORM_GATED>() + bwd_dstate_smem<VBT, KD, FORM_GATED>(); }

template <typename T, int VBT, int KD, int VD>
__global__ __launch_bounds__(512) void gdn_bwd_scans_kernel(BwdParams p) {
    extern __shared__ __align__(16) char smem[];
    static_assert(bwd_state_smem<VBT, KD, FORM_GATED>() % 16 == 0, "the second set of tiles starts 16-byte aligned");
    if (threadIdx.x < 256) bwd_state_body<T, true, false, VBT, KD, VD, FORM_GATED, 4>(p, smem, threadIdx.x, blockIdx.x, gridDim.x);
    else bwd_dstate_body<T, true, false, VBT, KD, VD, FORM_GATED, 4>(p, smem + bwd_state_smem<VBT, KD, FORM_GATED>(), threadIdx.x - 256, blockIdx.x, gridDim.x);
}

// Both scans in one launch, in workgroups of their own: the first `nrev` workgroups walk backwards (the longer steps) over VBR value
// columns each, the others forwards over VBT.  Where the two together need no more workgroups than there are CUs the launch takes the
// time of the longer scan; where they need more, the CUs that one scan's last round would leave idle go on with the other (16000
// packed tokens in 12 sequences, 32 heads: the step 1355 us with one scan after the other, 1245 us with both in a launch, longest
// sequences first).
template <int VBT, int VBR, int KD, int FORM> constexpr size_t bwd_scans_apart_smem() {
    return bwd_state_smem<VBT, KD, FORM>() > bwd_dstate_smem<VBR, KD, FORM>() ? bwd_state_smem<VBT, KD, FORM>() : bwd_dstate_smem<VBR, KD, FORM>();
}
template <typename T, int VBT, int VBR, int KD, int VD, int FORM, bool EXACT>
__global__ __launch_bounds__(64 * scan_waves<VBT>()) void gdn_bwd_scans_apart_kernel(BwdParams p, int64_t nrev) {
    extern __shared__ __align__(16) char smem[];
    static_assert(scan_waves<VBT>() == scan_waves<VBR>(), "workgroups of one size");
    if (blockIdx.x < nrev) bwd_dstate_body<T, false, EXACT, VBR, KD, VD, FORM, scan_waves<VBR>()>(p, smem, threadIdx.x, blockIdx.x, (unsigned)nrev);
    else bwd_state_body<T, false, EXACT, VBT, KD, VD, FORM, scan_waves<VBT>()>(p, smem, threadIdx.x, blockIdx.x - (unsigned)nrev, gridDim.x - (unsigned)nrev);
}

// The chunk-parallel front of the backward pass (included by gdn_chunk_bwd.hip, inside the namespace): one WAVE per (chunk, value head),
// no workgroup barrier.  From q, k, g, beta:
//
//   gam = cumsum(g);  A = (I + diag(beta) stril(k k^T o D))^-1;  P = scale tril(q k^T o D);  D_ij = e^(gam_i - gam_j)
//
// both [64][64] row-major in the operand type; gam and beta as the scans and the last kernel want them (after their activations); a
// bound on the chunk's transition; and with the l2 normalisation of q and k taken in here (L2) the normalised rows and their factors,
// left by the first of the value heads that share them.  The rows are loaded straight into matrix-core operand registers and serve as
// both factors of k k^T; results go from registers to memory, four columns of a row per lane.  P is formed a column of tiles at a time and
// on its way to memory before k k^T is begun, so that the rows of k stay in registers also at 256 features (128 registers, and two of q's
// four row tiles, 64) and need no normalising pass before: memory bounds the kernel, 1.26 GB at 5.2 TB/s there.  Two waves per SIMD: three,
// which 164 registers would let in at 128 features, only push one another's rows out of the caches (122 -> 136 us).
// 16000 packed tokens, 16 q/k and 32 value heads of 128, normalisation inside: 122 us; as four waves per unit with row-major LDS tiles, which also formed
// w = A (beta e^gam k) and u = A (beta v) - 32 KB per unit that the scans now do without - 264 us.
// 8 x 2048 tokens, 32 heads of 256, normalisation inside: 240 us; in two passes over q and k of their own before, whose rows were then
// read 128 features of k and q at a time: 320 us.
constexpr int BP_WAVES = 4;

template <typename T, int KD, bool L2>
__global__ __launch_bounds__(64 * BP_WAVES) __attribute__((amdgpu_waves_per_eu(2, 2))) void gdn_bwd_prepare_kernel(BwdParams p, int64_t units) {
    typedef typename Mma<T>::V8 V8;
    typedef typename Mma<T>::V4 V4;
    constexpr int NS = KD / 32;                                      // operands of 32 features per row tile
    constexpr int QT = KD <= 128 ? 4 : 2;                            // q's row tiles in registers at a time
    __shared__ __align__(16) float smem[BP_WAVES * PW_FLOATS];
    const int tid = threadIdx.x, lane = tid & 63, c16 = lane & 15, g = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int64_t u = (int64_t)blockIdx.x * BP_WAVES + w;            // (chunk, value head), heads fastest
    if (u >= units) return;
    float* tiles = smem + w * PW_FLOATS;
    float* sLd = tiles;                                              // [4][16 i][16 j] diagonal blocks of L, by rows
    float* sG = tiles + 1024; float* sBeta = sG + 64; float* sK2 = tiles + 4 * 16 * TP;
    auto lds_sync = [] { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); };

    const uint32_t HVg = (uint32_t)(p.HV / p.nb), ch = (uint32_t)u / HVg;
    const int hv = (int)((uint32_t)u - ch * HVg), G = (int)HVg / p.H, hq = hv / G;
    const ChunkAt c = chunk_at(p, ch);
    uint32_t rg = 0, rb = 0;
    if (lane < c.valid) {
        rg = p.g ? load_scalar_bits(p.g, (c.tok0 + lane) * HVg + hv, p.gb_dtype) : 0;
        rb = load_scalar_bits(p.beta, (c.tok0 + lane) * HVg + hv, p.beta_dtype);
    }
    const int64_t row0 = (c.tok0 * p.H + hq) * KD;
    const T* kg = (const T*)(L2 ? p.k_raw : p.k) + row0;
    const T* qg = (const T*)(L2 ? p.q_raw : p.q) + row0;
    // one 32-bit offset per lane (its row of a tile, its 8 features of 32); tile and block select a wave-uniform base
    const uint32_t lane_off = ((uint32_t)c16 * (uint32_t)(p.H * KD) + 8u * g) * (uint32_t)sizeof(T);
    auto fragment = [&](const T* rows, int t, int col0) {
        const char* bp = (const char*)(rows + (int64_t)(16 * t) * p.H * KD + col0);
        if (c.valid == CH || 16 * t + c16 < c.valid) return *(const u32x4*)(bp + lane_off);
        return u32x4{0u, 0u, 0u, 0u};
    };
    // the rows of a tile divided by their lengths, rounded as gdn_l2norm_fwd does it (the sum over a row's four lanes)
    auto unit_rows = [&](u32x4 (&f)[NS]) {
        float ss = 0.f;
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            const V8 x = __builtin_bit_cast(V8, f[s]);
#pragma unroll
            for (int e = 0; e < 8; ++e) ss += (float)x[e] * (float)x[e];
        }
        const float r = rsqrtf(sum_over_g(ss) + 1e-6f);
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            if constexpr (std::is_same<T, f16_t>::value) asm volatile("" : "+v"(f[s]));      // (or the sum's 32-bit values are kept till here)
            V8 x = __builtin_bit_cast(V8, f[s]);
#pragma unroll
            for (int e = 0; e < 8; ++e) x[e] = (T)((float)x[e] * r);
            f[s] = __builtin_bit_cast(u32x4, x);
        }
        return r;
    };
    // row tile t normalised; the first of the value heads that share the rows leaves them, with their factors
    auto normalise = [&](u32x4 (&f)[NS], int t, const void* rows, const float* factors) {
        const float n = unit_rows(f);
        if (hq * G == hv && 16 * t + c16 < c.valid) {
            char* bp = (char*)((T*)rows + row0 + (int64_t)(16 * t) * p.H * KD);
#pragma unroll
            for (int s = 0; s < NS; ++s) *(u32x4*)(bp + lane_off + 64 * s) = f[s];
            if (g == 0) ((float*)factors)[(c.tok0 + 16 * t + c16) * p.H + hq] = n;
        }
        __builtin_amdgcn_sched_barrier(0);                               // (one tile's values in 32 bits at a time)
    };
    u32x4 fk[4][NS], fq[QT][NS];
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int s = 0; s < NS; ++s) fk[t][s] = fragment(kg, t, 32 * s);
#pragma unroll
    for (int t = 0; t < QT; ++t)
#pragma unroll
        for (int s = 0; s < NS; ++s) fq[t][s] = fragment(qg, t, 32 * s);
    __builtin_amdgcn_sched_barrier(0);
    float x = scalar_of_bits(rg, p.gb_dtype), beta = scalar_of_bits(rb, p.beta_dtype);
    if (lane < c.valid) {
        if (p.A_log && p.g) x = -__expf(p.A_log[hv]) * softplus_f(x + (p.dt_bias ? p.dt_bias[hv] : 0.f));
        if (p.flags & GDN_FLAG_BETA_SIGMOID) beta = sigmoid_f(beta) * ((p.flags & GDN_FLAG_NEG_EIGVAL) ? 2.f : 1.f);
    }
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const float y = __shfl_up(x, off, 64);
        if (lane >= off) x += y;
    }
    sG[lane] = x * RCP_LN2_F;
    sBeta[lane] = beta;
    p.ws.Gam[u * 64 + lane] = x;
    p.ws.Bet[u * 64 + lane] = beta;
    lds_sync();
    if constexpr (L2) {
#pragma unroll
        for (int t = 0; t < 4; ++t) normalise(fk[t], t, p.k, p.k_rstd);
    }
    // P, then L: transposed tiles (rows: key tokens j, column: token i).  P's first, a column of tiles at a time, and on its way to memory
    // before L's are begun: either alone leaves room for the rows.
    // (select, never multiply by a mask: e^(gam_i - gam_j) may overflow for i < j)
    auto decay = [&](int a, int b, int r, int first, float gi, const f32x4& gj) {
        return a < b || c16 >= 4 * g + r + first ? fast_exp2(gi - gj[r]) : 0.f;
    };
    T* Pu = (T*)p.ws.Pm + u * 64 * 64;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
        if constexpr (L2) normalise(fq[b % QT], b, p.q, p.q_rstd);
        f32x4 QK[4];
#pragma unroll
        for (int a = 0; a < 4; ++a) QK[a] = ZERO4;
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            const V8 q8 = __builtin_bit_cast(V8, fq[b % QT][s]);
#pragma unroll
            for (int a = 0; a <= b; ++a) QK[a] = Mma<T>::run(__builtin_bit_cast(V8, fk[a][s]), q8, QK[a]);
        }
        if (b + QT < 4) {
#pragma unroll
            for (int s = 0; s < NS; ++s) fq[b % QT][s] = fragment(qg, b + QT, 32 * s);
        }
        const int i = 16 * b + c16;
        const float gi = sG[i];
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            f32x4 pt = ZERO4;
            if (a <= b) {
                const f32x4 gj = *(const f32x4*)(sG + 16 * a + 4 * g);
#pragma unroll
                for (int r = 0; r < 4; ++r) pt[r] = p.scale * QK[a][r] * decay(a, b, r, 0, gi, gj);
            }
            *(V4*)(Pu + i * 64 + 16 * a + 4 * g) = pack4<T>(pt);
        }
    }
    f32x4 U[4][4];
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int a = 0; a <= b; ++a) {
            U[a][b] = ZERO4;
#pragma unroll
            for (int s = 0; s < NS; ++s) U[a][b] = Mma<T>::run(__builtin_bit_cast(V8, fk[a][s]), __builtin_bit_cast(V8, fk[b][s]), U[a][b]);
        }
    // |k_t|^2 is the diagonal of k k^T
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        float d = 0.f;
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (r == (c16 & 3)) d = U[t][t][r];
        if ((c16 >> 2) == g) sK2[16 * t + c16] = d;
    }
    lds_sync();
    {
        // how much this chunk's transition can stretch a state, in log2 units: every token's factor gamma_t (I - beta_t k_t k_t^T)
        float lb = fabsf(1.f - beta * sK2[lane]);
        lb = lb > 1.f ? __log2f(lb) : 0.f;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) lb += __shfl_xor(lb, off, 64);
        if (lane == 63) p.ws.Bound[u] = x * RCP_LN2_F + lb;
    }
#pragma unroll
    for (int b = 0; b < 4; ++b) {
        const float gi = sG[16 * b + c16], bi = sBeta[16 * b + c16];
#pragma unroll
        for (int a = 0; a <= b; ++a) {
            const f32x4 gj = *(const f32x4*)(sG + 16 * a + 4 * g);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float d = decay(a, b, r, 1, gi, gj);
                U[a][b][r] = a < b || c16 > 4 * g + r ? bi * U[a][b][r] * d : 0.f;
            }
        }
    }
#pragma unroll
    for (int a = 0; a < 4; ++a) *(f32x4*)(sLd + a * 256 + c16 * 16 + 4 * g) = U[a][a];       // L[i = c16][j = 4g + r]
    lds_sync();
    f32x4 X[4][4];
    inverse_transposed(tiles, U, X, c16, g);
    T* Au = (T*)p.ws.Am + u * 64 * 64;
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int a = 0; a < 4; ++a) *(V4*)(Au + (16 * b + c16) * 64 + 16 * a + 4 * g) = a <= b ? pack4<T>(X[a][b]) : V4{(T)0.f, (T)0.f, (T)0.f, (T)0.f};
}

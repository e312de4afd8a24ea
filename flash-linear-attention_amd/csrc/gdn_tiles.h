// Building blocks of the chunk kernels that keep their operands as row-major LDS tiles (the backward pass of the gated delta
// rule, the chunked KDA forward): where a chunk lies in a packed batch, tiles on their way from global memory through
// registers into LDS, matrix-core operand fragments read from such tiles, small cross-lane sums.
// A product's two operands have the same register layout (lane (c16, g) holds index c16 and the 8 contraction indices
// 8g .. 8g+7 of a 32-wide step), so there are just two ways to fetch an operand fragment from a row-major tile: `frag_rows`
// (the contraction runs along a row: one 16-byte read) and `frag_cols` (the contraction runs down a column: two transposing
// LDS reads).  The result of run(a, b) holds, in lane (c16, g), column c16 (b's index) and rows 4g .. 4g+3 (a's index).
#pragma once
#include "gdn_chunk_common.h"

namespace gdn {

constexpr int BD = 128;              // value columns of these kernels; key features: KD = 128 KT with KT = 1 or 2 (a template argument)
constexpr int P128 = BD + 8;         // LDS pitch, in elements, of a [64][128] tile ([64][KD] tiles: KD + 8)
constexpr int P64 = CH + 8;          // ... of a [64][64] tile
constexpr int PL = CH + 4;           // pitch of the fp32 matrix L


// Params types used with chunk_at / seq_at carry: cu_seqlens, chunk_table, chunk_offsets, flags, T, NT.
// ---- geometry ------------------------------------------------------------------------------
struct ChunkAt { int64_t tok0; int valid; };
template <typename P>
__device__ __forceinline__ ChunkAt chunk_at(const P& p, int64_t ci) {
    const bool cu32 = p.flags & GDN_FLAG_CU_INT32;
    if (p.cu_seqlens) {
        const int64_t n = load_index_uniform(p.chunk_table, 2 * ci, cu32), it = load_index_uniform(p.chunk_table, 2 * ci + 1, cu32);
        const int64_t bos = load_index_uniform(p.cu_seqlens, n, cu32), eos = load_index_uniform(p.cu_seqlens, n + 1, cu32);
        const int64_t t0 = bos + it * CH;
        return ChunkAt{t0, (int)min((int64_t)CH, eos - t0)};
    }
    // (32-bit: the entries refuse calls with 2^31 chunks or more, and a 64-bit division costs some hundred instructions)
    const uint32_t b = (uint32_t)ci / (uint32_t)p.NT, it = (uint32_t)ci - b * (uint32_t)p.NT;
    return ChunkAt{(int64_t)b * p.T + (int64_t)it * CH, (int)min((int64_t)CH, p.T - (int64_t)it * CH)};
}
// Unit u = chunk * HV + v-head of the kernels that walk over the units: its v-head, q/k head and chunk.  (32-bit arithmetic,
// as above: these kernels are bound by the rate at which one or two waves per SIMD issue instructions.)
struct UnitAt { int hv, hq; ChunkAt c; };
template <typename P>
__device__ __forceinline__ UnitAt unit_at(const P& p, int64_t u) {
    const uint32_t HV = (uint32_t)p.HV, ch = (uint32_t)u / HV, hv = (uint32_t)u - ch * HV, G = HV / (uint32_t)p.H;
    return UnitAt{(int)hv, (int)(G == 1 ? hv : hv / G), chunk_at(p, ch)};
}
struct SeqAt { int64_t bos, len, cbase, nc; };
template <typename P>
__device__ __forceinline__ SeqAt seq_at(const P& p, int64_t n) {
    const bool cu32 = p.flags & GDN_FLAG_CU_INT32;
    SeqAt s;
    if (p.cu_seqlens) {
        s.bos = load_index_uniform(p.cu_seqlens, n, cu32);
        s.len = load_index_uniform(p.cu_seqlens, n + 1, cu32) - s.bos;
        s.cbase = load_index_uniform(p.chunk_offsets, n, cu32);
    } else {
        s.bos = n * p.T; s.len = p.T; s.cbase = n * p.NT;
    }
    s.nc = (s.len + CH - 1) / CH;
    return s;
}

// ---- tiles ---------------------------------------------------------------------------------
// 64 rows of NCOLS elements from global memory (row r at g + r * stride; rows from `valid` on read as zero) into a
// row-major LDS tile, by all 256 threads.  Loads first, stores after: the loads of one tile are in flight together.
template <int NCOLS, typename T>
__device__ __forceinline__ void load_tile(T* s, int pitch, const T* g, int64_t stride, int valid, int tid) {
    constexpr int PPR = NCOLS / 8, TOTAL = 64 * PPR, N = (TOTAL + 255) / 256;
    u32x4 x[N];
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const int idx = tid + 256 * i, row = idx / PPR, pc = idx % PPR;
        x[i] = u32x4{0u, 0u, 0u, 0u};
        if (idx < TOTAL && row < valid) x[i] = *(const u32x4*)(g + row * stride + pc * 8);
    }
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const int idx = tid + 256 * i, row = idx / PPR, pc = idx % PPR;
        if (idx < TOTAL) *(u32x4*)(s + row * pitch + pc * 8) = x[i];
    }
}

// The same in two halves, for loops that fetch the next tile while they work on the current one.
template <int NCOLS, int NTH = 256>
struct TileRegs { u32x4 x[64 * (NCOLS / 8) >= NTH ? 64 * (NCOLS / 8) / NTH : 1]; };
template <int NCOLS, int NTH = 256, typename T>
__device__ __forceinline__ void fetch_tile(TileRegs<NCOLS, NTH>& r, const T* g, int64_t stride, int valid, int tid) {
    constexpr int PPR = NCOLS / 8, TOTAL = 64 * PPR, N = TOTAL >= NTH ? TOTAL / NTH : 1, RPI = NTH / PPR;      // a thread's pieces lie RPI rows apart
    static_assert(TOTAL % NTH == 0 || TOTAL < NTH, "whole rounds of the workgroup's threads, or less than one");
    const int row0 = tid / PPR, pc = tid % PPR;
    const char* at = (const char*)(g + (int64_t)row0 * stride + pc * 8);
    const int64_t step = (int64_t)RPI * stride * (int64_t)sizeof(T);
    if (valid >= 64 && TOTAL >= NTH) {                          // (the same for the whole workgroup) full chunk: plain loads
#pragma unroll
        for (int i = 0; i < N; ++i) r.x[i] = *(const u32x4*)(at + i * step);
    } else {
#pragma unroll
        for (int i = 0; i < N; ++i) {
            r.x[i] = u32x4{0u, 0u, 0u, 0u};
            if (row0 + RPI * i < valid && tid < TOTAL) r.x[i] = *(const u32x4*)(at + i * step);
        }
    }
}
// The same for loops that keep stores in flight behind the next tile's loads: as many loads whatever `valid` (1 or more) is - behind a branch or a mask that leaves
// some out the compiler no longer knows how many accesses are younger and waits for all of them.  Past the end they repeat the last row; cleared on their way to LDS.
template <int NCOLS, int NTH, typename T>
__device__ __forceinline__ void fetch_rows(TileRegs<NCOLS, NTH>& r, const T* g, int64_t stride, int valid, int tid) {
    constexpr int PPR = NCOLS / 8, N = 64 * PPR / NTH, RPI = NTH / PPR;
    static_assert(64 * PPR % NTH == 0, "whole rounds of the workgroup's threads");
    const int row0 = tid / PPR;
    const char* at = (const char*)(g + (int64_t)row0 * stride + tid % PPR * 8);
    const int64_t step = (int64_t)RPI * stride * (int64_t)sizeof(T);
    if (valid >= 64) {
#pragma unroll
        for (int i = 0; i < N; ++i) r.x[i] = *(const u32x4*)(at + i * step);
    } else {
#pragma unroll
        for (int i = 0; i < N; ++i) r.x[i] = *(const u32x4*)(at + (int64_t)min(RPI * i, valid - 1 - row0) * stride * (int64_t)sizeof(T));
    }
}
template <int NCOLS, int NTH>
__device__ __forceinline__ void clear_rows(TileRegs<NCOLS, NTH>& r, int valid, int tid) {
    constexpr int PPR = NCOLS / 8, N = sizeof(r.x) / sizeof(r.x[0]), RPI = NTH / PPR;
    if (valid >= 64) return;
#pragma unroll
    for (int i = 0; i < N; ++i)
        if (tid / PPR + RPI * i >= valid) r.x[i] = u32x4{0u, 0u, 0u, 0u};
}
template <int NCOLS, int NTH = 256, typename T>
__device__ __forceinline__ void put_tile(T* s, int pitch, const TileRegs<NCOLS, NTH>& r, int tid) {
    constexpr int PPR = NCOLS / 8, TOTAL = 64 * PPR, N = TOTAL >= NTH ? TOTAL / NTH : 1, RPI = NTH / PPR;
    T* at = s + (tid / PPR) * pitch + (tid % PPR) * 8;
    if (TOTAL < NTH && tid >= TOTAL) return;
#pragma unroll
    for (int i = 0; i < N; ++i) *(u32x4*)(at + i * RPI * pitch) = r.x[i];
}
// ROWS rows of NCOLS elements of an LDS tile out to global memory (row r at g + r * stride), 16 bytes a lane along the rows:
// whole cache lines per group of lanes, where the lanes that hold a result as matrix-instruction output would write 8-byte pieces.
// (`valid`: rows from there on are left alone)
template <int ROWS, int NCOLS, int NTH, typename T>
__device__ __forceinline__ void copy_rows_out(T* g, int64_t stride, const T* s, int pitch, int tid, int valid = ROWS) {
    constexpr int PPR = NCOLS / 8, TOTAL = ROWS * PPR, N = TOTAL / NTH;
    static_assert(TOTAL % NTH == 0, "whole rounds of the workgroup's threads");
    u32x4 x[N];
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const int idx = tid + NTH * i;
        x[i] = *(const u32x4*)(s + (idx / PPR) * pitch + (idx % PPR) * 8);
    }
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const int idx = tid + NTH * i;
        if (valid >= ROWS || idx / PPR < valid) *(u32x4*)(g + (int64_t)(idx / PPR) * stride + (idx % PPR) * 8) = x[i];
    }
}
// A state in the workspace lies as the operand fragments that its readers take from it: 16 key features (tile a) x 32 of VD value columns (step s) after one
// another, in them 16 bytes a lane - key 16a + c16, value columns 32s + 8g .. +7.  A wave's load is 1 KB in a row (from rows of VD elements its lanes would go
// to sixteen rows, which the memory pipeline takes one lane at a time).  Step of 8 x 2048 tokens, 32 heads of 256: 3255 -> 3225 us; 16000 packed tokens, 32 heads
// of 128: 1081 -> 1074; 8 x 1024 tokens, 8 heads of 64: 120.8 -> 119.5.
template <int VD> __device__ __forceinline__ int state_frag(int a, int s, int lane) { return ((a * (VD / 32) + s) * 64 + lane) * 8; }
// ... and out of a row-major LDS tile of KD rows of NCOLS of the value columns, from step s0 on
template <int KD, int NCOLS, int VD, int NTH, typename T>
__device__ __forceinline__ void copy_state_out(T* g, int s0, const T* t, int pitch, int tid) {
    constexpr int SN = NCOLS / 32, N = KD * NCOLS / 8 / NTH;
    static_assert(N * NTH * 8 == KD * NCOLS, "whole rounds of the workgroup's threads");
    const int lane = tid & 63, w = tid >> 6;
    u32x4 x[N];
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const int f = w + NTH / 64 * i;
        x[i] = *(const u32x4*)(t + (16 * (f / SN) + (lane & 15)) * pitch + 32 * (f % SN) + 8 * (lane >> 4));
    }
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const int f = w + NTH / 64 * i;
        *(u32x4*)(g + state_frag<VD>(f / SN, s0 + f % SN, lane)) = x[i];
    }
}
// operand fragment whose contraction runs along a row: index r0 + c16, contraction c0 + 8g + e
template <typename T>
__device__ __forceinline__ typename Mma<T>::V8 frag_rows(const T* s, int pitch, int r0, int c0, int lane) {
    return *(const typename Mma<T>::V8*)(s + (r0 + (lane & 15)) * pitch + c0 + 8 * (lane >> 4));
}
// operand fragment whose contraction runs down a column: index c0 + c16, contraction r0 + 8g + e
template <typename T>
__device__ __forceinline__ typename Mma<T>::V8 frag_cols(const T* s, int pitch, int r0, int c0, int lane) {
    const int a = lane & 15;
    const T* at = s + (r0 + 8 * (lane >> 4) + (a >> 2)) * pitch + c0 + 4 * (a & 3);
    return join<typename Mma<T>::V8>(Mma<T>::tr_read(at), Mma<T>::tr_read(at + 4 * pitch));
}
// ... of 16 rows and columns: column c0 + c16, rows r0 + 4g + e
template <typename T>
__device__ __forceinline__ typename Mma<T>::V4 tile_cols(const T* s, int pitch, int r0, int c0, int lane) {
    const int a = lane & 15;
    return Mma<T>::tr_read(s + (r0 + 4 * (lane >> 4) + (a >> 2)) * pitch + c0 + 4 * (a & 3));
}
// ---- tiles in blocks -----------------------------------------------------------------------
// 64 rows of COLS elements without padding: blocks of four rows, in a block groups of sixteen 16-byte slots, group n the pieces (8 elements) 4n .. 4n+3 of its
// rows; piece c of row 4j + r in slot 4r + ((c & 3) ^ block_flip(j)) of its group.  A CU's LDS serves 256 bytes a cycle: of a 16-byte read the lanes {0-3, 12-15,
// 20-27} and {4-11, 16-19, 28-31} of each half wave together, of an 8-byte read (transposing or not) a half wave, of a store sixteen lanes.  block_flip puts
// what each of them meets on different banks: block_rows, block_cols and 8-byte accesses to (16t + c16, 4g).  (Rows padded by 16 bytes, as in the tiles above,
// put two rows of an operand read on a bank: 8.1 cycles an instruction, here 4.2; block_cols 2.5 each, there 4.2.)  Unlike pieces that trade places
// over a whole row, tiles and steps of a product are constants in the address.
__device__ __forceinline__ constexpr int block_flip(int j) { return (4 - j) & 3; }
// The address of an access is the tile, constants (or scalars) for where in it, and a lane's share in bytes that is the same for all tiles of a width: the caller
// computes it once and keeps it (`opaque`: the compiler would take it apart and add it up again at every access).  Odd 16-column tiles lie 32 bytes apart: the share ^ 32.
__device__ __forceinline__ int opaque(int x) { asm volatile("" : "+v"(x)); return x; }
template <int COLS> __device__ __forceinline__ constexpr int block_off(int r0, int c0) { return (r0 * COLS + (c0 >> 5) * 128) * 2; }      // r0, c0: multiples of 16
// element (r, c) of a 16 x 16 tile
template <int COLS> __device__ __forceinline__ constexpr int block_lane(int r, int c) {
    return ((r & ~3) * COLS + 32 * (r & 3) + (((c >> 3) ^ block_flip((r >> 2) & 3)) << 3) + (c & 7)) * 2;
}
// as frag_rows and frag_cols: the shares of lane (c16, g), then the reads
template <int COLS> __device__ __forceinline__ int block_rows_lane(int lane) {
    return ((lane & 12) * COLS + 32 * (lane & 3) + 8 * ((lane >> 4) ^ block_flip((lane >> 2) & 3))) * 2;
}
template <int COLS, typename T>
__device__ __forceinline__ typename Mma<T>::V8 block_rows(const T* s, int r0, int c0, int share) {
    return *(const typename Mma<T>::V8*)((const char*)s + block_off<COLS>(r0, c0) + share);
}
struct ColsLane { int a, b; };                                  // of the two transposing reads (of an even 16-column tile)
template <int COLS> __device__ __forceinline__ ColsLane block_cols_lane(int lane) {
    const int a = lane & 15, g = lane >> 4, x = ((a >> 1) & 1) ^ (2 * (g & 1)), at = 8 * g * COLS + 32 * (a >> 2) + 4 * (a & 1);
    return ColsLane{(at + 8 * x) * 2, (at + 4 * COLS + 8 * (x ^ 3)) * 2};
}
template <int COLS, typename T>
__device__ __forceinline__ typename Mma<T>::V8 block_cols(const T* s, int r0, int c0, ColsLane share) {
    const char* at = (const char*)s + block_off<COLS>(r0, c0);
    return join<typename Mma<T>::V8>(Mma<T>::tr_read((const T*)(at + share.a)), Mma<T>::tr_read((const T*)(at + share.b)));
}
__device__ __forceinline__ ColsLane odd_tile(ColsLane x) { return ColsLane{x.a ^ 32, x.b ^ 32}; }
// as fetch_tile and put_tile: a thread's pieces are those of the slots tid, tid + NTH, ..., four lanes on 64 bytes of a row
// (rows from `valid` on are fetched from the last valid one, and zeros by the time they are put)
template <int NCOLS, int NTH, typename T>
__device__ __forceinline__ void fetch_blocks(TileRegs<NCOLS, NTH>& r, const T* g, int64_t stride, int valid, int tid) {
    constexpr int SLOTS = NCOLS / 2, N = 64 * NCOLS / 8 / NTH, RPI = NTH / SLOTS * 4;      // a thread's pieces lie RPI rows apart
    static_assert(N >= 1 && N * NTH * 8 == 64 * NCOLS && RPI % 16 == 0, "whole rounds of the workgroup's threads");
    const int row0 = 4 * (tid / SLOTS) + ((tid >> 2) & 3), pc = 4 * ((tid % SLOTS) >> 4) + ((tid & 3) ^ block_flip((tid / SLOTS) & 3));
#pragma unroll
    for (int i = 0; i < N; ++i) r.x[i] = *(const u32x4*)((const char*)g + ((uint32_t)min(row0 + RPI * i, valid - 1) * (uint32_t)(stride * sizeof(T)) + (uint32_t)(pc * 16)));
}
template <int NCOLS, int NTH, typename T>
__device__ __forceinline__ void put_blocks(T* s, const TileRegs<NCOLS, NTH>& r, int valid, int tid) {
    constexpr int SLOTS = NCOLS / 2, N = 64 * NCOLS / 8 / NTH, RPI = NTH / SLOTS * 4;
    const int row0 = 4 * (tid / SLOTS) + ((tid >> 2) & 3);
#pragma unroll
    for (int i = 0; i < N; ++i) {
        u32x4 x = r.x[i];
        if (valid < 64) { if (row0 + RPI * i >= valid) x = u32x4{0u, 0u, 0u, 0u}; }
        *(u32x4*)(s + (tid + NTH * i) * 8) = x;
    }
}
// The same straight into the LDS, without registers: issued here, landed when the issuing waves have waited for their vector-memory operations
// (wait_vm_at_most) and met at a barrier.  Rows from `valid` on are zeros.  Nobody may still read the tile.
template <int NCOLS, int NW, typename T>
__device__ __forceinline__ void copy_blocks(T* s, const T* g, int64_t stride, int valid, int w, int lane) {
    constexpr int SLOTS = NCOLS / 2, N = NCOLS / 8 / NW;
    static_assert(N * NW * 8 == NCOLS && SLOTS <= 64, "whole rounds of the workgroup's waves, a block or two each");
    const uint32_t lds = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)s;
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const int k = w + NW * i, b = k * (64 / SLOTS) + lane / SLOTS, row = 4 * b + ((lane >> 2) & 3), pc = 4 * ((lane % SLOTS) >> 4) + ((lane & 3) ^ block_flip(b & 3));
        const uint32_t voff = (uint32_t)row * (uint32_t)(stride * sizeof(T)) + 16 * pc;
        if (valid >= 64) gather_1k_to_lds((const char*)g, voff, lds + k * 1024);
        else {
            gather_1k_to_lds_masked((const char*)g, voff, lds + k * 1024, __builtin_amdgcn_ballot_w64(row < valid));
            if (row >= valid) *(u32x4*)(s + (k * 64 + lane) * 8) = u32x4{0u, 0u, 0u, 0u};
        }
    }
}
template <typename T>
__device__ __forceinline__ typename Mma<T>::V4 pack4(f32x4 x) {
    return typename Mma<T>::V4{(T)x[0], (T)x[1], (T)x[2], (T)x[3]};
}
// Sums across lanes without LDS traffic (a ds_bpermute each, some hundred cycles apart, bounded the kernels that walk over units):
// rows of 16 lanes trade places with v_permlane16_swap / v_permlane32_swap (which need two wait states after the write of their
// operands), lanes inside a row with DPP.
__device__ __forceinline__ float sum_over_g(float x) {          // over the four lanes that share c16
    float y = x;
    asm("s_nop 1\n\tv_permlane16_swap_b32 %0, %1" : "+v"(x), "+v"(y));
    x += y;
    y = x;
    asm("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(x), "+v"(y));
    return x + y;
}
template <int CTRL> __device__ __forceinline__ float add_dpp(float x) {
    return x + __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xF, 0xF, true));
}
__device__ __forceinline__ float sum_over_c16(float x) {        // over the sixteen lanes that share g
    x = add_dpp<0xB1>(x);                                       // quad_perm [1,0,3,2]
    x = add_dpp<0x4E>(x);                                       // quad_perm [2,3,0,1]
    x = add_dpp<0x141>(x);                                      // row_half_mirror: the other quad of the eight
    return add_dpp<0x140>(x);                                   // row_mirror: the other eight
}
// x summed over the four lanes of a quad (lanes 4n .. 4n+3), in every one of them
__device__ __forceinline__ float sum_over_quad(float x) { return add_dpp<0x4E>(add_dpp<0xB1>(x)); }
#define ZERO4 (f32x4{0.f, 0.f, 0.f, 0.f})


// A = (I + L)^-1 for a strictly lower triangular 64 x 64 L, by forward substitution in fp32:
// A[i][c] = [i == c] - sum_{j < i} L[i][j] A[j][c].  Four waves, wave w the columns 16w .. 16w+15: a quad of lanes per
// column c, lane gq of the quad keeps A[j][c] for j = gq mod 4 and adds up its part of the sum.  sL holds entry (i, j)
// at [i][j % 4][j / 4] (pitch PL; zeros from the diagonal on within the 16 x 16 diagonal blocks); A goes to sA (pitch
// P64) in the operand type.  The caller's barriers separate it from the writers of sL and the readers of sA.
template <typename T>
__device__ __forceinline__ void solve_unit_lower(const float* sL, T* sA, int w, int lane) {
    const int c = 16 * w + (lane >> 2), gq = lane & 3;
    float a[16];
#pragma unroll
    for (int m = 0; m < 16; ++m) a[m] = 0.f;
#pragma unroll
    for (int i = 0; i < 64; ++i) {
        float part0 = 0.f, part1 = 0.f;
#pragma unroll
        for (int m4 = 0; 16 * m4 < i; ++m4) {                   // entries j = 4m + gq < i; those from i on are stored as zeros
            const f32x4 l = *(const f32x4*)(sL + i * PL + gq * 16 + 4 * m4);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if (4 * (4 * m4 + e) < i) {
                    if (e & 1) part1 += l[e] * a[4 * m4 + e];
                    else part0 += l[e] * a[4 * m4 + e];
                }
            }
        }
        const float ai = (i == c ? 1.f : 0.f) - sum_over_quad(part0 + part1);
        if (gq == (i & 3)) { a[i >> 2] = ai; sA[i * P64 + c] = (T)ai; }
    }
}

// The same inverse by blocks of 16, for the same four waves (all of them must call it: it holds two barriers).  Wave a first
// inverts the diagonal block a on its own (X_a (I + L_aa) = I by rows from the right: lane c16 owns row c16, 16 short steps
// without any exchange between lanes) and leaves X_a in LDS; then wave b computes block column b of A from
//     A_bb = X_b,   A_ab = -X_a sum_{b <= m < a} L_am A_mb   (a > b)
// on the matrix cores in fp32 (v_mfma_f32_16x16x4_f32): the left factors L_am and X_a come from LDS, the right factors are
// the blocks just computed, which an accumulator holds in the layout a right factor needs.  64 dependent steps become 16
// plus at most nine 16 x 16 products.  sX: 1024 floats of scratch, which may be the memory of sA itself.
template <typename T>
__device__ __forceinline__ void solve_unit_lower_blocks(const float* sL, float* sX, T* sA, int w, int lane) {
    const int c16 = lane & 15, g = lane >> 4;
    {
        float x[16], acc[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[i] = 0.f;
#pragma unroll
        for (int i = 15; i >= 0; --i) {
            x[i] = ((i == c16) ? 1.f : 0.f) - acc[i];
            // row i of the diagonal block: entry j = 4q + e at [e][4w + q]
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if (e >= i) continue;
                const f32x4 l = *(const f32x4*)(sL + (16 * w + i) * PL + e * 16 + 4 * w);
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    if (4 * q + e < i) acc[4 * q + e] += l[q] * x[i];
            }
        }
        if (g == 0) {
#pragma unroll
            for (int q = 0; q < 4; ++q) *(f32x4*)(sX + w * 256 + c16 * 16 + 4 * q) = f32x4{x[4 * q], x[4 * q + 1], x[4 * q + 2], x[4 * q + 3]};
        }
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    f32x4 A[4];
#pragma unroll
    for (int a = 0; a < 4; ++a) {
        A[a] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (a < w) continue;
        if (a == w) {
            const float* t = sX + a * 256;
            A[a] = f32x4{t[(4 * g) * 16 + c16], t[(4 * g + 1) * 16 + c16], t[(4 * g + 2) * 16 + c16], t[(4 * g + 3) * 16 + c16]};
            continue;
        }
        f32x4 t = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int m = 0; m < a; ++m) {
            if (m < w) continue;
            // left factor L_am by rows: entry (16a + c16, 16m + 4g + e) at [e][4m + g]
#pragma unroll
            for (int e = 0; e < 4; ++e)
                t = __builtin_amdgcn_mfma_f32_16x16x4f32(sL[(16 * a + c16) * PL + e * 16 + 4 * m + g], A[m][e], t, 0, 0, 0);
        }
        const f32x4 xa = *(const f32x4*)(sX + a * 256 + c16 * 16 + 4 * g);
        f32x4 r = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int e = 0; e < 4; ++e) r = __builtin_amdgcn_mfma_f32_16x16x4f32(xa[e], t[e], r, 0, 0, 0);
        A[a] = -r;
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");     // (every wave has read the X tiles: sA may take their place)
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int r = 0; r < 4; ++r) sA[(16 * a + 4 * g + r) * P64 + 16 * w + c16] = (T)A[a][r];
}

}  // namespace gdn

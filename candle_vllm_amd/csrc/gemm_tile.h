// The main loop of the 16-bit prompt products (y = x W^T, x [T][K] and W [N][K] both k-contiguous): one workgroup of eight waves makes a
// tile of BM tokens x BN weight rows.  Used by dense_gemv.hip (16-bit checkpoints) and hybrid_kernels.hip (layer-list models).
//
//   * K in units of 64: a unit's rows are 128 B, i.e. whole cache lines, and go global -> LDS by DMA (`global_load_lds_dwordx4`, asm: hipcc
//     would drain a DMA it can see at every barrier).  S buffers; ONE barrier per unit, in its middle: by then every wave has the
//     fragments of the unit's second half in registers, so the buffer is free for unit u + S, and unit u + 1 -- requested S - 1 units
//     earlier, a unit being 64 MFMAs of each of a SIMD's two waves at 256 x 256: 2048 cycles -- has landed.
//   * The fragments of the next half unit are read from LDS while the current half is multiplied (two register sets), so neither the
//     LDS nor the barrier stands between two MFMAs of a wave.
//   * x and row-major W: LDS rows of 128 B, the 16-byte chunk c of row r at chunk c ^ (r & 7) (the swizzle is applied to the lane's SOURCE
//     address; the DMA destination is lane-linear): fragment reads are free of bank conflicts.  Tiled W (dense_tile_index): its 1 KiB
//     fragments are copied verbatim and read lane-linear.
//   * Operand order of the MFMA: weights first, so a lane ends with FOUR CONSECUTIVE output columns of one token (one 8- or 16-byte store)
//     instead of four tokens of one column.
// What bounds it: the matrix cores and their power; LDS reads are 12 KiB per 32 MFMAs of a wave (three quarters of the LDS' rate at
// 256 x 256, all of it at 128 x 128 tiles), which is why the large tile is preferred wherever its last round is not too empty.
#pragma once
#include "common.h"

typedef _Float16 gt_f16x8_t __attribute__((ext_vector_type(8)));

template <int DT>
__device__ __forceinline__ f32x4_t gt_mfma(const uint4& a, const uint4& b, const f32x4_t& c) {
    if constexpr (DT == MI355_DTYPE_BF16)
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(gt_f16x8_t, a), __builtin_bit_cast(gt_f16x8_t, b), c, 0, 0, 0);
}

// one KiB global -> LDS: lane l's 16 bytes at base + off land at dst + 16 l
__device__ __forceinline__ void gt_dma(const uint8_t* base, uint32_t off, uint32_t dst) {
    uint32_t keep;
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %3\n\ts_mov_b32 m0, %0"
                 : "=&s"(keep) : "s"(dst), "v"(off), "s"(base) : "memory");
}

// the same from 64-bit addresses
__device__ __forceinline__ void gt_dma(const uint8_t* src, uint32_t dst) {
    uint32_t keep;
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, off\n\ts_mov_b32 m0, %0"
                 : "=&s"(keep) : "s"(dst), "v"(src) : "memory");
}

// a value every lane holds alike, in scalar registers (what the compiler works out through a division is in vector registers)
__device__ __forceinline__ const uint8_t* gt_uniform(const uint8_t* p) {
    const uint64_t v = (uint64_t)(uintptr_t)p;
    return reinterpret_cast<const uint8_t*>((uintptr_t)((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v) |
                                                        (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(v >> 32)) << 32));
}

// Workgroups go to the eight XCDs in turn: give every XCD a contiguous run of tiles, token tiles fastest inside groups of at most six, so
// that the 32 workgroups of an XCD share about six token tiles and five weight tiles through its L2.
struct GtPlace { int m, n; };
__device__ __forceinline__ GtPlace gt_place(int id, int n_m, int n_n) {
    const int total = n_m * n_n, xcd = id & 7, q = total >> 3, r = total & 7;
    const int t = xcd * q + (xcd < r ? xcd : r) + (id >> 3);
    const int groups = (n_m + 5) / 6, gm = (n_m + groups - 1) / groups;
    const int g = t / (gm * n_n), left = n_m - g * gm, here = left < gm ? left : gm, w = t - g * gm * n_n;
    return {__builtin_amdgcn_readfirstlane(g * gm + w % here), __builtin_amdgcn_readfirstlane(w / here)};
}

template <int DT, int WM, int WN, int MF, int NF, int S, bool TILED>
struct GemmTile {
    static_assert(WM * WN == 8, "eight waves");
    static constexpr int BM = WM * MF * 16, BN = WN * NF * 16, THREADS = 512;
    static constexpr uint32_t A_BYTES = BM * 128u, STAGE = (BM + BN) * 128u, LDS = S * STAGE;
    static constexpr int AR = BM / 64, BR = BN / 64;                  // DMA instructions per wave and unit

    struct Frags { uint4 a[MF], b[NF]; };
    f32x4_t acc[MF][NF];
    const uint8_t* smem;
    uint32_t lds0;
    int wave, lane, wm, wn;
    uint32_t a_rd, b_rd;                                              // this lane's fragment address of half 0 (half 1: ^ 64 / + 1024)

    __device__ __forceinline__ GemmTile(uint8_t* s) : smem(s) {
        lane = threadIdx.x & 63;
        wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
        wm = wave / WN; wn = wave % WN;
        lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(size_t)(__attribute__((address_space(3))) void*)s);
        const int m16 = lane & 15, kg = lane >> 4;
        a_rd = (uint32_t)(wm * MF * 16 + m16) * 128u + (uint32_t)((kg ^ (m16 & 7)) * 16);
        b_rd = A_BYTES + (TILED ? (uint32_t)(wn * NF) * 2048u + (uint32_t)lane * 16u
                                : (uint32_t)(wn * NF * 16 + m16) * 128u + (uint32_t)((kg ^ (m16 & 7)) * 16));
    }
    // row of the tile (0 .. BM or BN) that this lane stages with DMA instruction r, and the 16-byte chunk of it
    __device__ __forceinline__ int stage_row(int r) const { return 8 * (wave + 8 * r) + (lane >> 3); }
    __device__ __forceinline__ uint32_t stage_chunk() const { return (uint32_t)(((lane & 7) ^ (lane >> 3)) * 16); }
    // tiled weights: row tile (0 .. BN / 16) and fragment (0, 1) of this wave's DMA instruction r
    __device__ __forceinline__ int stage_tile(int r) const { return (wave + 8 * r) >> 1; }
    __device__ __forceinline__ int stage_frag() const { return wave & 1; }

    // fragment n of a half unit in the order the products want them: all of b, then a
    __device__ __forceinline__ void read(Frags& f, uint32_t buf, int half, int n) const {
        if (n < NF) f.b[n] = *reinterpret_cast<const uint4*>(smem + buf + (TILED ? b_rd + (half ? 1024u : 0u) : (b_rd ^ (half ? 64u : 0u))) + (size_t)n * 2048);
        else f.a[n - NF] = *reinterpret_cast<const uint4*>(smem + buf + (a_rd ^ (half ? 64u : 0u)) + (size_t)(n - NF) * 2048);
    }
    // a_base + a_off[r]: source of DMA instruction r in unit 0 (units are 128 B apart); b_base[r] + b_off[r] likewise, b_step bytes apart.
    // Offsets of 64 bits: rows gathered from anywhere
    template <class AOff>
    __device__ __forceinline__ void run(const uint8_t* a_src, const AOff (&a_off)[AR], const uint8_t* const (&b_src)[BR],
                                        const uint32_t (&b_off)[BR], uint32_t b_step, int units) {
        const uint8_t* a_base = gt_uniform(a_src);
        const uint8_t* b_base[BR];
#pragma unroll
        for (int r = 0; r < BR; ++r) b_base[r] = gt_uniform(b_src[r]);
#pragma unroll
        for (int i = 0; i < MF; ++i)
#pragma unroll
            for (int j = 0; j < NF; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        auto dma = [&](int u, uint32_t buf, int n) {                      // instruction n of unit u into the buffer at `buf`
            const uint32_t dst = lds0 + buf + (uint32_t)wave * 1024u;
            if (n < BR) gt_dma(b_base[n] + (size_t)u * b_step, b_off[n], dst + A_BYTES + (uint32_t)n * 8192u);
            else if constexpr (sizeof(AOff) == 8) gt_dma(a_base + (size_t)u * 128 + a_off[n - BR], dst + (uint32_t)(n - BR) * 8192u);
            else gt_dma(a_base + (size_t)u * 128, a_off[n - BR], dst + (uint32_t)(n - BR) * 8192u);
        };
        Frags f0, f1;
        // one half unit: MF steps of NF products; the reads of the next half (and the DMA of unit `fill`) are spread over the first steps.
        // Left alone, hipcc sinks every read to just above its product and the two register sets become one
        constexpr int RS = (MF + NF + MF - 2) / (MF - 1), DS = (AR + BR + MF - 1) / MF;   // reads, DMA instructions per step
        auto half = [&](const Frags& f, Frags& nf, uint32_t rbuf, int rhalf, bool rd, int fill, uint32_t fbuf) {
#pragma unroll
            for (int i = 0; i < MF; ++i) {
                if (fill >= 0) {
#pragma unroll
                    for (int n = i * DS; n < (i + 1) * DS; ++n) if (n < AR + BR) dma(fill, fbuf, n);
                }
                if (rd) {
#pragma unroll
                    for (int n = i * RS; n < (i + 1) * RS; ++n) if (n < MF + NF) read(nf, rbuf, rhalf, n);
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int j = 0; j < NF; ++j) acc[i][j] = gt_mfma<DT>(f.b[j], f.a[i], acc[i][j]);
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        // at unit u's barrier units u + 1 .. u + S - 1 are under way and u + 1 has to have landed; behind it this buffer takes unit u + S
        uint32_t buf = 0;
        auto unit = [&](int u, bool refill, bool next) {
            const uint32_t after = buf + STAGE == LDS ? 0u : buf + STAGE;
            half(f0, f1, buf, 1, true, -1, 0);
            if (refill) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" :: "n"((S - 2) * (AR + BR)) : "memory");
            else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");   // the last units: nothing younger is under way
            __builtin_amdgcn_s_barrier();                                  // everyone's share landed, everyone's reads of this buffer are done
            asm volatile("" ::: "memory");
            half(f1, f0, after, 0, next, refill ? u + S : -1, buf);
            buf = after;
        };
#pragma unroll
        for (int n = 0; n < AR + BR; ++n) dma(0, 0, n);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(0xC07F);                               // lgkmcnt(0), as hipcc counts: no scalar load is pending in the loop, its LDS waits stay exact
#pragma unroll
        for (int v = 1; v < S; ++v)
            if (v < units) {
#pragma unroll
                for (int n = 0; n < AR + BR; ++n) dma(v, v * STAGE, n);
            }
#pragma unroll
        for (int n = 0; n < MF + NF; ++n) read(f0, 0, 0, n);
        int u = 0;
        for (; u + S < units; ++u) unit(u, true, true);
        for (; u + 1 < units; ++u) unit(u, false, true);
        unit(u, false, false);
    }
    // output column of acc[i][j][v] inside the tile is col(j) + v, its token row(i)
    __device__ __forceinline__ int row(int i) const { return wm * MF * 16 + i * 16 + (lane & 15); }
    __device__ __forceinline__ int col(int j) const { return wn * NF * 16 + j * 16 + 4 * (lane >> 4); }
};

// ---- which tile.  us: a unit of 64 k of one round (per_cu workgroups on every CU); the launch takes the tile and K split whose rounds end
// first, never below the time of the weights' stream from HBM.  The 64- and 128-token tiles of one workgroup per CU have six and four
// buffers: where a launch is a stream over the weights, what counts is the bytes under way.
// 192 x 128 is for the launches whose 128 x 128 tiles are a little more than one per CU, which 256 x 256 ones leave half empty.  us, two 128 x 128
// per CU / one 192 x 128 (f32 results): 2100 x 2048 x 2048 29.3 / 25.3, x 6144 73.8 / 59.2; 1100 x 4096 x 4096 50.1 / 44.4; 300 x 14336 x 4096 64.9 / 49.0;
// where its second round is not full the pick stays: 1100 x 9216 x 2048 192 x 256 44.4 / 50.9, 1100 x 14336 x 4096 135.5 / 144.2.  From 16 units (k >= 1024) on:
// below, a launch is mostly its start and its stores (2100 x 2048 x 128 9.3 / 8.5, x 704 15.7 / 13.2).  256 x 128 as a seventh tile won nowhere by more than 2 %.
// With K in ranges (16-bit results, us, without it / with it): in place of 256 x 256 tiles 933 x 2784 x 8448 61.7 / 53.3 (sixteen such sizes 0.83 .. 0.91 of the time); of the other
// two-buffered ones up to four row tiles, 162 x 4272 x 8192 34.3 / 26.9, 373 x 3712 x 11264 46.5 / 42.1 (60 sizes 0.78 .. 0.99), and not beyond (1418 x 768 x 10496 42.4 / 38.8, but
// 1094 x 1216 x 5888 31.4 / 34.5: 0.87 .. 1.10); never in place of tiles 3 and 4, whose rounds the sum below makes look 1 .. 5 % longer than its short ranges and which
// are faster (185 x 6864 x 3072 16.8 / 22.9, 903 x 1136 x 7936 29.3 / 34.6, 960 x 2848 x 6400 40.9 / 45.6: 24 sizes 1.02 .. 1.37).
struct GtTile { int bm, bn, per_cu; float us; };
constexpr int GT_NARROW = 5;
static constexpr GtTile kGtTiles[] = {{256, 256, 1, 1.46f}, {192, 256, 1, 1.28f}, {128, 128, 2, 0.93f}, {128, 128, 1, 0.5f}, {64, 128, 1, 0.42f}, {192, 128, 1, 0.72f}};
// CALL with the six tiles' template arguments, by number
#define GT_TILES(which, CALL) do { switch (which) { \
    case 0: CALL(2, 4, 8, 4, 2); break; case 1: CALL(2, 4, 6, 4, 2); break; case 2: CALL(2, 4, 4, 2, 2); break; \
    case 3: CALL(2, 4, 4, 2, 4); break; case 4: CALL(2, 4, 2, 2, 6); break; default: CALL(4, 2, 3, 4, 4); break; } } while (0)
struct GtChoice { int tile, splits; float us; };
// tile and K ranges of this thread's last launch, 100 tile + ranges (tests: mi355_internal_last_gemm)
inline thread_local int gt_last_launch = -1;
// tiles(t): workgroups of the launch with tile t; stream_us: the weights' read; part_us: write or read of one range's partial sums
template <class F>
static inline GtChoice gt_pick(F tiles, int units, float stream_us, int max_split, float part_us, unsigned allowed, const GtTile* table = kGtTiles, int n_table = 6) {
    const int cus = mi355_num_cus();
    GtChoice best{-1, 1, 0.f};
    auto consider = [&](int i, int most) {
        if (!(allowed >> i & 1)) return;
        for (int s = 1; s <= most; ++s) {
            const int64_t wgs = (int64_t)cus * table[i].per_cu, rounds = (tiles(table[i]) * s + wgs - 1) / wgs;
            const float t = (float)rounds * (float)((units + s - 1) / s + 2) * table[i].us;
            const float c = (t > stream_us ? t : stream_us) + (s > 1 ? 5.f + part_us * (float)(s + 1) : 0.f);
            if (best.tile < 0 || c < best.us) best = {i, s, c};
        }
    };
    for (int i = 0; i < n_table; ++i) if (i != GT_NARROW) consider(i, max_split);
    if (n_table > GT_NARROW && units >= 16) {
        const bool ranges = best.tile == 0 || (best.tile > 0 && best.tile < 3 && tiles(GtTile{table[GT_NARROW].bm, 1 << 30, 1, 0.f}) <= 4);
        consider(GT_NARROW, ranges ? max_split : 1);
    }
    return best;
}

// Skinny (decode-shaped) linear layers on the reference's NATIVE weight layouts, for the safetensors path:
//   K10  dense 16-bit   `Linear::forward`  y = x.W^T (+b)        src/openai/models/linear.rs:124-172
//   K12  marlin_4bit_{bf16,f16}            y = x.(s*(q-8))       src/backend/gptq.rs:132-178
//   K13  marlin_awq_4bit_*                 y = x.(s*(q-z))       src/backend/gptq.rs:116-131,148-162
//   K14  gemm_half_q_half_alt (f16, act-order g_idx)             src/backend/gptq.rs:181-197
//   K15  gptq_repack / awq_repack                                src/backend/gptq.rs:313-332
// Decode is an HBM stream of the weights (2 B resp. ~0.53 B per weight, each read once); MFMA does the
// contraction with the tokens on the M rows (16 tokens per M tile; activations are exactly 16-bit so no hi/lo
// split is needed).  No LDS staging: weight fragments come straight from global memory in fragment order
// (a 16x16x32 B-fragment is 8 consecutive k of one output row = 16 B of a dense row, or ONE u32 of a GPTQ
// k-packed column), activation fragments straight from L2.
//
// Our packed 4-bit layout IS the GPTQ checkpoint layout qweight[k/8][n] (bits 4i.. = code of k = 8*row+i):
// `gptq_repack` is therefore a copy and `awq_repack` is the only real transform (AWQ packs along n with the
// interleave [0,2,4,6,1,3,5,7]).  Scales (and AWQ zero points) arrive Marlin-permuted from the reference's host
// code (`marlin_permute_scales`, linear.rs:341-379; examples/convert_awq_marlin.py:72-115) and are un-permuted
// by index arithmetic here.
#include "common.h"
#include "scratch.h"
#include "gemm_tile.h"
#include "../../include/mi355_vllm.h"
#include <hip/hip_runtime.h>
#include <algorithm>
#include <utility>

typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef unsigned int dg_u32x4 __attribute__((ext_vector_type(4)));

// DW_GPTQ4: checkpoint layout qweight[k/8][n] u32.  DW_GPTQ4T: the same words in 16-column x 256-k tiles (gptq_tile_index below):
// one wave's share of a k-block is two contiguous 1 KiB runs (two dwordx4 loads per lane) instead of eight loads that each
// touch four 64-byte segments a row apart -- what gptq_repack / awq_repack / mi355_marlin_format_repack produce at load time.
enum { DW_DENSE = 0, DW_GPTQ4 = 1, DW_GPTQ4T = 2 };
// word index of qweight[kr][n] (kr = k/8) in the tiled image: [tile n/16][k-block kr/32][half][lane = 16*(kr%4) + n%16][4]
// holding rows kr = 32 kb + 4 (4 half + jj) + lane/16 -- the fragment order of dense_body's 4-bit arm
__host__ __device__ __forceinline__ size_t gptq_tile_index(int kr, int n, int nkb) {
    const int kb = kr >> 5, rem = kr & 31, j = rem >> 2, kg = rem & 3;
    return ((((size_t)(n >> 4) * nkb + kb) * 2 + (j >> 2)) * 64 + kg * 16 + (n & 15)) * 4 + (j & 3);
}
// 16-bit weights [N][K] in the same 16-row x 256-k tiles (element index): [tile n/16][k-block k/256][j = (k%256)/32][lane = 16*((k%32)/8) + n%16][k%8]
// -- fragment j of a (tile, k-block) is 1 KiB contiguous, the whole (tile, k-block) 8 KiB; a row-major row tile is sixteen 512-byte
// pieces 2 K bytes apart, and a wave instruction touches 16 rows x 64 B of it (measured: 3.9 TB/s at best from that pattern)
__host__ __device__ __forceinline__ size_t dense_tile_index(int n, int k, int nkb) {
    const int kb = k >> 8, kk = k & 255, j = kk >> 5, kg = (kk & 31) >> 3, e = kk & 7;
    return (((((size_t)(n >> 4) * nkb + kb) * 8 + j) * 64 + kg * 16 + (n & 15)) << 3) + e;
}
enum { SP_NONE = 0, SP_GROUPED = 1, SP_SINGLE = 2 };

// attention.rs:644-719 after the projections: q,k -> f32 -> rope -> model dtype, then the cache write of k and v
struct DenseRope {
    const float* cos_t; const float* sin_t;         // [max_seq][head_dim / 2] f32
    const int64_t* positions; const int64_t* slots; // [T]
    uint16_t* kcache; uint16_t* vcache;             // this layer's bf16 cache
    int32_t n_kv_heads, head_dim, block_size, flash;
};
struct DenseArgs {
    const void* w;            // DENSE: 16-bit [N][ldw] (wtiled: the 16 x 256 tile image, dense_tile_index) ; GPTQ4: u32 [K/8][N]
    int32_t ldw;
    int32_t wtiled;           // DENSE only: 1 = w is the tiled image (N % 16 == 0, K % 256 == 0; ldw unused)
    const void* scales;       // GPTQ4: 16-bit [K/g][N]
    const uint32_t* qzeros;   // packed zero points [K/g][N/8] or null
    int32_t zmode, sperm;     // MI355_ZERO_* ; SP_*
    int32_t group_size;       // resolved: multiple of 32, <= K
    const void* x;            // 16-bit [T][ldx]
    int32_t ldx, T, N, K;
    void* out;                // 16-bit [T][ldo]
    int32_t ldo;
    const void* bias;         // 16-bit [N] or null
    const void* resid;        // 16-bit [T][ldo] (EPI_RESID)
    int32_t epi;              // MI355_EPI_STORE / RESID / SILU_MUL
    int32_t pair_offset;      // SILU_MUL: rows of `up` start at pair_offset (packed gate_up weight, mlp.rs:324-352)
    const void* norm_w;       // dense_small_kernel only: RmsNorm weight [K] (bf16) applied to x while it is staged, or null
    float norm_eps;
    const float* ss_in;       // with norm_w: [T][K/16] partial sums of squares of x's rows, left by the launch that produced x
    // dense_small3r_kernel only (q / k / v of a decode step): RoPE and the KV-cache write in the projection's epilogue
    int32_t rope_mode;        // 0 none; 1 = q (rotate, store); 2 = k (rotate, store, write the key cache); 3 = v (store, write the value cache)
    float* ss_out;            // dense_small_kernel only: where this launch leaves [T][ldo/16] partial sums of squares of its output
    struct DenseNormTail* tail;   // host only: the RmsNorm that reads this product's output, or null
};
// out [T][N] = RmsNorm(the product's output) * w, bf16; done: the launch made it (only split sums do, resid_norm_tail)
struct DenseNormTail { void* out; const void* w; float eps; bool done; };

template <int DT> __device__ __forceinline__ float h2f(uint16_t h) {
    return DT == MI355_DTYPE_BF16 ? bf16_to_f32(h) : f16_bits_to_f32(h);
}
template <int DT> __device__ __forceinline__ uint16_t f2h(float f) {
    return DT == MI355_DTYPE_BF16 ? f32_to_bf16(f) : f32_to_f16_bits(f);
}
template <int DT> __device__ __forceinline__ float rnd(float f) { return h2f<DT>(f2h<DT>(f)); }

template <int DT>
__device__ __forceinline__ f32x4_t mfma32(const uint4& a, const uint4& b, const f32x4_t& c) {
    if constexpr (DT == MI355_DTYPE_BF16)
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
}

// position of natural column n inside a Marlin-permuted row (inverse of linear.rs:341-379)
//   grouped: new[64c + 8i + j] = old[64c + i + 8j]
//   single : new[32c + 8i + jj] = old[32c + 2i + {0,1,8,9,16,17,24,25}[jj]]
__host__ __device__ __forceinline__ int marlin_scale_pos(int n, int sperm) {
    if (sperm == SP_GROUPED) {
        const int c = n & 63;
        return (n & ~63) + 8 * (c & 7) + (c >> 3);
    }
    if (sperm == SP_SINGLE) {
        const int c = n & 31;
        return (n & ~31) + 8 * ((c >> 1) & 3) + 2 * (c >> 3) + (c & 1);
    }
    return n;
}

__device__ __forceinline__ float zero_point(const DenseArgs& a, int g, int col) {
    if (a.zmode == MI355_ZERO_SYM8 || !a.qzeros) return 8.f;
    if (a.zmode == MI355_ZERO_GPTQ_PLUS1)   // AutoGPTQ v1: stored zero = z - 1, nibble n%8 of qzeros[g][n/8]
        return (float)(((a.qzeros[(size_t)g * (a.N / 8) + col / 8] >> (4 * (col & 7))) & 0xF) + 1);
    // marlin zero points (convert_awq_marlin.py:72-91): scale_perm, then interleave [0,2,4,6,1,3,5,7], then pack
    const int p1 = marlin_scale_pos(col, SP_GROUPED);
    const int u = p1 & 7;
    const int t = ((u & 1) << 2) | (u >> 1);            // argsort([0,2,4,6,1,3,5,7]) = [0,4,1,5,2,6,3,7]
    const int p2 = (p1 & ~7) + t;
    return (float)((a.qzeros[(size_t)g * (a.N / 8) + p2 / 8] >> (4 * (p2 & 7))) & 0xF);
}

// the rounding chain of one output element: y (and the `up` value u of a gate/up pair) -> the model dtype
template <int DT>
__device__ __forceinline__ float dense_epilogue(const DenseArgs& a, const int m, const int row, const float y, const float up) {
    const uint16_t* b16 = static_cast<const uint16_t*>(a.bias);
    // candle rounds the matmul result to the model dtype, then the bias add rounds again (linear.rs:124-172)
    float o = rnd<DT>(y);
    if (b16) o = rnd<DT>(o + h2f<DT>(b16[row]));
    if (a.epi == MI355_EPI_SILU_MUL) {
        float u = rnd<DT>(up);
        if (b16) u = rnd<DT>(u + h2f<DT>(b16[a.pair_offset + row]));
        o = rnd<DT>(rnd<DT>(o / (1.f + __expf(-o))) * u);               // silu(gate) * up (mlp.rs:457)
    } else if (a.epi == MI355_EPI_RESID) {
        o = rnd<DT>(o + h2f<DT>(static_cast<const uint16_t*>(a.resid)[(size_t)m * a.ldo + row]));
    }
    static_cast<uint16_t*>(a.out)[(size_t)m * a.ldo + row] = f2h<DT>(o);
    return o;
}

// One workgroup = R row tiles (R = 2 for the packed gate/up pair) x all of K; the waves split the 256-wide
// k-blocks; MT = ceil(T/16) M tiles.  GJ (4-bit only) = 32-wide k runs per quantisation group inside a k-block
// (group 32/64/128/>=256 -> 1/2/4/8): the MFMA chain runs over a whole group and the scale is applied once.
// rp (dense3r_kernel: q / k / v of a decode step of 5..32 tokens): RoPE and the cache write in the epilogue; q and k then run as row-tile
// PAIRS (j, j + D/2) of one head, as in dense_small_body
template <int DT, int WTYPE, int MT, int R, int GJ>
__device__ __forceinline__ void dense_body(const DenseArgs& a, const int bx, const DenseRope* rp = nullptr) {
    extern __shared__ __attribute__((aligned(16))) float dg_red[];   // [NW][R][MT][16 m][16 rows]
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, NW = blockDim.x >> 6;
    const int r16 = lane & 15, kg = lane >> 4;
    const int nkb = a.K >> 8;
    int row0[R];
    row0[0] = bx * 16;
    if (R == 2) row0[R - 1] = a.pair_offset + bx * 16;
    if (R == 2 && rp) {                                            // RoPE pairs: rows (h, j) and (h, j + D/2) of one head
        const int tph = rp->head_dim >> 5;                         // 16-row pair tiles per head
        row0[0] = (bx / tph) * rp->head_dim + (bx % tph) * 16;
        row0[R - 1] = row0[0] + (rp->head_dim >> 1);
    }
    const uint16_t* x16 = static_cast<const uint16_t*>(a.x);

    f32x4_t y[R][MT];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) y[r][mt] = f32x4_t{0.f, 0.f, 0.f, 0.f};

    // (tried in round 3 for the few-tile 16-bit launches of a batch-32 step: the next k-block's weights and activations requested
    // before the current one is multiplied, two register sets -- 215 VGPRs, wo / down 25.3 -> 28.2 us, q|k|v 22.3 -> 25.5: slower)
    for (int kb = wave; kb < nkb; kb += NW) {
        // ---- all loads of this k-block first: 8 weight fragments per tile, 8 activation fragments per M tile
        uint4 bw[R][8];
        uint4 aw[MT][8];
        if constexpr (WTYPE == DW_DENSE) {
#pragma unroll
            for (int r = 0; r < R; ++r) {
                // row-major: row r16 of the tile, 32 j + 8 kg inside the k-block; tiled: fragment j is 64 lanes x 16 B contiguous
                const uint16_t* wp = a.wtiled ? static_cast<const uint16_t*>(a.w) + ((((size_t)(row0[r] >> 4) * nkb + kb) * 8) * 64 + lane) * 8
                                              : static_cast<const uint16_t*>(a.w) + (size_t)(row0[r] + r16) * a.ldw + (size_t)kb * 256 + 8 * kg;
                const int jstride = a.wtiled ? 512 : 32;
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const dg_u32x4 v = __builtin_nontemporal_load(reinterpret_cast<const dg_u32x4*>(wp + (size_t)j * jstride));
                    bw[r][j] = make_uint4(v.x, v.y, v.z, v.w);
                }
            }
        } else {
#pragma unroll
            for (int r = 0; r < R; ++r) {
                if constexpr (WTYPE == DW_GPTQ4T) {
                    const dg_u32x4* tp = reinterpret_cast<const dg_u32x4*>(a.w) + ((size_t)(row0[r] >> 4) * nkb + kb) * 128 + lane;
                    const dg_u32x4 v0 = __builtin_nontemporal_load(tp), v1 = __builtin_nontemporal_load(tp + 64);
                    bw[r][0].x = v0.x; bw[r][1].x = v0.y; bw[r][2].x = v0.z; bw[r][3].x = v0.w;
                    bw[r][4].x = v1.x; bw[r][5].x = v1.y; bw[r][6].x = v1.z; bw[r][7].x = v1.w;
                } else {
                    const uint32_t* qp = static_cast<const uint32_t*>(a.w) + (size_t)(kb * 32 + kg) * a.N + row0[r] + r16;
#pragma unroll
                    for (int j = 0; j < 8; ++j) bw[r][j].x = __builtin_nontemporal_load(qp + (size_t)(4 * j) * a.N);
                }
            }
        }
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            const int m = min(mt * 16 + r16, a.T - 1);
            const uint16_t* xp = x16 + (size_t)m * a.ldx + (size_t)kb * 256 + 8 * kg;
#pragma unroll
            for (int j = 0; j < 8; ++j) aw[mt][j] = *reinterpret_cast<const uint4*>(xp + 32 * j);
        }
        // ---- contraction
        // (the machine scheduler otherwise sinks every load to just above its MFMA to save registers -- 48-60 VGPRs, eight dependent
        // memory round trips per k-block instead of one; Llama-3-8B bf16 at batch 32: wo 13.2 -> 12.9 us, down 43.9 -> 40.5)
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (WTYPE == DW_DENSE) {
#pragma unroll
            for (int r = 0; r < R; ++r)
#pragma unroll
                for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                    for (int j = 0; j < 8; ++j) y[r][mt] = mfma32<DT>(aw[mt][j], bw[r][j], y[r][mt]);
        } else {
            // 128+q (bf16) / 1024+q (f16): OR the 4-bit code into the mantissa of a constant; code pairs
            // (n_i, n_{i+4}) give the element order {0,4,1,5,2,6,3,7} -> permute the activations to match.
            constexpr uint32_t KOFF = (DT == MI355_DTYPE_BF16) ? 0x43004300u : 0x64006400u;
            constexpr float OFF = (DT == MI355_DTYPE_BF16) ? 128.f : 1024.f;
            constexpr uint32_t ONE2 = (DT == MI355_DTYPE_BF16) ? 0x3F803F80u : 0x3C003C00u;
            uint32_t nib = 0x000F000Fu;
            asm volatile("" : "+v"(nib));
            const uint4 ones = make_uint4(ONE2, ONE2, ONE2, ONE2);
            const f32x4_t zero4 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const uint4 v = aw[mt][j];        // v.x=(x0,x1) v.y=(x2,x3) v.z=(x4,x5) v.w=(x6,x7)
                    aw[mt][j].x = __builtin_amdgcn_perm(v.z, v.x, 0x05040100u);   // (x0, x4)
                    aw[mt][j].y = __builtin_amdgcn_perm(v.z, v.x, 0x07060302u);   // (x1, x5)
                    aw[mt][j].z = __builtin_amdgcn_perm(v.w, v.y, 0x05040100u);   // (x2, x6)
                    aw[mt][j].w = __builtin_amdgcn_perm(v.w, v.y, 0x07060302u);   // (x3, x7)
                }
#pragma unroll
            for (int gq = 0; gq < 8 / GJ; ++gq) {
                // groups of 32 / 64 / 128 are exactly GJ runs wide: no run-time division in the loop (GJ == 8: groups of >= 256)
                const int g = GJ < 8 ? kb * (8 / GJ) + gq : (kb * 256) / a.group_size;
                // row sums of x over the group (every column of a ones-MFMA result holds it)
                f32x4_t xs[MT];
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) {
                    xs[mt] = zero4;
#pragma unroll
                    for (int jj = 0; jj < GJ; ++jj) xs[mt] = mfma32<DT>(aw[mt][gq * GJ + jj], ones, xs[mt]);
                }
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const int col = row0[r] + r16;
                    const float s = h2f<DT>(static_cast<const uint16_t*>(a.scales)[(size_t)g * a.N + marlin_scale_pos(col, a.sperm)]);
                    const float c = -(OFF + zero_point(a, g, col)) * s;
                    f32x4_t acc[MT];
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt) acc[mt] = zero4;
#pragma unroll
                    for (int jj = 0; jj < GJ; ++jj) {
                        const uint32_t w = bw[r][gq * GJ + jj].x;
                        uint4 b;
                        b.x = (w & nib) | KOFF;
                        b.y = ((w >> 4) & nib) | KOFF;
                        b.z = ((w >> 8) & nib) | KOFF;
                        b.w = ((w >> 12) & nib) | KOFF;
#pragma unroll
                        for (int mt = 0; mt < MT; ++mt) acc[mt] = mfma32<DT>(aw[mt][gq * GJ + jj], b, acc[mt]);
                    }
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                        for (int v = 0; v < 4; ++v) y[r][mt][v] = fmaf(s, acc[mt][v], fmaf(c, xs[mt][v], y[r][mt][v]));   // (explicit: the same association in every instantiation)
                }
            }
        }
    }

    // ---- cross-wave reduction: C layout lane (col = weight row r16, rows m = 4kg+v)
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int v = 0; v < 4; ++v)
                dg_red[((((size_t)wave * R + r) * MT + mt) * 16 + 4 * kg + v) * 16 + r16] = y[r][mt][v];
    __syncthreads();
    const int nout = MT * 16 * 16;
    for (int idx = threadIdx.x; idx < nout; idx += blockDim.x) {
        const int rr = idx & 15, m = idx >> 4;
        if (m >= a.T) continue;
        float val[R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            float s = 0.f;
            for (int w = 0; w < NW; ++w) s += dg_red[((((size_t)w * R + r) * MT + (m >> 4)) * 16 + (m & 15)) * 16 + rr];
            val[r] = s;
        }
        if (rp) {
            // the rounding chain of the projection (+bias), then for q and k "f32 -> rope -> model dtype" (attention.rs:644-690;
            // rope_cache_bf16_kernel's arithmetic), then the cache write of k / v (attention.rs:707-719) -- dense_small_body's epilogue
            const uint16_t* b16 = static_cast<const uint16_t*>(a.bias);
            const int Dh = rp->head_dim, hf = Dh >> 1, bs = rp->block_size, Hkv = rp->n_kv_heads;
            const int64_t slot = rp->slots[m];
            const int64_t blk = slot >= 0 ? slot / bs : 0;
            const int off = slot >= 0 ? (int)(slot % bs) : 0;
            uint16_t* o16 = static_cast<uint16_t*>(a.out);
            float o0 = rnd<DT>(val[0]);
            if (b16) o0 = rnd<DT>(o0 + h2f<DT>(b16[row0[0] + rr]));
            if (R == 2) {
                float o1 = rnd<DT>(val[R - 1]);
                if (b16) o1 = rnd<DT>(o1 + h2f<DT>(b16[row0[R - 1] + rr]));
                const int h = row0[0] / Dh, j = row0[0] % Dh + rr;
                const int64_t pos = rp->positions[m];
                const float cc = rp->cos_t[pos * hf + j], sn = rp->sin_t[pos * hf + j];
                float f0, f1;
                rope_rotate(o0, o1, cc, sn, f0, f1);
                const uint16_t r0 = f2h<DT>(f0), r1 = f2h<DT>(f1);
                o16[(size_t)m * a.ldo + row0[0] + rr] = r0;
                o16[(size_t)m * a.ldo + row0[R - 1] + rr] = r1;
                if (a.rope_mode == 2 && slot >= 0) {
                    const int d0 = j, d1 = j + hf;
                    if (rp->flash) { rp->kcache[(slot * Hkv + h) * Dh + d0] = r0; rp->kcache[(slot * Hkv + h) * Dh + d1] = r1; }
                    else {
                        rp->kcache[((((blk * Hkv + h) * (Dh / 8) + d0 / 8) * bs + off) * 8) + d0 % 8] = r0;
                        rp->kcache[((((blk * Hkv + h) * (Dh / 8) + d1 / 8) * bs + off) * 8) + d1 % 8] = r1;
                    }
                }
            } else {
                const uint16_t r0 = f2h<DT>(o0);
                const int row = row0[0] + rr, h = row / Dh, d = row % Dh;
                o16[(size_t)m * a.ldo + row] = r0;
                if (a.rope_mode == 3 && slot >= 0)
                    rp->vcache[rp->flash ? (slot * Hkv + h) * Dh + d : ((blk * Hkv + h) * Dh + d) * (int64_t)bs + off] = r0;
            }
            continue;
        }
        dense_epilogue<DT>(a, m, row0[0] + rr, val[0], val[R - 1]);
    }
}
template <int DT, int WTYPE, int MT, int R, int GJ>
__global__ void __launch_bounds__(512) dense_kernel(const DenseArgs a) { dense_body<DT, WTYPE, MT, R, GJ>(a, (int)blockIdx.x); }
// q, k and v projections of one attention block in ONE launch (same x, k, tokens and weight format; three outputs): the k and
// v launches of a grouped-query model are 32 workgroups of 6 us each (Qwen2-7B: 2 of the 3 launches for 1/8 of the bytes).
// The workgroup index selects the matrix -- a uniform branch in front of one body.
template <int DT, int WTYPE, int MT, int GJ>
__global__ void __launch_bounds__(512) dense3_kernel(const DenseArgs a0, const DenseArgs a1, const DenseArgs a2, const int t0, const int t1) {
    const int bx = (int)blockIdx.x;
    if (bx < t0) dense_body<DT, WTYPE, MT, 1, GJ>(a0, bx);
    else if (bx < t0 + t1) dense_body<DT, WTYPE, MT, 1, GJ>(a1, bx - t0);
    else dense_body<DT, WTYPE, MT, 1, GJ>(a2, bx - t0 - t1);
}

// the same with RoPE and the cache write in the epilogue (decode steps of 5..32 tokens, bf16 cache, full non-interleaved rotary): q and k
// as pairs of row tiles half a head apart (t0, t1 count PAIRS), v one tile per workgroup -- no rope_cache launch behind it
template <int DT, int WTYPE, int MT, int GJ>
__global__ void __launch_bounds__(512) dense3r_kernel(const DenseArgs a0, const DenseArgs a1, const DenseArgs a2, const int t0, const int t1,
                                                      const DenseRope rp) {
    const int bx = (int)blockIdx.x;
    if (bx < t0) dense_body<DT, WTYPE, MT, 2, GJ>(a0, bx, &rp);
    else if (bx < t0 + t1) dense_body<DT, WTYPE, MT, 2, GJ>(a1, bx - t0, &rp);
    else dense_body<DT, WTYPE, MT, 1, GJ>(a2, bx - t0 - t1, &rp);
}

// ------------------------------------------------------------------------------------------------ 5..32 tokens x 16-bit weights, many row tiles (pairs: 5..16); 5..48, long K
// dense_body gives a workgroup ONE row tile (or gate/up pair) and lets its waves split K: every wave then fetches its own copy of
// the activations of its k-blocks -- at 32 tokens 16 KB of x (from L2) for every 8 KB of weights, and all of a k-block's loads are
// requested, waited for and consumed before the next k-block's go out (measured on BASELINE configs[2], Llama-3-8B bf16 at batch
// 32: gate/up 235 MB in 86.7 us = 2.7 TB/s, lm_head 2.7 TB/s).  Here the waves of a workgroup own DIFFERENT row tiles and sweep K
// together:
//   * one image of the activations per k-block in LDS, staged once by all threads and shared by the NW tiles (rows padded to
//     528 B: the 16 rows of an A-fragment read land on 16 different bank quads), double-buffered, one barrier per k-block;
//   * every wave keeps TWO k-blocks of its tile's weights in flight (a 2-slot register ring; the activations of the next
//     k-block are requested in between, so the counted vmcnt waits never drain the ring);
//   * a wave owns all of K for its tile: no cross-wave reduction, the epilogue runs out of the accumulators.
// Taken when the launch has enough row tiles for that shape (gate/up, lm_head); the few-tile projections (wo, down, q/k/v) keep
// the K-split of dense_body.
constexpr int DWD_LDX = 264;                        // 16-bit elements per staged row: 256 + 8 pad
//   * round 5: few-tile launches with a long K (down: 256 tiles x 56 k-blocks at Llama-3-8B) split K ACROSS workgroups (gridDim.y, two
//     workgroups per CU) and leave f32 partial sums [split][token][row] for gptq_wide_epilogue_kernel (split order: deterministic) --
//     on dense_body they ran at 2.7 TB/s (one k-block per wave at a time, every wave its own activations).
template <int DT, int MT, int R, int NW>
__global__ void __launch_bounds__(64 * NW) dense_wide_kernel(const DenseArgs a, float* __restrict__ part, const int ldp, const int kb_per_split) {
    extern __shared__ __attribute__((aligned(16))) uint16_t dwd_x[];          // [2][MT * 16][DWD_LDX]
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r16 = lane & 15, kg = lane >> 4;
    const int nkb_all = a.K >> 8, T = a.T;
    const int kb_lo = (int)blockIdx.y * kb_per_split, nkb = min(nkb_all, kb_lo + kb_per_split) - kb_lo;   // this workgroup's K range
    if (nkb <= 0) return;
    // every workgroup starts its sweep at a different k-block: in step, all waves of the launch would ask for the same 512-byte column
    // of rows 8 KB apart (the order of the f32 sum changes with the workgroup, not from run to run)
    const int rot = (int)((blockIdx.x * 7u) % (unsigned)nkb);
#define DWD_KB(KB_) (kb_lo + ((KB_) + rot) % nkb)
    const int ntiles = (R == 2 ? a.pair_offset : a.N) >> 4;
    const int tile = min((int)blockIdx.x * NW + wave, ntiles - 1);            // a surplus wave shadows the last tile (stores skipped)
    const bool live = (int)blockIdx.x * NW + wave < ntiles;
    int row0[R];
    row0[0] = tile * 16;
    if (R == 2) row0[R - 1] = a.pair_offset + tile * 16;
    const uint16_t* x16 = static_cast<const uint16_t*>(a.x);
    const uint16_t* wrow[R];
#pragma unroll
    for (int r = 0; r < R; ++r)
        wrow[r] = a.wtiled ? static_cast<const uint16_t*>(a.w) + (((size_t)(row0[r] >> 4) * nkb_all) * 512 + lane) * 8
                           : static_cast<const uint16_t*>(a.w) + (size_t)(row0[r] + r16) * a.ldw + 8 * kg;
    const int wkstride = a.wtiled ? 4096 : 256, wjstride = a.wtiled ? 512 : 32;      // elements per k-block / per fragment

    // ---- staging: MT * 512 pieces of 16 B per k-block over NW * 64 threads (piece p: row p / 32, 16-byte column p % 32)
    constexpr int XP = MT * 8 / NW;
    static_assert(XP >= 1 && XP * NW == MT * 8, "pieces must divide evenly");
    const int xcol = threadIdx.x & 31, xrow0 = threadIdx.x >> 5;             // piece i of this thread: row xrow0 + 2 NW i
    const uint16_t* xsrc[XP];
#pragma unroll
    for (int i = 0; i < XP; ++i) xsrc[i] = x16 + (size_t)min(xrow0 + 2 * NW * i, T - 1) * a.ldx + 8 * xcol;
    uint16_t* const xdst = dwd_x + (size_t)xrow0 * DWD_LDX + 8 * xcol;
    uint4 xr[XP];
#define DWD_X_LOAD(KB_) _Pragma("unroll") for (int i_ = 0; i_ < XP; ++i_) xr[i_] = *reinterpret_cast<const uint4*>(xsrc[i_] + (size_t)DWD_KB(KB_) * 256)
#define DWD_X_STORE(BUF_) _Pragma("unroll") for (int i_ = 0; i_ < XP; ++i_) \
        *reinterpret_cast<uint4*>(xdst + ((size_t)(BUF_) * MT * 16 + 2 * NW * i_) * DWD_LDX) = xr[i_]
    uint4 bw[2][R][8];
    // past the end: one 16-byte request per instruction (see dense_small_body)
#define DWD_W_LOAD(SLOT_, KB_) do { \
        const bool ok_ = (KB_) < nkb; \
        const size_t koff_ = ok_ ? (size_t)DWD_KB(KB_) * wkstride : 0; \
        _Pragma("unroll") for (int r_ = 0; r_ < R; ++r_) { \
            const uint16_t* wp_ = (ok_ ? wrow[r_] : static_cast<const uint16_t*>(a.w)) + koff_; \
            _Pragma("unroll") for (int j_ = 0; j_ < 8; ++j_) { \
                const dg_u32x4 v_ = __builtin_nontemporal_load(reinterpret_cast<const dg_u32x4*>(wp_ + (ok_ ? wjstride * j_ : 0))); \
                bw[SLOT_][r_][j_] = make_uint4(v_.x, v_.y, v_.z, v_.w); \
            } \
        } } while (0)
    DWD_X_LOAD(0);
    DWD_W_LOAD(0, 0);
    DWD_W_LOAD(1, 1);
    f32x4_t y[R][MT];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) y[r][mt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    DWD_X_STORE(0);
    __syncthreads();

#define DWD_COMPUTE(SLOT_, BUF_) do { \
        const uint16_t* xb_ = dwd_x + ((size_t)(BUF_) * MT * 16 + r16) * DWD_LDX + 8 * kg; \
        _Pragma("unroll") for (int j_ = 0; j_ < 8; ++j_) { \
            uint4 aw_[MT]; \
            _Pragma("unroll") for (int mt_ = 0; mt_ < MT; ++mt_) aw_[mt_] = *reinterpret_cast<const uint4*>(xb_ + (size_t)mt_ * 16 * DWD_LDX + 32 * j_); \
            _Pragma("unroll") for (int r_ = 0; r_ < R; ++r_) \
                _Pragma("unroll") for (int mt_ = 0; mt_ < MT; ++mt_) y[r_][mt_] = mfma32<DT>(aw_[mt_], bw[SLOT_][r_][j_], y[r_][mt_]); \
        } } while (0)
    for (int kb0 = 0; kb0 < nkb; kb0 += 2) {
        // slot 0
        {
            const int kb = kb0;
            DWD_X_LOAD(min(kb + 1, nkb - 1));                                // next k-block's activations ride between the ring's loads
            DWD_COMPUTE(0, 0);
            DWD_W_LOAD(0, kb + 2);
            DWD_X_STORE(1);
            __syncthreads();
        }
        if (kb0 + 1 < nkb) {                                                 // workgroup-uniform
            const int kb = kb0 + 1;
            DWD_X_LOAD(min(kb + 1, nkb - 1));
            DWD_COMPUTE(1, 1);
            DWD_W_LOAD(1, kb + 2);
            DWD_X_STORE(0);
            __syncthreads();
        }
    }
#undef DWD_X_LOAD
#undef DWD_X_STORE
#undef DWD_W_LOAD
#undef DWD_COMPUTE
#undef DWD_KB
    if (!live) return;
    if (part) {
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    part[((size_t)blockIdx.y * (MT * 16) + mt * 16 + 4 * kg + v) * ldp + row0[r] + r16] = y[r][mt][v];
        return;
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int m = mt * 16 + 4 * kg + v;
            if (m < T) dense_epilogue<DT>(a, m, row0[0] + r16, y[0][mt][v], y[R - 1][mt][v]);
        }
}

// ------------------------------------------------------------------------------------------------ 1..4 tokens x 4-bit weights
// The decode step of a GPTQ / AWQ model at batch 1..4 is a chain of small weight streams (Qwen2-7B: 6 / 8 / 34 / 68 MB), each
// against the launch floor (~4.5 us): what a launch reaches is (bytes in flight) / (memory latency), and what the step reaches is
// mostly the NUMBER of launches.  dense_body asks for one k-block per wave at a time and its activation and scale loads queue
// BEHIND the weight loads (VMEM returns in order).  Here:
//   * every wave stages the activations of ITS k-blocks once, into its own LDS region -- already in the (x0,x4,x1,x5,..) order
//     of the 4-bit code pairs -- one round trip together with the first weight loads, no workgroup barrier;
//   * when `norm_w` is set the staging applies RmsNorm: inv = rsqrt(sum(x^2)/K + eps) comes from `ss_in`, per-tile partial sums of
//     squares that the PRODUCER of the residual stream left behind in its epilogue (`ss_out`; fixed summation order on both
//     sides) -- the two norm launches of a layer disappear without a second pass over x (measured first: every workgroup
//     redoing the two-pass norm behind a barrier cost as much as the launches it saved);
//   * every wave keeps D k-blocks of weights + the dwords holding their scales / zero points in flight (a register ring of D
//     slots; the only VMEM instructions in the loop are the ring's loads, so the counted vmcnt waits leave D-1 slots outstanding).
// Same arithmetic as dense_body's 4-bit arm (128+q / 1024+q codes, scale applied once per group, ones-MFMA row sums).
// (wave_sum_dpp, common.h: __shfl_xor reductions measured 6 us on the 28 us gate/up launch when every wave reduced four tokens'
// partial sums that way)
constexpr int DS_X_BYTES_MAX = 40 * 1024;          // staged activations: T * K * 2 bytes (T = 1: K <= 20480)
template <int DT, int WTYPE, int R, int GJ, int D, bool ZP, int NCH>
__device__ __forceinline__ void dense_small_body(const DenseArgs& a, const int bx, const DenseRope* rp = nullptr) {
    static_assert(WTYPE != DW_DENSE, "4-bit weights only");
    constexpr int NG = 8 / GJ;                     // quantisation groups per k-block (GJ == 8: one group of >= 256)
    extern __shared__ __attribute__((aligned(16))) uint8_t ds_lds[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), NW = blockDim.x >> 6;
    const int r16 = lane & 15, kg = lane >> 4;
    const int nkb = a.K >> 8, T = a.T, K = a.K;
    const int nmine = (nkb - wave + NW - 1) / NW;                  // NW <= nkb: every wave has at least one k-block
    const int nmax = (nkb + NW - 1) / NW;
    uint16_t* xw = reinterpret_cast<uint16_t*>(ds_lds) + (size_t)wave * nmax * T * 256;    // this wave's [nmine][T][256], pair order
    float* red = reinterpret_cast<float*>(ds_lds + (size_t)NW * nmax * T * 512);           // [NW][R][4][16]
    int row0[R];
    row0[0] = bx * 16;
    if (R == 2) row0[R - 1] = a.pair_offset + bx * 16;
    if (R == 2 && rp) {                                            // RoPE pairs: rows (h, j) and (h, j + D/2) of one head
        const int tph = rp->head_dim >> 5;                         // 16-row pair tiles per head
        row0[0] = (bx / tph) * rp->head_dim + (bx % tph) * 16;
        row0[R - 1] = row0[0] + (rp->head_dim >> 1);
    }

    // ---- activation (and norm) loads first, then the ring's first D slots
    const uint16_t* x16 = static_cast<const uint16_t*>(a.x);
    const uint16_t* nw16 = static_cast<const uint16_t*>(a.norm_w);
    // entry f = i * T + t: 256 values = 32 lanes x 16 B, two entries per pass, NCH * 4 passes (the launch checks F <= NCH * 8).
    // Everything below is straight-line code: a run-time loop around loads in front of the ring makes the compiler's wait-count
    // pass give up on counted waits in the main loop (it drains the whole ring at the loop header).
    const int F = nmine * T, half = lane >> 5, piece = lane & 31;
    constexpr int SC = NCH * 4;
    float inv[4] = {1.f, 1.f, 1.f, 1.f};
    // Loads that have nothing to fetch (token >= T, pass beyond F) are still issued -- conditional loads make the wait-count pass
    // drain everything -- but with every lane on the SAME 16 bytes: one 64-byte request instead of a KiB (unpredicated and
    // clamped, a wave of the gate/up launch pulled 16 KB of partial sums, activations and norm weights for its 8 KB of weights).
    f32x4_t ssp[4][2];
    const f32x4_t z4 = {0.f, 0.f, 0.f, 0.f};
    if (nw16) {
        const int ntp = K >> 4;                                          // the producer's tiles (<= 512: K <= 8192 when normed), 4 per lane and load
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const bool ok = t < T && 256 * c < ntp;
                ssp[t][c] = *reinterpret_cast<const f32x4_t*>(a.ss_in + (ok ? (size_t)t * ntp + min(4 * lane + 256 * c, ntp - 4) : 0));   // masked at use
            }
    }
    uint4 xv[SC], gv[SC];
#pragma unroll
    for (int c = 0; c < SC; ++c) {
        const bool ok = 2 * c < F;
        const int f = min(2 * c + half, F - 1), i = f / T, t = f - i * T;
        const size_t k0 = (size_t)(wave + i * NW) * 256 + 8 * piece;
        xv[c] = *reinterpret_cast<const uint4*>(x16 + (ok ? (size_t)t * a.ldx + k0 : 0));
        if (nw16) gv[c] = *reinterpret_cast<const uint4*>(nw16 + (ok ? k0 : 0));
    }

    // sc: the aligned DWORD that holds the 16-bit scale (extracted at use): 16-bit loads get packed two to a VGPR by the compiler
    // right after they are issued -- a wait on the NEWEST loads of the ring, i.e. on all of it
    struct Slot { uint32_t q[R][8]; uint32_t sc[R][NG]; uint32_t zw[R][NG]; };
    int spos[R], zidx[R], zsh[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int col = row0[r] + r16;
        spos[r] = marlin_scale_pos(col, a.sperm);
        int zp = col;
        if (a.zmode == MI355_ZERO_AWQ_MARLIN) {        // marlin zero points (convert_awq_marlin.py:72-91), as zero_point()
            const int p1 = marlin_scale_pos(col, SP_GROUPED), u = p1 & 7;
            zp = (p1 & ~7) + (((u & 1) << 2) | (u >> 1));
        }
        zidx[r] = zp >> 3; zsh[r] = 4 * (zp & 7);
    }
    const float zadd = a.zmode == MI355_ZERO_GPTQ_PLUS1 ? 1.f : 0.f;
    const uint16_t* sc16 = static_cast<const uint16_t*>(a.scales);
    // Past the wave's last k-block the slot is still loaded (conditional loads in the ring make the compiler's wait-count pass drain
    // everything: measured), but every lane reads the SAME 16 bytes of the last block: one 64-byte request instead of a KiB.
    auto issue = [&](Slot& sl, const int kb_in) {
        const bool ok = kb_in < nkb;
        const int kb = ok ? kb_in : nkb - 1, ln = ok ? lane : 0;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            if constexpr (WTYPE == DW_GPTQ4T) {
                const dg_u32x4* tp = reinterpret_cast<const dg_u32x4*>(a.w) + ((size_t)(row0[r] >> 4) * nkb + kb) * 128 + ln;
                const dg_u32x4 v0 = __builtin_nontemporal_load(tp), v1 = __builtin_nontemporal_load(tp + (ok ? 64 : 0));
                sl.q[r][0] = v0.x; sl.q[r][1] = v0.y; sl.q[r][2] = v0.z; sl.q[r][3] = v0.w;
                sl.q[r][4] = v1.x; sl.q[r][5] = v1.y; sl.q[r][6] = v1.z; sl.q[r][7] = v1.w;
            } else {
                const uint32_t* qp = static_cast<const uint32_t*>(a.w) + (size_t)(kb * 32 + (ok ? kg : 0)) * a.N + row0[r] + (ok ? r16 : 0);
#pragma unroll
                for (int j = 0; j < 8; ++j) sl.q[r][j] = __builtin_nontemporal_load(qp + (size_t)(ok ? 4 * j : 0) * a.N);
            }
#pragma unroll
            for (int gq = 0; gq < NG; ++gq) {
                const int g = GJ < 8 ? kb * NG + gq : (kb * 256) / a.group_size;
                sl.sc[r][gq] = __builtin_nontemporal_load(reinterpret_cast<const uint32_t*>(sc16 + (size_t)g * a.N + (ok ? (spos[r] & ~1) : 0)));
                if constexpr (ZP) sl.zw[r][gq] = a.qzeros[(size_t)g * (a.N / 8) + (ok ? zidx[r] : 0)];
            }
        }
    };
    Slot ring[D];
#pragma unroll
    for (int d = 0; d < D; ++d) issue(ring[d], wave + d * NW);

    // ---- activations -> this wave's LDS region (rms_norm_bf16_kernel's arithmetic, elementwise.hip, when normed)
    if (nw16) {
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            if (t >= T) break;
            const int ntp = K >> 4;
            const f32x4_t p0 = 4 * lane < ntp ? ssp[t][0] : z4, p1 = 4 * lane + 256 < ntp ? ssp[t][1] : z4;    // (t < T here)
            float v = ((p0[0] + p0[1]) + (p0[2] + p0[3])) + ((p1[0] + p1[1]) + (p1[2] + p1[3]));
            inv[t] = rsqrtf(wave_sum_dpp(v) / (float)K + a.norm_eps);
        }
    }
#pragma unroll
    for (int c = 0; c < SC; ++c) {
        const int f = 2 * c + half;
        if (f < F) {
            uint4 v = xv[c];
            if (nw16) {
                const int t = f % T;
                const float iv = t == 0 ? inv[0] : t == 1 ? inv[1] : t == 2 ? inv[2] : inv[3];
                const uint32_t u[4] = {v.x, v.y, v.z, v.w}, gw[4] = {gv[c].x, gv[c].y, gv[c].z, gv[c].w};
                uint32_t o[4];
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    o[e] = pack_bf16x2(bf16lo_to_f32(u[e]) * iv * bf16lo_to_f32(gw[e]), bf16hi_to_f32(u[e]) * iv * bf16hi_to_f32(gw[e]));
                v = make_uint4(o[0], o[1], o[2], o[3]);
            }
            uint4 pq;                                                        // code pairs (n_i, n_{i+4}): element order {0,4,1,5,2,6,3,7}
            pq.x = __builtin_amdgcn_perm(v.z, v.x, 0x05040100u);
            pq.y = __builtin_amdgcn_perm(v.z, v.x, 0x07060302u);
            pq.z = __builtin_amdgcn_perm(v.w, v.y, 0x05040100u);
            pq.w = __builtin_amdgcn_perm(v.w, v.y, 0x07060302u);
            *reinterpret_cast<uint4*>(xw + (size_t)f * 256 + 8 * piece) = pq;
        }
    }

    constexpr uint32_t KOFF = (DT == MI355_DTYPE_BF16) ? 0x43004300u : 0x64006400u;
    constexpr float OFF = (DT == MI355_DTYPE_BF16) ? 128.f : 1024.f;
    constexpr uint32_t ONE2 = (DT == MI355_DTYPE_BF16) ? 0x3F803F80u : 0x3C003C00u;
    uint32_t nib = 0x000F000Fu;
    asm volatile("" : "+v"(nib));
    const uint4 ones = make_uint4(ONE2, ONE2, ONE2, ONE2);
    const f32x4_t zero4 = {0.f, 0.f, 0.f, 0.f};
    f32x4_t y[R];
#pragma unroll
    for (int r = 0; r < R; ++r) y[r] = zero4;
    const uint16_t* xrow = xw + (size_t)min(r16, T - 1) * 256 + 8 * kg;

    auto compute = [&](const Slot& sl, const int i) {
        uint4 aw[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) aw[j] = *reinterpret_cast<const uint4*>(xrow + (size_t)i * T * 256 + 32 * j);
#pragma unroll
        for (int gq = 0; gq < NG; ++gq) {
            f32x4_t xs = zero4;
#pragma unroll
            for (int jj = 0; jj < GJ; ++jj) xs = mfma32<DT>(aw[gq * GJ + jj], ones, xs);
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const float s = h2f<DT>((uint16_t)(sl.sc[r][gq] >> (16 * (spos[r] & 1))));
                float z = 8.f;
                if constexpr (ZP) z = (float)((sl.zw[r][gq] >> zsh[r]) & 0xFu) + zadd;
                const float c = -(OFF + z) * s;
                f32x4_t acc = zero4;
#pragma unroll
                for (int jj = 0; jj < GJ; ++jj) {
                    const uint32_t w = sl.q[r][gq * GJ + jj];
                    uint4 b;
                    b.x = (w & nib) | KOFF;
                    b.y = ((w >> 4) & nib) | KOFF;
                    b.z = ((w >> 8) & nib) | KOFF;
                    b.w = ((w >> 12) & nib) | KOFF;
                    acc = mfma32<DT>(aw[gq * GJ + jj], b, acc);
                }
#pragma unroll
                for (int v = 0; v < 4; ++v) y[r][v] += s * acc[v] + c * xs[v];
            }
        }
    };
    for (int i0 = 0; i0 < nmine; i0 += D) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
            const int i = i0 + d;
            if (i < nmine) compute(ring[d], i);
            issue(ring[d], wave + (i + D) * NW);
        }
    }

    // ---- cross-wave reduction: C layout lane (col = weight row r16, rows m = 4kg+v): tokens 0..3 sit in kg == 0
    if (kg == 0) {
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int v = 0; v < 4; ++v) red[((wave * R + r) * 4 + v) * 16 + r16] = y[r][v];
    }
    __syncthreads();
    if ((int)threadIdx.x < T * 16) {
        const int rr = threadIdx.x & 15, m = threadIdx.x >> 4;
        float val[R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            float sum = 0.f;
            for (int w = 0; w < NW; ++w) sum += red[((w * R + r) * 4 + m) * 16 + rr];
            val[r] = sum;
        }
        if (rp) {
            // q / k / v of a decode step: the rounding chain of the projection (+bias), then for q and k "f32 -> rope -> model
            // dtype" (attention.rs:644-690; rope_cache_bf16_kernel's arithmetic), then the cache write of k / v (attention.rs:707-719)
            const uint16_t* b16 = static_cast<const uint16_t*>(a.bias);
            const int Dh = rp->head_dim, hf = Dh >> 1, bs = rp->block_size, Hkv = rp->n_kv_heads;
            const int64_t slot = rp->slots[m];
            const int64_t blk = slot >= 0 ? slot / bs : 0;
            const int off = slot >= 0 ? (int)(slot % bs) : 0;
            uint16_t* o16 = static_cast<uint16_t*>(a.out);
            float o0 = rnd<DT>(val[0]);
            if (b16) o0 = rnd<DT>(o0 + h2f<DT>(b16[row0[0] + rr]));
            if (R == 2) {
                float o1 = rnd<DT>(val[R - 1]);
                if (b16) o1 = rnd<DT>(o1 + h2f<DT>(b16[row0[R - 1] + rr]));
                const int h = row0[0] / Dh, j = row0[0] % Dh + rr;
                const int64_t pos = rp->positions[m];
                const float cc = rp->cos_t[pos * hf + j], sn = rp->sin_t[pos * hf + j];
                float f0, f1;
                rope_rotate(o0, o1, cc, sn, f0, f1);
                const uint16_t r0 = f2h<DT>(f0), r1 = f2h<DT>(f1);
                o16[(size_t)m * a.ldo + row0[0] + rr] = r0;
                o16[(size_t)m * a.ldo + row0[R - 1] + rr] = r1;
                if (a.rope_mode == 2 && slot >= 0) {
                    const int d0 = j, d1 = j + hf;
                    if (rp->flash) { rp->kcache[(slot * Hkv + h) * Dh + d0] = r0; rp->kcache[(slot * Hkv + h) * Dh + d1] = r1; }
                    else {
                        rp->kcache[((((blk * Hkv + h) * (Dh / 8) + d0 / 8) * bs + off) * 8) + d0 % 8] = r0;
                        rp->kcache[((((blk * Hkv + h) * (Dh / 8) + d1 / 8) * bs + off) * 8) + d1 % 8] = r1;
                    }
                }
            } else {
                const uint16_t r0 = f2h<DT>(o0);
                const int row = row0[0] + rr, h = row / Dh, d = row % Dh;
                o16[(size_t)m * a.ldo + row] = r0;
                if (a.rope_mode == 3 && slot >= 0)
                    rp->vcache[rp->flash ? (slot * Hkv + h) * Dh + d : ((blk * Hkv + h) * Dh + d) * (int64_t)bs + off] = r0;
            }
            return;
        }
        const float o = dense_epilogue<DT>(a, m, row0[0] + rr, val[0], val[R - 1]);
        if (a.ss_out) {                                                  // sum of squares of this tile's 16 outputs of token m (fixed order)
            int q2 = __float_as_int(o * o);                            // row (16-lane) sum by DPP shifts: lane 15 of the row ends up with it
            q2 = __float_as_int(__int_as_float(q2) + __int_as_float(__builtin_amdgcn_update_dpp(0, q2, 0x111, 0xf, 0xf, true)));
            q2 = __float_as_int(__int_as_float(q2) + __int_as_float(__builtin_amdgcn_update_dpp(0, q2, 0x112, 0xf, 0xf, true)));
            q2 = __float_as_int(__int_as_float(q2) + __int_as_float(__builtin_amdgcn_update_dpp(0, q2, 0x114, 0xf, 0xf, true)));
            q2 = __float_as_int(__int_as_float(q2) + __int_as_float(__builtin_amdgcn_update_dpp(0, q2, 0x118, 0xf, 0xf, true)));
            if (rr == 15) a.ss_out[(size_t)m * (a.ldo >> 4) + bx] = __int_as_float(q2);
        }
    }
}
template <int DT, int WTYPE, int R, int GJ, int D, bool ZP, int NCH>
__global__ void __launch_bounds__(512) dense_small_kernel(const DenseArgs a) { dense_small_body<DT, WTYPE, R, GJ, D, ZP, NCH>(a, (int)blockIdx.x); }
template <int DT, int WTYPE, int GJ, int D>
__global__ void __launch_bounds__(512) dense_small3_kernel(const DenseArgs a0, const DenseArgs a1, const DenseArgs a2, const int t0, const int t1) {
    const int bx = (int)blockIdx.x;
    if (bx < t0) dense_small_body<DT, WTYPE, 1, GJ, D, false, 1>(a0, bx);
    else if (bx < t0 + t1) dense_small_body<DT, WTYPE, 1, GJ, D, false, 1>(a1, bx - t0);
    else dense_small_body<DT, WTYPE, 1, GJ, D, false, 1>(a2, bx - t0 - t1);
}

// q, k, v of a decode step with RoPE and the cache write in the epilogue: q and k as row-tile PAIRS (j, j + D/2) of one head
template <int DT, int WTYPE, int GJ>
__global__ void __launch_bounds__(512) dense_small3r_kernel(const DenseArgs a0, const DenseArgs a1, const DenseArgs a2, const int t0, const int t1,
                                                            const DenseRope rp) {
    const int bx = (int)blockIdx.x;
    if (bx < t0) dense_small_body<DT, WTYPE, 2, GJ, 2, false, 1>(a0, bx, &rp);
    else if (bx < t0 + t1) dense_small_body<DT, WTYPE, 2, GJ, 2, false, 1>(a1, bx - t0, &rp);
    else dense_small_body<DT, WTYPE, 1, GJ, 4, false, 1>(a2, bx - t0 - t1, &rp);
}

// ------------------------------------------------------------------------------------------------ launch
template <int DT, int WTYPE, int MT, int R>
static int dense_launch_gj(const DenseArgs& a, int gj, int nw, hipStream_t st) {
    const int tiles = (a.epi == MI355_EPI_SILU_MUL ? a.pair_offset : a.N) / 16;
    const size_t lds = (size_t)nw * R * MT * 256 * sizeof(float);
    dim3 grid(tiles), block(nw * 64);
    if constexpr (WTYPE == DW_DENSE) {
        hipLaunchKernelGGL((dense_kernel<DT, WTYPE, MT, R, 8>), grid, block, lds, st, a);
    } else {
        switch (gj) {
            case 1: hipLaunchKernelGGL((dense_kernel<DT, WTYPE, MT, R, 1>), grid, block, lds, st, a); break;
            case 2: hipLaunchKernelGGL((dense_kernel<DT, WTYPE, MT, R, 2>), grid, block, lds, st, a); break;
            case 4: hipLaunchKernelGGL((dense_kernel<DT, WTYPE, MT, R, 4>), grid, block, lds, st, a); break;
            default: hipLaunchKernelGGL((dense_kernel<DT, WTYPE, MT, R, 8>), grid, block, lds, st, a); break;
        }
    }
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

// ---- the 1..4-token launch of 4-bit weights (dense_small_kernel): -4 = this shape stays on dense_kernel
// Tokens from which a 16-bit projection takes the MFMA GEMM of gemm_tile.h (tuning key 36; from 17 where the launch has 768 row tiles or pairs).
// us per launch, streaming kernels against the GEMM: gate/up 28672 x 4096 T = 16 43.9 / 42.3, 32 47.0 / 42.3, 40 90.3 / 43.1 (two sweeps over
// the weights from 33 tokens), 64 96.5 / 44.0; down 4096 x 14336 T = 32 28.5 / 28.6, 40 31.0 / 29.5, 64 64.9 / 32.3; wo 4096 x 4096
// T = 16 9.3 / 13.7, 32 12.3 / 14.0, 40 16.1 / 13.7; 12288 x 2048 T = 32 17.0 / 12.9; at 5 .. 16 tokens either may win (16384 pairs of 3072: 18.7 / 22.1)
// 4-bit, against token chunks of the decode kernels: down 3584 x 18944 T = 32 21.6 / 27.4, 33 29.1 / 28.1, 49 72.7 / 29.1; 4608 x 3584 T = 33 20.8 / 16.0;
// wo 3584 x 3584 33 14.8 / 15.0, 64 19.2 / 16.5; gate/up 37888 x 3584 48 42.1 / 54.5, 64 48.3 / 58.3, 65 64.3 / 58.8
// (to 64 tokens the sizes decide: dense_streams, gptq_stream_us)
enum { DENSE_GEMM_MIN_T = 33, DENSE_GEMM_ANY_T = 96, GPTQ_GEMM_MIN_T = 33, GPTQ_GEMM_MIN_PAIR_T = 65 };
static int g_tune_gemm_min_t = DENSE_GEMM_MIN_T;
static int g_tune_gptq_gemm_off = 0;   // tuning key 39: 1 = 4-bit prompt steps run the decode kernel in 64-token chunks (A/B)
static int g_tune_wide_nw = 4;         // tuning key 38: waves (row tiles) per workgroup of dense_wide_kernel: 2 | 4
static int g_tune_wide_off = 0;        // tuning key 37: 1 = 16-bit launches with many row tiles stay on dense_kernel (A/B)
static int g_tune_small_nw = 0;        // tuning key 30: waves per workgroup (0 = chosen from the k-blocks)
static int g_tune_small_nw_big = 0;    // tuning key 35: the same for K > 8192
static int g_tune_gemm_tall = 0;       // tuning key 30 bits 32, 64: the 16-bit prompt GEMM always takes its 256 x 256 tile and never splits K
static int g_tune_small_off = 0;       // tuning key 31: 1 = keep 1..4 tokens on dense_kernel (A/B measurements)
static int g_tune_gptq_wide_nosplit = 0;   // tuning key 30 bit 256: gate/up pairs of the 5..32-token 4-bit launches stay on one wave each (A/B)
static int g_tune_gptq_wide_off = 0;   // tuning key 30 bit 128: 1 = 5..64-token launches of tiled 4-bit weights stay on dense_kernel (A/B; round 5)
static int g_tune_small_norope = 0;    // tuning key 34: 1 = RoPE and the cache write stay in their own launch
static int g_tune_small_nonorm = 0;    // tuning key 32: 1 = never norm on the way in (the host layer launches the norm separately)
// tuning key 30 (product): bit mask of folded launches switched OFF -- 1 = the 1..4-token 4-bit kernel, 2 = no norm on the way in,
// 4 = RoPE and the cache write in their own launch, 8 = the LDS-shared-activation 16-bit kernel, 16 = the one-pass 4-bit prompt GEMM;
// 32, 64 (switch ON) = the 256 x 256 tile of the 16-bit prompt GEMM wherever that GEMM runs (tests).
// Probe builds: 33 / 35 waves per workgroup of the 1..4-token kernel (hidden-sized K / long K), 36 tokens from which 16-bit
// projections take the MFMA GEMM, 38 waves per workgroup of the LDS-shared-activation kernel.
void mi355_dense_set_small(int key, int v) {
    if (key == 30) {
        g_tune_small_off = v & 1; g_tune_small_nonorm = (v >> 1) & 1; g_tune_small_norope = (v >> 2) & 1;
        g_tune_wide_off = (v >> 3) & 1; g_tune_gptq_gemm_off = (v >> 4) & 1; g_tune_gemm_tall = (v >> 5) & 3;
        g_tune_gptq_wide_off = (v >> 7) & 1;
        g_tune_gptq_wide_nosplit = (v >> 8) & 1;
    }
    else if (key == 33) g_tune_small_nw = v;
    else if (key == 35) g_tune_small_nw_big = v;
    else if (key == 36 && v > 0) g_tune_gemm_min_t = v;
    else if (key == 38) g_tune_wide_nw = v;
}
static inline int dense_small_gj(int group_size) {
    if (group_size >= 256) return (group_size % 256) ? -1 : 8;
    return group_size == 128 ? 4 : group_size == 64 ? 2 : group_size == 32 ? 1 : -1;
}
static inline int dense_small_nw(int nkb) {
    if (g_tune_small_nw >= 1 && g_tune_small_nw <= 8 && g_tune_small_nw <= nkb && nkb <= 32) return g_tune_small_nw;   // experiments: hidden-sized K only
    if (g_tune_small_nw_big >= 1 && g_tune_small_nw_big <= 8 && nkb > 32) return g_tune_small_nw_big;
    if (nkb < 4) return nkb;
    // hidden-sized K (<= 16 k-blocks: 4096): four waves -- more, smaller workgroups per CU balance the launch better than more
    // waves on fewer (Qwen2-7B gate/up, 1184 workgroups: 19.5 us with 2..4 waves, 22.3 us with 7; q/k/v and wo within 0.4 us)
    if (nkb <= 16) return 4;
    int best = 1, best_slots = 1 << 30;
    for (int nw = 8; nw >= 4; --nw) {                               // fewest idle wave-slots, the larger workgroup on a tie
        const int slots = (nkb + nw - 1) / nw * nw;
        if (slots < best_slots) { best_slots = slots; best = nw; }
    }
    return best;
}
// staging passes a wave needs: ceil(k-blocks per wave * T / 8); the kernel is built for 1 and 2
static inline int dense_small_nch(const DenseArgs& a) {
    const int nkb = a.K >> 8, nw = dense_small_nw(nkb);
    return (((nkb + nw - 1) / nw) * a.T + 7) / 8;
}
static inline bool dense_small_ok(const DenseArgs& a, int dt) {
    if (g_tune_small_off || a.T < 1 || a.T > 4 || (a.N & 15) || (a.K & 255) || (size_t)a.T * a.K * 2 > (size_t)DS_X_BYTES_MAX) return false;
    if (a.norm_w && (dt != MI355_DTYPE_BF16 || g_tune_small_nonorm || !a.ss_in || a.K > 8192)) return false;
    if (((uintptr_t)a.x & 15) || (a.ldx & 7)) return false;
    return dense_small_gj(a.group_size) > 0 && dense_small_nch(a) <= 2;
}
template <int DT, int R, int D, bool ZP, int NCH>
static int dense_small_launch_gj(const DenseArgs& a, int gj, hipStream_t st) {
    const int tiles = (R == 2 ? a.pair_offset : a.N) / 16;
    const int nw = dense_small_nw(a.K >> 8);
    const size_t lds = (size_t)nw * (((a.K >> 8) + nw - 1) / nw) * a.T * 512 + (size_t)nw * R * 64 * sizeof(float);
    dim3 grid(tiles), block(nw * 64);
    switch (gj) {
        case 1: hipLaunchKernelGGL((dense_small_kernel<DT, DW_GPTQ4T, R, 1, D, ZP, NCH>), grid, block, lds, st, a); break;
        case 2: hipLaunchKernelGGL((dense_small_kernel<DT, DW_GPTQ4T, R, 2, D, ZP, NCH>), grid, block, lds, st, a); break;
        case 4: hipLaunchKernelGGL((dense_small_kernel<DT, DW_GPTQ4T, R, 4, D, ZP, NCH>), grid, block, lds, st, a); break;
        default: hipLaunchKernelGGL((dense_small_kernel<DT, DW_GPTQ4T, R, 8, D, ZP, NCH>), grid, block, lds, st, a); break;
    }
    return hipGetLastError() == hipSuccess ? 0 : -1;
}
template <int DT, int R, int D, bool ZP>
static int dense_small_launch_nch(const DenseArgs& a, int gj, hipStream_t st) {
    return dense_small_nch(a) <= 1 ? dense_small_launch_gj<DT, R, D, ZP, 1>(a, gj, st) : dense_small_launch_gj<DT, R, D, ZP, 2>(a, gj, st);
}
// the tiled weight image only: the checkpoint layout (mi355_gptq_linear) stays on dense_kernel
template <int DT, int WTYPE>
static int dense_small_launch(const DenseArgs& a, hipStream_t st) {
    if constexpr (WTYPE != DW_GPTQ4T) return -4;
    else {
        if (!dense_small_ok(a, DT)) return -4;
        const int gj = dense_small_gj(a.group_size);
        const bool zp = a.zmode != MI355_ZERO_SYM8 && a.qzeros;
        if (a.epi == MI355_EPI_SILU_MUL)
            return zp ? dense_small_launch_nch<DT, 2, 2, true>(a, gj, st) : dense_small_launch_nch<DT, 2, 2, false>(a, gj, st);
        return zp ? dense_small_launch_nch<DT, 1, 4, true>(a, gj, st) : dense_small_launch_nch<DT, 1, 4, false>(a, gj, st);
    }
}
template <int DT, int WTYPE>
static int dense_small3_launch(const DenseArgs (&a)[3], const DenseRope* rp, hipStream_t st) {
    if constexpr (WTYPE != DW_GPTQ4T) return -4;
    else {
        for (int i = 0; i < 3; ++i)
            if (!dense_small_ok(a[i], DT) || a[i].zmode != MI355_ZERO_SYM8 || dense_small_nch(a[i]) != 1) return -4;
        const int gj = dense_small_gj(a[0].group_size);
        const int nw = dense_small_nw(a[0].K >> 8);
        if (rp) {
            // RoPE + cache write in the epilogue: whole heads of an even, 32-divisible width (pairs of 16-row tiles half a head apart)
            if (g_tune_small_norope || DT != MI355_DTYPE_BF16 || (rp->head_dim & 31) || a[0].N % rp->head_dim || a[1].N != rp->n_kv_heads * rp->head_dim ||
                a[2].N != a[1].N)
                return -4;
            DenseArgs b[3] = {a[0], a[1], a[2]};
            b[0].rope_mode = 1; b[1].rope_mode = 2; b[2].rope_mode = 3;
            const int t0 = a[0].N / 32, t1 = a[1].N / 32, t2 = a[2].N / 16;
            const size_t lds = (size_t)nw * (((a[0].K >> 8) + nw - 1) / nw) * a[0].T * 512 + (size_t)nw * 2 * 64 * sizeof(float);
            dim3 grid(t0 + t1 + t2), block(nw * 64);
#define DS3R(GJ_) hipLaunchKernelGGL((dense_small3r_kernel<DT, DW_GPTQ4T, GJ_>), grid, block, lds, st, b[0], b[1], b[2], t0, t1, *rp)
            switch (gj) { case 1: DS3R(1); break; case 2: DS3R(2); break; case 4: DS3R(4); break; default: DS3R(8); break; }
#undef DS3R
            return hipGetLastError() == hipSuccess ? 0 : -1;
        }
        const int t0 = a[0].N / 16, t1 = a[1].N / 16, t2 = a[2].N / 16;
        const size_t lds = (size_t)nw * (((a[0].K >> 8) + nw - 1) / nw) * a[0].T * 512 + (size_t)nw * 64 * sizeof(float);
        dim3 grid(t0 + t1 + t2), block(nw * 64);
#define DS3(GJ_) hipLaunchKernelGGL((dense_small3_kernel<DT, DW_GPTQ4T, GJ_, 4>), grid, block, lds, st, a[0], a[1], a[2], t0, t1)
        switch (gj) { case 1: DS3(1); break; case 2: DS3(2); break; case 4: DS3(4); break; default: DS3(8); break; }
#undef DS3
        return hipGetLastError() == hipSuccess ? 0 : -1;
    }
}

// waves per workgroup of dense_kernel: K split so that tiles * waves covers the chip several times, capped by the k-blocks
static int dense_waves(int tiles, int nkb, int mt) {
    int nw = 8;
    while (nw > 1 && (nw > nkb || (size_t)tiles * nw > 256 * 32)) nw >>= 1;
    return mt >= 3 && nw > 4 ? 4 : nw;
}
#include "gptq_wide.inc"   // 5..64 tokens x tiled 4-bit weights: LDS-shared activations, split-K for few-tile launches
template <int DT, int WTYPE>
static int dense_launch_dt(const DenseArgs& a, hipStream_t st) {
    if (a.T < 1 || a.T > 64 || (a.N & 15) || (a.K & 255)) return -2;
    {
        const int rs = dense_small_launch<DT, WTYPE>(a, st);
        if (rs != -4) return rs;
        if (a.norm_w) return -4;                   // only the small kernel norms on the way in: the caller norms separately
    }
    const bool pair = a.epi == MI355_EPI_SILU_MUL;
    const int mt = (a.T + 15) / 16;
    if constexpr (WTYPE == DW_GPTQ4T) {
        const int rw = gptq_wide_launch<DT>(a, st);
        if (rw != -4) return rw;
    }
    if constexpr (WTYPE == DW_DENSE) {
        // enough row tiles for one tile (or gate/up pair) per wave on every CU: the LDS-shared-activation sweep.  Round 5: ALSO the few-tile
        // launches with a long K (down: 256 tiles x 56 k-blocks at Llama-3-8B), split over K until two workgroups sit on every CU; their
        // partial sums meet in gptq_wide_epilogue_kernel (short-K few-tile launches -- wo, q / k / v -- keep dense_kernel: a sweep of 4
        // k-blocks plus the epilogue launch is not faster than its one launch)
        const int wtiles = (pair ? a.pair_offset : a.N) / 16;
        const int nkb_w = a.K >> 8;
        const bool many = wtiles >= 4 * 192 && (mt == 1 || (mt == 2 && !pair)), longk = !pair && nkb_w >= 32 && mt <= 3;   // (more tokens: the prompt GEMM, dense_run)
        if (!g_tune_wide_off && a.T > 4 && (many || longk) && !((uintptr_t)a.x & 15) && !(a.ldx & 7) &&
            !((uintptr_t)a.w & 15) && (a.wtiled || !(a.ldw & 7))) {
            const int nwv = many && g_tune_wide_nw == 2 ? 2 : 4;
            const int gx = (wtiles + nwv - 1) / nwv;
            int ks = 1;
            if (!many) {
                g_num_cus_dg = mi355_num_cus();                         // per device (common.h)
                ks = (2 * g_num_cus_dg + gx - 1) / gx;
                if (ks > nkb_w / 4) ks = nkb_w / 4;
                if (ks < 1) ks = 1;
            }
            const int kps = (nkb_w + ks - 1) / ks;
            ks = (nkb_w + kps - 1) / kps;
            const int tpad = mt * 16, ldp = a.N;
            void* pp = nullptr;
            Mi355ScratchTurn turn(MI355_SCR_GPTQ_WIDE, st);
            const bool room = ks == 1 || mi355_scratch_get(&pp, MI355_SCR_GPTQ_WIDE, (size_t)ks * tpad * ldp * sizeof(float), st, false) == 0;
            float* part = static_cast<float*>(pp);
            if (room) {                                                 // (else dense_kernel below)
                const dim3 grid(gx, ks), block(64 * nwv);
                const size_t lds = (size_t)2 * mt * 16 * DWD_LDX * 2;
#define DWD_GO2(MT_, R_, NW_) do { \
                    static bool attr = false; \
                    if (!attr) { (void)hipFuncSetAttribute((const void*)dense_wide_kernel<DT, MT_, R_, NW_>, hipFuncAttributeMaxDynamicSharedMemorySize, 80 * 1024); attr = true; } \
                    hipLaunchKernelGGL((dense_wide_kernel<DT, MT_, R_, NW_>), grid, block, lds, st, a, part, ldp, kps); } while (0)
#define DWD_GO(MT_, R_) do { if (nwv == 2) DWD_GO2(MT_, R_, 2); else DWD_GO2(MT_, R_, 4); } while (0)
                if (pair) DWD_GO(1, 2); else if (mt == 1) DWD_GO(1, 1); else if (mt == 2) DWD_GO(2, 1); else DWD_GO2(3, 1, 4);
#undef DWD_GO2
#undef DWD_GO
                if (hipGetLastError() != hipSuccess) return -1;
                if (ks > 1) {
                    if (!resid_norm_tail<DT>(a, part, ldp, ks, tpad, st))
                        hipLaunchKernelGGL((gptq_wide_epilogue_kernel<DT>), dim3((a.N + 255) / 256, a.T), dim3(256), 0, st, a, part, ldp, ks, tpad);
                    if (hipGetLastError() != hipSuccess) return -1;
                }
                return 0;
            }
        }
    }
    int gj = 8;
    if (WTYPE != DW_DENSE) {
        if (a.group_size >= 256) { if (a.group_size % 256) return -2; gj = 8; }
        else if (a.group_size == 128) gj = 4;
        else if (a.group_size == 64) gj = 2;
        else if (a.group_size == 32) gj = 1;
        else return -2;
    }
    const int nw = dense_waves((pair ? a.pair_offset : a.N) / 16, a.K >> 8, mt);
#define DG_CASE(MT_, R_) return dense_launch_gj<DT, WTYPE, MT_, R_>(a, gj, nw, st)
    if (pair) {
        switch (mt) { case 1: DG_CASE(1, 2); case 2: DG_CASE(2, 2); default: return -3; }
    }
    switch (mt) { case 1: DG_CASE(1, 1); case 2: DG_CASE(2, 1); case 3: DG_CASE(3, 1); default: DG_CASE(4, 1); }
#undef DG_CASE
}

template <int DT, int WTYPE>
static int dense3_launch_dt(const DenseArgs (&a)[3], const DenseRope* rp, hipStream_t st) {
    {
        const int rs = dense_small3_launch<DT, WTYPE>(a, rp, st);
        if (rs != -4) return rs;
        if (a[0].norm_w) return -4;                // only the 1..4-token kernel norms on the way in
    }
    const int mt = (a[0].T + 15) / 16;
    if (rp) {
        // RoPE + cache write in the epilogue of the 5..32-token kernel: whole heads of an even, 32-divisible width, bf16
        if (g_tune_small_norope || DT != MI355_DTYPE_BF16 || mt > 2 || (rp->head_dim & 31) || a[0].N % rp->head_dim ||
            a[1].N != rp->n_kv_heads * rp->head_dim || a[2].N != a[1].N)
            return -4;
    }
    int gj = 8;
    if (WTYPE != DW_DENSE) {
        const int g = a[0].group_size;
        if (g >= 256) { if (g % 256) return -2; }
        else if (g == 128) gj = 4;
        else if (g == 64) gj = 2;
        else if (g == 32) gj = 1;
        else return -2;
    }
    const int t0 = a[0].N / 16, t1 = a[1].N / 16, t2 = a[2].N / 16, tiles = t0 + t1 + t2;
    const int nkb = a[0].K >> 8;
    const int nw = dense_waves(tiles, nkb, mt);
    if (rp) {
        DenseArgs b[3] = {a[0], a[1], a[2]};
        b[0].rope_mode = 1; b[1].rope_mode = 2; b[2].rope_mode = 3;
        const int p0 = t0 / 2, p1 = t1 / 2;
        const size_t ldr = (size_t)nw * 2 * mt * 256 * sizeof(float);
        dim3 gridr(p0 + p1 + t2), block(nw * 64);
#define DG3R(MT_, GJ_) hipLaunchKernelGGL((dense3r_kernel<DT, WTYPE, MT_, GJ_>), gridr, block, ldr, st, b[0], b[1], b[2], p0, p1, *rp)
#define DG3R_MT(GJ_) if (mt == 1) DG3R(1, GJ_); else DG3R(2, GJ_);
        if (WTYPE == DW_DENSE) { DG3R_MT(8) }
        else switch (gj) { case 1: DG3R_MT(1) break; case 2: DG3R_MT(2) break; case 4: DG3R_MT(4) break; default: DG3R_MT(8) break; }
#undef DG3R_MT
#undef DG3R
        return hipGetLastError() == hipSuccess ? 0 : -1;
    }
    const size_t lds = (size_t)nw * mt * 256 * sizeof(float);
    dim3 grid(tiles), block(nw * 64);
#define DG3(MT_, GJ_) hipLaunchKernelGGL((dense3_kernel<DT, WTYPE, MT_, GJ_>), grid, block, lds, st, a[0], a[1], a[2], t0, t1)
#define DG3_MT(GJ_) switch (mt) { case 1: DG3(1, GJ_); break; case 2: DG3(2, GJ_); break; case 3: DG3(3, GJ_); break; default: DG3(4, GJ_); break; }
    if (WTYPE == DW_DENSE) { DG3_MT(8) }
    else switch (gj) { case 1: DG3_MT(1) break; case 2: DG3_MT(2) break; case 4: DG3_MT(4) break; default: DG3_MT(8) break; }
#undef DG3_MT
#undef DG3
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

template <int DT>
static int dense_dispatch_dt(const DenseArgs& a, int wtype, hipStream_t st) {
    if (wtype == DW_DENSE) return dense_launch_dt<DT, DW_DENSE>(a, st);
    if (wtype == DW_GPTQ4T) return dense_launch_dt<DT, DW_GPTQ4T>(a, st);
    return dense_launch_dt<DT, DW_GPTQ4>(a, st);
}
static int dense_dispatch(const DenseArgs& a, int wtype, int dt, hipStream_t st) {
    if (dt == MI355_DTYPE_BF16) return dense_dispatch_dt<MI355_DTYPE_BF16>(a, wtype, st);
    if (dt == MI355_DTYPE_F16) return dense_dispatch_dt<MI355_DTYPE_F16>(a, wtype, st);
    return -2;
}

// ---- prompt steps (T >= DENSE_GEMM_MIN_T, dense 16-bit weights): the matmul is compute-bound -> a hand-written MFMA GEMM
// (`Linear::forward` on prompt chunks, linear.rs:124-172; packed gate_up of mlp.rs:324-352,440-458) around the main loop of gemm_tile.h.
//   * candle's rounding chain in the epilogue, from the f32 accumulators: round to the dtype, + bias (rounded), then
//     + residual (rounded) or silu(gate) rounded * up rounded -- no separate chain kernel, no f32 / 16-bit staging of y;
//   * SILU_MUL: the weight tile holds BN / 2 gate rows and the matching up rows (pair_offset apart in W), fragments j and j + NF / 2 of a
//     wave are the two halves of the same output columns, so gate and up meet in registers;
//   * up to three matrices over one x (q, k, v) are one launch: their column tiles follow each other.
struct DenseGemm3 {
    DenseArgs a[3];
    int32_t tiles[3], n_m;               // column tiles of each matrix (0: none), token tiles
    int32_t splits, units_per_split;     // K in `splits` ranges whose partial sums go to `part` [splits][token][ldp], a matrix's from column col0 on
    float* part;
    int32_t ldp, col0[3];
};
// candle's rounding of one value by the hardware's conversion (the same round-to-nearest-even; a NaN keeps its sign)
template <int DT> __device__ __forceinline__ uint32_t gemm_pack(float lo, float hi) {
    if constexpr (DT == MI355_DTYPE_BF16) return cvt_pk_bf16(lo, hi);
    else return (uint32_t)f2h<DT>(lo) | (uint32_t)f2h<DT>(hi) << 16;
}
template <int DT> __device__ __forceinline__ float gemm_rnd(float v) {
    if constexpr (DT == MI355_DTYPE_BF16) return __uint_as_float(cvt_pk_bf16(v, 0.f) << 16);
    else return rnd<DT>(v);
}
// Epilogue of the prompt GEMMs: acc[i][j][v] is token t_first + 16 i, column col_first + 16 j + v (SILU_MUL: fragments j and j + NF / 2 are gate
// and up of the same columns): four consecutive columns of one token per fragment
template <int DT, int EPI, int MF, int NF>
__device__ __forceinline__ void gemm_store(const DenseArgs& a, const f32x4_t (&acc)[MF][NF], const int t_first, const int col_first) {
    constexpr bool silu = EPI == MI355_EPI_SILU_MUL;
    const int n_cols = silu ? a.pair_offset : a.N;
    const uint16_t* bias = static_cast<const uint16_t*>(a.bias);
    const uint16_t* resid = static_cast<const uint16_t*>(a.resid);
    uint16_t* out = static_cast<uint16_t*>(a.out);
    const bool wide = !((a.ldo & 3) | (n_cols & 3)) && !(((uintptr_t)out | (uintptr_t)resid) & 7);
#pragma unroll
    for (int i = 0; i < MF; ++i) {
        const int t = t_first + 16 * i;
        if (t >= a.T) continue;
#pragma unroll
        for (int j = 0; j < (silu ? NF / 2 : NF); ++j) {
            float o[4];
            int col;
            if (silu) {
                col = col_first + 16 * j;
                if (col >= n_cols) continue;
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    float gv = gemm_rnd<DT>(acc[i][j][v]), u = gemm_rnd<DT>(acc[i][(j + NF / 2) % NF][v]);
                    if (bias && col + v < n_cols) { gv = gemm_rnd<DT>(gv + h2f<DT>(bias[col + v])); u = gemm_rnd<DT>(u + h2f<DT>(bias[a.pair_offset + col + v])); }
                    o[v] = gemm_rnd<DT>(gv / (1.f + __expf(-gv))) * u;        // silu(gate) * up (mlp.rs:457); the store rounds
                }
            } else {
                col = col_first + 16 * j;
                if (col >= n_cols) continue;
                uint16_t rr[4];
                if (EPI == MI355_EPI_RESID) {
                    const uint16_t* rp = resid + (size_t)t * a.ldo + col;
                    if (wide) {
                        const uint2 r2 = *reinterpret_cast<const uint2*>(rp);
                        rr[0] = (uint16_t)r2.x; rr[1] = (uint16_t)(r2.x >> 16); rr[2] = (uint16_t)r2.y; rr[3] = (uint16_t)(r2.y >> 16);
                    } else {
#pragma unroll
                        for (int v = 0; v < 4; ++v) rr[v] = col + v < n_cols ? rp[v] : (uint16_t)0;
                    }
                }
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    o[v] = gemm_rnd<DT>(acc[i][j][v]);
                    if (bias && col + v < n_cols) o[v] = gemm_rnd<DT>(o[v] + h2f<DT>(bias[col + v]));
                    if (EPI == MI355_EPI_RESID) o[v] = o[v] + h2f<DT>(rr[v]);
                }
            }
            uint16_t* op = out + (size_t)t * a.ldo + col;
            if (wide) {
                *reinterpret_cast<uint2*>(op) = make_uint2(gemm_pack<DT>(o[0], o[1]), gemm_pack<DT>(o[2], o[3]));
            } else {
#pragma unroll
                for (int v = 0; v < 4; ++v) if (col + v < n_cols) op[v] = (uint16_t)gemm_pack<DT>(o[v], 0.f);
            }
        }
    }
}

template <int DT, int EPI, int WM, int WN, int MF, int NF, int S, bool TILED>
__global__ void __launch_bounds__(512, 2) dense_gemm_kernel(const DenseGemm3 g) {
    typedef GemmTile<DT, WM, WN, MF, NF, S, TILED> Tile;
    extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
    const int n_tiles = g.n_m * (g.tiles[0] + g.tiles[1] + g.tiles[2]);
    const int split = blockIdx.x / n_tiles;                              // the splits of a tile are as far apart as they can be: their reads do not meet
    const GtPlace at = gt_place(blockIdx.x - split * n_tiles, g.n_m, g.tiles[0] + g.tiles[1] + g.tiles[2]);
    int bn = at.n;
    const int which = bn < g.tiles[0] ? 0 : bn < g.tiles[0] + g.tiles[1] ? 1 : 2;
    if (which > 0) bn -= g.tiles[0];
    if (which > 1) bn -= g.tiles[1];
    const DenseArgs& a = g.a[which];
    Tile tile(smem);
    constexpr bool silu = EPI == MI355_EPI_SILU_MUL;
    const int t0 = at.m * Tile::BM;
    const int n_cols = silu ? a.pair_offset : a.N;                      // output columns
    const int c0 = bn * (silu ? Tile::BN / 2 : Tile::BN);               // first output column of this tile
    // weight row held by row j of the tile's weight side (clamped: rows beyond the matrix are multiplied and never stored)
    auto wrow = [&](int j) {
        int n = c0 + j, lim = a.N - 1;
        if (silu) {
            const int w = j / (NF * 16), in = j % (NF * 16), up = in >= NF * 8;
            n = c0 + w * (NF * 8) + (up ? in - NF * 8 : in);
            lim = a.pair_offset - 1;
            n = (n > lim ? lim : n) + (up ? a.pair_offset : 0);
            return n;
        }
        return n > lim ? lim : n;
    };
    const uint8_t* wb = static_cast<const uint8_t*>(a.w);
    const uint8_t* a_base = static_cast<const uint8_t*>(a.x) + (size_t)t0 * a.ldx * 2;
    uint32_t a_off[Tile::AR], b_off[Tile::BR];
    const uint8_t* b_base[Tile::BR];
#pragma unroll
    for (int r = 0; r < Tile::AR; ++r) {
        int row = tile.stage_row(r);
        if (row > a.T - 1 - t0) row = a.T - 1 - t0;
        a_off[r] = (uint32_t)row * (uint32_t)a.ldx * 2u + tile.stage_chunk();
    }
#pragma unroll
    for (int r = 0; r < Tile::BR; ++r) {
        if constexpr (TILED) {                                          // 8 KiB per (row tile, 256 k), 2 KiB per unit, 1 KiB per fragment
            b_base[r] = wb + (size_t)(wrow(16 * tile.stage_tile(r)) >> 4) * (a.K >> 8) * 8192 + tile.stage_frag() * 1024;
            b_off[r] = tile.lane * 16u;
        } else {
            const int first = wrow(8 * (tile.wave + 8 * r)), row = wrow(tile.stage_row(r));
            b_base[r] = wb + (size_t)first * a.ldw * 2;
            b_off[r] = (uint32_t)(row - first) * (uint32_t)a.ldw * 2u + tile.stage_chunk();
        }
    }
    constexpr uint32_t b_step = TILED ? 2048u : 128u;
    int units = a.K / 64;
    if (g.splits > 1) {
        const int u0 = split * g.units_per_split;
        units = min(units - u0, g.units_per_split);
        a_base += (size_t)u0 * 128;
#pragma unroll
        for (int r = 0; r < Tile::BR; ++r) b_base[r] += (size_t)u0 * b_step;
    }
    tile.run(a_base, a_off, b_base, b_off, b_step, units);
    if (g.splits > 1) {                                                  // gptq_wide_epilogue_kernel adds the ranges in their order and rounds
        float* part = g.part + (size_t)split * a.T * g.ldp + g.col0[which];
#pragma unroll
        for (int i = 0; i < MF; ++i) {
            const int t = t0 + tile.row(i);
            if (t >= a.T) continue;
#pragma unroll
            for (int j = 0; j < NF; ++j) {
                int col = c0 + tile.col(j);
                if (silu) col = c0 + tile.wn * (NF * 8) + (j % (NF / 2)) * 16 + 4 * (tile.lane >> 4);
                if (col >= n_cols) continue;
                if (silu && j >= NF / 2) col += a.pair_offset;
                *reinterpret_cast<f32x4_t*>(part + (size_t)t * g.ldp + col) = tile.acc[i][j];
            }
        }
        return;
    }
    gemm_store<DT, EPI, MF, NF>(a, tile.acc, t0 + tile.row(0), c0 + (silu ? tile.wn * NF * 8 : tile.wn * NF * 16) + 4 * (tile.lane >> 4));
}

#include "gptq_gemm.inc"
template <int DT, int EPI, bool SYM, int XG, int WM, int WN, int MF, int NF, int S>
static void gptq_gemm_go(const GptqGemm& g, hipStream_t st) {
    constexpr int BM = WM * MF * 16, BN = WN * NF * 16;
    constexpr uint32_t lds = S * (BM * 256u + BN * 64u) + (S + 1) * (GG_UNIT / XG) * (1024u + BN * 4u);
    static_assert(lds <= 160 * 1024, "a CU's LDS");
    static Mi355DevOnce attr_done;
    if (!attr_done.done()) {
        (void)hipFuncSetAttribute((const void*)gptq_gemm_kernel<DT, EPI, SYM, XG, WM, WN, MF, NF, S>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        attr_done.set();
    }
    hipLaunchKernelGGL((gptq_gemm_kernel<DT, EPI, SYM, XG, WM, WN, MF, NF, S>), dim3(g.n_m * (g.tiles[0] + g.tiles[1] + g.tiles[2]) * g.splits), dim3(512), lds, st, g);
}
static constexpr GtTile kGgTiles[] = {{128, 256, 1, 2.0f}, {128, 128, 1, 1.2f}, {64, 128, 1, 0.9f}};   // us: a unit of 128 k
template <int DT, int EPI, bool SYM, int XG>
static void gptq_gemm_tile(const GptqGemm& g, int which, hipStream_t st) {
    switch (which) {
        case 0: if constexpr (XG == GG_UNIT) gptq_gemm_go<DT, EPI, SYM, XG, 2, 4, 4, 4, 3>(g, st); break;   // (groups of 64: 8 .. 31 registers too many)
        case 1: gptq_gemm_go<DT, EPI, SYM, XG, 2, 4, 4, 2, 3>(g, st); break;
        default: gptq_gemm_go<DT, EPI, SYM, XG, 2, 4, 2, 2, 5>(g, st); break;
    }
}
template <int DT, bool SYM, int XG>
static void gptq_gemm_epi(const GptqGemm& g, int which, hipStream_t st) {
    if (g.a[0].epi == MI355_EPI_SILU_MUL) gptq_gemm_tile<DT, MI355_EPI_SILU_MUL, SYM, XG>(g, which, st);
    else if (g.a[0].epi == MI355_EPI_RESID) gptq_gemm_tile<DT, MI355_EPI_RESID, SYM, XG>(g, which, st);
    else gptq_gemm_tile<DT, MI355_EPI_STORE, SYM, XG>(g, which, st);
}
template <int DT>
static int gptq_gemm_dt(const GptqGemm& g, uint16_t* xp, float* xs, int which, hipStream_t st) {
    const DenseArgs& a = g.a[0];
    const int xg = a.group_size % GG_UNIT ? 64 : GG_UNIT;
    int64_t xb = ((int64_t)a.T * (a.K >> 3) + 255) / 256, pb[3], all = xb;
    for (int i = 0; i < 3; ++i) { pb[i] = g.tiles[i] ? ((int64_t)(a.K / a.group_size) * g.a[i].N + 255) / 256 : 0; all += pb[i]; }
    if (all > 0x7FFFFFFF) return (int)hipErrorNotSupported;
    if (xg == 64) hipLaunchKernelGGL((gptq_gemm_prep_kernel<DT, 64>), dim3((unsigned)all), dim3(256), 0, st, g, xp, xs, (int)xb, (int)pb[0], (int)pb[1]);
    else hipLaunchKernelGGL((gptq_gemm_prep_kernel<DT, 128>), dim3((unsigned)all), dim3(256), 0, st, g, xp, xs, (int)xb, (int)pb[0], (int)pb[1]);
    const bool sym = a.zmode == MI355_ZERO_SYM8 || !a.qzeros;
    if (xg == 64) { if (sym) gptq_gemm_epi<DT, true, 64>(g, which, st); else gptq_gemm_epi<DT, false, 64>(g, which, st); }
    else { if (sym) gptq_gemm_epi<DT, true, 128>(g, which, st); else gptq_gemm_epi<DT, false, 128>(g, which, st); }
    return (int)hipGetLastError();
}
// The workspaces of the prompt GEMMs are kept, so they are bounded: partial sums of at most 128 MiB, and of a 4-bit prompt at most 128 MiB of permuted
// x and its sums at a time (3 328 tokens of 18 944, 19 712 of 3 584; a launch of that many is at its rate, and the panel in front of each costs 1 % of it)
constexpr int64_t GEMM_PART_BYTES = 128ll << 20, GPTQ_GEMM_X_BYTES = 128ll << 20;
static int gemm_max_split(const DenseArgs& a, int64_t rows, int most) {
    return (int)std::min<int64_t>(std::min(16, most), std::max<int64_t>(1, GEMM_PART_BYTES / ((int64_t)a.T * rows * 4)));
}
static int gptq_gemm_slab(int k) { return (int)std::max<int64_t>(1, GPTQ_GEMM_X_BYTES / ((int64_t)k * 2 + k / 16) / 256) * 256; }
// rows t0 .. of a launch of T tokens, at most n of them
static DenseArgs dense_rows(const DenseArgs& a, int t0, int n) {
    DenseArgs c = a;
    c.T = a.T - t0 < n ? a.T - t0 : n;
    c.x = static_cast<const uint16_t*>(a.x) + (size_t)t0 * a.ldx;
    c.out = static_cast<uint16_t*>(a.out) + (size_t)t0 * a.ldo;
    if (a.resid) c.resid = static_cast<const uint16_t*>(a.resid) + (size_t)t0 * a.ldo;
    if (c.T < a.T) c.tail = nullptr;                                   // (its buffer starts with the first row)
    return c;
}
// The sums of q | k | v in ranges of K, RoPE (halves) and the cache write: four pairs of q or k or four channels of v per thread, units of a token one behind the other.
// The products' own rounding, then rope_kernel's and the cache's: what the launches that it stands for do.  Three small products with K in ranges and this launch
// in place of the products over all of K, RoPE and the cache write, us: 4608 x 3584 in 4 bits, 50 tokens 17.1 for 37.8; 3072 x 2048 in 16 bits, 99 tokens 15.9 for 22.9.
__global__ void __launch_bounds__(256) sum3_rope_cache_kernel(const DenseGemm3 g, const DenseRope rp, const int n_units) {
    constexpr int DT = MI355_DTYPE_BF16;
    const int u = blockIdx.x * 256 + threadIdx.x;
    if (u >= n_units) return;
    const int D = rp.head_dim, half = D >> 1, G = rp.n_kv_heads, H = g.a[0].N / D, qk = (H + G) * (half >> 2), per_tok = qk + G * (D >> 2);
    const int t = u / per_tok, r = u - t * per_tok;
    const int64_t slot = rp.slots[t];
    const int64_t blk = slot >= 0 ? slot / rp.block_size : 0;
    const int off = slot >= 0 ? (int)(slot % rp.block_size) : 0;
    const size_t step = (size_t)g.a[0].T * g.ldp;
    const int h = r < qk ? r / (half >> 2) : 0, m = r >= qk ? 2 : h < H ? 0 : 1;
    const int col = r < qk ? (m ? h - H : h) * D + (r - h * (half >> 2)) * 4 : (r - qk) * 4;   // in matrix m
    const int second = m < 2 ? half : 0;
    const float* p = g.part + (size_t)t * g.ldp + g.col0[m] + col;
    f32x4_t x = {0.f, 0.f, 0.f, 0.f}, y = x;
#pragma unroll 8
    for (int s = 0; s < g.splits; ++s, p += step) {
        x += *reinterpret_cast<const f32x4_t*>(p);
        y += *reinterpret_cast<const f32x4_t*>(p + second);
    }
    const uint16_t* bias = static_cast<const uint16_t*>(g.a[m].bias);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        x[i] = gemm_rnd<DT>(x[i]); y[i] = gemm_rnd<DT>(y[i]);
        if (bias) { x[i] = gemm_rnd<DT>(x[i] + h2f<DT>(bias[col + i])); y[i] = gemm_rnd<DT>(y[i] + h2f<DT>(bias[col + second + i])); }
    }
    if (m == 2) {
        if (slot < 0) return;
        const int hh = col / D, d = col - hh * D;
        if (rp.flash) *reinterpret_cast<uint2*>(rp.vcache + (slot * G + hh) * D + d) = make_uint2(pack_bf16x2(x[0], x[1]), pack_bf16x2(x[2], x[3]));
        else {
#pragma unroll
            for (int i = 0; i < 4; ++i) rp.vcache[((blk * G + hh) * D + d + i) * (int64_t)rp.block_size + off] = f32_to_bf16(x[i]);
        }
        return;
    }
    const int hh = col / D, j = col - hh * D;
    const float4 c = *reinterpret_cast<const float4*>(rp.cos_t + rp.positions[t] * half + j), s = *reinterpret_cast<const float4*>(rp.sin_t + rp.positions[t] * half + j);
    const float cc[4] = {c.x, c.y, c.z, c.w}, ss[4] = {s.x, s.y, s.z, s.w};
    float o[4], o2[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) rope_rotate(x[i], y[i], cc[i], ss[i], o[i], o2[i]);
    uint16_t *pa, *pb;
    if (m == 0) { pa = static_cast<uint16_t*>(g.a[0].out) + (size_t)t * g.a[0].ldo + col; pb = pa + half; }
    else if (slot < 0) return;
    else if (rp.flash) { pa = rp.kcache + (slot * G + hh) * D + j; pb = pa + half; }
    else { pa = rp.kcache + (((blk * G + hh) * (D / 8) + j / 8) * rp.block_size + off) * 8 + j % 8; pb = pa + (int64_t)(half / 8) * rp.block_size * 8; }
    *reinterpret_cast<uint2*>(pa) = make_uint2(pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3]));
    *reinterpret_cast<uint2*>(pb) = make_uint2(pack_bf16x2(o2[0], o2[1]), pack_bf16x2(o2[2], o2[3]));
}
// Whether the launch above takes the sums of these three, and its units
static int64_t sum3_units(const DenseArgs* a, const DenseRope& rp, int dt) {
    if (dt != MI355_DTYPE_BF16 || rp.head_dim % 16 || a[0].N % rp.head_dim || a[1].N != rp.n_kv_heads * rp.head_dim || a[2].N != a[1].N) return 0;
    if (((uintptr_t)a[0].out | (uintptr_t)rp.kcache | (uintptr_t)rp.vcache | (uintptr_t)rp.cos_t | (uintptr_t)rp.sin_t) & 15 || a[0].ldo % 8 || rp.block_size < 1) return 0;
    const int64_t units = (int64_t)a[0].T * ((a[0].N + a[1].N) / 8 + a[2].N / 4);
    return units < (1ll << 31) - 256 ? units : 0;
}
// us that the streaming kernels take for one matrix and 33 .. 64 tokens, from what their time follows: the k-blocks in a row of the slowest wave.
//   * gptq_wide_kernel, K in one range: 4.3 + 1.29 a block (512 .. 12288 rows x 1024 9.4 .. 9.8, 16384 x 8192 45.7; more waves per CU are slower by 6 % each);
//     K in ranges (and an epilogue launch that adds them): the rounds of two workgroups per CU, the last range's share of a second round
//     counted as far as its workgroups are a quarter of the CUs (4096 x 14336: 7 blocks 22.3, 4608: 14 31.8; 4608 x 11008: 6 + 1 22.9);
//   * dense_kernel: its waves' share of K, once per round of the row tiles over the CUs (4096 rows x 2048 33 tokens 9.3, 48 10.3, 64 12.1; 8192 x 2048 13.1,
//     15.7, 18.6).
// With gptq_gemm_us it picks the faster side, or one within 5 %, at 748 of 759 measured sizes (512 .. 32000 rows, k of 256 .. 18944, groups, zero points, epilogues)
static float gptq_stream_us(const DenseArgs& a) {
    const int cus = mi355_num_cus(), tiles = a.N / 16, nkb = a.K >> 8, mt = (a.T + 15) / 16;
    if (gptq_wide_takes(a)) {
        const GptqWideSplit w = gptq_wide_split(tiles, nkb, cus);
        if (w.ks == 1) return 4.3f + (float)nkb * (1.29f + 0.08f * (float)(w.nw - 4)) * (float)((w.gx + cus - 1) / cus);
        const int wgs = w.gx * w.ks, over = wgs - 2 * cus;
        const float sweep = (float)w.kps + (over > 0 ? (float)(nkb - w.kps * (w.ks - 1)) * std::min(1.f, 4.f * (float)over / (float)cus) : 0.f);
        const float one = 5.f + 0.3f * (float)w.ks + 1.3f * sweep, two = 12.f + 1.55f * sweep;      // one workgroup per CU, two
        return one + (two - one) * std::min(1.f, std::max(0.f, 2.f * (float)(wgs - cus) / (float)cus));
    }
    const int nw = dense_waves(tiles, nkb, mt), blocks = (nkb + nw - 1) / nw, rounds = (tiles + cus - 1) / cus;
    const float t1 = mt <= 3 ? 2.93f + 0.018f * (float)(a.T - 33) : 3.95f + 0.02f * (float)(a.T - 49);    // a block, one tile per CU
    const float t2 = mt <= 3 ? 2.53f + 0.036f * (float)(a.T - 33) : 3.6f;                                  // a block and a tile of several
    const bool small = a.group_size < 128, zp = a.qzeros && a.zmode != MI355_ZERO_SYM8;                     // more scales, zero points to unpack
    const float f = (small ? 1.05f : 1.f) * (!zp ? 1.f : small ? 1.25f : 1.1f);
    return 3.3f + f * (float)blocks * (rounds == 1 ? t1 : t2 * (float)rounds) + (a.epi == MI355_EPI_RESID ? (mt <= 3 ? 1.f : 1.7f) : 0.f);
}
// the GEMM's, from its choice: beside the rounds there are the launch in front, the partial sums and their launch, and a start on cold weights
static float gptq_gemm_us(const GtChoice& c, int T, float weights_us) {
    const float cold = std::min(1.7f, weights_us);
    return c.splits == 1 ? 0.88f * c.us + 3.5f + cold : c.us + 0.2f * (float)(c.splits - 1) + 1.9f * cold + 0.03f * (float)(T - 33);
}
// n matrices over the same x, of one group size and zero mode; at most gptq_gemm_slab(K) tokens
// (rope, three matrices: K may go in ranges, and then RoPE and the cache write are done too, *roped)
static int gptq_prompt_gemm(const DenseArgs* ms, int n, int dt, hipStream_t st, const DenseRope* rope = nullptr, bool* roped = nullptr) {
    const DenseArgs& a = ms[0];
    const int gs = a.group_size;
    const bool silu = a.epi == MI355_EPI_SILU_MUL;
    if (dt != MI355_DTYPE_BF16 && dt != MI355_DTYPE_F16) return (int)hipErrorNotSupported;
    if (g_tune_gptq_gemm_off || (a.K & 255) || a.T < 4 || gs < 64 || (gs % 64) || (a.K % gs) || (gs > 128 && gs % 256)) return (int)hipErrorNotSupported;   // (the groups of the token chunks, but 32)
    if ((a.ldx * 2) % 16 || ((uintptr_t)a.x & 15) || (int64_t)a.K * 512 >= (1ll << 32)) return (int)hipErrorNotSupported;
    int64_t rows = 0, words = 0;
    for (int i = 0; i < n; ++i) {
        if ((ms[i].N & 15) || ((uintptr_t)ms[i].w & 15) || ms[i].epi != a.epi || ms[i].zmode != a.zmode || !ms[i].qzeros != !a.qzeros) return (int)hipErrorNotSupported;
        rows += ms[i].N;
        words += ((int64_t)(a.K / gs) * ms[i].N + 63) / 64 * 64;
    }
    if (silu && (a.pair_offset <= 0 || a.N != 2 * a.pair_offset || (a.pair_offset & 15))) return (int)hipErrorNotSupported;
    GptqGemm g{};
    auto tiles = [&](const GtTile& t) {
        int64_t c = 0;
        for (int i = 0; i < n; ++i) c += g.tiles[i] = silu ? (a.pair_offset + t.bn / 2 - 1) / (t.bn / 2) : (ms[i].N + t.bn - 1) / t.bn;
        return c * ((a.T + t.bm - 1) / t.bm);
    };
    // us per launch (Qwen2-7B's layers, groups of 128; the 128 x 64 kernel that unpacked 128 k per wave and step, then this one): gate/up 37888 x 3584
    // at 700 tokens 695 / 236, at 2048 2030 / 560; down 3584 x 18944 at 700 470 / 118 (three ranges), at 64 (chunks of the decode kernel) 78 / 30
    // (64-token tiles, eight ranges), at 96 102 / 36.
    const int units = a.K / GG_UNIT;
    const float weights_us = (float)rows * (float)a.K / 2.f / 5.0e6f;
    const float part_us = (float)a.T * 4.f / 4.5e6f;
    GtChoice best = gt_pick(tiles, units, weights_us, n == 1 && a.T <= 65535 ? gemm_max_split(a, a.N, std::max(1, units / 4)) : 1, part_us * (float)a.N, gs % GG_UNIT ? 6 : 7, kGgTiles, 3);
    const int64_t units3 = n == 3 && rope ? sum3_units(ms, *rope, dt) : 0;
    if (units3) {
        const GtChoice c = gt_pick(tiles, units, weights_us, gemm_max_split(a, rows, std::max(1, units / 4)), part_us * (float)rows, gs % GG_UNIT ? 6 : 7, kGgTiles, 3);
        if (c.splits > 1) best = c;
    }
    // To 64 tokens one matrix is also one sweep of the streaming kernels.  us, streaming / this (33 tokens unless given): 4096 x 512 7.0 / 8.9, x 1024 9.6 / 11.8,
    // x 2048 9.3 / 12.8, x 4096 15.5 / 15.8, x 5120 18.4 / 17.7, x 14336 22.3 / 24.7; 2048 x 14336 18.7 / 19.2, 1024 x 14336 48 tokens 15.7 / 21.6; 4608 x 14336 31.8 / 25.9;
    // 16384 x 2048 15.1 / 18.9, x 8192 45.7 / 37.9; 28672 x 8192 51 / 58; 64 tokens 4096 x 1024 8.0 / 12.2, 2048 x 3072 16.3 / 12.5
    if (n == 1 && a.T <= 64 && !silu && gptq_stream_us(a) <= gptq_gemm_us(best, a.T, weights_us)) return (int)hipErrorNotSupported;
    const GtTile& t = kGgTiles[best.tile];
    for (int i = 0; i < 3; ++i) g.a[i] = ms[i < n ? i : 0];
    g.n_m = (a.T + t.bm - 1) / t.bm; g.t_pad = (a.T + 255) / 256 * 256 + 256;   // (a DMA of the sums reads 256 tokens from the tile's first)
    g.units_per_split = (units + best.splits - 1) / best.splits;
    g.splits = (units + g.units_per_split - 1) / g.units_per_split;
    if (tiles(t) * g.splits > 0x7FFFFFFF) return (int)hipErrorNotSupported;
    // workspace: permuted x | sums | panels | partial sums
    const size_t xp_b = (size_t)a.T * a.K * 2, xs_b = (size_t)(a.K / 64) * g.t_pad * 4, pn_b = (size_t)words * 4;
    g.ldp = n == 1 ? a.N : (int)rows;
    for (int i = 1; i < n; ++i) g.col0[i] = g.col0[i - 1] + ms[i - 1].N;
    const size_t pt_b = g.splits > 1 ? (size_t)g.splits * a.T * g.ldp * 4 : 0;
    void* ws = nullptr;
    Mi355ScratchTurn turn(MI355_SCR_GPTQ_GEMM, st);
    if (mi355_scratch_get(&ws, MI355_SCR_GPTQ_GEMM, xp_b + xs_b + pn_b + pt_b, st, false, (size_t)(GPTQ_GEMM_X_BYTES + GEMM_PART_BYTES)))
        return n == 3 && pt_b ? gptq_prompt_gemm(ms, n, dt, st) : (int)hipErrorNotSupported;   // (no room while a stream is captured: token chunks)
    uint8_t* base = static_cast<uint8_t*>(ws);
    uint16_t* xp = reinterpret_cast<uint16_t*>(base);
    float* xs = reinterpret_cast<float*>(base + xp_b);
    uint32_t* panel = reinterpret_cast<uint32_t*>(base + xp_b + xs_b);
    g.xp = xp; g.xs = xs; g.part = reinterpret_cast<float*>(base + xp_b + xs_b + pn_b);
    for (int i = 0; i < n; ++i) { g.panel[i] = panel; panel += ((int64_t)(a.K / gs) * ms[i].N + 63) / 64 * 64; }
    gt_last_launch = 100 * best.tile + g.splits;
    const int rc = dt == MI355_DTYPE_BF16 ? gptq_gemm_dt<MI355_DTYPE_BF16>(g, xp, xs, best.tile, st) : gptq_gemm_dt<MI355_DTYPE_F16>(g, xp, xs, best.tile, st);
    if (rc || g.splits <= 1) return rc;
    if (n == 3) {
        DenseGemm3 s{};
        for (int i = 0; i < 3; ++i) { s.a[i] = ms[i]; s.col0[i] = g.col0[i]; }
        s.splits = g.splits; s.part = g.part; s.ldp = g.ldp;
        hipLaunchKernelGGL(sum3_rope_cache_kernel, dim3((unsigned)((units3 + 255) / 256)), dim3(256), 0, st, s, *rope, (int)units3);
        *roped = true;
        return (int)hipGetLastError();
    }
    if (dt == MI355_DTYPE_BF16 && resid_norm_tail<MI355_DTYPE_BF16>(a, g.part, a.N, g.splits, a.T, st)) return (int)hipGetLastError();
    const dim3 grid(((silu ? a.pair_offset : a.N) + 255) / 256, a.T);
    if (dt == MI355_DTYPE_BF16) hipLaunchKernelGGL((gptq_wide_epilogue_kernel<MI355_DTYPE_BF16>), grid, dim3(256), 0, st, a, g.part, a.N, g.splits, a.T);
    else hipLaunchKernelGGL((gptq_wide_epilogue_kernel<MI355_DTYPE_F16>), grid, dim3(256), 0, st, a, g.part, a.N, g.splits, a.T);
    return (int)hipGetLastError();
}

template <int DT, int EPI, int WM, int WN, int MF, int NF, int S, bool TILED>
static void dense_gemm_go(const DenseGemm3& g, hipStream_t st) {
    typedef GemmTile<DT, WM, WN, MF, NF, S, TILED> Tile;
    static Mi355DevOnce attr_done;
    if (!attr_done.done()) {
        (void)hipFuncSetAttribute((const void*)dense_gemm_kernel<DT, EPI, WM, WN, MF, NF, S, TILED>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)Tile::LDS);
        attr_done.set();
    }
    hipLaunchKernelGGL((dense_gemm_kernel<DT, EPI, WM, WN, MF, NF, S, TILED>), dim3(g.n_m * (g.tiles[0] + g.tiles[1] + g.tiles[2]) * g.splits), dim3(512), Tile::LDS, st, g);
}
template <int DT, int EPI, bool TILED>
static void dense_gemm_tile(const DenseGemm3& g, int which, hipStream_t st) {
#define DG_GO(WM_, WN_, MF_, NF_, S_) dense_gemm_go<DT, EPI, WM_, WN_, MF_, NF_, S_, TILED>(g, st)
    GT_TILES(which, DG_GO);
#undef DG_GO
}
template <int DT, bool TILED>
static void dense_gemm_epi(const DenseGemm3& g, int which, hipStream_t st) {
    if (g.a[0].epi == MI355_EPI_SILU_MUL) dense_gemm_tile<DT, MI355_EPI_SILU_MUL, TILED>(g, which, st);
    else if (g.a[0].epi == MI355_EPI_RESID) dense_gemm_tile<DT, MI355_EPI_RESID, TILED>(g, which, st);
    else dense_gemm_tile<DT, MI355_EPI_STORE, TILED>(g, which, st);
}
// Whether the streaming kernels make a 16-bit product sooner than the GEMM in its choice c, of those it would take below 65 tokens (33 .. 64; 17 .. 32 against 768
// row tiles).  With a row tile or two per CU they need one launch and a wave's share of K; the GEMM walks all units in one workgroup, or there is the partial sums'
// launch.  Both times as they were measured with the weights in HBM: the side taken is the faster one or within 5 % at 1064 of 1098 sizes (512 .. 32000 rows,
// k of 256 .. 18944, both layouts, with and without a residual).  us, streaming / GEMM: 33 tokens 4096 x 1024 6.6 / 9.6, x 2048 9.4 / 12.2, x 3072 11.7 / 13.9, x 5120
// 16.7 / 16.1; 2048 x 512 4.8 / 6.0, x 2048 8.8 / 9.9, x 3072 11.1 / 10.7; 48 tokens 4096 x 3072 13.4 / 14.5; 64 tokens 4096 x 1024 8.5 / 10.6, x 3072 16.6 / 15.1; two tiles per CU
// 33 tokens 8192 x 1024 9.2 / 10.1, 64 12.6 / 11.1; a residual adds 1 .. 2 to the streaming kernels and next to nothing to the GEMM, row-major weights 0.5 .. 2; a long K in ranges
// (few rows, activations shared through LDS) 48 tokens 1024 x 8192 14.0 / 15.8, 64 x 8192 12.4 / 11.1, row-major 1024 x 11008 19.0 / 16.9; 32 tokens 12288 x 512 7.3 / 8.1, x 1536
// 13.3 / 14.2, x 2048 17.6 / 17.5, row-major 12288 x 1024 11.8 / 10.7
static bool dense_streams(const DenseArgs& a, const GtChoice& c, float weights_us) {
    if (a.T > 64 || a.epi == MI355_EPI_SILU_MUL || (a.N & 15) || (a.K & 255)) return false;
    const int cus = mi355_num_cus(), tiles = a.N / 16, nkb = a.K >> 8, mt = (a.T + 15) / 16, rounds = (tiles + cus - 1) / cus;
    if (a.T <= 32) return a.K >= 512 && a.K <= (a.wtiled ? 1536 : tiles <= 4 * cus ? 512 : 0);
    if (mt == 3 && a.wtiled && a.K >= 8192 && tiles >= 32 && tiles * 4 <= cus) return true;
    if (rounds > 2) return false;
    const bool resid = a.epi == MI355_EPI_RESID;
    const int nw = dense_waves(tiles, nkb, mt);
    const float blocks = 0.5f * (float)((nkb + nw - 1) / nw) + 0.5f * (float)nkb / (float)nw;         // the slowest wave's, and the mean
    const float block = (mt == 3 ? 2.46f + 0.04f * (float)(a.T - 33) : 3.3f + 0.04f * (float)(a.T - 49)) + (a.wtiled ? 0.f : 0.7f);
    const float stream = 3.5f - (nw == 2 ? 1.5f : nw == 1 ? 1.4f : 0.f) + (rounds == 2 ? 0.8f : 0.3f * (float)a.N / 4096.f) +
                         block * (rounds == 2 ? 2.05f : 1.f) * blocks + (resid ? mt == 3 ? 1.35f : 1.75f : 0.f);
    const float cold = 1.3f * std::min(weights_us, 3.f);                                              // what of the weights' first bytes nothing hides
    const float gemm = c.splits == 1 ? 0.67f * c.us + 2.4f + cold + 0.02f * (float)(a.T - 33) + (resid ? 0.5f : 0.f)
                                     : 0.95f * c.us - (c.splits <= 3 ? 0.9f : 1.6f) + cold + 0.21f * (float)(c.splits - 1) + 0.03f * (float)(a.T - 33) + (resid ? 0.15f : 0.f);
    return stream <= gemm;
}
// n matrices over the same x: all tiled or all row-major, one dtype
static int dense_prompt_gemm(const DenseArgs* a, int n, int dt, hipStream_t st, const DenseRope* rope = nullptr, bool* roped = nullptr) {   // (rope: as gptq_prompt_gemm)
    if (dt != MI355_DTYPE_BF16 && dt != MI355_DTYPE_F16) return (int)hipErrorNotSupported;
    for (int i = 0; i < n; ++i) {
        if (a[i].K % 64 || a[i].T < 1 || a[i].N < 1 || a[i].wtiled != a[0].wtiled || a[i].epi != a[0].epi) return (int)hipErrorNotSupported;
        if ((a[i].ldx * 2) % 16 || (!a[i].wtiled && (a[i].ldw * 2) % 16) || (((uintptr_t)a[i].x | (uintptr_t)a[i].w) & 15)) return (int)hipErrorNotSupported;   // 16-byte DMA pieces
        if (a[i].epi == MI355_EPI_SILU_MUL && (a[i].pair_offset <= 0 || a[i].N != 2 * a[i].pair_offset)) return (int)hipErrorNotSupported;
        if (a[i].epi == MI355_EPI_SILU_MUL && a[i].wtiled && (a[i].pair_offset & 15)) return (int)hipErrorNotSupported;
        if ((int64_t)a[i].ldx * 512 >= (1ll << 32) || (int64_t)a[i].ldw * 512 >= (1ll << 32)) return (int)hipErrorNotSupported;   // 32-bit offsets inside a tile
    }
    auto tiles = [&](const GtTile& t, DenseGemm3* g) {
        int64_t cols = 0;
        for (int i = 0; i < 3; ++i) {
            const bool silu = i < n && a[i].epi == MI355_EPI_SILU_MUL;
            const int c = i >= n ? 0 : silu ? (a[i].pair_offset + t.bn / 2 - 1) / (t.bn / 2) : (a[i].N + t.bn - 1) / t.bn;
            if (g) g->tiles[i] = c;
            cols += c;
        }
        return cols * ((a[0].T + t.bm - 1) / t.bm);
    };
    const int units = a[0].K / 64;
    int64_t rows = 0;
    for (int i = 0; i < n; ++i) rows += a[i].N;
    // A split adds a write and a read of f32 partial sums and a launch; it needs whole groups of four columns.  us per launch (T x N x K) with
    // the 128 x 128 tile of four waves and two buffers drained at every step, and now: 3001 x 28672 x 4096 742 / 580 (256 x 256; 192 x 256 570,
    // 128 x 128 640), 3001 x 4096 x 14336 480 / 292 (192 x 256: exactly one round; 256 x 256 331), 2048 x 28672 x 4096 550 / 375,
    // 2048 x 4096 x 14336 215 (128 x 128, two per CU), 700 x 4096 x 14336 94 (two ranges; one: 175), 96 x 4096 x 14336 33 (64-token tiles,
    // eight ranges; one: 113), 64 x 28672 x 4096 96 / 44.
    const int max_split = n == 1 && a[0].T <= 65535 && !(a[0].N & 3) && !(a[0].epi == MI355_EPI_SILU_MUL && (a[0].pair_offset & 3)) ? gemm_max_split(a[0], a[0].N, std::max(1, units / 8)) : 1;
    const float weights_us = (float)rows * (float)a[0].K * 2.f / 5.4e6f;
    GtChoice best = gt_pick([&](const GtTile& t) { return tiles(t, nullptr); }, units, weights_us, max_split,
                            (float)a[0].T * (float)a[0].N * 4.f / 4.5e6f, 63);
    if (n == 1 && g_tune_gemm_min_t == DENSE_GEMM_MIN_T && !g_tune_gemm_tall && dense_streams(a[0], best, weights_us)) return (int)hipErrorNotSupported;
    const int64_t units3 = n == 3 && rope ? sum3_units(a, *rope, dt) : 0;
    if (units3) {
        const GtChoice c = gt_pick([&](const GtTile& t) { return tiles(t, nullptr); }, units, weights_us, gemm_max_split(a[0], rows, std::max(1, units / 8)),
                                   (float)a[0].T * (float)rows * 4.f / 4.5e6f, 63);
        if (c.splits > 1) best = c;
    }
    if (g_tune_gemm_tall) best = {0, 1, 0.f};
    DenseGemm3 g{};
    g.ldp = n == 1 ? a[0].N : (int)rows;
    for (int i = 1; i < n; ++i) g.col0[i] = g.col0[i - 1] + a[i - 1].N;
    for (int i = 0; i < 3; ++i) g.a[i] = a[i < n ? i : 0];
    g.n_m = (a[0].T + kGtTiles[best.tile].bm - 1) / kGtTiles[best.tile].bm;
    g.units_per_split = (units + best.splits - 1) / best.splits;
    g.splits = (units + g.units_per_split - 1) / g.units_per_split;
    Mi355ScratchTurn turn(MI355_SCR_GPTQ_WIDE, st);
    if (g.splits > 1) {
        void* p = nullptr;
        if (mi355_scratch_get(&p, MI355_SCR_GPTQ_WIDE, (size_t)g.splits * a[0].T * g.ldp * sizeof(float), st, false, (size_t)GEMM_PART_BYTES)) { g.splits = 1; g.units_per_split = units; }
        g.part = static_cast<float*>(p);
    }
    if (tiles(kGtTiles[best.tile], &g) * g.splits > 0x7FFFFFFF) return (int)hipErrorNotSupported;
    gt_last_launch = 100 * best.tile + g.splits;
    if (dt == MI355_DTYPE_BF16) { if (a[0].wtiled) dense_gemm_epi<MI355_DTYPE_BF16, true>(g, best.tile, st); else dense_gemm_epi<MI355_DTYPE_BF16, false>(g, best.tile, st); }
    else { if (a[0].wtiled) dense_gemm_epi<MI355_DTYPE_F16, true>(g, best.tile, st); else dense_gemm_epi<MI355_DTYPE_F16, false>(g, best.tile, st); }
    if (g.splits > 1 && n == 3) {
        hipLaunchKernelGGL(sum3_rope_cache_kernel, dim3((unsigned)((units3 + 255) / 256)), dim3(256), 0, st, g, *rope, (int)units3);
        *roped = true;
    } else if (g.splits > 1 && dt == MI355_DTYPE_BF16 && resid_norm_tail<MI355_DTYPE_BF16>(a[0], g.part, a[0].N, g.splits, a[0].T, st)) {
    } else if (g.splits > 1) {
        const int n_out = a[0].epi == MI355_EPI_SILU_MUL ? a[0].pair_offset : a[0].N;
        const dim3 grid((n_out + 255) / 256, a[0].T);
        if (dt == MI355_DTYPE_BF16) hipLaunchKernelGGL((gptq_wide_epilogue_kernel<MI355_DTYPE_BF16>), grid, dim3(256), 0, st, a[0], g.part, a[0].N, g.splits, a[0].T);
        else hipLaunchKernelGGL((gptq_wide_epilogue_kernel<MI355_DTYPE_F16>), grid, dim3(256), 0, st, a[0], g.part, a[0].N, g.splits, a[0].T);
    }
    return (int)hipGetLastError();
}

// x or w of a prompt that do not start on 16 bytes: the GEMM over copies that do (a pass over each, against a sweep of the weights per 64 tokens)
static int dense_prompt_gemm_staged(const DenseArgs& a, int dt, hipStream_t st) {
    DenseArgs c = a;
    const size_t x_b = ((size_t)(a.T - 1) * a.ldx + a.K) * 2, w_b = ((size_t)(a.N - 1) * a.ldw + a.K) * 2, x_room = (x_b + 255) & ~(size_t)255;
    const bool x_off = (uintptr_t)a.x & 15, w_off = (uintptr_t)a.w & 15;
    void* ws = nullptr;
    Mi355ScratchTurn turn(MI355_SCR_GPTQ_WIDE, st);                     // (the GEMM's, which takes it again)
    if ((!x_off && !w_off) || a.K % 64 || mi355_scratch_get(&ws, MI355_SCR_DENSE_WS, x_room + (w_off ? w_b : 0), st, false)) return (int)hipErrorNotSupported;
    uint8_t* base = static_cast<uint8_t*>(ws);
    hipError_t e = hipSuccess;
    if (x_off) { e = hipMemcpyAsync(base, a.x, x_b, hipMemcpyDeviceToDevice, st); c.x = base; }
    if (w_off && e == hipSuccess) { e = hipMemcpyAsync(base + x_room, a.w, w_b, hipMemcpyDeviceToDevice, st); c.w = base + x_room; }
    return e != hipSuccess ? (int)e : dense_prompt_gemm(&c, 1, dt, st);
}

// SILU_MUL with more than 32 tokens, or any T > 64: run in token chunks
static int dense_run(DenseArgs a, int wtype, int dt, hipStream_t st) {
    // (rows and k that are not whole tiles of the streaming kernels are served from DENSE_GEMM_ANY_T tokens, and refused below)
    const bool whole = !(a.N & 15) && !(a.K & 255);
    if (wtype == DW_DENSE && (a.T >= DENSE_GEMM_ANY_T || whole) &&
        (a.T >= g_tune_gemm_min_t || (g_tune_gemm_min_t == DENSE_GEMM_MIN_T && a.T > 16 && (a.epi == MI355_EPI_SILU_MUL ? a.pair_offset : a.N) >= 16 * 768))) {
        int rc = dense_prompt_gemm(&a, 1, dt, st);
        if (rc == (int)hipErrorNotSupported && a.T >= DENSE_GEMM_ANY_T) rc = dense_prompt_gemm_staged(a, dt, st);
        if (rc != (int)hipErrorNotSupported) return rc;                    // odd K, few tokens off the 16-byte grid: keep streaming in token chunks
    }
    if (wtype == DW_GPTQ4T && a.T >= (a.epi == MI355_EPI_SILU_MUL ? GPTQ_GEMM_MIN_PAIR_T : GPTQ_GEMM_MIN_T)) {
        const int slab = gptq_gemm_slab(a.K);
        if (a.T > slab) {
            for (int t0 = 0; t0 < a.T; t0 += slab)
                if (const int rc = dense_run(dense_rows(a, t0, slab), wtype, dt, st)) return rc;
            return 0;
        }
        const int rc = gptq_prompt_gemm(&a, 1, dt, st);
        if (rc != (int)hipErrorNotSupported) return rc;                    // groups of 32, odd strides: token chunks of the decode kernel
    }
    const int chunk = a.epi == MI355_EPI_SILU_MUL ? 32 : 64;
    const int T = a.T;
    if (T < 1) return -2;
    for (int t0 = 0; t0 < T; t0 += chunk) {
        const int rc = dense_dispatch(dense_rows(a, t0, chunk), wtype, dt, st);
        if (rc) return rc;
    }
    return 0;
}

// ------------------------------------------------------------------------------------------------ K15 repack
// 16-bit [N][ld_in] row-major -> the tiled image (dense_tile_index): one thread per 16-byte chunk of the output
__global__ void __launch_bounds__(256) dense_tile_kernel(const uint16_t* __restrict__ in, uint16_t* __restrict__ out, int N, int K, int64_t ld_in) {
    const size_t o = (size_t)blockIdx.x * blockDim.x + threadIdx.x;                 // chunk index = (((tile * nkb + kb) * 8 + j) * 64 + lane)
    const int nkb = K >> 8;
    if (o >= (size_t)(N >> 4) * nkb * 512) return;
    const int lane = (int)(o & 63), j = (int)((o >> 6) & 7);
    const size_t tk = o >> 9;
    const int kb = (int)(tk % nkb), tile = (int)(tk / nkb);
    const int n = tile * 16 + (lane & 15), k = kb * 256 + j * 32 + (lane >> 4) * 8;
    *reinterpret_cast<uint4*>(out + o * 8) = *reinterpret_cast<const uint4*>(in + (size_t)n * ld_in + k);
}
// checkpoint layout [K/8][n_in] (columns [0, n_in)) -> tiles tile0 .. of the tiled image (gptq_tile_index); K % 256 == 0, n_in % 16 == 0
__global__ void gptq_tile_kernel(const uint32_t* __restrict__ in, uint32_t* __restrict__ out, int K, int n_in, int tile0) {
    const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (size_t)(K / 8) * n_in) return;
    const int n = (int)(idx % n_in), kr = (int)(idx / n_in);
    out[gptq_tile_index(kr, n + 16 * tile0, K >> 8)] = in[idx];
}
// the inverse (tests / the exllama arm of a model that changes its mind): tiled image -> [K/8][N]
__global__ void gptq_untile_kernel(const uint32_t* __restrict__ in, uint32_t* __restrict__ out, int K, int N) {
    const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (size_t)(K / 8) * N) return;
    out[idx] = in[gptq_tile_index((int)(idx / N), (int)(idx % N), K >> 8)];
}
static inline bool gptq_tileable(int k, int n) { return k > 0 && n > 0 && !(k & 255) && !(n & 15); }

__global__ void awq_repack_kernel(const uint32_t* __restrict__ in, uint32_t* __restrict__ out, int K, int NP, int tiled) {
    // in [K][NP] : nibble i of in[k][c] = code(k, 8c + {0,2,4,6,1,3,5,7}[i])   [EXT: AutoAWQ order_map]
    // out [K/8][8 NP] : nibble i of out[kr][n] = code(8kr + i, n), stored at gptq_tile_index(kr, n) when `tiled`
    const int N = NP * 8;
    const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (size_t)(K / 8) * N) return;
    const int n = (int)(idx % N), kr = (int)(idx / N);
    const int u = n & 7;
    const int pos = ((u & 1) << 2) | (u >> 1);
    uint32_t o = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) o |= ((in[(size_t)(8 * kr + i) * NP + (n >> 3)] >> (4 * pos)) & 0xFu) << (4 * i);
    out[tiled ? gptq_tile_index(kr, n, K >> 8) : idx] = o;
}

// ------------------------------------------------------------------------------------------------ K14 exllama
// act-order GPTQ: every k has its own group g_idx[k], so the scale cannot be factored out of an MFMA chain; the
// weights are dequantised to f16 (w = s * (q - (z+1)) rounded to f16, as a half-precision dequant kernel does)
// and contracted on MFMA.  One workgroup per 16-column tile, its 4 waves split K.
template <int MT, int BITS>
__global__ void __launch_bounds__(256) exllama_kernel(const uint16_t* __restrict__ x, const uint32_t* __restrict__ qw,
                                                      const uint32_t* __restrict__ qz, const uint16_t* __restrict__ sc,
                                                      const int32_t* __restrict__ g_idx, uint16_t* __restrict__ out,
                                                      int T, int N, int K, int group_size) {
    __shared__ float red[4][MT][16][16];
    constexpr int PF = 32 / BITS;                                   // codes per u32: 8 (4-bit) or 4 (8-bit, linear.rs:215-217)
    constexpr uint32_t QM = (1u << BITS) - 1u;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int r16 = lane & 15, kg = lane >> 4;
    const int col = blockIdx.x * 16 + r16;
    f32x4_t y[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) y[mt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    for (int k32 = wave; k32 < K / 32; k32 += 4) {
        const int k0 = k32 * 32 + 8 * kg;
        uint32_t w[8 / PF];                                         // the 8 consecutive k of this lane: 1 word (4-bit) / 2 words (8-bit)
#pragma unroll
        for (int u = 0; u < 8 / PF; ++u) w[u] = qw[(size_t)(k0 / PF + u) * N + col];
        f16x8_t bf;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int g = g_idx ? g_idx[k0 + i] : (k0 + i) / group_size;
            const float s = f16_bits_to_f32(sc[(size_t)g * N + col]);
            const int z = (int)((qz[(size_t)g * (N / PF) + col / PF] >> (BITS * (col % PF))) & QM) + 1;
            bf[i] = (_Float16)(s * (float)((int)((w[i / PF] >> (BITS * (i % PF))) & QM) - z));
        }
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            const int m = min(mt * 16 + r16, T - 1);
            const f16x8_t af = *reinterpret_cast<const f16x8_t*>(x + (size_t)m * K + k0);
            y[mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af, bf, y[mt], 0, 0, 0);
        }
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int v = 0; v < 4; ++v) red[wave][mt][4 * kg + v][r16] = y[mt][v];
    __syncthreads();
    for (int idx = threadIdx.x; idx < MT * 256; idx += 256) {
        const int rr = idx & 15, m = idx >> 4;
        if (m >= T) continue;
        const float s = red[0][m >> 4][m & 15][rr] + red[1][m >> 4][m & 15][rr] + red[2][m >> 4][m & 15][rr] + red[3][m >> 4][m & 15][rr];
        out[(size_t)m * N + blockIdx.x * 16 + rr] = f32_to_f16_bits(s);
    }
}

// ------------------------------------------------------------------------------------------------ Marlin-format checkpoints
// `checkpoint_format == "marlin"` (linear.rs:222-239,279-290): the file holds B [k/16, 2n] u32 already in the Marlin
// tile order (IST-DASLab marlin `Layer.pack` [EXT]): codes (k, n) -> 16x16 tiles, tile-row major; every 1024
// consecutive values of a tile row (4 tiles) permuted by `_perm`, then 8 values per word with the nibble
// interleave [0,2,4,6,1,3,5,7].  The reference hands B to marlin_4bit_* without a repack; this path's mat-mul streams
// the GPTQ layout qweight[k/8][n], so a Marlin-format B is un-permuted ONCE at load time.
//   perm1(i)[4*blk + e] = 16*row_e(i) + i/4 + 8*blk,  row_e = {2(i%4), 2(i%4)+1, 2(i%4+4), 2(i%4+4)+1}
//   perm = concat_i concat_j (perm1(i) + 256 j), then within every 8: [0,2,4,6,1,3,5,7]
__device__ __forceinline__ int marlin_perm_at(int j) {              // j in [0,1024): source index inside the 1024 chunk
    const int e8 = j & 7, grp = j >> 3;                             // 8-group; interleave picks element {0,2,4,6,1,3,5,7}[e8]
    const int src8 = (e8 < 4) ? 2 * e8 : 2 * (e8 - 4) + 1;
    const int q = grp * 8 + src8;                                   // index into the un-interleaved perm
    const int i = q >> 5, jj = (q >> 3) & 3, t = q & 7;             // 32 entries per i: 4 (j) x 8 (perm1)
    const int blk = t >> 2, e = t & 3;
    const int r = (e < 2) ? 2 * (i & 3) + e : 2 * ((i & 3) + 4) + (e - 2);
    return 16 * r + (i >> 2) + 8 * blk + 256 * jj;
}
__global__ void __launch_bounds__(256) marlin_to_gptq_kernel(const uint32_t* __restrict__ B, uint32_t* __restrict__ out, int K, int N, int tiled) {
    __shared__ uint16_t inv[1024];
    for (int j = threadIdx.x; j < 1024; j += 256) inv[marlin_perm_at(j)] = (uint16_t)j;
    __syncthreads();
    const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (size_t)(K / 8) * N) return;
    const int n = (int)(idx % N), kr = (int)(idx / N);
    uint32_t o = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int k = 8 * kr + i;
        const int src = (n >> 4) * 256 + (k & 15) * 16 + (n & 15);  // position inside tile row k/16 before the permutation
        const int col = (src & ~1023) + inv[src & 1023];
        o |= ((B[(size_t)(k >> 4) * (2 * N) + (col >> 3)] >> (4 * (col & 7))) & 0xFu) << (4 * i);
    }
    out[tiled ? gptq_tile_index(kr, n, K >> 8) : idx] = o;
}

// ------------------------------------------------------------------------------------------------ C ABI
static int marlin_common(const void* in, const int32_t* qweight, const void* scales, const void* zeros, void* out,
                         int m, int k, int n, int group_size, int dt, int awq, int64_t stream) {
    DenseArgs a{};
    a.w = qweight; a.scales = scales;
    a.group_size = (group_size <= 0 || group_size > k) ? k : group_size;
    a.sperm = a.group_size < k ? SP_GROUPED : SP_SINGLE;
    a.qzeros = awq ? static_cast<const uint32_t*>(zeros) : nullptr;
    a.zmode = awq ? MI355_ZERO_AWQ_MARLIN : MI355_ZERO_SYM8;
    a.x = in; a.ldx = k; a.T = m; a.N = n; a.K = k;
    a.out = out; a.ldo = n; a.epi = MI355_EPI_STORE;
    return dense_run(a, DW_GPTQ4T, dt, (hipStream_t)stream);          // the image gptq_repack / awq_repack / mi355_marlin_format_repack made
}

template <int BITS>
static void exllama_launch(const uint16_t* x, const uint32_t* qw, const uint32_t* qz, const uint16_t* sc, const int32_t* g_idx,
                           uint16_t* o, int T, int n, int k, hipStream_t st) {
    // without g_idx the whole of k is one group: the op does not pass group_size, and the reference always loads g_idx
    // for gptq checkpoints (linear.rs:298-314)
    if (T <= 16) hipLaunchKernelGGL((exllama_kernel<1, BITS>), dim3(n / 16), dim3(256), 0, st, x, qw, qz, sc, g_idx, o, T, n, k, k);
    else hipLaunchKernelGGL((exllama_kernel<2, BITS>), dim3(n / 16), dim3(256), 0, st, x, qw, qz, sc, g_idx, o, T, n, k, k);
}
extern "C" {

// The reference's FFI symbols return nothing.  A call this library cannot serve must not leave the caller with an
// uninitialised output that looks like data: the failure is recorded (mi355_last_error) and the output is filled with
// 0xFFFF (NaN in f16 and bf16) whenever its pointer and shape are usable.
static void ffi_fail(int code, void* out, int64_t m, int64_t n, int64_t stream) {
    mi355_note_error(code ? code : (int)hipErrorInvalidValue);
    if (out && m > 0 && n > 0) (void)hipMemsetAsync(out, 0xFF, (size_t)m * n * 2, (hipStream_t)stream);
}
static void marlin_ffi(const void* in, const int32_t* qweight, const void* scales, const void* zeros, void* out, int m, int k, int n,
                       int group_size, int dt, int awq, int64_t stream) {
    if (m == 0) return;
    if (!in || !qweight || !scales || !out || m < 0 || k <= 0 || n <= 0 || (k & 255) || (n & 15) || (awq && !zeros)) {
        ffi_fail((int)hipErrorInvalidValue, out, m, n, stream);
        return;
    }
    const int rc = marlin_common(in, qweight, scales, zeros, out, m, k, n, group_size, dt, awq, stream);
    if (rc) ffi_fail(rc, out, m, n, stream);
}
void marlin_4bit_f16(const void* in, const int32_t* qweight, const void* scales, const void* zeros, const void* g_idx,
                     void* out, int32_t m, int32_t k, int32_t n, const void* workspace, int32_t group_size, int64_t stream) {
    (void)g_idx; (void)workspace;
    marlin_ffi(in, qweight, scales, zeros, out, m, k, n, group_size, MI355_DTYPE_F16, 0, stream);
}
void marlin_4bit_bf16(const void* in, const int32_t* qweight, const void* scales, const void* zeros, const void* g_idx,
                      void* out, int32_t m, int32_t k, int32_t n, const void* workspace, int32_t group_size, int64_t stream) {
    (void)g_idx; (void)workspace;
    marlin_ffi(in, qweight, scales, zeros, out, m, k, n, group_size, MI355_DTYPE_BF16, 0, stream);
}
void marlin_awq_4bit_f16(const void* in, const int32_t* qweight, const void* scales, const void* zeros, const void* g_idx,
                         void* out, int32_t m, int32_t k, int32_t n, const void* workspace, int32_t group_size, int64_t stream) {
    (void)g_idx; (void)workspace;
    marlin_ffi(in, qweight, scales, zeros, out, m, k, n, group_size, MI355_DTYPE_F16, 1, stream);
}
void marlin_awq_4bit_bf16(const void* in, const int32_t* qweight, const void* scales, const void* zeros, const void* g_idx,
                          void* out, int32_t m, int32_t k, int32_t n, const void* workspace, int32_t group_size, int64_t stream) {
    (void)g_idx; (void)workspace;
    marlin_ffi(in, qweight, scales, zeros, out, m, k, n, group_size, MI355_DTYPE_BF16, 1, stream);
}

void gemm_half_q_half_alt(const void* a, const uint32_t* b_q_weight, const uint32_t* b_gptq_qzeros, const void* b_gptq_scales,
                          const int32_t* b_g_idx, void* c, int32_t m, int32_t n, int32_t k, int32_t bit, int64_t stream) {
    if (m == 0) return;
    // the reference admits 4 | 8 bits on this arm (linear.rs:215-217) and forwards `bits` (gptq.rs:181-194)
    if ((bit != 4 && bit != 8) || !a || !b_q_weight || !b_gptq_qzeros || !b_gptq_scales || !c || m < 0 || n <= 0 || k <= 0 ||
        (n & 15) || (k & 31)) {
        ffi_fail((int)hipErrorInvalidValue, c, m, n, stream);
        return;
    }
    hipStream_t st = (hipStream_t)stream;
    for (int t0 = 0; t0 < m; t0 += 32) {
        const int T = m - t0 < 32 ? m - t0 : 32;
        const uint16_t* x = static_cast<const uint16_t*>(a) + (size_t)t0 * k;
        uint16_t* o = static_cast<uint16_t*>(c) + (size_t)t0 * n;
        if (bit == 4) exllama_launch<4>(x, b_q_weight, b_gptq_qzeros, static_cast<const uint16_t*>(b_gptq_scales), b_g_idx, o, T, n, k, st);
        else exllama_launch<8>(x, b_q_weight, b_gptq_qzeros, static_cast<const uint16_t*>(b_gptq_scales), b_g_idx, o, T, n, k, st);
    }
    const int rc = (int)hipGetLastError();
    if (rc) ffi_fail(rc, c, m, n, stream);
}

/* gptq_repack (marlin gptq_marlin_repack.cu's slot, linear.rs:845-853): checkpoint qweight [k/8][n] -> the weight image the
 * marlin_* entry points stream.  Every shape those entry points accept (k % 256 == 0, n % 16 == 0) gets the 16 x 256 tile order
 * (gptq_tile_index); any other shape is copied as is (marlin_* refuses it loudly either way).  in != out. */
void gptq_repack(const void* in, void* out, int32_t k_packed, int32_t n, int64_t stream) {
    if (!in || !out || k_packed <= 0 || n <= 0 || in == out) { mi355_note_error((int)hipErrorInvalidValue); return; }
    if (gptq_tileable(k_packed * 8, n)) {
        const size_t total = (size_t)k_packed * n;
        hipLaunchKernelGGL(gptq_tile_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                           static_cast<const uint32_t*>(in), static_cast<uint32_t*>(out), k_packed * 8, n, 0);
        const int rc = (int)hipGetLastError();
        if (rc) mi355_note_error(rc);
        return;
    }
    const hipError_t e = hipMemcpyAsync(out, in, (size_t)k_packed * n * sizeof(uint32_t), hipMemcpyDeviceToDevice, (hipStream_t)stream);
    if (e != hipSuccess) mi355_note_error((int)e);
}
/* the tile order on its own: columns [0, n_in) of a checkpoint-layout tensor -> tiles tile0 .. of `out` (a tensor of any width
 * >= 16 (tile0 + n_in / 16)): the host layer packs gate_proj and up_proj side by side this way.  And its inverse. */
int mi355_gptq_tile_repack(const void* in, void* out, int32_t k, int32_t n_in, int32_t tile0, int64_t stream) {
    if (!in || !out || in == out || !gptq_tileable(k, n_in) || tile0 < 0) return (int)hipErrorInvalidValue;
    const size_t total = (size_t)(k / 8) * n_in;
    hipLaunchKernelGGL(gptq_tile_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                       static_cast<const uint32_t*>(in), static_cast<uint32_t*>(out), k, n_in, tile0);
    return (int)hipGetLastError();
}
int mi355_gptq_tile_unpack(const void* in, void* out, int32_t k, int32_t n, int64_t stream) {
    if (!in || !out || in == out || !gptq_tileable(k, n)) return (int)hipErrorInvalidValue;
    const size_t total = (size_t)(k / 8) * n;
    hipLaunchKernelGGL(gptq_untile_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                       static_cast<const uint32_t*>(in), static_cast<uint32_t*>(out), k, n);
    return (int)hipGetLastError();
}
void awq_repack(const void* in, void* out, int32_t k, int32_t n_packed, int32_t bits, int64_t stream) {
    if (bits != 4 || (k & 7) || !in || !out || k <= 0 || n_packed <= 0) {
        // the output is a weight image, not activations: poison it as NaN-scaled codes cannot be expressed -- record and leave
        mi355_note_error((int)hipErrorInvalidValue);
        return;
    }
    const size_t total = (size_t)(k / 8) * n_packed * 8;
    hipLaunchKernelGGL(awq_repack_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                       static_cast<const uint32_t*>(in), static_cast<uint32_t*>(out), k, n_packed, gptq_tileable(k, n_packed * 8) ? 1 : 0);
    const int rc = (int)hipGetLastError();
    if (rc) mi355_note_error(rc);
}

/* Marlin-FORMAT checkpoint weight B [k/16, 2n] u32 -> the layout the marlin_* entry points stream ([k/8][n] u32).  The
 * integration calls this once per tensor on the `marlin_format` branch of qlinear (linear.rs:279-290), where the reference
 * passes B through untouched. */
int mi355_marlin_format_repack(const void* in_B, void* out, int32_t k, int32_t n, int64_t stream) {
    if (!in_B || !out || k <= 0 || n <= 0 || (k & 15) || (n & 63)) return (int)hipErrorInvalidValue;
    const size_t total = (size_t)(k / 8) * n;
    hipLaunchKernelGGL(marlin_to_gptq_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                       static_cast<const uint32_t*>(in_B), static_cast<uint32_t*>(out), k, n, gptq_tileable(k, n) ? 1 : 0);
    return (int)hipGetLastError();
}
/* host statement of the tile order (unit-tested on CPU against oracle/gptq.py's gptq_tile); -1 for a shape that is not tiled */
int64_t mi355_gptq_tile_index(int32_t kr, int32_t n, int32_t k, int32_t n_total) {
    if (!gptq_tileable(k, n_total) || kr < 0 || kr >= k / 8 || n < 0 || n >= n_total) return -1;
    return (int64_t)gptq_tile_index(kr, n, k >> 8);
}
/* host statement of the same permutation (unit-tested on CPU against the numpy restatement of marlin's `_get_perms`) */
int32_t mi355_marlin_weight_perm(int32_t j) {
    if (j < 0 || j >= 1024) return -1;
    const int e8 = j & 7, grp = j >> 3;
    const int src8 = (e8 < 4) ? 2 * e8 : 2 * (e8 - 4) + 1;
    const int q = grp * 8 + src8;
    const int i = q >> 5, jj = (q >> 3) & 3, t = q & 7;
    const int blk = t >> 2, e = t & 3;
    const int r = (e < 2) ? 2 * (i & 3) + e : 2 * ((i & 3) + 4) + (e - 2);
    return 16 * r + (i >> 2) + 8 * blk + 256 * jj;
}

/* host-side index arithmetic of the Marlin permutations (unit-tested on CPU against the reference's Python) */
int32_t mi355_marlin_scale_pos(int32_t n, int32_t grouped) { return marlin_scale_pos(n, grouped ? SP_GROUPED : SP_SINGLE); }
int32_t mi355_marlin_zero_pos(int32_t n) {
    const int p1 = marlin_scale_pos(n, SP_GROUPED);
    const int u = p1 & 7;
    return (p1 & ~7) + (((u & 1) << 2) | (u >> 1));
}

/* 16-bit weights [n][k] (row stride ld_in elements) -> the 16-row x 256-k tile image mi355_linear_tiled streams; in != out */
int mi355_dense_tile_repack(const void* in, void* out, int32_t n, int32_t k, int64_t ld_in, int64_t stream) {
    if (!in || !out || in == out || n <= 0 || k <= 0 || (n & 15) || (k & 255) || ld_in < k || (ld_in & 7) || ((uintptr_t)in & 15) || ((uintptr_t)out & 15))
        return (int)hipErrorInvalidValue;
    const size_t chunks = (size_t)(n >> 4) * (k >> 8) * 512;
    hipLaunchKernelGGL(dense_tile_kernel, dim3((unsigned)((chunks + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                       static_cast<const uint16_t*>(in), static_cast<uint16_t*>(out), n, k, ld_in);
    return (int)hipGetLastError();
}
/* host statement of the tile order (element index of w[n][k]; -1 for a shape that is not tiled) */
int64_t mi355_dense_tile_index(int32_t n_row, int32_t k_col, int32_t n, int32_t k) {
    if (n <= 0 || k <= 0 || (n & 15) || (k & 255) || n_row < 0 || n_row >= n || k_col < 0 || k_col >= k) return -1;
    return (int64_t)dense_tile_index(n_row, k_col, k >> 8);
}
static int linear_impl(int tiled, void* out, const void* x, const void* w, const void* bias, const void* residual, int32_t num_tokens,
                       int32_t n, int32_t k, int32_t dtype, int32_t epilogue, int64_t stream) {
    if (tiled && ((n & 15) || (k & 255))) return -2;
    DenseArgs a{};
    a.w = w; a.ldw = k; a.wtiled = tiled;
    a.x = x; a.ldx = k; a.T = num_tokens; a.K = k; a.N = n;
    a.bias = bias; a.resid = residual; a.epi = epilogue; a.out = out;
    if (epilogue == MI355_EPI_SILU_MUL) { a.pair_offset = n / 2; a.ldo = n / 2; } else a.ldo = n;
    if (epilogue == MI355_EPI_RESID && !residual) return -2;
    return dense_run(a, DW_DENSE, dtype, (hipStream_t)stream);
}
/* `Linear::forward` over the tiled weight image (mi355_dense_tile_repack); everything else as mi355_linear */
int mi355_linear_tiled(void* out, const void* x, const void* w_tiled, const void* bias, const void* residual, int32_t num_tokens,
                       int32_t n, int32_t k, int32_t dtype, int32_t epilogue, int64_t stream) {
    return linear_impl(1, out, x, w_tiled, bias, residual, num_tokens, n, k, dtype, epilogue, stream);
}
int mi355_linear(void* out, const void* x, const void* w, const void* bias, const void* residual, int32_t num_tokens,
                 int32_t n, int32_t k, int32_t dtype, int32_t epilogue, int64_t stream) {
    DenseArgs a{};
    a.w = w; a.ldw = k; a.x = x; a.ldx = k; a.T = num_tokens; a.K = k; a.N = n;
    a.bias = bias; a.resid = residual; a.epi = epilogue; a.out = out;
    if (epilogue == MI355_EPI_SILU_MUL) { a.pair_offset = n / 2; a.ldo = n / 2; } else a.ldo = n;
    if (epilogue == MI355_EPI_RESID && !residual) return -2;
    return dense_run(a, DW_DENSE, dtype, (hipStream_t)stream);
}

/* a residual product and the RmsNorm behind it: out = residual + x . w^T as mi355_linear / _linear_tiled / _gptq_linear_tiled (kind 0, 1, 2; symmetric
 * zero points); *normed != 0: norm_out holds the norm of out too (else the caller makes it).  Internal to the host layer. */
int mi355_internal_resid_norm_linear(void* out, const void* x, const void* w, const void* scales, const void* residual, int32_t num_tokens, int32_t n, int32_t k,
                                     int32_t group_size, int32_t kind, int32_t dtype, void* norm_out, const void* norm_w, float eps, int32_t* normed, int64_t stream) {
    if (!residual || !norm_out || !norm_w || !normed || num_tokens < 1 || kind < 0 || kind > 2) return -1;
    DenseNormTail tail{norm_out, norm_w, eps, false};
    DenseArgs a{};
    a.w = w; a.ldw = k; a.wtiled = kind == 1; a.scales = scales; a.zmode = kind == 2 ? MI355_ZERO_SYM8 : 0; a.sperm = SP_NONE;
    a.group_size = (group_size <= 0 || group_size > k) ? k : group_size;
    a.x = x; a.ldx = k; a.T = num_tokens; a.K = k; a.N = n; a.resid = residual; a.epi = MI355_EPI_RESID; a.out = out; a.ldo = n;
    a.tail = &tail;
    const int rc = dense_run(a, kind == 2 ? DW_GPTQ4T : DW_DENSE, dtype, (hipStream_t)stream);
    *normed = tail.done;
    return rc;
}

static int gptq_linear_impl(int wtype, void* out, const void* x, const void* qweight, const void* scales, const void* qzeros,
                            int32_t zero_mode, int32_t scales_permuted, const void* bias, const void* residual,
                            int32_t num_tokens, int32_t n, int32_t k, int32_t group_size, int32_t dtype, int32_t epilogue,
                            int64_t stream) {
    DenseArgs a{};
    a.w = qweight; a.scales = scales; a.qzeros = static_cast<const uint32_t*>(qzeros); a.zmode = zero_mode;
    a.group_size = (group_size <= 0 || group_size > k) ? k : group_size;
    a.sperm = !scales_permuted ? SP_NONE : (a.group_size < k ? SP_GROUPED : SP_SINGLE);
    a.x = x; a.ldx = k; a.T = num_tokens; a.K = k; a.N = n;
    a.bias = bias; a.resid = residual; a.epi = epilogue; a.out = out;
    if (epilogue == MI355_EPI_SILU_MUL) { a.pair_offset = n / 2; a.ldo = n / 2; } else a.ldo = n;
    if (epilogue == MI355_EPI_RESID && !residual) return -2;
    return dense_run(a, wtype, dtype, (hipStream_t)stream);
}
int mi355_gptq_linear(void* out, const void* x, const void* qweight, const void* scales, const void* qzeros,
                      int32_t zero_mode, int32_t scales_permuted, const void* bias, const void* residual,
                      int32_t num_tokens, int32_t n, int32_t k, int32_t group_size, int32_t dtype, int32_t epilogue,
                      int64_t stream) {
    return gptq_linear_impl(DW_GPTQ4, out, x, qweight, scales, qzeros, zero_mode, scales_permuted, bias, residual, num_tokens, n, k,
                            group_size, dtype, epilogue, stream);
}
/* host layer only: the tiled sym-8 op on the 1..4-token kernel, with its two extras: RmsNorm(norm_w, eps) applied to x on the
 * way in (inv from `ss_in`, the per-tile sums of squares the producer of x left behind) and `ss_out`, the same sums of this
 * launch's own output rows for the next consumer.  -4 when the shape is not served by that kernel: the caller then norms
 * separately, calls mi355_gptq_linear_tiled, and treats ss_out as not written. */
int mi355_internal_gptq_small_linear(void* out, const void* x, const void* qweight_tiled, const void* scales, const void* bias,
                                     const void* residual, const void* norm_w, float norm_eps, const float* ss_in, float* ss_out,
                                     int32_t num_tokens, int32_t n, int32_t k, int32_t group_size, int32_t dtype, int32_t epilogue,
                                     int64_t stream) {
    if (num_tokens < 1 || num_tokens > 4 || (epilogue == MI355_EPI_RESID && !residual)) return -4;
    DenseArgs a{};
    a.w = qweight_tiled; a.scales = scales; a.zmode = MI355_ZERO_SYM8;
    a.group_size = (group_size <= 0 || group_size > k) ? k : group_size;
    a.sperm = SP_NONE;
    a.x = x; a.ldx = k; a.T = num_tokens; a.K = k; a.N = n;
    a.bias = bias; a.resid = residual; a.epi = epilogue; a.out = out;
    a.norm_w = norm_w; a.norm_eps = norm_eps; a.ss_in = ss_in; a.ss_out = ss_out;
    if (epilogue == MI355_EPI_SILU_MUL) { a.pair_offset = n / 2; a.ldo = n / 2; } else a.ldo = n;
    hipStream_t st = (hipStream_t)stream;
    if (dtype == MI355_DTYPE_BF16) return dense_small_launch<MI355_DTYPE_BF16, DW_GPTQ4T>(a, st);
    if (dtype == MI355_DTYPE_F16) return dense_small_launch<MI355_DTYPE_F16, DW_GPTQ4T>(a, st);
    return -4;
}
/* the same op over the TILED weight image (gptq_repack / mi355_gptq_tile_repack); scales and zero points as above */
int mi355_gptq_linear_tiled(void* out, const void* x, const void* qweight_tiled, const void* scales, const void* qzeros,
                            int32_t zero_mode, int32_t scales_permuted, const void* bias, const void* residual,
                            int32_t num_tokens, int32_t n, int32_t k, int32_t group_size, int32_t dtype, int32_t epilogue,
                            int64_t stream) {
    return gptq_linear_impl(DW_GPTQ4T, out, x, qweight_tiled, scales, qzeros, zero_mode, scales_permuted, bias, residual, num_tokens,
                            n, k, group_size, dtype, epilogue, stream);
}

int mi355_internal_linear3_prompt(void* const* outs, const void* x, const void* const* ws, const void* const* scales,
                                  const void* const* biases, const int32_t* ns, int32_t num_tokens, int32_t k, int32_t group_size,
                                  int32_t is_gptq, int32_t dtype, const void* norm_w, float norm_eps, const float* ss_in, const void* rope,
                                  const void* prompt_rope, int32_t* roped, int64_t stream);
/* q, k, v projections (plain store epilogue, optional bias) in one launch; returns -4 when the shapes do not qualify
 * (the caller then issues three mi355_linear / mi355_gptq_linear calls).  norm_w != NULL: x is the residual stream and the
 * launch applies RmsNorm(norm_w, eps) on the way in, inv from the producer's sums of squares `ss_in` (1..4 tokens of 4-bit
 * weights only; -4 otherwise and the caller norms separately).  rope != NULL (a DenseRope): the launch also rotates q and k
 * and writes k and v into the layer's bf16 cache -- the work of mi355_internal_rope_cache -- in its epilogue (same kernel only;
 * -4 otherwise and the caller keeps the separate launch).  Internal to the host layer (dense_model.cpp). */
int mi355_internal_linear3(void* const* outs, const void* x, const void* const* ws, const void* const* scales,
                           const void* const* biases, const int32_t* ns, int32_t num_tokens, int32_t k, int32_t group_size,
                           int32_t is_gptq, int32_t dtype, const void* norm_w, float norm_eps, const float* ss_in, const void* rope,
                           int64_t stream) {
    return mi355_internal_linear3_prompt(outs, x, ws, scales, biases, ns, num_tokens, k, group_size, is_gptq, dtype, norm_w, norm_eps, ss_in, rope, nullptr, nullptr, stream);
}
/* the same for a prompt step (rope NULL): *roped != 0: the launch also rotated q and wrote the rotated k and v into the cache as prompt_rope says (k's and v's outs are not
 * written then); else the caller does */
int mi355_internal_linear3_prompt(void* const* outs, const void* x, const void* const* ws, const void* const* scales,
                                  const void* const* biases, const int32_t* ns, int32_t num_tokens, int32_t k, int32_t group_size,
                                  int32_t is_gptq, int32_t dtype, const void* norm_w, float norm_eps, const float* ss_in, const void* rope,
                                  const void* prompt_rope, int32_t* roped, int64_t stream) {
    if (roped) *roped = 0;
    // One GEMM launch for the three (K in one range), or the streaming kernel over all their row tiles (to 64 tokens).  us, streaming / GEMM, weights from HBM
    // (q + k + v rows x k): 16-bit 2048 + 2 x 512 x 2048 33 tokens 9.3 / 11.0, 49 11.4 / 16.0, 64 12.9 / 17.0; 3 x 2048 x 2048 33 14.5 / 16.0, 48 17.3 / 16.9; 4096 + 2 x 1024
    // x 1024 33 9.3 / 10.1, 48 10.7 / 10.5, x 4096 33 24.1 / 27.9, 48 29.4 / 29.3, 49 31.5 / 29.3; 5120 + 2 x 1024 x 5120 40 32.5 / 36.8, 48 36.6 / 38.2, 56 42.3 / 39.3; 3 x 2048 x 512 33
    // 6.5 / 6.3, 3 x 4096 x 4096 34.9 / 30.4, 8192 + 2 x 1024 x 8192 62.9 / 54.0.  4-bit (its GEMM has a launch in front) 2048 + 2 x 512 x 4096 64 tokens 20.6 / 29.9; 3584 + 2 x 512 x
    // 3584 48 24.8 / 27.1, 52 29.0 / 27.2, groups of 64 29.3 / 30.8, 60 31.2 / 30.9; 4096 + 2 x 1024 x 1024 49 11.0 / 12.3, 64 12.3 / 12.6; 3 x 4096 x 4096 33 34.6 / 31.2
    const int64_t rows3 = ns ? (int64_t)ns[0] + ns[1] + ns[2] : 0;
    const int gemm_t = is_gptq == 2 ? (rows3 < 4096 ? 65 : rows3 >= 10240 ? (k <= 1024 ? 49 : (int)GPTQ_GEMM_MIN_T) : k <= 1024 ? 65 : group_size > 0 && group_size < 128 ? 57 : 49)
                                    : std::max(g_tune_gemm_min_t, rows3 < 4096 ? 65 : rows3 < 10240 && k >= 1024 ? 48 : 0);
    const bool prompt = !norm_w && !rope && is_gptq != 1 && num_tokens >= gemm_t;
    if (num_tokens < 1 || (num_tokens > 64 && !prompt) || (k & 255)) return -4;
    const DenseRope* rp = static_cast<const DenseRope*>(rope);
    DenseArgs a[3];
    for (int i = 0; i < 3; ++i) {
        if (!ws[i] || !outs[i] || ns[i] <= 0 || (ns[i] & 15)) return -4;
        a[i] = DenseArgs{};
        a[i].w = ws[i]; a[i].ldw = k; a[i].wtiled = is_gptq == 3 ? 1 : 0; a[i].x = x; a[i].ldx = k; a[i].T = num_tokens; a[i].K = k; a[i].N = ns[i];
        a[i].bias = biases ? biases[i] : nullptr; a[i].epi = MI355_EPI_STORE; a[i].out = outs[i]; a[i].ldo = ns[i];
        a[i].norm_w = norm_w; a[i].norm_eps = norm_eps; a[i].ss_in = ss_in;
        if (is_gptq == 1 || is_gptq == 2) {
            a[i].scales = scales[i]; a[i].qzeros = nullptr; a[i].zmode = MI355_ZERO_SYM8;
            a[i].group_size = (group_size <= 0 || group_size > k) ? k : group_size;
            a[i].sperm = SP_NONE;
        }
    }
    hipStream_t st = (hipStream_t)stream;
    if (prompt) {
        int rc = 0;
        const int slab = is_gptq == 2 ? gptq_gemm_slab(k) : num_tokens;
        const DenseRope* pr = slab >= num_tokens && roped ? static_cast<const DenseRope*>(prompt_rope) : nullptr;
        bool did = false;
        for (int t0 = 0; t0 < num_tokens && rc == 0; t0 += slab) {
            const DenseArgs c[3] = {dense_rows(a[0], t0, slab), dense_rows(a[1], t0, slab), dense_rows(a[2], t0, slab)};
            rc = is_gptq == 2 ? gptq_prompt_gemm(c, 3, dtype, st, pr, &did) : dense_prompt_gemm(c, 3, dtype, st, pr, &did);
        }
        if (roped) *roped = did;
        if (rc != (int)hipErrorNotSupported) return rc;
        if (num_tokens > 64) return -4;
    }
    if (dtype == MI355_DTYPE_BF16)
        return is_gptq == 2 ? dense3_launch_dt<MI355_DTYPE_BF16, DW_GPTQ4T>(a, rp, st)
               : is_gptq == 1 ? dense3_launch_dt<MI355_DTYPE_BF16, DW_GPTQ4>(a, rp, st) : dense3_launch_dt<MI355_DTYPE_BF16, DW_DENSE>(a, rp, st);
    if (dtype == MI355_DTYPE_F16)
        return is_gptq == 2 ? dense3_launch_dt<MI355_DTYPE_F16, DW_GPTQ4T>(a, rp, st)
               : is_gptq == 1 ? dense3_launch_dt<MI355_DTYPE_F16, DW_GPTQ4>(a, rp, st) : dense3_launch_dt<MI355_DTYPE_F16, DW_DENSE>(a, rp, st);
    return -4;
}

}  // extern "C"

// The gated delta rule of the layer-list host layer (include/mi355_hybrid.h): per head a state S [d, vd] in f32, per token
//   S <- diag(g) S;  u = beta (v - S^T k);  S <- S + k u^T;  o = S^T q
// with unit q (times d^-1/2) and k, decays g per head or per key channel.  Two forms: a walk over the tokens (decoded tokens, short portions, odd
// sizes) and pieces of 16 tokens on the f32 matrix cores (portions of prompts).
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <math.h>
#include <algorithm>

#include "common.h"
#include "hybrid_device.h"
#include "scratch.h"
#include "../../include/mi355_hybrid.h"

namespace {

struct DeltaArgs {
    float* o; float* state; int64_t state_stride;
    const float* qkv; int ldq;
    const float* proj; int ldp, b_off;
    const float* decay_in; int ldd, decay_channels;
    const float* a_log; const float* dt_bias;
    const uint32_t* ctx; const uint32_t* cu_q; const int32_t* slots;
    int H, G, d, vd; float unit_eps;
};
// Everything of the rule that does not depend on the state is computed for all new tokens at once, one wave per (token, head):
// prep [T, P] = unit q times d^-1/2 and unit k per q/k head, the decays per head (or per head and key channel), beta per head.
__global__ __launch_bounds__(64) void delta_prep_kernel(DeltaArgs p, float* prep, int P, int T) {
    const int t = blockIdx.x, h = blockIdx.y, lane = threadIdx.x;
    const int d = p.d, hpg = p.H / p.G, g = h / hpg;
    float* out = prep + (size_t)t * P;
    const int q_off = 0, k_off = p.G * d, g_off = 2 * p.G * d, dd = p.decay_channels ? d : 1, b_off = g_off + p.H * dd;
    if (h % hpg == 0) {
        const float* row = p.qkv + (size_t)t * p.ldq;
        float qq = 0.f, kk = 0.f;
        for (int i = lane; i < d; i += 64) { const float a = row[g * d + i], b = row[p.G * d + g * d + i]; qq += a * a; kk += b * b; }
        qq = wave_sum(qq); kk = wave_sum(kk);
        const float qi = (1.f / sqrtf((float)d)) / sqrtf(qq + p.unit_eps), ki = 1.f / sqrtf(kk + p.unit_eps);
        for (int i = lane; i < d; i += 64) {
            out[q_off + g * d + i] = row[g * d + i] * qi;
            out[k_off + g * d + i] = row[p.G * d + g * d + i] * ki;
        }
    }
    const float a_rate = expf(p.a_log[h]);
    if (p.decay_channels) {
        for (int i = lane; i < d; i += 64) {
            const int ch = h * d + i;
            out[g_off + ch] = expf(-a_rate * softplusf_(p.decay_in[(size_t)t * p.ldd + ch] + p.dt_bias[ch]));
        }
    } else if (lane == 0) {
        out[g_off + h] = expf(-a_rate * softplusf_(p.decay_in[(size_t)t * p.ldd + h] + p.dt_bias[h]));
    }
    if (lane == 0) out[b_off + h] = sigmoidf_(p.proj[(size_t)t * p.ldp + p.b_off + h]);
}

// The scan.  A workgroup of 256 threads owns 256 / LPC columns of one (sequence, head)'s state S [d, vd]; LPC neighbouring lanes share
// a column, each holding DP = ceil(d / LPC) of its rows in registers, and walk the new tokens in order:
//   S <- diag(g) S;  u = beta (v - S^T k);  S <- S + k u^T;  o = S^T q
// (the two sums over d are finished by lane exchanges among the LPC lanes).  The walk is a chain of dependent steps, so its time per
// token is the latency of one step: the more lanes share a column the shorter the step (LPC = 16 at d >= 64).  q, k, g of CH tokens
// at a time sit in LDS, rows padded so that the parts fall into different banks; the next CH tokens are fetched into registers
// while the current ones are used.
template <int DP, int LPC, int CH> __global__ __launch_bounds__(256) void delta_scan_kernel(DeltaArgs p, const float* __restrict__ prep, int P) {
    constexpr int RS = DP + 4, ROW = LPC * DP, TOT = CH * ROW, NPT = (TOT + 255) / 256, CPB = 256 / LPC;
    __shared__ __align__(16) float sq[2][CH][LPC][RS], sk[2][CH][LPC][RS], sg[2][CH][LPC][RS];
    __shared__ float sb[2][CH], sgh[2][CH];
    const int s = blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
    const int col = blockIdx.z * CPB + tid / LPC, part = tid % LPC;
    const int d = p.d, vd = p.vd, g = h / (p.H / p.G);
    const int tb = (int)p.cu_q[s], te = (int)p.cu_q[s + 1];
    if (te <= tb) return;
    const int start_pos = (int)p.ctx[s] - (te - tb);
    const bool own = col < vd, chan = p.decay_channels != 0;
    float* stt = p.state + (size_t)p.slots[s] * p.state_stride + (size_t)h * d * vd;
    float S[DP];
#pragma unroll
    for (int r = 0; r < DP; ++r) { const int i = part * DP + r; S[r] = (own && i < d && start_pos > 0) ? stt[(size_t)i * vd + col] : 0.f; }
    const int q_off = g * d, k_off = p.G * d + g * d, g_off = 2 * p.G * d + (chan ? h * d : h), b_off = 2 * p.G * d + p.H * (chan ? d : 1) + h;
    const int v_col = 2 * p.G * d + h * vd + col;
    float rq[NPT], rk[NPT], rg[NPT], rv[CH], rbeta = 0.f, rgh = 1.f;
    auto fetch = [&](int t0) {
#pragma unroll
        for (int n = 0; n < NPT; ++n) {
            const int idx = tid + n * 256, c = idx / ROW, ii = idx - c * ROW, t = t0 + c;
            const bool ok_ = idx < TOT && t < te && ii < d;
            const float* row = prep + (size_t)(ok_ ? t : tb) * P;
            rq[n] = ok_ ? row[q_off + ii] : 0.f;
            rk[n] = ok_ ? row[k_off + ii] : 0.f;
            rg[n] = (ok_ && chan) ? row[g_off + ii] : 1.f;
        }
#pragma unroll
        for (int c = 0; c < CH; ++c) rv[c] = (own && t0 + c < te) ? p.qkv[(size_t)(t0 + c) * p.ldq + v_col] : 0.f;
        if (tid < CH && t0 + tid < te) {
            rbeta = prep[(size_t)(t0 + tid) * P + b_off];
            rgh = chan ? 1.f : prep[(size_t)(t0 + tid) * P + g_off];
        }
    };
    auto stage = [&](int buf) {
#pragma unroll
        for (int n = 0; n < NPT; ++n) {
            const int idx = tid + n * 256;
            if (idx < TOT) {
                const int c = idx / ROW, ii = idx - c * ROW, pp = ii / DP, r = ii - pp * DP;
                sq[buf][c][pp][r] = rq[n]; sk[buf][c][pp][r] = rk[n]; sg[buf][c][pp][r] = rg[n];
            }
        }
        if (tid < CH) { sb[buf][tid] = rbeta; sgh[buf][tid] = rgh; }
    };
    fetch(tb);
    stage(0);
    __syncthreads();
    int buf = 0;
    for (int t0 = tb; t0 < te; t0 += CH, buf ^= 1) {
        float vc[CH];
#pragma unroll
        for (int c = 0; c < CH; ++c) vc[c] = rv[c];
        const bool more = t0 + CH < te;
        if (more) fetch(t0 + CH);
        const int cn = min(CH, te - t0);
#pragma unroll
        for (int c = 0; c < CH; ++c) {
            if (c < cn) {
                float kv = 0.f;
                if (chan) {
#pragma unroll
                    for (int r = 0; r < DP; ++r) { S[r] *= sg[buf][c][part][r]; kv = fmaf(S[r], sk[buf][c][part][r], kv); }
                } else {
                    const float gh = sgh[buf][c];
#pragma unroll
                    for (int r = 0; r < DP; ++r) { S[r] *= gh; kv = fmaf(S[r], sk[buf][c][part][r], kv); }
                }
                kv = column_sum<LPC>(kv);
                const float u = sb[buf][c] * (vc[c] - kv);
                float o = 0.f;
#pragma unroll
                for (int r = 0; r < DP; ++r) { S[r] = fmaf(sk[buf][c][part][r], u, S[r]); o = fmaf(S[r], sq[buf][c][part][r], o); }
                o = column_sum<LPC>(o);
                if (own && part == 0) p.o[((size_t)(t0 + c) * p.H + h) * vd + col] = o;
            }
        }
        if (more) stage(buf ^ 1);
        __syncthreads();
    }
    if (own)
#pragma unroll
        for (int r = 0; r < DP; ++r) { const int i = part * DP + r; if (i < d) stt[(size_t)i * vd + col] = S[r]; }
}

// The rule by pieces of 16 tokens, for portions of prompts.  With G_t the products of a piece's decays up to and including token t, the walk
// over a piece that starts from S is
//   (I + A) U = diag(beta) (V - K_G S),  A[t, s] = beta_t sum_c k_t k_s prod_(s < r <= t) g_r  (s < t),  K_G[t] = G_t k_t
//   O = Q_G S + M U,  M[t, s] = sum_c q_t k_s prod_(s < r <= t) g_r  (s <= t),  Q_G[t] = G_t q_t
//   S <- diag(G_16) S + K_hat^T U,  K_hat[s] = k_s prod_(s < r) g_r
// so that everything but U, O and S is known for all pieces at once: `prepare` makes W = (I + A)^-1 diag(beta) K_G and X = (I + A)^-1 diag(beta) V
// by forward substitution, and the scan is U = X - W S and the two lines below it, on the f32 matrix cores.  Only products of decays are
// formed, never their quotients: nothing over- or underflows that the walk keeps.
// What is summed enters what it is added to by one rounding (forward substitution, K_hat^T U into the state, M U), the unit vectors' factors are
// rounded once, and the decays' products G are formed in 64 bits.  Error against 64 bits (2-norm) of outputs / state, 16 heads of 128, 2048 tokens:
// walk 1.81e-7 / 1.55e-7, pieces with every step in f32 and sums run on from their start 1.95e-7 / 1.76e-7, as here 1.46e-7 / 1.25e-7;
// 200 tokens 1.77 / 1.59, 1.85 / 1.71, 1.26 / 1.18; at the same time (195 us; 64-wide heads 163 -> 167).
// What bounds it: the chain over the pieces, about 24
// f32 MFMAs of 32 cycles and one barrier each (0.88 us per 16 tokens against 0.36 us per ONE token of the walk); `prepare` (83 us for 2048
// tokens) the logarithms and exponentials of the decays and the walks of the keys inside a piece.
// A record per (piece, head), in the order the scan's lanes read it, 16 B each: W, Q_G [d / 16][lane = 16 (c % 16 / 4) + t][c % 4],
// K_hat [d / 16][lane = 16 (t / 4) + c % 16][t % 4], G_16 [d], M [lane = 16 (s / 4) + t][s % 4], X [vd / 16][lane = 16 (t / 4) + c % 16][t % 4].
constexpr int DPC = 16;
struct DeltaPieces { float* rec; int n_seqs; int64_t rec_floats; int first, count; };   // this launch's window of piece numbers; rec holds theirs
__host__ __device__ __forceinline__ int64_t delta_rec_floats(int d, int vd) { return 3 * DPC * (int64_t)d + d + DPC * DPC + DPC * (int64_t)vd; }
// pieces of sequence s start at number cu_q[s] / 16 + s: room for every sequence's last, shorter piece without a table
__device__ __forceinline__ int delta_first_piece(const uint32_t* cu_q, int s) { return (int)(cu_q[s] / DPC) + s; }

// x / sqrt(s), rounded about once: the f32 root and quotient with one step of Newton's method in 64 bits, as the sum of two f32
// (where that step has no value, s = 0 or infinite, the quotient stands)
struct DeltaRoot { float hi, lo; };
__device__ __forceinline__ DeltaRoot delta_rsqrt(double s) {
    const float y = 1.f / sqrtf((float)s);
    const double e = fma(-s * (double)y, (double)y, 1.), z = fma(0.5 * (double)y, e, (double)y);
    if (!(fabs(e) < 1.)) return {y, 0.f};
    return {(float)z, (float)(z - (double)(float)z)};
}
__device__ __forceinline__ float delta_scaled(float x, const DeltaRoot& r) { return fmaf(x, r.hi, x * r.lo); }

template <int DP> __global__ __launch_bounds__(256, 3) void delta_piece_prepare_kernel(DeltaArgs p, DeltaPieces q) {
    constexpr int D = 16 * DP, RS = D + 4;                             // channels of a row, rounded up; floats per LDS row
    __shared__ __align__(16) float sq[DPC][RS], sk[DPC][RS], sg[DPC][RS];
    // 2^25 (decay - sg), 11 bits of it: a decay is at most 1, so this is too.  (Not for 256 channels: three workgroups of 52 KB fill a CU's LDS,
    // and two took 154 us instead of 139 for 8 x 128 tokens; the error is below the walk's there without it)
    constexpr bool LOW = DP <= 8;
    __shared__ __align__(16) _Float16 sl[LOW ? DPC : 1][RS];
    __shared__ float sA[DPC][DPC], sb[DPC], sM[DPC][DPC];
    const int piece = q.first + (int)blockIdx.x, h = blockIdx.y, tid = threadIdx.x, row = tid >> 4, part = tid & 15;
    const int d = p.d, vd = p.vd, g = h / (p.H / p.G);
    int s = 0;
    while (s + 1 < q.n_seqs && delta_first_piece(p.cu_q, s + 1) <= piece) ++s;
    const int t0 = (int)p.cu_q[s] + (piece - delta_first_piece(p.cu_q, s)) * DPC, te = (int)p.cu_q[s + 1];
    if (t0 >= te) return;
    // ---- token t0 + row: unit q times d^-1/2, unit k, decays (1 beyond the portion, k = q = 0 there), 16 lanes per row
    {
        const int t = t0 + row;
        const bool live = t < te;
        const float* src = p.qkv + (size_t)(live ? t : t0) * p.ldq;
        float qv[DP], kv[DP], qq = 0.f, kk = 0.f;
#pragma unroll
        for (int r = 0; r < DP; ++r) {
            const int i = part + 16 * r;
            qv[r] = (live && i < d) ? src[g * d + i] : 0.f;
            kv[r] = (live && i < d) ? src[p.G * d + g * d + i] : 0.f;
            qq += qv[r] * qv[r]; kk += kv[r] * kv[r];
        }
        qq = column_sum<16>(qq); kk = column_sum<16>(kk);
        const DeltaRoot qi = delta_rsqrt((double)d * ((double)qq + (double)p.unit_eps)), ki = delta_rsqrt((double)kk + (double)p.unit_eps);
        const float rate = expf(p.a_log[h]);
        double gh = 1.;
        if (!p.decay_channels && live) gh = exp((double)(-rate * softplusf_(p.decay_in[(size_t)t * p.ldd + h] + p.dt_bias[h])));
#pragma unroll
        for (int r = 0; r < DP; ++r) {
            const int i = part + 16 * r;
            sq[row][i] = delta_scaled(qv[r], qi); sk[row][i] = delta_scaled(kv[r], ki);
        }
#pragma unroll 2
        for (int r = 0; r < DP; ++r) {                                   // (all at once they take the registers of two more waves)
            const int i = part + 16 * r;
            double gv = gh;
            if (p.decay_channels && live && i < d) gv = exp((double)(-rate * softplusf_(p.decay_in[(size_t)t * p.ldd + h * d + i] + p.dt_bias[h * d + i])));
            const float gf = (float)gv;
            sg[row][i] = gf;
            if constexpr (LOW) sl[row][i] = (_Float16)((float)(gv - (double)gf) * 0x1p25f);
        }
        if (part == 0) sb[row] = live ? sigmoidf_(p.proj[(size_t)t * p.ldp + p.b_off + h]) : 0.f;
    }
    __syncthreads();
    float* rec = q.rec + ((size_t)blockIdx.x * p.H + h) * q.rec_floats;
    // ---- A, M, K_hat: row s's key walks on through the decays (16 lanes per row, DP channels each)
    {
        float x[DP];
#pragma unroll
        for (int r = 0; r < DP; ++r) x[r] = sk[row][part * DP + r];
#pragma unroll 2
        for (int t = 0; t < DPC; ++t) {
            float a = 0.f, m = 0.f;
#pragma unroll
            for (int r = 0; r < DP; ++r) {
                const int c = part * DP + r;
                if (t > row) x[r] *= sg[t][c];
                a = fmaf(x[r], sk[t][c], a);
                m = fmaf(x[r], sq[t][c], m);
            }
            a = column_sum<16>(a); m = column_sum<16>(m);
            if (part == 0) { sA[t][row] = t > row ? sb[t] * a : 0.f; sM[t][row] = t >= row ? m : 0.f; }
        }
        float* kh = rec + 2 * DPC * (size_t)d;
#pragma unroll
        for (int r = 0; r < DP; ++r) {
            const int c = part * DP + r;
            if (c < d) kh[(size_t)(c >> 4) * 256 + (16 * (row >> 2) + (c & 15)) * 4 + (row & 3)] = x[r];
        }
    }
    __syncthreads();
    float* mrec = rec + 3 * DPC * (size_t)d + d;
    mrec[(16 * (part >> 2) + row) * 4 + (part & 3)] = sM[row][part];
    // ---- a column of K_G or V per thread: forward substitution
    for (int c = tid; c < d + vd; c += 256) {
        const bool key = c < d;
        float x[DPC];
        double G = 1.;
#pragma unroll
        for (int t = 0; t < DPC; ++t) {
            float v, a = 0.f;
            if (key) {
                G *= LOW ? (double)sg[t][c] + (double)((float)sl[LOW ? t : 0][c] * 0x1p-25f) : (double)sg[t][c];
                const float Gf = (float)G;
                v = sk[t][c] * Gf;
                rec[DPC * (size_t)d + (size_t)(c >> 4) * 256 + (16 * ((c & 15) >> 2) + t) * 4 + (c & 3)] = sq[t][c] * Gf;
            } else {
                v = t0 + t < te ? p.qkv[(size_t)(t0 + t) * p.ldq + 2 * p.G * d + h * vd + (c - d)] : 0.f;
            }
            v *= sb[t];
            if (t & 1) asm volatile("" ::: "memory");                    // two rows of A in registers at a time, not all of them (172 registers: half the waves)
#pragma unroll
            for (int r = 0; r < t; ++r) a = fmaf(sA[t][r], x[r], a);
            x[t] = v - a;                                                // (the sum by itself: its roundings are smaller than v's)
        }
        if (key) {
            rec[3 * DPC * (size_t)d + c] = (float)G;
#pragma unroll
            for (int t = 0; t < DPC; ++t) rec[(size_t)(c >> 4) * 256 + (16 * ((c & 15) >> 2) + t) * 4 + (c & 3)] = x[t];
        } else {
            float* xr = mrec + DPC * DPC + (size_t)((c - d) >> 4) * 256 + ((c - d) & 15) * 4;
#pragma unroll
            for (int t = 0; t < DPC; t += 4) *reinterpret_cast<f32x4_t*>(xr + (t >> 2) * 64) = f32x4_t{x[t], x[t + 1], x[t + 2], x[t + 3]};
        }
    }
}

// The scan: a workgroup owns 16 columns of one (sequence, head)'s state.  Wave w < 4 holds rows 16 ND w .. of them as ND accumulator tiles, whose
// registers ARE the right operand of the products with the state (a step's four k are rows 4 kg + v of a tile); the waves' shares of W S
// meet in LDS behind one barrier per piece, and Q_G S is made while they are read.  Wave 4 makes the outputs, a piece behind, so that they
// are not on the chain.  Records are requested two pieces ahead.
template <int ND, bool FULL> __global__ __launch_bounds__(320) void delta_piece_scan_kernel(DeltaArgs p, DeltaPieces q) {
    __shared__ f32x4_t sw[2][4][64], so[2][4][64];
    const int s = blockIdx.x / p.H, h = blockIdx.x % p.H, ct = blockIdx.y, lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), m16 = lane & 15, kg = lane >> 4;
    const int d = p.d, vd = p.vd, nd = d >> 4;
    // this sequence's tokens in the window: from piece `skip` of it (its state is in the slot by then), n pieces
    const int cu0 = (int)p.cu_q[s], cu1 = (int)p.cu_q[s + 1], first = delta_first_piece(p.cu_q, s) - q.first, skip = max(-first, 0);
    const int tb = cu0 + skip * DPC, te = min(cu1, cu0 + (q.count - first) * DPC);
    if (te <= tb) return;
    const int n = (te - tb + DPC - 1) / DPC, start_pos = (int)p.ctx[s] - (cu1 - cu0) + skip;
    const float* rec0 = q.rec + ((size_t)(first + skip) * p.H + h) * q.rec_floats;
    const size_t rstep = (size_t)p.H * q.rec_floats, m_at = 3 * DPC * (size_t)d + d + lane * 4, x_at = 3 * DPC * (size_t)d + d + DPC * DPC + (size_t)ct * 256 + lane * 4;
    auto ld4 = [](const float* a) { return *reinterpret_cast<const f32x4_t*>(a); };
    auto meet = [] {                                                     // own LDS accesses done; everyone's
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    auto sum4 = [&](const f32x4_t (&b)[4][64]) { return (b[0][lane] + b[1][lane]) + (b[2][lane] + b[3][lane]); };
    if (wave == 4) {
        struct Rec { f32x4_t m, x; };
        auto fetch = [&](Rec& r, int i) { const float* rec = rec0 + (size_t)(i < n ? i : n - 1) * rstep; r.m = ld4(rec + m_at); r.x = ld4(rec + x_at); };
        auto piece = [&](Rec& r, int i) {
            const f32x4_t U = r.x - sum4(sw[i & 1]), m = r.m;
            fetch(r, i + 3);
            meet();                                                      // Q_G S of piece i (and W S of piece i + 1)
            f32x4_t qs = sum4(so[i & 1]), o = f32x4_t{0.f, 0.f, 0.f, 0.f};
            asm volatile("" : "+v"(qs));                                 // in hand first: these products are not on the chain, and a wave that is shares their SIMD
#pragma unroll
            for (int v = 0; v < 4; ++v) o = __builtin_amdgcn_mfma_f32_16x16x4f32(m[v], U[v], o, 0, 0, 0);   // (the sum by itself, as the state's)
            if (__any(o[0] != o[0])) {
                // The zeros of M are no zeros times an infinity or a NaN: tokens in front of such a U are summed without it, as the walk does.
                // (a U behind the first token that is not finite leaves a NaN in the first row, whose M is zero there: one comparison sees them all)
                o = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int s2 = 0; s2 < DPC; ++s2) {
                    const float us = __shfl(U[s2 & 3], 16 * (s2 >> 2) + m16);
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        const float ms = __shfl(m[s2 & 3], 16 * (s2 >> 2) + 4 * kg + v);
                        if (s2 <= 4 * kg + v) o[v] = fmaf(ms, us, o[v]);
                    }
                }
            }
            o += qs;
            const int t = tb + i * DPC + 4 * kg;
#pragma unroll
            for (int v = 0; v < 4; ++v)
                if (t + v < te) p.o[((size_t)(t + v) * p.H + h) * vd + 16 * ct + m16] = o[v];
        };
        Rec r0, r1, r2;                                                  // (in turn, never copied: a copy waits for the load)
        fetch(r0, 0); fetch(r1, 1); fetch(r2, 2);
        meet();                                                          // W S of piece 0
        for (int i = 0; i < n; i += 3) {
            piece(r0, i);
            if (i + 1 < n) piece(r1, i + 1);
            if (i + 2 < n) piece(r2, i + 2);
        }
        return;
    }
    float* stt = p.state + (size_t)p.slots[s] * p.state_stride + (size_t)h * d * vd + 16 * ct + m16;
    bool own[ND];
    f32x4_t S[ND];
#pragma unroll
    for (int j = 0; j < ND; ++j) {
        const int tile = wave * ND + j;
        own[j] = FULL || tile < nd;                                       // FULL: d = 64 ND
#pragma unroll
        for (int v = 0; v < 4; ++v) S[j][v] = (own[j] && start_pos > 0) ? stt[(size_t)(16 * tile + 4 * kg + v) * vd] : 0.f;
    }
    struct Rec { f32x4_t w[ND], qg[ND], kh[ND], gd[ND], x; };
    auto fetch = [&](Rec& r, int i) {
        const float* rec = rec0 + (size_t)(i < n ? i : n - 1) * rstep;
#pragma unroll
        for (int j = 0; j < ND; ++j) {
            const size_t tile = own[j] ? wave * ND + j : 0;              // (a tile beyond d reads the first one's; its state stays zero)
            r.w[j] = ld4(rec + tile * 256 + lane * 4);
            r.qg[j] = ld4(rec + DPC * (size_t)d + tile * 256 + lane * 4);
            r.kh[j] = ld4(rec + 2 * DPC * (size_t)d + tile * 256 + lane * 4);
            r.gd[j] = ld4(rec + 3 * DPC * (size_t)d + 16 * tile + 4 * kg);
        }
        r.x = ld4(rec + x_at);
    };
    auto piece = [&](const Rec& r, int i) {
        f32x4_t pw[ND], po[ND];
#pragma unroll
        for (int j = 0; j < ND; ++j) pw[j] = po[j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int v = 0; v < 4; ++v)
#pragma unroll
            for (int j = 0; j < ND; ++j) pw[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(r.w[j][v], S[j][v], pw[j], 0, 0, 0);
#pragma unroll
        for (int j = 1; j < ND; ++j) pw[0] += pw[j];
        sw[i & 1][wave][lane] = pw[0];
        __builtin_amdgcn_sched_barrier(0);                               // (hipcc moves half of the products below in front of the barrier and the reads behind them)
        meet();
        const f32x4_t a0 = sw[i & 1][0][lane], a1 = sw[i & 1][1][lane], a2 = sw[i & 1][2][lane], a3 = sw[i & 1][3][lane];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int v = 0; v < 4; ++v)
#pragma unroll
            for (int j = 0; j < ND; ++j) po[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(r.qg[j][v], S[j][v], po[j], 0, 0, 0);
        f32x4_t U = r.x - ((a0 + a1) + (a2 + a3));
        if (i == n - 1) {                                                // rows beyond the portion: nothing times a state that is not finite
#pragma unroll
            for (int v = 0; v < 4; ++v) if (tb + i * DPC + 4 * kg + v >= te) U[v] = 0.f;
        }
#pragma unroll
        for (int j = 0; j < ND; ++j) pw[j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int v = 0; v < 4; ++v)
#pragma unroll
            for (int j = 0; j < ND; ++j) pw[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(r.kh[j][v], U[v], pw[j], 0, 0, 0);
#pragma unroll
        for (int j = 0; j < ND; ++j)
            if (own[j])                                                  // (the sum by itself: one rounding of the state per piece)
#pragma unroll
                for (int v = 0; v < 4; ++v) S[j][v] = fmaf(S[j][v], r.gd[j][v], pw[j][v]);
#pragma unroll
        for (int j = 1; j < ND; ++j) po[0] += po[j];
        so[i & 1][wave][lane] = po[0];
    };
    Rec r0, r1, r2;
    fetch(r0, 0);
    fetch(r1, 1);
    for (int i = 0; i < n; i += 3) {
        fetch(r2, i + 2);
        piece(r0, i);
        fetch(r0, i + 3);
        if (i + 1 < n) piece(r1, i + 1);
        fetch(r1, i + 4);
        if (i + 2 < n) piece(r2, i + 2);
    }
    meet();                                                              // the last piece's Q_G S
#pragma unroll
    for (int j = 0; j < ND; ++j)
        if (own[j]) {
#pragma unroll
            for (int v = 0; v < 4; ++v) stt[(size_t)(16 * (wave * ND + j) + 4 * kg + v) * vd] = S[j][v];
        }
}

constexpr int DELTA_MIN_TOKENS = 64, DELTA_MIN_TOKENS_WIDE = 80, DELTA_MIN_PER_SEQ = 48;
constexpr int64_t DELTA_WINDOW_BYTES = 256ll << 20;

}  // namespace

extern "C" {

int mi355_hyb_delta_rule_scratch_floats(int32_t num_tokens, int32_t heads, int32_t kv_heads, int32_t dim, int32_t decay_channels) {
    return num_tokens * (2 * kv_heads * dim + heads * (decay_channels ? dim : 1) + heads);
}

int mi355_hyb_delta_rule(float* o, float* state, int64_t state_stride, const float* qkv, int32_t ldq, const float* proj, int32_t ldp,
                         int32_t b_off, const float* decay_in, int32_t ldd, int32_t decay_channels, const float* a_log,
                         const float* dt_bias, const uint32_t* context_lens, const uint32_t* cu_seqlens_q, const int32_t* state_slots,
                         int32_t num_seqs, int32_t num_tokens, int32_t heads, int32_t kv_heads, int32_t dim, int32_t vdim, float unit_eps,
                         float* scratch, int64_t stream) {
    if (!o || !state || !qkv || !proj || !decay_in || !a_log || !dt_bias || !context_lens || !cu_seqlens_q || !state_slots || !scratch) return -1;
    if (heads <= 0 || kv_heads <= 0 || heads % kv_heads || dim <= 0 || dim > 256 || vdim <= 0) return -1;
    if (num_seqs <= 0 || num_tokens <= 0) return 0;
    DeltaArgs p{o, state, state_stride, qkv, ldq, proj, ldp, b_off, decay_in, ldd, decay_channels, a_log, dt_bias,
                context_lens, cu_seqlens_q, state_slots, heads, kv_heads, dim, vdim, unit_eps};
    hipStream_t s_ = to_stream(stream);
    // Whole 16-row tiles and portions of prompts: by pieces.  us per call, walk / pieces.  16 heads of 128 x 128: one portion of 64 tokens 32 / 27, 200 81 / 37,
    // 2048 740 / 195; two of 1050 396 / 145; 4 of 64 40 / 39, 8 of 64 56 / 57, 8 of 400 246 / 230; one of 500 beside 7 single tokens 266 / 89.  32 heads of
    // 64: 64 tokens 25 / 20, 2048 590 / 174.  8 heads of 256: 64 tokens 44 / 48, 80 51 / 49, 200 111 / 63, 2048 1018 / 310.
    // The lengths are on the device; what is known here is their mean.  Portions that fill the chip by themselves would be walked a little faster (16 of 50
    // 79 / 102, 16 of 100 135 / 158), but a batch of the same mean with one long portion in it would take three times as long, so the mean decides
    // Their records take 8.6 KB per token and 16 heads of 128: windows of at most 256 MiB (7 800 such tokens), one behind the other, with the state in
    // its slot in between
    const int64_t pieces = num_tokens / DPC + num_seqs, piece_bytes = heads * delta_rec_floats(dim, vdim) * 4, room = DELTA_WINDOW_BYTES / piece_bytes;
    if (dim % 16 == 0 && vdim % 16 == 0 && num_tokens >= (dim > 128 ? DELTA_MIN_TOKENS_WIDE : DELTA_MIN_TOKENS) && num_tokens / num_seqs >= DELTA_MIN_PER_SEQ && vdim <= 65535 * 16 && room > 0) {
        const int64_t windows = (pieces + room - 1) / room, window = (pieces + windows - 1) / windows;             // of one size: the scan of a short one is as long
        void* ws = nullptr;
        Mi355ScratchTurn turn(MI355_SCR_DELTA, s_);
        if (heads <= 65535 && mi355_scratch_get(&ws, MI355_SCR_DELTA, (size_t)(window * piece_bytes), s_, false, (size_t)DELTA_WINDOW_BYTES) == 0) {   // (no room while a stream is captured: the walk)
            for (int64_t first = 0; first < pieces; first += window) {
                const DeltaPieces q{static_cast<float*>(ws), num_seqs, delta_rec_floats(dim, vdim), (int)first, (int)std::min(window, pieces - first)};
                const dim3 pg((unsigned)q.count, heads), sg(num_seqs * heads, vdim / 16);
#define DELTA_SCAN(ND) do { if (dim == 64 * (ND)) delta_piece_scan_kernel<ND, true><<<sg, 320, 0, s_>>>(p, q); else delta_piece_scan_kernel<ND, false><<<sg, 320, 0, s_>>>(p, q); } while (0)
                if (dim <= 64) { delta_piece_prepare_kernel<4><<<pg, 256, 0, s_>>>(p, q); DELTA_SCAN(1); }
                else if (dim <= 128) { delta_piece_prepare_kernel<8><<<pg, 256, 0, s_>>>(p, q); DELTA_SCAN(2); }
                else { delta_piece_prepare_kernel<16><<<pg, 256, 0, s_>>>(p, q); DELTA_SCAN(4); }
#undef DELTA_SCAN
            }
            LAUNCH_OK(); return 0;
        }
    }
    const int P = 2 * kv_heads * dim + heads * (decay_channels ? dim : 1) + heads;
    delta_prep_kernel<<<dim3(num_tokens, heads), 64, 0, s_>>>(p, scratch, P, num_tokens);
    LAUNCH_OK();
    if (dim < 64) {
        const dim3 grid(num_seqs, heads, (vdim + 63) / 64);
        if (dim <= 16) delta_scan_kernel<4, 4, 8><<<grid, 256, 0, s_>>>(p, scratch, P);
        else if (dim <= 32) delta_scan_kernel<8, 4, 8><<<grid, 256, 0, s_>>>(p, scratch, P);
        else delta_scan_kernel<16, 4, 8><<<grid, 256, 0, s_>>>(p, scratch, P);
    } else {
        const dim3 grid(num_seqs, heads, (vdim + 15) / 16);
        if (dim <= 64) delta_scan_kernel<4, 16, 8><<<grid, 256, 0, s_>>>(p, scratch, P);
        else if (dim <= 128) delta_scan_kernel<8, 16, 8><<<grid, 256, 0, s_>>>(p, scratch, P);
        else delta_scan_kernel<16, 16, 8><<<grid, 256, 0, s_>>>(p, scratch, P);
    }
    LAUNCH_OK(); return 0;
}

}  // extern "C"

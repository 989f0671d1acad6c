// gfx950 kernels of the head that follows the encoder (the reference's `KneeBaseline` context and
// per-finding attention pooling, src/knee/models/baseline.py:870-932,954-977,1083-1170) and their C
// ABI, d8s_head (include/d8s_hip.h).
//
// Per study (W windows of D-dim encoder features, a few hundred KB) the head is a few small matrix
// products with row-wise normalisations around them: latency, not arithmetic, is its cost (a call of 8
// studies is 13 us of float32 MFMA work at peak).  So the work is arranged for few dependent launches
// (six for all studies of a call), in float32; the small products Mo and Mf below are summed in float64.
// The logits use the context's output only through its dots with attn.weight and cls_w (the 2T rows V of D
// values), so with
//   Mo = V ctx_out (2T x CD),  Mf = Mo ff2 (2T x FF)
// every window's dots are V (z + slot_emb) + Mo h1 + Mf u + const, and neither the ff2 and ctx_out
// products over the windows nor the features f2 are formed (55 % of the multiplications before):
//   1. k_head_prod<SLOT>: (z + slot_emb) [ctx_in | V]^T, split over K into raw sums; Mo's raw sums
//   2. k_head_rows:       per window h = sums + b + ctx_pos[w % per], LN1(h), the feature dots; Mo;
//                         V ctx_out_b; whether the window's slot is present
//   3. k_head_prod:       qkv = LN1(h) in_proj^T + b; Mf = Mo ff2
//   4. k_head_attn:       per (study, head, 16 queries) softmax(q k^T / sqrt(dh), keys of absent slots
//                         masked) v, times the head's columns of out_proj (one partial sum per head;
//                         beyond 4 heads the attention itself, and a product for out_proj)
//   5. k_head_ff:         per 16 windows and 128 hidden units h1 = h + partial sums + b, LN2,
//                         u = relu(. ff1^T + b), the partial dots Mf u and (a share of) Mo h1
//   6. k_head_pool:       per study: a = attn(f2) masked, softmax over windows,
//                         logits = sum_w a (f2 . cls_w) + cls_b
// (one context layer: the final model's configuration.)  Mo and Mf are formed again in every call, beside
// the products that do not need them yet: nothing is kept from one call for the next.
//
// The products run on v_mfma_f32_16x16x4_f32 with 16-byte operand reads: lane l holds row (A) or column (B)
// l % 16 and, in step s of a 16-deep group, k = 4 (l / 16) + s, the same permutation of k for both.
// Measured with HIP events per call (every input resident): 8 studies of 88 windows 65 us,
// 1 study of 44 windows 49 us (15 launches with the products staged through LDS: 118 and 79 us).
#include <hip/hip_runtime.h>

#include <math.h>
#include <stdint.h>

#include <algorithm>
#include <mutex>
#include <string>

#include "d8s_hip.h"
#include "d8s_host.h"

#define DEV __device__ __forceinline__

namespace {

constexpr int NT = 256;
constexpr int KC = 64;                       // k per chunk of a product
constexpr int WMAX = 128;                    // windows per study
constexpr int TMAX = 16;                     // findings
constexpr int FS = 64;                       // hidden units per workgroup of k_head_ff
constexpr int HFUSE = 4;                     // heads up to which out_proj is one partial sum per head

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef double f64x4 __attribute__((ext_vector_type(4)));
// four consecutive floats at any float's address (one 16-byte load: the hardware takes 4-byte alignment)
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));

DEV f32x4 mfma_f32(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// x, or +0 where off (an integer mask: a select of a loaded value is turned back into a branch around the
// load, and a load under a branch waits for every load in flight before it)
DEV float keep(float x, bool on) {
    uint32_t m = on ? ~0u : 0u;
    asm volatile("" : "+v"(m));
    return __uint_as_float(__float_as_uint(x) & m);
}
DEV f32x4 ld4(const float* row, int k) { return *(const f32x4u*)(row + k); }
// values k .. k + 3 of a row of K, zeros past its end
DEV f32x4 ld4_tail(const float* row, int k, int K) {
    f32x4 v;
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = keep(row[min(k + i, K - 1)], k + i < K);
    return v;
}

// A product C[z][r][n] = sum over the split z's k of A[r][k] B[n][k] (+ bias[n] + R[r][n] when bias is
// given), and beside it a second one of the same depth in float64, with B2 stored [k][n]: the grid's row
// tiles from `rt` on are its 32 rows.  Column n of B is row n of B0, or of Bt, Bc for the T columns from
// N0 and the T after them; row t of the second A is row t of A2a, or of A2b from T2 on, or of A2d.
struct ProdP {
    const float* A;
    int M, K, rt;                            // rt: row tiles of the first product
    const float* slot_emb;                   // SLOT: A row r gets + slot_emb[slot_of[r % W]] (nothing for
    const int32_t* slot_of;                  // a slot outside 0 .. S-1)
    int W, S;
    const float *B0, *Bt, *Bc;
    int N0, T, N;
    const float *bias, *R;
    float* C;
    const float *A2a, *A2b, *B2;
    const double* A2d;
    int T2, M2, N2;
    double* C2;                              // [splits][M2][N2]; C2f: the same in float32
    float* C2f;
    int kc;                                  // chunks of KC per split (gridDim.z splits)
};

// Rows r0 .. r0 + 15 x 16 columns of the second product, in float64 (what Mo and Mf are rounded by is the
// same for every window, so it does not average out over them as the windows' own roundings do: with
// float32 sums the logits were 3.3e-7 from float64's, the products they replace 1.1e-7).  The MFMA's
// result rows are 4 v + l / 16 (float32's: 4 (l / 16) + v).
template <class TA>
DEV void prod_second(const ProdP& p, const TA* ar, int r0, int n0, int i16, int q, int g0, int g1) {
    constexpr int PF = 4;
    typedef TA vec __attribute__((ext_vector_type(4), aligned(sizeof(TA))));
    const float* bc = p.B2 + min(n0 + i16, p.N2 - 1);
    f64x4 acc = {0.0, 0.0, 0.0, 0.0};
    vec a[PF];
    float b[PF][4];
    const int gf = min(g1, p.K / 16);
    auto load = [&](int u, int g) __attribute__((always_inline)) {
        const int k = 16 * g + 4 * q;
        a[u] = *(const vec*)(ar + k);
#pragma unroll
        for (int i = 0; i < 4; ++i) b[u][i] = bc[(int64_t)(k + i) * p.N2];
    };
    auto step = [&](int u) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; ++i) acc = __builtin_amdgcn_mfma_f64_16x16x4f64((double)a[u][i], (double)b[u][i], acc, 0, 0, 0);
    };
    if (g0 < gf) {
#pragma unroll
        for (int u = 0; u < PF; ++u) load(u, min(g0 + u, gf - 1));
        int g = g0;
        for (; g + PF <= gf; g += PF) {
#pragma unroll
            for (int u = 0; u < PF; ++u) {
                step(u);
                load(u, min(g + PF + u, gf - 1));
            }
        }
        if (g < gf) step(0);
        if (g + 1 < gf) step(1);
        if (g + 2 < gf) step(2);
    }
    if (g1 > gf) {                           // the last, partial group
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int k = 16 * gf + 4 * q + i, kc = min(k, p.K - 1);
            a[0][i] = (TA)keep((float)ar[kc], k < p.K);      // (only the float32 operand has partial groups)
            b[0][i] = keep(bc[(int64_t)kc * p.N2], k < p.K);
        }
        step(0);
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const int ro = r0 + 4 * v + q, no = n0 + i16;
        if (ro >= p.M2 || no >= p.N2) continue;
        const int64_t at = ((int64_t)blockIdx.z * p.M2 + ro) * p.N2 + no;
        if (p.C2 != nullptr) p.C2[at] = acc[v];
        if (p.C2f != nullptr) p.C2f[at] = (float)acc[v];
    }
}

// One workgroup = a 64 x 64 tile, its four waves the 32 x 32 quarters.  K in chunks of KC staged through LDS:
// 16 lanes read 256 consecutive bytes of a row and the MFMA operands come from LDS (a lane's operand
// straight from memory makes every lane of a load touch another row: 29 us for the first product of 8
// studies, against 17-19).  The next chunk's values are in registers, in flight during the MFMAs.
// The grid's row tiles from `rt` on are the second product, its waves two rows by two columns of 16 x 16
// tiles.
template <bool SLOT>
__global__ void __launch_bounds__(NT) k_head_prod(ProdP p) {
    __shared__ __attribute__((aligned(16))) float sA[64][KC + 4], sB[64][KC + 4];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, i16 = lane & 15, q = lane >> 4;
    if ((int)blockIdx.x >= p.rt) {
        const int g1 = min(((int)blockIdx.z + 1) * p.kc * (KC / 16), (p.K + 15) / 16), g0 = blockIdx.z * p.kc * (KC / 16);
        const int r0 = 16 * (wave & 1), n0 = 32 * (((int)blockIdx.x - p.rt) * gridDim.y + blockIdx.y) + 16 * (wave >> 1);
        if (r0 >= p.M2 || n0 >= p.N2) return;
        const int r = min(r0 + i16, p.M2 - 1);
        if (p.A2d != nullptr)
            prod_second(p, p.A2d + (int64_t)r * p.K, r0, n0, i16, q, g0, g1);
        else
            prod_second(p, r < p.T2 ? p.A2a + (int64_t)r * p.K : p.A2b + (int64_t)(r - p.T2) * p.K, r0, n0, i16, q, g0, g1);
        return;
    }
    const int M = p.M, N = p.N, r0 = (int)blockIdx.x * 64, n0 = blockIdx.y * 64;
    const int kbeg = blockIdx.z * p.kc * KC, kend = min(p.K, kbeg + p.kc * KC);
    // this thread stages columns 4 (tid % 16) .. + 3 of rows tid / 16 + 16 j of both operands (rows past M
    // and columns past N read the last one: their sums are not stored)
    const int k4 = 4 * (tid & 15), s0 = tid >> 4;
    const float *ar[4], *sr[4], *br[4];
    uint32_t smask = 0u;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int r = min(r0 + s0 + 16 * j, M - 1), n = min(n0 + s0 + 16 * j, N - 1);
        ar[j] = p.A + (int64_t)r * p.K;
        br[j] = n < p.N0 ? p.B0 + (int64_t)n * p.K
                         : n < p.N0 + p.T ? p.Bt + (int64_t)(n - p.N0) * p.K : p.Bc + (int64_t)(n - p.N0 - p.T) * p.K;
        sr[j] = nullptr;
        if constexpr (SLOT) {
            const int sl = p.slot_of[r % p.W];
            const bool has = (unsigned)sl < (unsigned)p.S;
            if (has) smask |= 1u << j;
            sr[j] = p.slot_emb + (int64_t)(has ? sl : 0) * p.K;
        }
    }
    f32x4 ra[4], rs[SLOT ? 4 : 1], rb[4], acc[2][2];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int c = 0; c < 2; ++c) acc[t][c] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    auto fetch = [&](int k0) __attribute__((always_inline)) {
        const int k = k0 + k4;
        if (k0 + KC <= p.K) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                ra[j] = ld4(ar[j], k);
                if constexpr (SLOT) rs[j] = ld4(sr[j], k);
                rb[j] = ld4(br[j], k);
            }
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                ra[j] = ld4_tail(ar[j], k, p.K);
                if constexpr (SLOT) rs[j] = ld4_tail(sr[j], k, p.K);
                rb[j] = ld4_tail(br[j], k, p.K);
            }
        }
    };
    fetch(kbeg);
    for (int k0 = kbeg; k0 < kend; k0 += KC) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            f32x4 v = ra[j];
            if constexpr (SLOT) {
#pragma unroll
                for (int i = 0; i < 4; ++i) v[i] += keep(rs[j][i], (smask >> j) & 1u);
            }
            *(f32x4*)&sA[s0 + 16 * j][k4] = v;
            *(f32x4*)&sB[s0 + 16 * j][k4] = rb[j];
        }
        __syncthreads();
        if (k0 + KC < kend) fetch(k0 + KC);
        // the chunk's even and odd groups in sums of their own: chains of 32 products, not of the split's
        // K (the feature dots are the largest term of a logit, and every window rounds by them)
        f32x4 part[2][2][2];
#pragma unroll
        for (int u = 0; u < 8; ++u) part[u >> 2][(u >> 1) & 1][u & 1] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int g = 0; g < KC / 16; ++g) {
            f32x4 a[2], b[2];
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                a[t] = *(const f32x4*)&sA[32 * (wave >> 1) + 16 * t + i16][16 * g + 4 * q];
                b[t] = *(const f32x4*)&sB[32 * (wave & 1) + 16 * t + i16][16 * g + 4 * q];
            }
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int t = 0; t < 2; ++t)
#pragma unroll
                    for (int c = 0; c < 2; ++c) part[g & 1][t][c] = mfma_f32(a[t][i], b[c][i], part[g & 1][t][c]);
        }
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int c = 0; c < 2; ++c) acc[t][c] += part[0][t][c] + part[1][t][c];
        __syncthreads();
    }
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        const int n = n0 + 32 * (wave & 1) + 16 * c + i16;
        if (n >= N) continue;
        const float bias = p.bias == nullptr ? 0.0f : p.bias[n];
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int r = r0 + 32 * (wave >> 1) + 16 * t + 4 * q + v;
                if (r >= M) continue;
                float x = acc[t][c][v] + bias;
                if (p.R != nullptr) x += p.R[(int64_t)r * N + n];
                p.C[((int64_t)blockIdx.z * M + r) * N + n] = x;
            }
    }
}

struct RowsP {
    const float* Cs;           // [splits][M][CD + 2T] raw sums
    const double* Ms;          // [splits][2T][CD] raw sums of Mo
    const float *bias, *pos, *ln_w, *ln_b, *ctx_out_b, *tw, *cw, *attn_b;
    const int32_t* slot_of;
    const uint8_t* slot_mask;
    float *h, *hn, *d0, *Mo, *dc;
    double* Mod;               // Mo in float64, for Mf
    uint8_t* valid;
    int M, W, CD, D, S, T, PER, splits;
};

// the splits' raw sums of NE elements i, i + 64, ...: eight splits' loads in flight, their values added in
// pairs (a fixed order)
template <int NE>
DEV void split_sums(float (&x)[NE], const float* src, int64_t stride, int64_t i, int splits) {
#pragma unroll
    for (int e = 0; e < NE; ++e) x[e] = 0.0f;
    for (int s0 = 0; s0 < splits; s0 += 8) {
        float v[NE][8];
#pragma unroll
        for (int u = 0; u < 8; ++u)
#pragma unroll
            for (int e = 0; e < NE; ++e) v[e][u] = src[min(s0 + u, splits - 1) * stride + i + 64 * e];
#pragma unroll
        for (int e = 0; e < NE; ++e) {
#pragma unroll
            for (int u = 0; u < 8; ++u) v[e][u] = keep(v[e][u], s0 + u < splits);
            x[e] += ((v[e][0] + v[e][1]) + (v[e][2] + v[e][3])) + ((v[e][4] + v[e][5]) + (v[e][6] + v[e][7]));
        }
    }
}

DEV float wave_sum(float x) {
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) x += __shfl_xor(x, d, 64);
    return x;
}

// A wave per window row (HC = CD / 64 values a lane, 0: any count): h = sums + b + pos, LN1(h) (biased
// variance in two passes over the values, as torch's layer_norm), the row's feature dots, its slot's
// presence.  Blocks past the rows: Mo, and dc[q] = V[q] . ctx_out_b (+ attn_b), a wave each.
template <int HC>
__global__ void __launch_bounds__(NT) k_head_rows(RowsP p) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int rb = (p.M + 3) / 4, N = p.CD + 2 * p.T;
    if ((int)blockIdx.x >= rb) {
        const int e = ((int)blockIdx.x - rb) * NT + threadIdx.x, n = 2 * p.T * p.CD;
        const int mb = (n + NT - 1) / NT;
        if ((int)blockIdx.x - rb < mb) {
            if (e < n) {
                double x = 0.0;
#pragma unroll 8
                for (int s = 0; s < p.splits; ++s) x += p.Ms[(int64_t)s * n + e];
                p.Mod[e] = x;
                p.Mo[e] = (float)x;
            }
            return;
        }
        const int t = ((int)blockIdx.x - rb - mb) * 4 + wave;
        if (t >= 2 * p.T) return;
        const float* v = t < p.T ? p.tw + (int64_t)t * p.D : p.cw + (int64_t)(t - p.T) * p.D;
        float x = 0.0f;
        for (int k0 = 0; k0 < p.D; k0 += 8 * 64) {
            float a[8], b[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int k = min(k0 + 64 * u + lane, p.D - 1);
                a[u] = v[k];
                b[u] = p.ctx_out_b[k];
            }
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const bool on = k0 + 64 * u + lane < p.D;
                x = __builtin_fmaf(keep(a[u], on), keep(b[u], on), x);
            }
        }
        x = wave_sum(x);
        if (lane == 0) p.dc[t] = t < p.T ? x + p.attn_b[t] : x;
        return;
    }
    const int r = blockIdx.x * 4 + wave;
    if (r >= p.M) return;
    const int w = r % p.W, b = r / p.W;
    const int64_t mn = (int64_t)p.M * N, row = (int64_t)r * N;
    if (lane < 2 * p.T) {
        float d[1];
        split_sums<1>(d, p.Cs, mn, row + p.CD + lane, p.splits);
        p.d0[(int64_t)r * 2 * p.T + lane] = d[0];
    }
    if (lane == 0) {
        const int sl = p.slot_of[w];
        p.valid[r] = (unsigned)sl < (unsigned)p.S && p.slot_mask[(int64_t)b * p.S + sl] ? 1 : 0;
    }
    const float* pos = p.pos + (int64_t)(w % p.PER) * p.CD;
    float* hr = p.h + (int64_t)r * p.CD;
    float* nr = p.hn + (int64_t)r * p.CD;
    float x[HC ? HC : 1], sum = 0.0f, ss = 0.0f;
    if constexpr (HC > 0) {
        split_sums<HC>(x, p.Cs, mn, row + lane, p.splits);
#pragma unroll
        for (int i = 0; i < HC; ++i) {
            const int c = 64 * i + lane;
            x[i] = x[i] + p.bias[c] + pos[c];
            hr[c] = x[i];
            sum += x[i];
        }
    } else {
        for (int c = lane; c < p.CD; c += 64) {
            float y[1];
            split_sums<1>(y, p.Cs, mn, row + c, p.splits);
            y[0] = y[0] + p.bias[c] + pos[c];
            hr[c] = y[0];
            sum += y[0];
        }
    }
    const float mean = wave_sum(sum) / (float)p.CD;
    if constexpr (HC > 0) {
#pragma unroll
        for (int i = 0; i < HC; ++i) ss = __builtin_fmaf(x[i] - mean, x[i] - mean, ss);
    } else {
        for (int c = lane; c < p.CD; c += 64) ss = __builtin_fmaf(hr[c] - mean, hr[c] - mean, ss);
    }
    const float rstd = 1.0f / sqrtf(wave_sum(ss) / (float)p.CD + 1e-5f);
    if constexpr (HC > 0) {
#pragma unroll
        for (int i = 0; i < HC; ++i) {
            const int c = 64 * i + lane;
            nr[c] = (x[i] - mean) * rstd * p.ln_w[c] + p.ln_b[c];
        }
    } else {
        for (int c = lane; c < p.CD; c += 64) nr[c] = (hr[c] - mean) * rstd * p.ln_w[c] + p.ln_b[c];
    }
}

struct AttnP {
    const float* qkv;      // [B*W][3 CD]
    const uint8_t* valid;  // [B][W] 1 = key of a present slot (absent slots are not keys)
    const float* wo;       // [CD][CD] out_proj
    float* out;            // FUSE: [heads][B*W][CD] partial out_proj sums; else [B*W][CD]
    int M, W, CD, heads;
};

// One workgroup per (study, head, 16 queries): scores of 16 queries x 16 keys a wave at a time (q, k and
// v straight from memory in the MFMA's layout), softmax over the keys of present slots (all keys when
// no slot of the study is present) through LDS, 16 lanes per query, then a wave's 16 output dims
// over all keys.  FUSE: the 64 output dims times the head's columns of out_proj.
template <bool FUSE>
__global__ void __launch_bounds__(NT) k_head_attn(AttnP p) {
    constexpr int DH = 64, KG = WMAX / 16;
    __shared__ __attribute__((aligned(16))) float sP[16][WMAX + 4];
    __shared__ __attribute__((aligned(16))) float sO[16][DH + 4];
    __shared__ float sInv[16];
    __shared__ uint8_t sKey[WMAX];
    __shared__ int sAny;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, i16 = lane & 15, q = lane >> 4;
    const int b = blockIdx.x, h = blockIdx.y, q0 = blockIdx.z * 16, ld = 3 * p.CD;
    const float* base = p.qkv + (int64_t)b * p.W * ld + h * DH;
    const int ng = (p.W + 15) / 16;                       // 16-key groups
    if (tid == 0) sAny = 0;
    f32x4 qa[4], ka[2][4];
    float va[KG][4];
    const float* qrow = base + (int64_t)min(q0 + i16, p.W - 1) * ld;
#pragma unroll
    for (int g = 0; g < 4; ++g) qa[g] = ld4(qrow, 16 * g + 4 * q);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const float* krow = base + p.CD + (int64_t)min(16 * (wave + 4 * j) + i16, p.W - 1) * ld;
#pragma unroll
        for (int g = 0; g < 4; ++g) ka[j][g] = ld4(krow, 16 * g + 4 * q);
    }
    // (values of keys past W are zeroed: their weight is 0, and 0 x NaN is not)
#pragma unroll
    for (int g = 0; g < KG; ++g)
#pragma unroll
        for (int i = 0; i < 4; ++i)
            va[g][i] = base[2 * p.CD + (int64_t)min(16 * g + 4 * q + i, p.W - 1) * ld + 16 * wave + i16];
    __syncthreads();
    if (tid < p.W) {
        const uint8_t v = p.valid[(int64_t)b * p.W + tid];
        sKey[tid] = v;
        if (v) atomicOr(&sAny, 1);
    }
    const float scale = 1.0f / sqrtf((float)DH);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int kt = wave + 4 * j;
        if (kt >= ng) break;
        f32x4 s = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int g = 0; g < 4; ++g)
#pragma unroll
            for (int i = 0; i < 4; ++i) s = mfma_f32(qa[g][i] * scale, ka[j][g][i], s);
#pragma unroll
        for (int v = 0; v < 4; ++v) sP[4 * q + v][16 * kt + i16] = s[v];
    }
    __syncthreads();
    {
        const int ql = tid >> 4, l = tid & 15;
        const bool any = sAny != 0;
        float sc[KG], mx = -INFINITY;
#pragma unroll
        for (int m = 0; m < KG; ++m) {
            const int j = l + 16 * m;
            sc[m] = -INFINITY;
            if (j < p.W && (!any || sKey[j])) sc[m] = sP[ql][j];
            mx = fmaxf(mx, sc[m]);
        }
#pragma unroll
        for (int d = 8; d >= 1; d >>= 1) mx = fmaxf(mx, __shfl_xor(mx, d, 16));
        float sum = 0.0f;
#pragma unroll
        for (int m = 0; m < KG; ++m) {
            const float e = sc[m] == -INFINITY ? 0.0f : expf(sc[m] - mx);
            sum += e;
            sP[ql][l + 16 * m] = e;
        }
#pragma unroll
        for (int d = 8; d >= 1; d >>= 1) sum += __shfl_xor(sum, d, 16);
        if (l == 0) sInv[ql] = 1.0f / sum;
    }
    __syncthreads();
    f32x4 o = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int g = 0; g < KG; ++g) {
        if (g >= ng) break;
        const f32x4 pa = *(const f32x4*)&sP[i16][16 * g + 4 * q];
#pragma unroll
        for (int i = 0; i < 4; ++i) o = mfma_f32(pa[i], keep(va[g][i], 16 * g + 4 * q + i < p.W), o);
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) o[v] *= sInv[4 * q + v];
    const int64_t r0 = (int64_t)b * p.W + q0;
    const int nq = p.W - q0;                              // queries of this workgroup (16 or the rest)
    if constexpr (!FUSE) {
#pragma unroll
        for (int v = 0; v < 4; ++v)
            if (4 * q + v < nq) p.out[(r0 + 4 * q + v) * p.CD + h * DH + 16 * wave + i16] = o[v];
    } else {
#pragma unroll
        for (int v = 0; v < 4; ++v) sO[4 * q + v][16 * wave + i16] = o[v];
        __syncthreads();
        float* out = p.out + (int64_t)h * p.M * p.CD;
        f32x4 oa[4];
#pragma unroll
        for (int g = 0; g < 4; ++g) oa[g] = *(const f32x4*)&sO[i16][16 * g + 4 * q];
#pragma unroll
        for (int j = 0; j < HFUSE; ++j) {
            const int n = 16 * (wave + 4 * j) + i16;
            if (n >= p.CD) break;
            const float* wrow = p.wo + (int64_t)n * p.CD + h * DH;
            f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f}, wb[4];
#pragma unroll
            for (int g = 0; g < 4; ++g) wb[g] = ld4(wrow, 16 * g + 4 * q);
#pragma unroll
            for (int g = 0; g < 4; ++g)
#pragma unroll
                for (int i = 0; i < 4; ++i) acc = mfma_f32(oa[g][i], wb[g][i], acc);
#pragma unroll
            for (int v = 0; v < 4; ++v)
                if (4 * q + v < nq) out[(r0 + 4 * q + v) * p.CD + n] = acc[v];
        }
    }
}

struct FfP {
    const float *h, *hp, *out_b;             // FUSE: h1 = h + out_b + the heads' partial sums hp
    const float* h1;                         // else: [M][CD]
    const float *ln_w, *ln_b, *ff1_w, *ff1_b, *ff2_b, *Mo, *Mf, *dc;
    float* part;                             // [slices][M][2T]
    int M, CD, FF, T, heads;
};

// One workgroup per 16 windows and FS hidden units (blockIdx.y): LN2(h1), u = relu(. ff1^T + b) (a 16-unit
// tile a wave), then the partial dots Mf u over those units and Mo (h1 + ff2_b) over this slice's share of
// the CD columns (+ the constants dc in the first), the waves' k groups added through LDS in wave
// order.  The weights' first groups are requested before h1 is summed, the dots' before ff1's loop.
template <bool FUSE>
__global__ void __launch_bounds__(NT) k_head_ff(FfP p) {
    constexpr int HC = FUSE ? 64 * HFUSE : 4;
    __shared__ __attribute__((aligned(16))) float sH[16][HC + 4];
    __shared__ __attribute__((aligned(16))) float sU[16][FS + 4];
    __shared__ float sR[4][16][2 * TMAX];
    __shared__ float sMean[16], sRstd[16];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, i16 = lane & 15, q = lane >> 4;
    const int r0 = blockIdx.x * 16, f0 = blockIdx.y * FS;
    const int row = tid >> 4, l16 = tid & 15;             // 16 lanes per row
    const int rc = min(r0 + row, p.M - 1);
    const float* grow = FUSE ? nullptr : p.h1 + (int64_t)rc * p.CD;
    constexpr int PF = 4;
    const int ng = p.CD / 16;                             // a multiple of 4
    const float* wrow = p.ff1_w + (int64_t)min(f0 + 16 * wave + i16, p.FF - 1) * p.CD;
    f32x4 wb[PF], lw[PF], lb[PF];
    auto load = [&](int u, int g) __attribute__((always_inline)) {
        const int k = 16 * g + 4 * q;
        wb[u] = ld4(wrow, k);
        lw[u] = ld4(p.ln_w, k);
        lb[u] = ld4(p.ln_b, k);
    };
#pragma unroll
    for (int u = 0; u < PF; ++u) load(u, u);
    float sum = 0.0f, ss = 0.0f;
    if constexpr (FUSE) {
        // lane l16 of a row: columns 4 l16 + 64 i
        f32x4 x[HFUSE];
        const int64_t mn = (int64_t)p.M * p.CD, at = (int64_t)rc * p.CD + 4 * l16;
#pragma unroll
        for (int i = 0; i < HFUSE; ++i) {
            x[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            if (64 * i >= p.CD) break;
            f32x4 v[HFUSE];
#pragma unroll
            for (int d = 0; d < HFUSE; ++d) v[d] = ld4(p.hp + min(d, p.heads - 1) * mn, at + 64 * i);
            f32x4 y = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int d = 0; d < HFUSE; ++d)
#pragma unroll
                for (int e = 0; e < 4; ++e) y[e] += keep(v[d][e], d < p.heads);
            x[i] = ld4(p.h, at + 64 * i) + (y + ld4(p.out_b, 4 * l16 + 64 * i));
            *(f32x4*)&sH[row][4 * l16 + 64 * i] = x[i];
            sum += (x[i][0] + x[i][1]) + (x[i][2] + x[i][3]);
        }
#pragma unroll
        for (int d = 8; d >= 1; d >>= 1) sum += __shfl_xor(sum, d, 16);
        const float mean = sum / (float)p.CD;
#pragma unroll
        for (int i = 0; i < HFUSE; ++i)
            if (64 * i < p.CD)
#pragma unroll
                for (int e = 0; e < 4; ++e) ss = __builtin_fmaf(x[i][e] - mean, x[i][e] - mean, ss);
        sum = mean;
    } else {
        for (int c = 4 * l16; c < p.CD; c += 64) {
            const f32x4 v = ld4(grow, c);
            sum += (v[0] + v[1]) + (v[2] + v[3]);
        }
#pragma unroll
        for (int d = 8; d >= 1; d >>= 1) sum += __shfl_xor(sum, d, 16);
        const float mean = sum / (float)p.CD;
        for (int c = 4 * l16; c < p.CD; c += 64) {
            const f32x4 v = ld4(grow, c);
#pragma unroll
            for (int e = 0; e < 4; ++e) ss = __builtin_fmaf(v[e] - mean, v[e] - mean, ss);
        }
        sum = mean;
    }
#pragma unroll
    for (int d = 8; d >= 1; d >>= 1) ss += __shfl_xor(ss, d, 16);
    if (l16 == 0) {
        sMean[row] = sum;
        sRstd[row] = 1.0f / sqrtf(ss / (float)p.CD + 1e-5f);
    }
    __syncthreads();
    // h1 of this lane's row (window i16 of the workgroup's) at column k
    const float* hrow = FUSE ? &sH[i16][0] : p.h1 + (int64_t)min(r0 + i16, p.M - 1) * p.CD;
    const float mean = sMean[i16], rstd = sRstd[i16];
    // the dots' weights: this wave's k group of the slice's units, and its first of the slice's columns
    f32x4 acc[2], bu[2], bo[2], b2;
    const float *mf[2], *mo[2];
    const int gs = min(wave, (p.FF - f0 + 15) / 16 - 1);  // (a wave past the units repeats the last, unused)
    const int per = (ng + (int)gridDim.y - 1) / (int)gridDim.y, go = (int)blockIdx.y * per + wave;
    const int ge = min(((int)blockIdx.y + 1) * per, ng), ko = 16 * min(go, ng - 1) + 4 * q;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        const int t = min(16 * c + i16, 2 * p.T - 1);
        mf[c] = p.Mf + (int64_t)t * p.FF;
        mo[c] = p.Mo + (int64_t)t * p.CD;
        bu[c] = ld4_tail(mf[c], f0 + 16 * gs + 4 * q, p.FF);
        bo[c] = ld4(mo[c], ko);
        acc[c] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    b2 = ld4(p.ff2_b, ko);
    {
        f32x4 u4 = {0.0f, 0.0f, 0.0f, 0.0f};
        const float bias = p.ff1_b[min(f0 + 16 * wave + i16, p.FF - 1)];
        for (int g = 0; g < ng; g += PF) {
#pragma unroll
            for (int u = 0; u < PF; ++u) {
                const f32x4 x = ld4(hrow, 16 * (g + u) + 4 * q);
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    u4 = mfma_f32((x[i] - mean) * rstd * lw[u][i] + lb[u][i], wb[u][i], u4);
                load(u, min(g + PF + u, ng - 1));
            }
        }
        const int f = 16 * wave + i16;
#pragma unroll
        for (int v = 0; v < 4; ++v) sU[4 * q + v][f] = f0 + f < p.FF ? fmaxf(u4[v] + bias, 0.0f) : 0.0f;
    }
    __syncthreads();
    if (f0 + 16 * wave < p.FF) {
        const f32x4 u = *(const f32x4*)&sU[i16][16 * wave + 4 * q];
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int c = 0; c < 2; ++c) acc[c] = mfma_f32(u[i], bu[c][i], acc[c]);
    }
    for (int g = go; g < ge; g += 4) {
        const f32x4 x = ld4(hrow, 16 * g + 4 * q);
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int c = 0; c < 2; ++c) acc[c] = mfma_f32(x[i] + b2[i], bo[c][i], acc[c]);
        const int kn = 16 * min(g + 4, ng - 1) + 4 * q;
        b2 = ld4(p.ff2_b, kn);
#pragma unroll
        for (int c = 0; c < 2; ++c) bo[c] = ld4(mo[c], kn);
    }
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int v = 0; v < 4; ++v) sR[wave][4 * q + v][16 * c + i16] = acc[c][v];
    __syncthreads();
    for (int e = tid; e < 16 * 2 * TMAX; e += NT) {
        const int r = e / (2 * TMAX), t = e % (2 * TMAX);
        if (r0 + r < p.M && t < 2 * p.T)
            p.part[((int64_t)blockIdx.y * p.M + r0 + r) * 2 * p.T + t] =
                ((sR[0][r][t] + sR[1][r][t]) + (sR[2][r][t] + sR[3][r][t])) + (blockIdx.y == 0 ? p.dc[t] : 0.0f);
    }
}

struct PoolP {
    const float *d0, *part;   // [M][2T]; [slices][M][2T]
    const uint8_t* valid;     // [B][W]
    const float* cls_b;       // [T]
    float* logits;            // [B][T]
    int M, W, T, slices;
};

// One workgroup per study: the windows' dots (features and partial sums), a[w][t] = the attention
// logits (masked to -inf for absent slots; all zeros when no slot is present), softmax over the windows,
// logits[t] = sum_w a[w][t] s[w][t] + cls_b[t].
constexpr int PT = 1024;                     // threads: a study's dots a few each, all in flight at once
__global__ void __launch_bounds__(PT) k_head_pool(PoolP p) {
    __shared__ float sA[WMAX][TMAX], sS[WMAX][TMAX];
    const int b = blockIdx.x, T2 = 2 * p.T;
    {
        // (past W * 2T: the last dot, unused)
        constexpr int PN = WMAX * 2 * TMAX / PT;
        const int n = p.W * T2;
        float v[PN];
        const float* d0 = p.d0 + (int64_t)b * n;
        const float* part = p.part + (int64_t)b * n;
        const int64_t stride = (int64_t)p.M * T2;
#pragma unroll
        for (int u = 0; u < PN; ++u) v[u] = d0[min((int)threadIdx.x + u * PT, n - 1)];
        for (int s0 = 0; s0 < p.slices; s0 += 8) {
            float y[8][PN];
#pragma unroll
            for (int s = 0; s < 8; ++s)
#pragma unroll
                for (int u = 0; u < PN; ++u)
                    y[s][u] = part[min(s0 + s, p.slices - 1) * stride + min((int)threadIdx.x + u * PT, n - 1)];
#pragma unroll
            for (int s = 0; s < 8; ++s)
#pragma unroll
                for (int u = 0; u < PN; ++u) v[u] += keep(y[s][u], s0 + s < p.slices);
        }
#pragma unroll
        for (int u = 0; u < PN; ++u) {
            const int i = (int)threadIdx.x + u * PT, w = i / T2, q = i % T2;
            if (i < n) {
                if (q < p.T)
                    sA[w][q] = v[u];
                else
                    sS[w][q - p.T] = v[u];
            }
        }
    }
    __shared__ uint8_t sV[WMAX];
    __shared__ int sAny;
    if (threadIdx.x == 0) sAny = 0;
    __syncthreads();
    for (int w = threadIdx.x; w < p.W; w += PT) {
        sV[w] = p.valid[(int64_t)b * p.W + w];
        if (sV[w]) atomicOr(&sAny, 1);
    }
    __syncthreads();
    // 16 lanes per finding t, lane l taking windows l, l + 16, ...: maximum, then the sums, reduced
    // over the 16 lanes
    const int t = threadIdx.x / 16, l = threadIdx.x % 16;
    const bool any = sAny != 0;
    float mx = -INFINITY;
    if (t < p.T)
        for (int w = l; w < p.W; w += 16) mx = fmaxf(mx, any ? (sV[w] ? sA[w][t] : -INFINITY) : 0.0f);
#pragma unroll
    for (int d = 8; d >= 1; d >>= 1) mx = fmaxf(mx, __shfl_xor(mx, d, 16));
    float sum = 0.0f, acc = 0.0f;
    if (t < p.T)
        for (int w = l; w < p.W; w += 16) {
            const float a = any ? (sV[w] ? sA[w][t] : -INFINITY) : 0.0f;
            const float e = expf(a - mx);
            sum += e;
            acc = __builtin_fmaf(e, sS[w][t], acc);
        }
#pragma unroll
    for (int d = 8; d >= 1; d >>= 1) {
        sum += __shfl_xor(sum, d, 16);
        acc += __shfl_xor(acc, d, 16);
    }
    if (t < p.T && l == 0) p.logits[(int64_t)b * p.T + t] = acc / sum + p.cls_b[t];
}

#define HREQ(cond, msg) \
    do { if (!(cond)) return d8s_host_fail((int)hipErrorInvalidValue, std::string(what) + ": " + (msg)); } while (0)

// K split of the first product: about 384 workgroups (with the second product's within two per CU, which is
// what its registers allow), at most 16 raw sums per value
struct Split {
    int splits, kc;
};

Split split_plan(int64_t M, int N, int K) {
    const int chunks = (K + KC - 1) / KC;
    const int64_t tiles = (M + 63) / 64 * ((N + 63) / 64);
    const int want = (int)std::min<int64_t>({chunks, 16, std::max<int64_t>(1, (384 + tiles - 1) / tiles)});
    const int kc = (chunks + want - 1) / want;
    return {(chunks + kc - 1) / kc, kc};
}

// Whether attention multiplies by out_proj itself (a partial sum per head): up to HFUSE heads, where the
// sums take no more room than the attention, h1 and hidden units would (the layout then stays within
// what callers sized for those)
bool fuse_out(const D8sHeadArgs* a) { return a->heads <= HFUSE && a->heads * a->CD <= 2 * a->CD + a->FF; }

struct Ws {
    float *h, *hn, *qkv, *cs, *hp, *att, *h1, *d0, *mo, *mf, *dc, *part;
    double *ms, *mod;
    uint8_t* valid;
    uint64_t bytes;
};

// The workspace: what lives from launch 2 to the end, and two regions used in turn by what does not.
//   region 1: launch 1's raw sums (read by 2), qkv (3 to 4), the partial dots (5 to 6);
//   region 2: LN1(h) (2 to 3) and Mo's raw sums (1 to 2), which become Mo in float64 in place (k_head_rows adds
//             the splits' sums of an element and writes it in one thread; read by 3); then what launch 4, or 4
//             and the out_proj product, leave for 5.
// So a call takes no more than one that kept every intermediate of the unfolded head (at most 8192 wide, 65536
// hidden units), whatever the K split.
Ws carve(const D8sHeadArgs* a, char* base) {
    Ws w{};
    const uint64_t M = (uint64_t)a->B * a->W, T2 = 2ull * a->T;
    uint64_t off = 0;
    auto take = [&](uint64_t n) {
        char* p = base ? base + off : nullptr;
        off += (4 * n + 255) / 256 * 256;
        return (float*)p;
    };
    const Split sp = split_plan((int64_t)M, a->CD + (int)T2, a->D);
    w.h = take(M * a->CD);
    w.d0 = take(M * T2);
    w.mo = take(T2 * a->CD);
    w.mf = take(T2 * a->FF);
    w.dc = take(T2);
    w.valid = (uint8_t*)take((M + 3) / 4);
    uint64_t o0 = off, end = off;
    auto region = [&]() { off = o0; };
    auto done = [&]() { end = std::max(end, off); };
    w.cs = take((uint64_t)sp.splits * M * (a->CD + T2));
    done(), region();
    w.qkv = take(3 * M * a->CD);
    done(), region();
    w.part = take((uint64_t)((a->FF + FS - 1) / FS) * M * T2);
    done();
    o0 = off = end;
    w.hn = take(M * a->CD);
    w.ms = (double*)take(2 * (uint64_t)sp.splits * T2 * a->CD);
    w.mod = w.ms;
    done(), region();
    if (fuse_out(a)) {
        w.hp = take((uint64_t)a->heads * M * a->CD);
    } else {
        w.att = take(M * a->CD);
        w.h1 = take(M * a->CD);
    }
    done();
    w.bytes = end;
    return w;
}

template <bool SLOT>
void launch_prod(ProdP p, const Split& sp, hipStream_t st) {
    p.rt = (p.M + 63) / 64;
    p.kc = sp.kc;
    const int gy = (p.N + 63) / 64, rt2 = ((p.N2 + 31) / 32 + gy - 1) / gy;
    k_head_prod<SLOT><<<dim3(p.rt + rt2, gy, sp.splits), NT, 0, st>>>(p);
}

void launch_rows(const RowsP& p, hipStream_t st) {
    const unsigned grid = (unsigned)((p.M + 3) / 4 + (2 * p.T * p.CD + NT - 1) / NT + (2 * p.T + 3) / 4);
    switch (p.CD / 64) {
        case 1: k_head_rows<1><<<grid, NT, 0, st>>>(p); break;
        case 2: k_head_rows<2><<<grid, NT, 0, st>>>(p); break;
        case 3: k_head_rows<3><<<grid, NT, 0, st>>>(p); break;
        case 4: k_head_rows<4><<<grid, NT, 0, st>>>(p); break;
        default: k_head_rows<0><<<grid, NT, 0, st>>>(p); break;
    }
}

}  // namespace

extern "C" int d8s_head_workspace(const D8sHeadArgs* a, uint64_t* bytes) {
    const char* what = "d8s_head_workspace";
    HREQ(a != nullptr && bytes != nullptr, "null arguments");
    HREQ(a->B >= 1 && a->W >= 1 && a->D >= 1 && a->T >= 1, "bad sizes");
    *bytes = carve(a, nullptr).bytes;
    return 0;
}

namespace {

// Checks the arguments (everything but the workspace) and returns the workspace layout's size.
int head_check(const D8sHeadArgs* a, const char* what) {
    HREQ(a != nullptr, "null arguments");
    HREQ(a->z && a->slot_of && a->slot_mask && a->slot_emb && a->attn_w && a->attn_b && a->cls_w &&
         a->cls_b && a->logits, "null pointer");
    HREQ(a->B >= 1 && a->B < 65536, "B must be 1 .. 65535");
    HREQ(a->W >= 1 && a->W <= WMAX, "W must be 1 .. 128 windows per study");
    HREQ(a->D >= 1 && a->S >= 1 && a->T >= 1 && a->T <= TMAX, "bad D, S or T (T <= 16)");
    HREQ(a->ctx_layers == 1, "ctx_layers must be 1 (one context layer)");
    {
        HREQ(a->ctx_in_w && a->ctx_in_b && a->ctx_pos && a->in_proj_w && a->in_proj_b && a->out_proj_w &&
             a->out_proj_b && a->ln1_w && a->ln1_b && a->ln2_w && a->ln2_b && a->ff1_w && a->ff1_b &&
             a->ff2_w && a->ff2_b && a->ctx_out_w && a->ctx_out_b, "null context weight");
        HREQ(a->heads >= 1 && a->CD == 64 * a->heads, "context width must be 64 x heads");
        HREQ(a->FF >= 1 && a->PER >= 1, "bad FF or PER");
    }
    HREQ((int64_t)a->B * a->W * a->D < (1ll << 31), "too many values");
    return 0;
}

// The launch sequence of the head over the workspace `ws` (laid out by carve).
void head_run(const D8sHeadArgs* a, char* ws, hipStream_t st) {
    const Ws w = carve(a, ws);
    const int M = a->B * a->W, T2 = 2 * a->T;
    const Split one = {1, (a->CD + KC - 1) / KC};
    // 1. (z + slot_emb) [ctx_in | attn | cls]^T and [attn | cls] ctx_out, raw sums per K split
    const Split sp = split_plan(M, a->CD + T2, a->D);
    ProdP p{};
    p.A = a->z; p.M = M; p.K = a->D;
    p.slot_emb = a->slot_emb; p.slot_of = a->slot_of; p.W = a->W; p.S = a->S;
    p.B0 = a->ctx_in_w; p.Bt = a->attn_w; p.Bc = a->cls_w; p.N0 = a->CD; p.T = a->T; p.N = a->CD + T2;
    p.C = w.cs;
    p.A2a = a->attn_w; p.A2b = a->cls_w; p.T2 = a->T; p.M2 = T2; p.B2 = a->ctx_out_w; p.N2 = a->CD; p.C2 = w.ms;
    launch_prod<true>(p, sp, st);
    // 2. h, LN1(h), the feature dots, Mo, the constants, the slots' presence
    launch_rows(RowsP{w.cs, w.ms, a->ctx_in_b, a->ctx_pos, a->ln1_w, a->ln1_b, a->ctx_out_b, a->attn_w, a->cls_w,
                      a->attn_b, a->slot_of, a->slot_mask, w.h, w.hn, w.d0, w.mo, w.dc, w.mod, w.valid, M, a->W, a->CD, a->D,
                      a->S, a->T, a->PER, sp.splits}, st);
    // 3. qkv = LN1(h) in_proj^T + b; Mf = Mo ff2
    p = ProdP{};
    p.A = w.hn; p.M = M; p.K = a->CD;
    p.B0 = a->in_proj_w; p.N0 = p.N = 3 * a->CD; p.bias = a->in_proj_b; p.C = w.qkv;
    p.A2d = w.mod; p.M2 = T2; p.B2 = a->ff2_w; p.N2 = a->FF; p.C2f = w.mf;
    launch_prod<false>(p, one, st);
    // 4. attention per (study, head), with out_proj
    const bool fuse = fuse_out(a);
    const AttnP at{w.qkv, w.valid, a->out_proj_w, fuse ? w.hp : w.att, M, a->W, a->CD, a->heads};
    const dim3 ag(a->B, a->heads, (a->W + 15) / 16);
    FfP f{w.h, w.hp, a->out_proj_b, w.h1, a->ln2_w, a->ln2_b, a->ff1_w, a->ff1_b, a->ff2_b, w.mo, w.mf, w.dc, w.part,
          M, a->CD, a->FF, a->T, a->heads};
    const dim3 fg((M + 15) / 16, (a->FF + FS - 1) / FS);
    if (fuse) {
        k_head_attn<true><<<ag, NT, 0, st>>>(at);
        k_head_ff<true><<<fg, NT, 0, st>>>(f);
    } else {
        k_head_attn<false><<<ag, NT, 0, st>>>(at);
        p = ProdP{};
        p.A = w.att; p.M = M; p.K = a->CD;
        p.B0 = a->out_proj_w; p.N0 = p.N = a->CD; p.bias = a->out_proj_b; p.R = w.h; p.C = w.h1;
        launch_prod<false>(p, one, st);
        k_head_ff<false><<<fg, NT, 0, st>>>(f);
    }
    // 6. pooling
    k_head_pool<<<a->B, PT, 0, st>>>(PoolP{w.d0, w.part, w.valid, a->cls_b, a->logits, M, a->W, a->T, (int)fg.y});
}

}  // namespace

extern "C" int d8s_head(const D8sHeadArgs* a, void* stream) {
    const char* what = "d8s_head";
    if (int rc = head_check(a, what)) return rc;
    HREQ(a->workspace, "null workspace");
    HREQ(a->ws_bytes >= carve(a, nullptr).bytes, "workspace smaller than d8s_head_workspace()");
    head_run(a, (char*)a->workspace, (hipStream_t)stream);
    return d8s_host_launched(what);
}

// ---- the entry point that allocates nothing -------------------------------------------------------
// Its workspace is this array, one copy per GPU, held until the process ends.  Host code never uses
// the array's name as an address (on the host it is a stand-in, not device memory): the device
// address of each GPU's copy comes from hipGetSymbolAddress, looked up once per device with that
// device current, and is what the kernels receive.  Every call on a GPU shares that GPU's copy, so
// calls that overlap on one GPU (different streams, no ordering between them) race.
static __device__ __align__(256) unsigned char scratch[D8S_HEAD_SCRATCH_BYTES];

namespace {

constexpr int MAX_DEVICES = 64;
std::mutex g_scratch_mu;
void* g_scratch[MAX_DEVICES] = {};

// The device address of the current device's scratch; `stream` must belong to that device.
int scratch_ptr(hipStream_t stream, void** out, const char* what) {
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    HREQ(e == hipSuccess, std::string("hipGetDevice: ") + hipGetErrorString(e));
    HREQ(dev >= 0 && dev < MAX_DEVICES, "device ordinal out of range");
    if (stream != nullptr) {
        hipDevice_t sdev = -1;
        e = hipStreamGetDevice(stream, &sdev);
        HREQ(e == hipSuccess, std::string("hipStreamGetDevice: ") + hipGetErrorString(e));
        HREQ(sdev == dev, "the stream belongs to another device than the current one");
    }
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (g_scratch[dev] == nullptr) {
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        HREQ(e == hipSuccess && p != nullptr,
             std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
        g_scratch[dev] = p;
    }
    *out = g_scratch[dev];
    return 0;
}

}  // namespace

extern "C" int d8s_head_noalloc(const D8sHeadArgs* a, void* stream) {
    const char* what = "d8s_head_noalloc";
    if (int rc = head_check(a, what)) return rc;
    const uint64_t need = carve(a, nullptr).bytes;
    HREQ(need <= D8S_HEAD_SCRATCH_BYTES,
         "workspace of " + std::to_string(need) + " bytes exceeds the static scratch of " +
             std::to_string((unsigned long long)D8S_HEAD_SCRATCH_BYTES) + " bytes (fewer studies per call)");
    void* ws = nullptr;
    if (int rc = scratch_ptr((hipStream_t)stream, &ws, what)) return rc;
    head_run(a, (char*)ws, (hipStream_t)stream);
    return d8s_host_launched(what);
}

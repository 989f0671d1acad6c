// gfx950 kernels of the upstream preprocessing (raw uint16 crops -> resize -> exact 1/99 percentiles
// -> uint8 -> side flip) and their C ABI, d8s_prep / d8s_prep_resize (include/d8s_hip.h).
//
// The work is byte and float bookkeeping bound by memory, not matrix work.  Design:
//   - uint16 regions (kind 0): the first pass evaluates the resize from the region and writes the
//     float32 stacks once to the workspace's scratch while it counts the first radix level; the
//     later passes read the stored stacks (k_prep_hist<1, 1, true>, then float_view).  Evaluating
//     the resize again in every pass instead was VALU-bound at about 40 instructions per pixel and
//     2-3x slower.  Float32 stacks (kind 1) are read as given by every pass;
//   - the order statistics k1, k1+1, k2, k2+1 are selected exactly by a three-level radix histogram
//     of the float's order key (11 + 11 + 10 bits).  Each level is one pass over the stack that
//     counts in LDS and adds the nonzero bins to a global histogram, then one workgroup per stack
//     finds the bins holding the four ranks;  equal ranks share a histogram (at most four per level);
//   - the last pass writes the uint8 value of every pixel (float64 arithmetic, the reference's exact
//     operations) at its flipped position.
// A pass works on blocks of output rows of one slice: the source rows a block needs are resized along x
// once into LDS, then every output pixel combines them along y (the bilinear formula is separable as
// written: fma(h0, top, h1 * bottom) with top and bottom the x interpolations of two source rows).  A
// histogram workgroup runs several blocks of one stack before it adds its LDS counts to the global
// histogram; the final pass runs one block per workgroup.
//
// Numerics (the file is compiled with -ffp-contract=off: only the explicit fmaf are fused):
//   rescale   (float)u * slope, then + intercept (raw_crop.py:520-522);
//   bilinear  torch's upsample_bilinear2d kernel with the fused multiply-adds its compiler forms
//             (src index fma(scale, d + 0.5, -0.5) clamped at 0; fma(h0, fma(w0, a, w1 b), h1 fma(w0, c,
//             w1 d))), raw_crop.py:431-432;
//   area      cv2's INTER_AREA tables (raw_crop.py:347-381) in float64 on the device, columns then rows,
//             each product and sum rounded, in table order with the zero padding taps
//             (raw_crop.py:396-416);
//   uint8     numpy's _lerp on the order statistics (float32 difference, float64 product and sum, the
//             t >= 0.5 form), scale = 255 / (hi - lo) (correctly rounded float64 division), then
//             ((double)x - lo) * scale clipped to [0, 255] and truncated (cache.py:319-340).
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include <math.h>
#include <stdint.h>

#include <algorithm>
#include <string>
#include <type_traits>

#include "d8s_hip.h"
#include "d8s_host.h"

#define DEV __device__ __forceinline__

namespace {

constexpr int NT = 256;                          // threads per workgroup
constexpr int NB1 = 2048, NB2 = 2048, NB3 = 1024;  // radix levels: key bits 31..21, 20..10, 9..0
constexpr int MAX_S = D8S_PREP_MAX_STACKS;
constexpr int MAX_T = D8S_PREP_MAX_TAPS;
constexpr int UP = 4;                            // output pixels per thread step (one 16-byte LDS read)
constexpr int STAGE = 10240;                     // LDS of the block kernels: 40 KB (resized rows + raw rows)

// per-stack workspace block, in 32-bit words
constexpr int W_H1 = 0;
constexpr int W_H2 = W_H1 + NB1;                 // 4 histograms of level 2
constexpr int W_H3 = W_H2 + 4 * NB2;             // 4 histograms of level 3
constexpr int W_NAN = W_H3 + 4 * NB3;            // nonzero if the stack holds a NaN
constexpr int W_SEL1 = W_NAN + 4;                // selection after level 1 (Sel, 16 words)
constexpr int W_SEL2 = W_SEL1 + 16;              // selection after level 2
constexpr int W_CLEAR = W_SEL2 + 16;             // words cleared at the start of d8s_prep
constexpr int W_TAPS = (W_CLEAR + 63) / 64 * 64; // area tables: ix, wx [img][Tx], iy, wy [img][Ty]
constexpr uint64_t WS_HEAD = 1024;               // D8sPrepStat[16] (512 bytes), then the stacks

static_assert(sizeof(D8sPrepStat) * MAX_S <= WS_HEAD, "stat header");

uint64_t stack_words(int img) { return ((uint64_t)W_TAPS + 4ull * img * MAX_T + 63) / 64 * 64; }

enum Mode { M_IDENT = 0, M_BILIN = 1, M_AREA = 2, M_FLOAT = 3 };

// The selection a level leaves for the next: `nslot` distinct key prefixes (one histogram each at the
// next level), and for each of the 4 ranks its slot and its rank among the keys of that prefix.
struct Sel {
    uint32_t nslot;
    uint32_t pre[4];
    uint32_t slot[4];
    uint32_t res[4];
    uint32_t pad_[3];
};
static_assert(sizeof(Sel) == 64, "Sel is 16 words");

struct PStack {
    const void* src;
    const float* resc;
    void* out;
    uint32_t* ws;
    float* sc;           // kind 0 in d8s_prep: the resized stack (slice kk at sc + kk img img)
    int K, hr, wr, y0, x0, h, w, k0, k1, flip, mode, Tx, Ty, r1, r2;
    float rh, rw;
    double g1, g2;
    int rb, bps, nblk;   // output rows per block, blocks per slice, blocks of the slices [k0, k1)
    int ns_max, rp, dpl; // source rows a block may read; LDS dwords per staged raw row; per lane
    int dbuf;            // 1: two raw buffers (block b+1 copied during block b's x pass); 0: one
    float inv_rp;
    int hb, hb2, nb;     // blocks per workgroup: level 1 of regions, float32 levels, final pass
    int wg_hist, wg_hist2, wg_norm;  // first workgroup of this stack in each grid
};

struct PArgs {
    PStack s[MAX_S];
    D8sPrepStat* stat;
    int n, img, upr;     // stacks, output side, UP-pixel units per output row (img / UP)
    float inv_img, inv_upr;
};

// ---- float order keys -------------------------------------------------------------------------
// unsigned key with the order of the floats: sign bit set for positives, all bits flipped for
// negatives.
DEV uint32_t order_key(float v) {
    const uint32_t b = __float_as_uint(v);
    return b ^ ((uint32_t)((int32_t)b >> 31) | 0x80000000u);
}
DEV float key_float(uint32_t k) {
    return __uint_as_float((k & 0x80000000u) ? (k ^ 0x80000000u) : ~k);
}

// ---- cv2 INTER_AREA table, one output index (raw_crop.py:347-381) --------------------------------
// Python float arithmetic is IEEE double: the same operations in the same order.  Writes up to
// `cap` taps (when idx != nullptr) and returns the row's number of taps.
__host__ __device__ inline int area_row(int ssize, int dsize, int d, int cap, int32_t* idx, float* w) {
    const double scale = 1.0 / ((double)dsize / (double)ssize);
    const double fsx1 = (double)d * scale;
    const double fsx2 = fsx1 + scale;
    const double rem = (double)ssize - fsx1;
    const double cw = rem < scale ? rem : scale;
    long sx1 = (long)ceil(fsx1), sx2 = (long)floor(fsx2);
    if (sx2 > ssize - 1) sx2 = ssize - 1;
    if (sx1 > sx2) sx1 = sx2;
    int n = 0;
    if ((double)sx1 - fsx1 > 1e-3) {
        if (idx && n < cap) { idx[n] = (int32_t)(sx1 - 1); w[n] = (float)(((double)sx1 - fsx1) / cw); }
        ++n;
    }
    for (long sx = sx1; sx < sx2; ++sx) {
        if (idx && n < cap) { idx[n] = (int32_t)sx; w[n] = (float)(1.0 / cw); }
        ++n;
    }
    if (fsx2 - (double)sx2 > 1e-3) {
        double a = fsx2 - (double)sx2;
        if (1.0 < a) a = 1.0;
        if (cw < a) a = cw;
        if (idx && n < cap) { idx[n] = (int32_t)sx2; w[n] = (float)(a / cw); }
        ++n;
    }
    return n;
}

int area_taps_max(int ssize, int dsize) {
    int T = 0;
    for (int d = 0; d < dsize; ++d) {
        const int n = area_row(ssize, dsize, d, 0, nullptr, nullptr);
        if (n > T) T = n;
    }
    return T;
}

// ---- evaluation of 8 output pixels -------------------------------------------------------------
DEV float src_index(float scale, int d) {
    const float s = __builtin_fmaf(scale, (float)d + 0.5f, -0.5f);
    return s < 0.0f ? 0.0f : s;
}

// n / d for 0 <= n < 2^22 and 1 <= d <= 4096 (inv = 1 / d): a float estimate, corrected.
DEV int fdiv(int n, int d, float inv) {
    int q = (int)((float)n * inv);
    q -= q * d > n ? 1 : 0;
    q += (q + 1) * d <= n ? 1 : 0;
    return q;
}

// A block: output rows [r0, r0 + rb) of slice kk, reading source rows [s0, s0 + ns) of the crop.
struct Geo {
    int kk, r0, rb, s0, ns;
};

template <int MODE>
DEV Geo block_geo(const PStack& st, const PArgs& a, int b) {
    Geo g;
    const int q = b / st.bps;
    g.kk = st.k0 + q;
    g.r0 = (b - q * st.bps) * st.rb;
    g.rb = min(st.rb, a.img - g.r0);
    if constexpr (MODE == M_FLOAT) {
        g.s0 = 0;
        g.ns = 0;
        return g;
    } else {
        int s1;
        if constexpr (MODE == M_IDENT) {
            g.s0 = g.r0;
            s1 = g.r0 + g.rb;
        } else if constexpr (MODE == M_BILIN) {
            g.s0 = (int)src_index(st.rh, g.r0);
            const int h1 = (int)src_index(st.rh, g.r0 + g.rb - 1);
            s1 = h1 + (h1 < st.h - 1 ? 1 : 0) + 1;
        } else {
            const int32_t* iy = (const int32_t*)st.ws + W_TAPS + 2 * a.img * st.Tx;
            const float* wy = (const float*)(iy + a.img * st.Ty);
            const int last = g.r0 + g.rb - 1;
            int t = st.Ty - 1;
            while (t > 0 && !(wy[last * st.Ty + t] > 0.0f)) --t;   // the padding taps have weight 0
            g.s0 = iy[g.r0 * st.Ty];
            s1 = iy[last * st.Ty] + t + 1;
        }
        g.ns = min(s1 - g.s0, st.ns_max);
        return g;
    }
}

constexpr int NW = NT / 64;  // waves per workgroup

// Copies source rows [s0, s0 + ns) of a block, crop columns [0, w), to LDS with gfx950's
// global_load_lds (memory to LDS without registers).  Wave v copies rows v, v + NW, ...; row r starts
// at element e_r = e0 + r wr of the dword-aligned series base, and its dwords [0, nd) from element
// e_r & ~1 (the first and last may hold 2 bytes of the neighbouring rows, nothing outside the dwords
// that hold the row) go to s_raw[r][0 .. nd); lanes past nd repeat the last dword, inside the row's
// 64-dword-padded slot.  The caller waits for the copies (vmcnt) and synchronises.
DEV void raw_stage(const PStack& st, const Geo& g, uint32_t* s_raw) {
    const int wv = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = (int)threadIdx.x & 63;
    const uint32_t* base = (const uint32_t*)((uintptr_t)st.src & ~(uintptr_t)3);
    const int e0 = (int)(((uintptr_t)st.src >> 1) & 1u) + (g.kk * st.hr + st.y0 + g.s0) * st.wr + st.x0;
    const int pitch = st.dpl * 64;
    for (int r = wv; r < g.ns; r += NW) {
        const int er = e0 + r * st.wr;
        const int nd = ((er & 1) + st.w + 1) >> 1;
        const uint32_t* row = base + (er >> 1);
        for (int m = 0; m < st.dpl; ++m) {
            const int d = min(lane + 64 * m, nd - 1);
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(row + d),
                                             (__attribute__((address_space(3))) void*)(s_raw + r * pitch + 64 * m),
                                             4, 0, 0);
        }
    }
}

template <bool HAS>
DEV float rescale(uint32_t u, float sl, float ic) {
    const float f = (float)u;
    if constexpr (!HAS) {
        return f;
    } else {
        const float p = f * sl;
        return p + ic;
    }
}

// The values of every block b0 .. b1-1 of stack st, UP consecutive pixels of a row at a time, handed to
// f(kk, dy, dx0, v).  Region modes: a block's raw rows are copied to LDS (two buffers: the copy of block
// b+1 runs while block b is computed), resized along x into
// s_st [ns][img] (bilinear `top`/`bottom` values fma(w0, a, w1 b), area column sums, identity values),
// and every pixel combines them along y.  A thread keeps the same output columns in the x pass, so
// their interpolation positions are computed once.  The workgroup calls this uniformly (it holds
// barriers).
//
// The area taps of an output index are consecutive source indices (raw_crop.py:361-369), so a tap's
// source is the first index + t; a zero-weight padding tap then reads a neighbour instead of index 0,
// which changes nothing for finite values (x * 0 = +-0 added to a sum that is never -0).
template <int MODE, bool HAS, bool WROW, int TH = NT, class F>
DEV void run_blocks(const PStack& st, const PArgs& a, int b0, int b1, float* s_st, F&& f) {
    const int img = a.img;
    if constexpr (MODE == M_FLOAT) {
        // a thread's units u = tid + TH i of a block in batches of FB: the batch's loads are issued
        // before any of its values is used (the histogram passes' LDS atomics would otherwise keep
        // each load behind the previous unit's counting); units past the block load its last unit
        // again and are not used
        constexpr int FB = 4;
        for (int b = b0; b < b1; ++b) {
            const Geo g = block_geo<MODE>(st, a, b);
            const int n = g.rb * a.upr;
            const float* base = (const float*)st.src + (int64_t)g.kk * img * img;
            for (int u0 = threadIdx.x; u0 < n; u0 += FB * TH) {
                float4 x[FB];
                int dy[FB], dx0[FB];
#pragma unroll
                for (int i = 0; i < FB; ++i) {
                    const int u = min(u0 + i * TH, n - 1);
                    const int row = fdiv(u, a.upr, a.inv_upr);
                    dx0[i] = (u - row * a.upr) * UP;
                    dy[i] = g.r0 + row;
                    x[i] = *(const float4*)(base + (int64_t)dy[i] * img + dx0[i]);
                }
#pragma unroll
                for (int i = 0; i < FB; ++i) {
                    if (u0 + i * TH < n) {
                        float v[UP] = {x[i].x, x[i].y, x[i].z, x[i].w};
                        f(g.kk, dy[i], dx0[i], v);
                    }
                }
            }
        }
        return;
    } else {
        constexpr int CMAX = 4;                      // output columns per thread in the x pass (img <= 1024)
        const int32_t* ix = (const int32_t*)st.ws + W_TAPS;
        const float* wx = (const float*)(ix + img * st.Tx);
        const int32_t* iy = (const int32_t*)(wx + img * st.Tx);
        const float* wy = (const float*)(iy + img * st.Ty);
        const int pitch = st.dpl * 64;               // dwords per staged raw row
        // raw buffers: with two, block b+1 is copied during block b's x pass; with one, during its
        // y pass
        uint32_t* s_raw0 = (uint32_t*)(s_st + st.ns_max * img);
        uint32_t* s_raw1 = st.dbuf ? s_raw0 + st.ns_max * pitch : s_raw0;
        // x-pass mapping: img >= NT: columns tid + c NT, every row; img < NT: column tid % img, rows
        // tid / img + P j (threads beyond P img rest)
        const int P = img >= NT ? 1 : NT / img;
        const int ph = img >= NT ? 0 : (int)threadIdx.x / img;
        const int col0 = (int)threadIdx.x - ph * img;
        const bool xact = ph < P;
        int ca[CMAX], cb[CMAX];          // uint16 index of the two taps (bilinear) / first tap (area)
        float cm0[CMAX], cm1[CMAX];      // bilinear weights / area: first and middle tap weights
        float cwl[CMAX];                 // area: last tap weight; cb = number of real taps
#pragma unroll
        for (int c = 0; c < CMAX; ++c) {
            const int dx = min(col0 + c * NT, img - 1);
            ca[c] = cb[c] = dx;
            cm0[c] = cm1[c] = 0.0f;
            if constexpr (MODE == M_BILIN) {
                const float sx = src_index(st.rw, dx);
                const int w1 = (int)sx;
                ca[c] = w1;
                cb[c] = w1 + (w1 < st.w - 1 ? 1 : 0);
                cm1[c] = sx - (float)w1;
                cm0[c] = 1.0f - cm1[c];
            } else if constexpr (MODE == M_AREA) {
                // a table row is [first, middle ..., last] with equal middle weights
                // (raw_crop.py:361-369), then zero padding: keep first / middle / last and the count
                cwl[c] = 0.0f;
                if (st.w != img) {
                    const float* tw = wx + dx * st.Tx;
                    ca[c] = ix[dx * st.Tx];
                    int n = 0;
                    for (int t = 0; t < st.Tx; ++t) n += tw[t] > 0.0f ? 1 : 0;
                    cb[c] = n;
                    cm0[c] = tw[0];
                    cm1[c] = n > 2 ? tw[1] : 0.0f;
                    cwl[c] = tw[n > 0 ? n - 1 : 0];
                }
            }
        }
        // uint16 parity of the crop rows: row index q starts at element (src / 2) + q wr + x0
        const int par0 = (int)((((uintptr_t)st.src >> 1) + (uintptr_t)st.x0) & 1u);
        const int last = st.ns_max - 1;
        // y-pass mapping: RS rows at a time, thread (tr, tc); with WROW (a row is a multiple of 64
        // units) every wave works on one row, so the row quantities are wave-uniform
        const int RS = NT / a.upr;
        int tr = (int)threadIdx.x / a.upr;
        if constexpr (WROW) tr = __builtin_amdgcn_readfirstlane(tr);
        const int dx0 = ((int)threadIdx.x - ((int)threadIdx.x / a.upr) * a.upr) * UP;
        const bool yact = tr < RS;
        // bilinear: the taps and weights of the thread's UP output columns dx0 .. dx0 + UP - 1
        int ba[UP], bb[UP];
        float bw0[UP], bw1[UP];
        if constexpr (MODE == M_BILIN) {
#pragma unroll
            for (int i = 0; i < UP; ++i) {
                const float sx = src_index(st.rw, dx0 + i);
                const int w1 = (int)sx;
                ba[i] = w1;
                bb[i] = w1 + (w1 < st.w - 1 ? 1 : 0);
                bw1[i] = sx - (float)w1;
                bw0[i] = 1.0f - bw1[i];
            }
        }
        Geo nxt = block_geo<MODE>(st, a, b0);
        raw_stage(st, nxt, s_raw0);
        for (int b = b0; b < b1; ++b) {
            const Geo g = nxt;
            const uint16_t* raw16 = (const uint16_t*)((b - b0) & 1 ? s_raw1 : s_raw0);
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
            if (st.dbuf && b + 1 < b1) {
                nxt = block_geo<MODE>(st, a, b + 1);
                raw_stage(st, nxt, (b - b0) & 1 ? s_raw0 : s_raw1);
            }
            const float sl = HAS ? st.resc[2 * g.kk] : 1.0f, ic = HAS ? st.resc[2 * g.kk + 1] : 0.0f;
            const int e0 = par0 + (g.kk * st.hr + st.y0 + g.s0) * st.wr;
            if constexpr (MODE == M_BILIN) {
                // one pass: thread (tr, tc) walks the contiguous rows tr rpg .. (tr + 1) rpg - 1 of the
                // block down its UP columns and keeps the horizontal interpolations of the two source
                // rows it combines in registers (consecutive output rows mostly share them when
                // upsampling); the same operations as the x and y passes below, in the same order
                if (yact) {
                    const int rpg = (g.rb + RS - 1) / RS;
                    const int rr1 = min(g.rb, (tr + 1) * rpg);
                    int cq0 = -1, cq1 = -1;
                    float X0[UP], X1[UP];
                    auto xrow = [&](int q, float* X) {
                        const uint16_t* row = raw16 + q * 2 * pitch + ((e0 + q * st.wr) & 1);
#pragma unroll
                        for (int i = 0; i < UP; ++i)
                            X[i] = __builtin_fmaf(bw0[i], rescale<HAS>(row[ba[i]], sl, ic),
                                                  bw1[i] * rescale<HAS>(row[bb[i]], sl, ic));
                    };
                    for (int rr = tr * rpg; rr < rr1; ++rr) {
                        const int dy = g.r0 + rr;
                        const float sy = src_index(st.rh, dy);
                        const int h1 = (int)sy;
                        const int h1p = h1 < st.h - 1 ? 1 : 0;
                        const float l1 = sy - (float)h1, l0 = 1.0f - l1;
                        const int q0 = min(h1 - g.s0, last), q1 = min(h1 + h1p - g.s0, last);
                        if (q0 != cq0) {
                            if (q0 == cq1) {
#pragma unroll
                                for (int i = 0; i < UP; ++i) X0[i] = X1[i];
                            } else {
                                xrow(q0, X0);
                            }
                            cq0 = q0;
                            cq1 = -1;
                        }
                        if (q1 != cq1) {
                            if (q1 == q0) {
#pragma unroll
                                for (int i = 0; i < UP; ++i) X1[i] = X0[i];
                            } else {
                                xrow(q1, X1);
                            }
                            cq1 = q1;
                        }
                        float v[UP];
#pragma unroll
                        for (int i = 0; i < UP; ++i) v[i] = __builtin_fmaf(l0, X0[i], l1 * X1[i]);
                        f(g.kk, dy, dx0, v);
                    }
                }
                if (!st.dbuf && b + 1 < b1) {
                    __syncthreads();                      // every thread is done with this block's rows
                    nxt = block_geo<MODE>(st, a, b + 1);
                    raw_stage(st, nxt, s_raw0);
                }
                continue;
            }
            if (xact) {
                for (int r = ph; r < g.ns; r += P) {
                    const uint16_t* row = raw16 + r * 2 * pitch + ((e0 + r * st.wr) & 1);
                    float* dst = s_st + r * img;
#pragma unroll
                    for (int c = 0; c < CMAX; ++c) {
                        const int dx = col0 + c * NT;
                        if (c * NT < img && dx < img) {
                            float v;
                            if constexpr (MODE == M_IDENT) {
                                v = rescale<HAS>(row[dx], sl, ic);
                            } else if constexpr (MODE == M_BILIN) {
                                const float xa = rescale<HAS>(row[ca[c]], sl, ic);
                                const float xb = rescale<HAS>(row[cb[c]], sl, ic);
                                v = __builtin_fmaf(cm0[c], xa, cm1[c] * xb);
                            } else if (st.w == img) {
                                v = rescale<HAS>(row[dx], sl, ic);
                            } else {
                                // every tap of the table in order; the padding taps (weight 0) read
                                // a neighbour (x * 0 adds nothing to a finite sum)
                                v = 0.0f;
                                const uint16_t* tp = row + ca[c];
                                const int lim = st.w - 1 - ca[c];
                                for (int t = 0; t < st.Tx; ++t) {
                                    const float wt = t == 0 ? cm0[c]
                                                   : t >= cb[c] ? 0.0f
                                                   : t == cb[c] - 1 ? cwl[c] : cm1[c];
                                    const float p = rescale<HAS>(tp[min(t, lim)], sl, ic) * wt;
                                    v = v + p;
                                }
                            }
                            dst[dx] = v;
                        }
                    }
                }
            }
            __syncthreads();
            if (!st.dbuf && b + 1 < b1) {
                nxt = block_geo<MODE>(st, a, b + 1);
                raw_stage(st, nxt, s_raw0);
            }
            // combine along y: thread (row phase tr, unit column tc) runs rows tr, tr + RS, ...
            if (yact) {
                for (int rr = tr; rr < g.rb; rr += RS) {
                    const int dy = g.r0 + rr;
                    float v[UP];
                    if constexpr (MODE == M_IDENT) {
                        const float* p = s_st + min(dy - g.s0, last) * img + dx0;
#pragma unroll
                        for (int i = 0; i < UP; ++i) v[i] = p[i];
                    } else if constexpr (MODE == M_BILIN) {
                        const float sy = src_index(st.rh, dy);
                        const int h1 = (int)sy;
                        const int h1p = h1 < st.h - 1 ? 1 : 0;
                        const float l1 = sy - (float)h1, l0 = 1.0f - l1;
                        const float* p0 = s_st + min(h1 - g.s0, last) * img + dx0;
                        const float* p1 = s_st + min(h1 + h1p - g.s0, last) * img + dx0;
#pragma unroll
                        for (int i = 0; i < UP; ++i) v[i] = __builtin_fmaf(l0, p0[i], l1 * p1[i]);
                    } else {
                        // the row's real taps in table order (its zero-weight padding taps add +0 to
                        // a finite sum and are skipped: their source row need not be staged)
                        const int y0t = iy[dy * st.Ty] - g.s0;
                        const float* tw = wy + dy * st.Ty;
#pragma unroll
                        for (int i = 0; i < UP; ++i) v[i] = 0.0f;
                        for (int j = 0; j < st.Ty; ++j) {
                            const float wyj = tw[j];
                            if (!(wyj > 0.0f)) break;
                            const float* p = s_st + min(y0t + j, last) * img + dx0;
#pragma unroll
                            for (int i = 0; i < UP; ++i) {
                                const float q = p[i] * wyj;
                                v[i] = v[i] + q;
                            }
                        }
                    }
                    f(g.kk, dy, dx0, v);
                }
            }
            __syncthreads();
        }
    }
}

// REGION: the kernel instance for uint16 regions (kind 0) or for float32 stacks (kind 1).  Runs
// body(mode, rescale, wave-uniform rows) with the stack's mode, whether it has a Rescale and whether
// an output row is a multiple of 64 units as constants.
template <int REGION, class B>
DEV void with_mode(const PStack& st, const PArgs& a, B&& body) {
    using T = std::true_type;
    using N = std::false_type;
    if constexpr (REGION) {
        const bool h = st.resc != nullptr;
        auto go = [&](auto m) {
            if (a.upr % 64 == 0)
                h ? body(m, T{}, T{}) : body(m, N{}, T{});
            else
                h ? body(m, T{}, N{}) : body(m, N{}, N{});
        };
        switch (st.mode) {
            case M_IDENT: go(std::integral_constant<int, M_IDENT>{}); break;
            case M_BILIN: go(std::integral_constant<int, M_BILIN>{}); break;
            default: go(std::integral_constant<int, M_AREA>{}); break;
        }
    } else {
        body(std::integral_constant<int, M_FLOAT>{}, N{}, N{});
    }
}

// grid 0: histogram level 1 of regions; 1: the float32 levels; 2: final pass and resize
DEV int first_wg(const PStack& p, int grid) { return grid == 0 ? p.wg_hist : grid == 1 ? p.wg_hist2 : p.wg_norm; }

DEV int stack_of(const PArgs& a, int grid) {
    int s = 0;
    for (int i = 1; i < a.n; ++i)
        if ((int)blockIdx.x >= first_wg(a.s[i], grid)) s = i;
    return s;
}

// ---- kernels ------------------------------------------------------------------------------------

// Clears the histograms and selections of every stack, writes the zeros of the output slices outside
// [k0, k1) (d8s_prep: clear = 1) and builds the area tables.
__global__ void __launch_bounds__(NT) k_prep_setup(PArgs a, int clear) {
    const PStack& st = a.s[blockIdx.y];
    const int gid = blockIdx.x * NT + threadIdx.x, gsz = gridDim.x * NT;
    if (clear) {
        for (int i = gid; i < W_CLEAR; i += gsz) st.ws[i] = 0u;
        const int per = a.img * a.img / 8;            // 8-byte words per slice
        const int outside = (st.K - (st.k1 - st.k0)) * per;
        for (int i = gid; i < outside; i += gsz) {
            int kk = i / per;
            kk = kk < st.k0 ? kk : kk + (st.k1 - st.k0);
            const int ko = st.flip == D8S_FLIP_SLICES ? st.K - 1 - kk : kk;
            ((uint2*)st.out)[(int64_t)ko * per + (i % per)] = make_uint2(0u, 0u);
        }
    }
    if (st.mode != M_AREA) return;
    int32_t* ix = (int32_t*)st.ws + W_TAPS;
    float* wx = (float*)(ix + a.img * st.Tx);
    int32_t* iy = (int32_t*)(wx + a.img * st.Tx);
    float* wy = (float*)(iy + a.img * st.Ty);
    for (int d = gid; d < a.img; d += gsz) {
        int32_t ti[MAX_T];
        float tw[MAX_T];
        if (st.w != a.img) {
            const int n = area_row(st.w, a.img, d, MAX_T, ti, tw);
            for (int j = 0; j < st.Tx; ++j) {
                ix[d * st.Tx + j] = j < n ? ti[j] : 0;
                wx[d * st.Tx + j] = j < n ? tw[j] : 0.0f;
            }
        }
        const int n = area_row(st.h, a.img, d, MAX_T, ti, tw);
        for (int j = 0; j < st.Ty; ++j) {
            iy[d * st.Ty + j] = j < n ? ti[j] : 0;
            wy[d * st.Ty + j] = j < n ? tw[j] : 0.0f;
        }
    }
}

// One radix level over the blocks [b0, b0 + hb) of one stack.  Float32 stacks run wide workgroups over
// many blocks (wide_view): noisy values fill most of a level-2 histogram, and each workgroup adds its
// nonzero bins to the global one, so their number is what that costs (level 2 of 8 stacks of 24 x 288^2:
// 25 us with 1012 workgroups of 256, 21 with 506 of 1024).
constexpr int WIDE = 1024;
template <int LEVEL, int REGION, bool STORE = false>
__global__ void __launch_bounds__(LEVEL == 1 && REGION ? NT : WIDE) k_prep_hist(PArgs a) {
    constexpr bool WD = LEVEL > 1 || !REGION;
    constexpr int TH = WD ? WIDE : NT;
    // level 1 of float32 stacks: copies of its histogram, a lane's by its index.  The keys' top bits put
    // neighbouring values in few bins, so 64 lanes adding to one copy would mostly wait for each other
    // (and runs kept per thread broke at almost every unit of noisy values: 22.5 us, now 19.3)
    constexpr int CP = LEVEL == 1 && !REGION ? 8 : 1;
    constexpr int NB = LEVEL == 1 ? NB1 : LEVEL == 2 ? NB2 : NB3;
    constexpr int NH = LEVEL == 1 ? 1 : 2;    // LDS histograms; slots 2 and 3 (rare) count in memory
    __shared__ uint32_t s_h[NH * NB * CP];
    __shared__ float s_st[REGION ? STAGE : 1];
    const int s = stack_of(a, WD ? 1 : 0);
    const PStack& st = a.s[s];
    for (int i = threadIdx.x; i < NH * NB * CP; i += TH) s_h[i] = 0u;
    uint32_t nslot = 0, pre[4] = {0u, 0u, 0u, 0u};
    if constexpr (LEVEL > 1) {
        const Sel* sel = (const Sel*)(st.ws + (LEVEL == 2 ? W_SEL1 : W_SEL2));
        nslot = sel->nslot;
#pragma unroll
        for (int t = 0; t < 4; ++t) pre[t] = sel->pre[t];
    }
    __syncthreads();
    const int hb = WD ? st.hb2 : st.hb;
    const int b0 = ((int)blockIdx.x - (WD ? st.wg_hist2 : st.wg_hist)) * hb;
    const int b1 = min(b0 + hb, st.nblk);
    bool nan = false;
    uint32_t run_bin = 0xffffffffu, run_n = 0u;   // the thread's current run of one histogram index
    uint32_t* gh = st.ws + (LEVEL == 1 ? W_H1 : LEVEL == 2 ? W_H2 : W_H3);
    auto run_flush = [&]() {
        if (LEVEL == 1 || run_bin < (uint32_t)(NH * NB))
            atomicAdd(&s_h[run_bin], run_n);
        else
            atomicAdd(gh + run_bin, run_n);
    };
    auto count = [&](int kk, int dy, int dx0, const float* v) {
        if constexpr (STORE)
            *(float4*)(st.sc + ((int64_t)kk * a.img + dy) * a.img + dx0) = make_float4(v[0], v[1], v[2], v[3]);
        // The UP values of a unit are counted in one step when every counted one continues the
        // thread's run (the common case: no branch taken); otherwise value by value.
        if constexpr (CP > 1) {
#pragma unroll
            for (int i = 0; i < UP; ++i) {
                nan |= v[i] != v[i];
                atomicAdd(&s_h[(order_key(v[i]) >> 21) * CP + (threadIdx.x & (CP - 1))], 1u);
            }
            return;
        }
        if constexpr (LEVEL == 1) {
            // a thread's values are neighbours (UP along x, then the next row of its column), so they
            // mostly share a (coarse) level-1 bin: the thread counts a run in a register and adds it
            // to LDS when the bin changes
            uint32_t b[UP];
            bool same = true;
#pragma unroll
            for (int i = 0; i < UP; ++i) {
                nan |= v[i] != v[i];
                b[i] = order_key(v[i]) >> 21;
                same &= b[i] == run_bin;
            }
            if (same) {
                run_n += UP;
                return;
            }
#pragma unroll
            for (int i = 0; i < UP; ++i) {
                if (b[i] != run_bin) {
                    if (run_n) run_flush();
                    run_bin = b[i];
                    run_n = 0u;
                }
                ++run_n;
            }
            return;
        }
        // the keys under one of the slots' prefixes (unused slots hold 0xffffffff, which no key has at
        // these levels); index = slot * NB + bin, slots from NH on count in memory.  Keys of the thread's
        // run (a value four of its neighbours shared, e.g. a zero background) count in a register; any
        // other adds to LDS by itself and leaves the run: within one level-1 bin the keys spread over the
        // 2048 finer ones, so lanes seldom meet.  (A run that followed every change of bin broke at
        // almost every unit of noisy values: level 2 of 8 stacks of 24 x 288^2 26.6 us, with the wide workgroups 21-25; a wave
        // counting only its uniform units in one add took 88 against 48 us at a study's two levels,
        // where background and body share waves.)
        uint32_t idx[UP];
        bool ok[UP], one = true;
#pragma unroll
        for (int i = 0; i < UP; ++i) {
            const uint32_t k = order_key(v[i]);
            const uint32_t p = LEVEL == 2 ? k >> 21 : k >> 10;
            const uint32_t bin = LEVEL == 2 ? (k >> 10) & (NB2 - 1) : k & (NB3 - 1);
            ok[i] = p == pre[0] || p == pre[1] || p == pre[2] || p == pre[3];
            const uint32_t t = p == pre[0] ? 0u : p == pre[1] ? 1u : p == pre[2] ? 2u : 3u;
            idx[i] = t * NB + bin;
            one &= ok[i] && idx[i] == idx[0];
        }
        if (one && idx[0] != run_bin) {
            if (run_n) run_flush();
            run_bin = idx[0];
            run_n = 0u;
        }
#pragma unroll
        for (int i = 0; i < UP; ++i) {
            const bool in = idx[i] == run_bin;
            run_n += ok[i] && in ? 1u : 0u;
            if (ok[i] && !in) {
                if (idx[i] < (uint32_t)(NH * NB))
                    atomicAdd(&s_h[idx[i]], 1u);
                else
                    atomicAdd(gh + idx[i], 1u);
            }
        }
    };
    with_mode<REGION>(st, a, [&](auto m, auto h, auto w) {
        run_blocks<decltype(m)::value, decltype(h)::value, decltype(w)::value, TH>(st, a, b0, b1, s_st, count);
    });
    if (run_n) run_flush();
    if constexpr (LEVEL == 1) {
        if (__ballot(nan) != 0ull && (int)__lane_id() == 0) atomicOr(st.ws + W_NAN, 1u);
    }
    __syncthreads();
    const int nh = LEVEL == 1 ? 1 : min((int)nslot, NH);
    for (int i = threadIdx.x; i < nh * NB; i += TH) {
        uint32_t c = 0u;
#pragma unroll
        for (int k = 0; k < CP; ++k) c += s_h[i * CP + k];
        if (c) atomicAdd(gh + i, c);
    }
}

// Exclusive prefix sums over the workgroup of four values per thread at once.
DEV void block_excl_scan4(uint32_t (&x)[4], uint32_t (*s_w)[4]) {
    const int lane = __lane_id(), wv = threadIdx.x >> 6;
    uint32_t incl[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) incl[t] = x[t];
#pragma unroll
    for (int d = 1; d < 64; d <<= 1)
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const uint32_t y = __shfl_up(incl[t], d, 64);
            if (lane >= d) incl[t] += y;
        }
    if (lane == 63)
#pragma unroll
        for (int t = 0; t < 4; ++t) s_w[wv][t] = incl[t];
    __syncthreads();
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        uint32_t base = 0;
#pragma unroll
        for (int i = 0; i < NT / 64; ++i) base += i < wv ? s_w[i][t] : 0u;
        x[t] = base + incl[t] - x[t];
    }
}

// The bins holding the 4 ranks at one level (one workgroup per stack); the last level also derives
// the percentiles, the scale and the bad flag.  Latency is its cost (one workgroup, between two passes that
// wait for it): the four ranks' histograms are loaded together, 16 bytes a load, and scanned together
// (rank by rank it took 6.1, 6.5 and 4.7 us, now 4.1-4.7 each).
template <int LEVEL>
__global__ void __launch_bounds__(NT) k_prep_select(PArgs a) {
    constexpr int NB = LEVEL == 1 ? NB1 : LEVEL == 2 ? NB2 : NB3;
    constexpr int PER = NB / NT;
    __shared__ uint32_t s_w[NT / 64][4];
    __shared__ uint32_t s_bin[4], s_res[4];
    const PStack& st = a.s[blockIdx.x];
    uint32_t rank[4], slot[4] = {0u, 0u, 0u, 0u}, pre[4] = {0u, 0u, 0u, 0u};
    if constexpr (LEVEL == 1) {
        rank[0] = (uint32_t)st.r1; rank[1] = (uint32_t)st.r1 + 1u;
        rank[2] = (uint32_t)st.r2; rank[3] = (uint32_t)st.r2 + 1u;
    } else {
        const Sel* sel = (const Sel*)(st.ws + (LEVEL == 2 ? W_SEL1 : W_SEL2));
#pragma unroll
        for (int t = 0; t < 4; ++t) { rank[t] = sel->res[t]; slot[t] = sel->slot[t] & 3u; pre[t] = sel->pre[t]; }
    }
    const uint32_t* gh = st.ws + (LEVEL == 1 ? W_H1 : LEVEL == 2 ? W_H2 : W_H3);
    if (threadIdx.x < 4) { s_bin[threadIdx.x] = 0u; s_res[threadIdx.x] = 0u; }
    static_assert(PER % 4 == 0, "whole 16-byte loads");
    uint32_t c[4][PER], sum[4], excl[4];
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int i = 0; i < PER; i += 4) {
            const uint4 v = *(const uint4*)(gh + slot[t] * NB + threadIdx.x * PER + i);
            c[t][i] = v.x; c[t][i + 1] = v.y; c[t][i + 2] = v.z; c[t][i + 3] = v.w;
        }
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        sum[t] = 0;
#pragma unroll
        for (int i = 0; i < PER; ++i) sum[t] += c[t][i];
        excl[t] = sum[t];
    }
    block_excl_scan4(excl, s_w);
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        if (excl[t] <= rank[t] && rank[t] < excl[t] + sum[t]) {
            uint32_t acc = excl[t];
#pragma unroll
            for (int i = 0; i < PER; ++i) {
                if (rank[t] >= acc && rank[t] < acc + c[t][i]) {
                    s_bin[t] = threadIdx.x * PER + i;
                    s_res[t] = rank[t] - acc;
                }
                acc += c[t][i];
            }
        }
    }
    __syncthreads();
    if (threadIdx.x != 0) return;
    uint32_t key[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const uint32_t b = s_bin[t];
        const uint32_t q = slot[t] == 0 ? pre[0] : slot[t] == 1 ? pre[1] : slot[t] == 2 ? pre[2] : pre[3];
        key[t] = LEVEL == 1 ? b : LEVEL == 2 ? ((q << 11) | b) : ((q << 10) | b);
    }
    if constexpr (LEVEL < 3) {
        // the distinct keys in order of first use (indexed by constants: no array in memory)
        Sel out;
        uint32_t nslot = 0;
#pragma unroll
        for (int t = 0; t < 4; ++t) out.pre[t] = 0xffffffffu;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            uint32_t j = nslot;
#pragma unroll
            for (int u = t - 1; u >= 0; --u) j = key[u] == key[t] ? out.slot[u] : j;
            out.slot[t] = j;
            out.res[t] = s_res[t];
#pragma unroll
            for (int s = 0; s < 4; ++s) out.pre[s] = (uint32_t)s == j ? key[t] : out.pre[s];
            nslot += j == nslot ? 1u : 0u;
        }
        out.nslot = nslot;
        out.pad_[0] = out.pad_[1] = out.pad_[2] = 0u;
        Sel* dst = (Sel*)(st.ws + (LEVEL == 1 ? W_SEL1 : W_SEL2));
        *dst = out;
    } else {
        // numpy's _lerp: difference in float32, product and sum in float64, the t >= 0.5 form
        const float pv[2] = {key_float(key[0]), key_float(key[2])};
        const float nx[2] = {key_float(key[1]), key_float(key[3])};
        const double g[2] = {st.g1, st.g2};
        double q[2];
        for (int i = 0; i < 2; ++i) {
            const float diff = nx[i] - pv[i];
            double lerp = (double)pv[i] + (double)diff * g[i];
            if (g[i] >= 0.5) lerp = (double)nx[i] - (double)diff * (1.0 - g[i]);
            q[i] = lerp;
        }
        const double lo = q[0], hi = q[1];
        const bool nan = st.ws[W_NAN] != 0u;
        const bool bad = nan || !isfinite(lo) || !isfinite(hi) || hi <= lo;
        D8sPrepStat r;
        r.lo = lo;
        r.hi = hi;
        r.scale = 255.0 / (hi - lo);
        r.bad = bad ? 1 : 0;
        r.pad_ = 0;
        a.stat[blockIdx.x] = r;
    }
}

// Final pass: uint8 of every pixel, written at its flipped position.
template <int REGION>
__global__ void __launch_bounds__(NT) k_prep_norm(PArgs a) {
    const int s = stack_of(a, 2);
    const PStack& st = a.s[s];
    const D8sPrepStat r = a.stat[s];
    const double nlo = -r.lo;
    __shared__ float s_st[REGION ? STAGE : 1];
    const int b0 = ((int)blockIdx.x - st.wg_norm) * st.nb;
    const int b1 = min(b0 + st.nb, st.nblk);
    uint8_t* out = (uint8_t*)st.out;
    auto write = [&](int kk, int dy, int dx0, const float* v) {
        uint32_t b[UP];
#pragma unroll
        for (int i = 0; i < UP; ++i) {
            // (x - lo) * scale clipped to [0, 255] and truncated; x + (-lo) is x - lo exactly
            double y = (double)v[i] + nlo;
            y = y * r.scale;
            y = __builtin_fmax(y, 0.0);
            y = __builtin_fmin(y, 255.0);
            b[i] = (uint32_t)y;
        }
        const int ko = st.flip == D8S_FLIP_SLICES ? st.K - 1 - kk : kk;
        uint32_t word;
        int xo = dx0;
        if (st.flip == D8S_FLIP_X) {
            xo = a.img - UP - dx0;
            word = b[3] | (b[2] << 8) | (b[1] << 16) | (b[0] << 24);
        } else {
            word = b[0] | (b[1] << 8) | (b[2] << 16) | (b[3] << 24);
        }
        *(uint32_t*)(out + ((int64_t)ko * a.img + dy) * a.img + xo) = word;
    };
    if (r.bad) {
        // a stack with non-finite or equal percentiles (or a NaN) is all zeros: its rows of the blocks
        const int per = a.img / 4;
        for (int b = b0; b < b1; ++b) {
            const int q = b / st.bps, kk = st.k0 + q, r0 = (b - q * st.bps) * st.rb;
            const int rb = min(st.rb, a.img - r0);
            const int ko = st.flip == D8S_FLIP_SLICES ? st.K - 1 - kk : kk;
            uint32_t* o = (uint32_t*)(out + ((int64_t)ko * a.img + r0) * a.img);
            for (int i = threadIdx.x; i < rb * per; i += NT) o[i] = 0u;
        }
        return;
    }
    with_mode<REGION>(st, a, [&](auto m, auto h, auto w) {
        run_blocks<decltype(m)::value, decltype(h)::value, decltype(w)::value>(st, a, b0, b1, s_st, write);
    });
}

// The resized float32 values themselves.
__global__ void __launch_bounds__(NT) k_prep_resize(PArgs a) {
    const int s = stack_of(a, 2);
    const PStack& st = a.s[s];
    __shared__ float s_st[STAGE];
    const int b0 = ((int)blockIdx.x - st.wg_norm) * st.nb;
    const int b1 = min(b0 + st.nb, st.nblk);
    float* out = (float*)st.out;
    auto write = [&](int kk, int dy, int dx0, const float* v) {
        *(float4*)(out + ((int64_t)kk * a.img + dy) * a.img + dx0) = make_float4(v[0], v[1], v[2], v[3]);
    };
    with_mode<1>(st, a, [&](auto m, auto h, auto w) {
        run_blocks<decltype(m)::value, decltype(h)::value, decltype(w)::value>(st, a, b0, b1, s_st, write);
    });
}

// ---- grid sampling (geometric TTA view) -------------------------------------------------------
// A thread owns one output pixel, or four consecutive ones of a row, for a group of images: the grid is
// shared by all images, so the source taps and weights are computed once and applied to each image
// (torch's grid_sampler_2d arithmetic in float32, as its compiler contracts it, rounded once to fp16).
// KIND 0 reads fp16 images, KIND 1 gathers uint8 slices through the u / 255 fp16 table.
constexpr int GIMG = 8;

// the source plane of image n (a slice index outside 0 .. SK-1 is clamped into it, so every read stays
// inside the volume)
template <int KIND>
DEV int64_t grid_plane(const D8sGridArgs& a, int n) {
    const int HW = a.H * a.W;
    if constexpr (KIND == 1) {
        const int b = n / a.M, m = n - b * a.M;
        int64_t si = ((const int64_t*)a.slice_idx)[m];
        si = si < 0 ? 0 : si >= a.SK ? (int64_t)a.SK - 1 : si;
        return ((int64_t)b * a.SK + si) * HW;
    } else {
        return (int64_t)n * HW;
    }
}

// Streaming stores: the output is not read back here, and kept out of the caches it leaves them to the
// source rows the neighbouring blocks share (88 x 3 windows of 512 x 512: 100 -> 83 us).
DEV void nt_store64(void* p, uint32_t lo, uint32_t hi) {
    __builtin_nontemporal_store((uint64_t)lo | (uint64_t)hi << 32, (uint64_t*)p);
}

// The fp16 bits of a float32 sum, which is opaque here: a conversion that the compiler sees behind an fma becomes
// one v_fma_mixlo_f16, which rounds once where the sum is to be rounded to float32 first.
DEV uint32_t half_bits(float x) {
    asm("" : "+v"(x));
    return (uint32_t)__half_as_ushort(__float2half_rn(x));
}

// Taps (nw, ne, sw, se), weights and which taps lie inside the image, of one output pixel.
struct Tap {
    int x0, y0;
    float w[4];
    bool ok[4];
};

DEV Tap grid_tap(const D8sGridArgs& a, uint32_t gbits) {
    Tap t;
    const __half2 g = __builtin_bit_cast(__half2, gbits);
    const float gx = __low2float(g), gy = __high2float(g);
    const float ix = __builtin_fmaf(gx + 1.0f, (float)a.W, -1.0f) * 0.5f;
    const float iy = __builtin_fmaf(gy + 1.0f, (float)a.H, -1.0f) * 0.5f;
    t.x0 = (int)floorf(ix);
    t.y0 = (int)floorf(iy);
    // (an infinite coordinate saturates: + 1 and the range checks are unsigned, so it wraps to outside.  Signed,
    // the compiler takes x1 >= 0 as x0 > -2, and the tap at INT_MAX + 1 counted as inside)
    const int x1 = (int)((uint32_t)t.x0 + 1u), y1 = (int)((uint32_t)t.y0 + 1u);
    t.w[0] = ((float)x1 - ix) * ((float)y1 - iy);
    t.w[1] = (ix - (float)t.x0) * ((float)y1 - iy);
    t.w[2] = ((float)x1 - ix) * (iy - (float)t.y0);
    t.w[3] = (ix - (float)t.x0) * (iy - (float)t.y0);
    const bool vx0 = (uint32_t)t.x0 < (uint32_t)a.W, vx1 = (uint32_t)x1 < (uint32_t)a.W;
    const bool vy0 = (uint32_t)t.y0 < (uint32_t)a.H, vy1 = (uint32_t)y1 < (uint32_t)a.H;
    t.ok[0] = vy0 && vx0;
    t.ok[1] = vy0 && vx1;
    t.ok[2] = vy1 && vx0;
    t.ok[3] = vy1 && vx1;
    return t;
}

// One pixel of NI images: every gather of every image issued before the first is used (taps outside the
// image read the plane's first pixel and are not added).  lut(u): the float32 value of byte u.
template <int KIND, int NI, class L>
DEV void grid_pixel(const D8sGridArgs& a, const Tap& t, const int64_t (&pl)[NI], float (&acc)[NI], L&& lut) {
    const int off[4] = {t.ok[0] ? t.y0 * a.W + t.x0 : 0, t.ok[1] ? t.y0 * a.W + t.x0 + 1 : 0,
                        t.ok[2] ? (t.y0 + 1) * a.W + t.x0 : 0, t.ok[3] ? (t.y0 + 1) * a.W + t.x0 + 1 : 0};
    uint16_t v[NI][4];
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            if constexpr (KIND == 1)
                v[i][k] = ((const uint8_t*)a.src)[pl[i] + off[k]];
            else
                v[i][k] = ((const uint16_t*)a.src)[pl[i] + off[k]];
        }
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        acc[i] = 0.0f;
#pragma unroll
        for (int k = 0; k < 4; ++k)
            if (t.ok[k]) acc[i] = __builtin_fmaf(KIND == 1 ? lut(v[i][k]) : __half2float(__ushort_as_half(v[i][k])), t.w[k], acc[i]);
    }
}

template <int KIND>
__global__ void __launch_bounds__(NT) k_grid_sample(D8sGridArgs a) {
    __shared__ uint16_t s_lut[256];
    if constexpr (KIND == 1) {
        s_lut[threadIdx.x] = ((const uint16_t*)a.lut)[threadIdx.x];
        __syncthreads();
    }
    const int HW = a.H * a.W;
    const int p = blockIdx.x * NT + threadIdx.x;
    const int n0 = blockIdx.y * GIMG, n1 = min(n0 + GIMG, a.N);
    if (p >= HW) return;
    int64_t pl[GIMG];
#pragma unroll
    for (int i = 0; i < GIMG; ++i) pl[i] = grid_plane<KIND>(a, min(n0 + i, n1 - 1));
    const Tap t = grid_tap(a, ((const uint32_t*)a.grid)[p]);
    float acc[GIMG];
    grid_pixel<KIND, GIMG>(a, t, pl, acc, [&](uint32_t u) { return __half2float(__ushort_as_half(s_lut[u])); });
#pragma unroll
    for (int i = 0; i < GIMG; ++i)
        if (n0 + i < n1) ((uint16_t*)a.out)[(int64_t)(n0 + i) * HW + p] = (uint16_t)half_bits(acc[i]);
}

// The gather alone (no grid): out = lut[slice], 8 consecutive pixels of a plane per thread (the last of a
// plane that is no multiple of 8 takes its pixels singly).  Planes of any size and address: the loads and
// stores are 8 bytes at byte (2-byte) alignment, which the hardware takes.  The table in 16 copies, a
// lane's by its index, keeps random bytes off one bank; 88 x 3 windows of 512 x 512: 131 -> 57 us (a byte
// and a 2-byte store a thread and image before), of 449 x 449 115 -> 62.
struct __attribute__((packed)) u64_any { uint64_t v; };
__global__ void __launch_bounds__(NT) k_grid_gather(D8sGridArgs a) {
    constexpr int GC = 16;
    __shared__ __attribute__((aligned(16))) uint32_t s_lut[256 * GC];
    {
        const uint32_t x = ((const uint16_t*)a.lut)[threadIdx.x];
#pragma unroll
        for (int c = 0; c < GC; c += 4) *(uint4*)&s_lut[threadIdx.x * GC + c] = make_uint4(x, x, x, x);
    }
    __syncthreads();
    const uint32_t lc = threadIdx.x % GC;
    const int HW = a.H * a.W;
    const int64_t p = 8 * ((int64_t)blockIdx.x * NT + threadIdx.x);
    const int n0 = blockIdx.y * GIMG, n1 = min(n0 + GIMG, a.N);
    if (p >= HW) return;
    const uint8_t* src = (const uint8_t*)a.src;
    if (p + 8 > HW) {
        for (int n = n0; n < n1; ++n) {
            const int64_t pl = grid_plane<1>(a, n);
            for (int64_t q = p; q < HW; ++q) ((uint16_t*)a.out)[(int64_t)n * HW + q] = (uint16_t)s_lut[src[pl + q] * GC + lc];
        }
        return;
    }
    int64_t pl[GIMG];
#pragma unroll
    for (int i = 0; i < GIMG; ++i) pl[i] = grid_plane<1>(a, min(n0 + i, n1 - 1));
    uint64_t v[GIMG];
#pragma unroll
    for (int i = 0; i < GIMG; ++i) v[i] = ((const u64_any*)(src + pl[i] + p))->v;
#pragma unroll
    for (int i = 0; i < GIMG; ++i) {
        if (n0 + i >= n1) break;
        uint16_t* out = (uint16_t*)a.out + (int64_t)(n0 + i) * HW + p;
        uint32_t o[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const uint32_t w = (uint32_t)(v[i] >> (16 * k));
            o[k] = s_lut[(w & 0xffu) * GC + lc] | (s_lut[((w >> 8) & 0xffu) * GC + lc] << 16);
        }
        if (((uintptr_t)out & 7) == 0) {
            nt_store64(out, o[0], o[1]);
            nt_store64(out + 4, o[2], o[3]);
        } else {
            ((u64_any*)out)->v = (uint64_t)o[0] | (uint64_t)o[1] << 32;
            ((u64_any*)(out + 4))->v = (uint64_t)o[2] | (uint64_t)o[3] << 32;
        }
    }
}

// Four consecutive output pixels of a row per thread (W a multiple of 4, the grid 16-byte aligned).  Where
// the four share their two source rows inside the image, their taps lie in a few columns of the two rows from
// the least left column on: two or three dwords (KIND 0: four or five) per row and image, each column converted
// once, a pixel's two picked by selects.  By o_k, pixel k's left column from the least:
//   NEAR  o_k in {k - 1, k}: zooms in up to about 1.6, shifts; 5 columns, a select a row and pixel;
//   IN    any o_k up to 3: further zooms in, mirrored images; 5 columns, three selects;
//   OUT   o_k in {k, k + 1}: zooms out to about 0.75; 6 columns, one select;
//   FAR   o_k in k .. 2 k: zooms out to 0.5; 8 columns, k selects.
// Pixels whose taps all lie outside the image store zeros; the others (borders, further zooms out, rotations)
// take the one-pixel kernel's taps, for fp16 images a lane per pixel where more than 8 lanes of a wave need it.
// A wave all NEAR decides nothing else; the lanes of any other take one form together where one fits.
// Per pixel the values, weights and fma order are the one-pixel kernel's, so the outputs are identical.
// What bounds the uint8 form is the table in LDS: ten to sixteen lookups of random entries a thread and image
// (sixteen through one table: about four lanes on one bank each), in a table of NC float32 copies, a lane's
// copy by its index; streaming stores leave the caches to the source.  88 x 3 windows, us by scale, this
// kernel and (in brackets) a single window rule of 8 aligned bytes for uint8, a pixel a thread for fp16:
//   uint8 512 px  0.5 92 (82)  0.7 109 (156)  0.9 108 (143)  1.1 52 (61)  1.8 65 (60)  2.5 65 (59)  -1.1 67 (60)
//   uint8 288 px  0.5 42 (34)  0.7 43 (66)    0.9 41 (55)    1.1 20 (27)  1.8 26 (27)  2.5 26 (27)  -1.1 27 (27)
//   fp16  288 px  0.4 35 (26)  0.5 31 (29)  0.7 38 (36)  0.9 29 (42)  1.1 16 (29)  2.5 19 (25)  -1.1 21 (29)
// The grid's x blocks are renumbered so that each XCD's share is consecutive rows (neighbouring blocks read the
// same source rows: one L2).
constexpr int NC = 16;
template <int KIND>
constexpr int G4IMG = KIND == 1 ? 4 : 8;     // images per thread
enum { NEAR, OUT, IN, FAR };
// pixel k's least left column, and how many further ones it may take
constexpr int lo_of(int mode, int k) { return mode == NEAR ? (k ? k - 1 : 0) : mode == IN ? 0 : k; }
constexpr int steps_of(int mode, int k) { return mode == IN ? 3 : mode == FAR ? k : k ? 1 : 0; }

template <int KIND>
__global__ void __launch_bounds__(NT, KIND == 1 ? 7 : 4) k_grid_sample4(D8sGridArgs a, int n_first) {
    constexpr int NI = G4IMG<KIND>;
    __shared__ __attribute__((aligned(16))) float s_lut[KIND == 1 ? 256 * NC : 4];
    if constexpr (KIND == 1) {
        const float x = __half2float(__ushort_as_half(((const uint16_t*)a.lut)[threadIdx.x]));
#pragma unroll
        for (int c = 0; c < NC; c += 4) *(float4*)&s_lut[threadIdx.x * NC + c] = make_float4(x, x, x, x);
        __syncthreads();
    }
    const int HW = a.H * a.W;
    const int per = (int)gridDim.x / 8;                       // (gridDim.x is a multiple of 8)
    // (at most 2^31 - 4: H * W < 2^31 makes at most 2^21 blocks, itself a multiple of 8)
    const int p0 = 4 * ((((int)blockIdx.x % 8) * per + (int)blockIdx.x / 8) * NT + (int)threadIdx.x);
    const int n0 = n_first + (int)blockIdx.y * NI, n1 = min(n0 + NI, a.N);
    if (p0 >= HW) return;
    int64_t pl[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) pl[i] = grid_plane<KIND>(a, min(n0 + i, n1 - 1));
    const uint4 gq = ((const uint4*)a.grid)[p0 >> 2];         // 4 pixels x (gx, gy) fp16
    const Tap t[4] = {grid_tap(a, gq.x), grid_tap(a, gq.y), grid_tap(a, gq.z), grid_tap(a, gq.w)};
    const uint32_t lane_off = (threadIdx.x % NC) * 4;
    auto lut = [&](uint32_t at) {                             // at = 4 NC u
        return *(const float*)((const char*)s_lut + (at | lane_off));
    };
    const int y0 = t[0].y0, x0 = t[0].x0;
    constexpr int AL = KIND == 1 ? 4 : 2;                     // pixels per dword
    const bool same = t[1].y0 == y0 && t[2].y0 == y0 && t[3].y0 == y0 && y0 >= 0 && y0 < a.H - 1;
    // what a lane's taps allow: near (here), in / out / far / none (further down)
    bool near = same && x0 >= 0 && (x0 & ~(AL - 1)) <= a.W - 8;
#pragma unroll
    for (int k = 1; k < 4; ++k) near &= (uint32_t)k - ((uint32_t)t[k].x0 - (uint32_t)x0) <= 1u;
    float acc[NI][4];
    // x: the least of the four left columns
    auto fast = [&](auto mode, int x) __attribute__((always_inline)) {
        constexpr int MODE = decltype(mode)::value, COLS = MODE == FAR ? 8 : MODE == OUT ? 6 : 5;
        constexpr int DW = KIND == 0 ? (COLS + 3) / 2 : COLS == 5 ? 2 : 3;
        constexpr int CI = KIND == 0 && MODE == FAR ? NI / 2 : NI;   // images whose dwords are in registers together
        const int r0 = y0 * a.W + (x & ~(AL - 1));
        const uint32_t sft = (uint32_t)(x & (AL - 1)) * (KIND == 1 ? 8 : 16);
        // pixel k's left column is LO + (how many of is[k][] hold)
        constexpr int STEPS = MODE == IN || MODE == FAR ? 3 : 1;
        bool is[4][STEPS];
#pragma unroll
        for (int k = 0; k < 4; ++k)
#pragma unroll
            for (int e = 0; e < STEPS; ++e) is[k][e] = t[k].x0 - x > lo_of(MODE, k) + e;
#pragma unroll
        for (int i0 = 0; i0 < NI; i0 += CI) {
            uint32_t d[CI][2][DW];
#pragma unroll
            for (int i = 0; i < CI; ++i)
#pragma unroll
                for (int r = 0; r < 2; ++r) {
                    const uint32_t* q = (const uint32_t*)((const uint8_t*)a.src + (KIND == 1 ? 1 : 2) * (pl[i0 + i] + r0 + r * a.W));
#pragma unroll
                    for (int w = 0; w < DW; ++w) d[i][r][w] = q[w];
                }
#pragma unroll
            for (int i = 0; i < CI; ++i) {
                float c[2][COLS + (COLS & 1)];
#pragma unroll
                for (int r = 0; r < 2; ++r) {
                    if constexpr (KIND == 1) {
                        const uint32_t lo = __builtin_amdgcn_alignbit(d[i][r][1], d[i][r][0], sft);
                        const uint32_t hi = __builtin_amdgcn_alignbit(d[i][r][DW - 1], d[i][r][1], sft);
                        constexpr uint32_t M = 255u * 4 * NC;
                        static_assert(NC == 16, "byte u at bit 6: 4 NC u");
                        c[r][0] = lut((lo << 6) & M);
                        c[r][1] = lut((lo >> 2) & M);
                        c[r][2] = lut((lo >> 10) & M);
                        c[r][3] = lut((lo >> 18) & M);
                        c[r][4] = lut((hi << 6) & M);
                        if constexpr (COLS > 5) c[r][5] = lut((hi >> 2) & M);
                        if constexpr (COLS > 6) c[r][6] = lut((hi >> 10) & M);
                        if constexpr (COLS > 6) c[r][7] = lut((hi >> 18) & M);
                    } else {
#pragma unroll
                        for (int w = 0; w < DW - 1; ++w) {
                            const __half2 v = __builtin_bit_cast(__half2, __builtin_amdgcn_alignbit(d[i][r][w + 1], d[i][r][w], sft));
                            c[r][2 * w] = __low2float(v);
                            if (2 * w + 1 < COLS) c[r][2 * w + 1] = __high2float(v);
                        }
                    }
                }
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    float s = 0.0f;
#pragma unroll
                    for (int r = 0; r < 2; ++r) {
                        const int lo = lo_of(MODE, k);
                        float l = c[r][lo], h = c[r][lo + 1];
#pragma unroll
                        for (int e = 0; e < steps_of(MODE, k); ++e) {
                            l = is[k][e] ? c[r][lo + e + 1] : l;
                            h = is[k][e] ? c[r][lo + e + 2] : h;
                        }
                        s = __builtin_fmaf(l, t[k].w[2 * r], s);
                        s = __builtin_fmaf(h, t[k].w[2 * r + 1], s);
                    }
                    acc[i0 + i][k] = s;
                }
            }
        }
    };
    // (an image past the last is the last again: a store under a branch would take its loads there with it)
    auto store = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const uint32_t lo = half_bits(acc[i][0]) | half_bits(acc[i][1]) << 16;
            const uint32_t hi = half_bits(acc[i][2]) | half_bits(acc[i][3]) << 16;
            nt_store64((uint16_t*)a.out + (int64_t)min(n0 + i, n1 - 1) * HW + p0, lo, hi);
        }
    };
    if (__all(near)) {
        fast(std::integral_constant<int, NEAR>{}, x0);
        store();
        return;
    }
    const int xmin = min(min(x0, t[1].x0), min(t[2].x0, t[3].x0)), xmax = max(max(x0, t[1].x0), max(t[2].x0, t[3].x0));
    const int base = xmin & ~(AL - 1);
    const bool rows = same && xmin >= 0 && base <= a.W - 8;
    bool in = rows && (uint32_t)xmax - (uint32_t)xmin <= 3u, out = rows, far = rows, none = true;
    {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const uint32_t o = (uint32_t)t[k].x0 - (uint32_t)xmin;
            out &= o == (uint32_t)k || (k > 0 && o == (uint32_t)k + 1u);
            far &= o >= (uint32_t)k && o <= 2u * k;
#pragma unroll
            for (int q = 0; q < 4; ++q) none &= !t[k].ok[q];
        }
        // (a zoom out's columns may reach into a further dword)
        out &= KIND == 0 || base <= a.W - 12;
        far &= base <= a.W - (KIND == 1 ? 12 : 10);
        if constexpr (KIND == 0) {
            const bool slow = !(in || out || far || none);
            if (__popcll(__ballot(slow)) > 8 && __ballot(true) == ~0ull) {
                // much of the wave has taps that lie nowhere together: a lane per pixel, 64 neighbours at a time
                const int pw = p0 - 3 * (int)__lane_id();
#pragma unroll 2
                for (int s = 0; s < 256; s += 64) {
                    const Tap ts = grid_tap(a, ((const uint32_t*)a.grid)[pw + s]);
                    float v[NI];
                    grid_pixel<KIND, NI>(a, ts, pl, v, lut);
#pragma unroll
                    for (int i = 0; i < NI; ++i)
                        ((uint16_t*)a.out)[(int64_t)min(n0 + i, n1 - 1) * HW + pw + s] = (uint16_t)half_bits(v[i]);
                }
                return;
            }
        }
        // one form for the wave's lanes where one will do (a lane's neighbours often need the wider form)
    }
    const bool use_in = __any(in && !near && !out), use_out = __any(out && !near), use_far = __any(far && !out && !in);
    if (use_far && far) {
        fast(std::integral_constant<int, FAR>{}, xmin);
    } else if (use_out && out) {
        fast(std::integral_constant<int, OUT>{}, xmin);
    } else if (use_in && in) {
        fast(std::integral_constant<int, IN>{}, xmin);
    } else if (near) {
        fast(std::integral_constant<int, NEAR>{}, x0);
    } else if (none) {
#pragma unroll
        for (int i = 0; i < NI; ++i)
#pragma unroll
            for (int k = 0; k < 4; ++k) acc[i][k] = 0.0f;
    } else {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            float v[NI];
            grid_pixel<KIND, NI>(a, t[k], pl, v, [&](uint32_t u) { return lut(u * 4 * NC); });
#pragma unroll
            for (int i = 0; i < NI; ++i) acc[i][k] = v[i];
        }
    }
    store();
}

// ---- host side ----------------------------------------------------------------------------------
#define PREQ(cond, msg) \
    do { if (!(cond)) return d8s_host_fail((int)hipErrorInvalidValue, std::string(what) + ": " + (msg)); } while (0)

// The workgroup ranges of every stack in the grids of regions and of the final pass (4 blocks per workgroup;
// the float32 levels' are wide_view's); returns the size of the per-block grid.
int assign_grids(PArgs& a) {
    int wh = 0, wn = 0;
    for (int i = 0; i < a.n; ++i) {
        PStack& p = a.s[i];
        p.hb = p.nb = 4;
        p.wg_hist = wh;
        p.wg_norm = wn;
        wh += (p.nblk + p.hb - 1) / p.hb;
        wn += (p.nblk + p.nb - 1) / p.nb;
    }
    return wn;
}

// The float32 view of a kind-0 call after the first pass: every stack reads its resized slices from
// the scratch buffer (M_FLOAT), in blocks of about 4096 pixels.
PArgs float_view(const PArgs& a) {
    PArgs f = a;
    const int rb = a.img >= 4096 ? 1 : 4096 / a.img;
    for (int i = 0; i < f.n; ++i) {
        PStack& p = f.s[i];
        p.src = p.sc;
        p.resc = nullptr;
        p.mode = M_FLOAT;
        p.rb = rb;
        p.bps = (a.img + rb - 1) / rb;
        p.nblk = (p.k1 - p.k0) * p.bps;
    }
    assign_grids(f);
    return f;
}

// The view the wide workgroups read: float32 stacks in blocks of about 16384 pixels (four 16-byte loads a
// thread of a wide workgroup), as many blocks a workgroup as make a grid of about four workgroups per CU, two
// of them resident at a time (a study's level 3 takes 38 us so, 44 with a grid of two per CU).
PArgs wide_view(const PArgs& a) {
    PArgs f = a;
    const int rb = a.img >= 16384 ? 1 : 16384 / a.img;
    int64_t blocks = 0;
    for (int i = 0; i < f.n; ++i) {
        PStack& p = f.s[i];
        p.rb = rb;
        p.bps = (a.img + rb - 1) / rb;
        p.nblk = (p.k1 - p.k0) * p.bps;
        blocks += p.nblk;
    }
    const int per = (int)std::max<int64_t>(1, blocks / (4 * d8s_host_cu_count()));
    int wg = 0;
    for (int i = 0; i < f.n; ++i) {
        PStack& p = f.s[i];
        p.hb2 = per;
        p.wg_hist2 = wg;
        wg += (p.nblk + per - 1) / per;
    }
    return f;
}

int prepare(const D8sPrepArgs* in, const char* what, bool resize_only, PArgs& a, int& setup_blocks) {
    PREQ(in != nullptr, "null arguments");
    PREQ(in->kind == 0 || in->kind == 1, "kind must be 0 (uint16 regions) or 1 (float32 stacks)");
    PREQ(!resize_only || in->kind == 0, "kind 1 has nothing to resize");
    PREQ(in->n_stacks >= 1 && in->n_stacks <= MAX_S, "n_stacks must be 1 .. 16");
    PREQ(in->img >= 8 && in->img <= 4096 && in->img % 8 == 0, "img must be a multiple of 8 in 8 .. 4096");
    PREQ(in->workspace != 0 && in->workspace % 256 == 0, "workspace null or not 256-byte aligned");
    uint64_t need = 0;
    d8s_prep_workspace(in->n_stacks, in->img, &need);
    PREQ(in->ws_bytes >= need, "workspace smaller than d8s_prep_workspace()");
    const int img = in->img;
    if (in->kind == 0 && !resize_only) {
        uint64_t sc = 0;
        for (int i = 0; i < in->n_stacks; ++i) {
            const int64_t sl = (int64_t)in->s[i].k1 - in->s[i].k0;
            sc += 4ull * (uint64_t)(sl > 0 ? sl : 0) * img * img;
        }
        PREQ(in->scratch != 0 && in->scratch % 16 == 0, "scratch null or not 16-byte aligned");
        PREQ(in->scratch_bytes >= sc, "scratch smaller than 4 * sum(k1 - k0) * img * img bytes");
    }
    a = PArgs{};
    a.n = in->n_stacks;
    a.img = img;
    a.upr = img / UP;
    a.stat = (D8sPrepStat*)in->workspace;
    a.inv_img = 1.0f / (float)img;
    a.inv_upr = 1.0f / (float)a.upr;
    PREQ(in->kind == 1 || img <= 1024, "img above 1024 is supported for float32 stacks (kind 1) only");
    const int rb_want = 4096 / img > 1 ? 4096 / img : 1;     // about 4096 output pixels per block
    int64_t sc_off = 0;
    for (int i = 0; i < a.n; ++i) {
        const D8sPrepStack& s = in->s[i];
        PStack& p = a.s[i];
        const std::string at = "stack " + std::to_string(i) + ": ";
        PREQ(s.src != 0 && s.out != 0, at + "null src or out");
        PREQ(s.K >= 1 && s.k0 >= 0 && s.k0 < s.k1 && s.k1 <= s.K, at + "slice range outside 0 .. K");
        const int64_t n = (int64_t)(s.k1 - s.k0) * img * img;
        PREQ((int64_t)s.K * img * img < (1ll << 31), at + "more than 2^31 - 1 pixels");
        if (!resize_only) {
            PREQ(n >= 4, at + "fewer than 4 pixels");
            PREQ(s.r1 >= 0 && (int64_t)s.r1 + 1 < n && s.r2 >= 0 && (int64_t)s.r2 + 1 < n,
                 at + "ranks outside the stack");
            PREQ(s.g1 >= 0.0 && s.g1 < 1.0 && s.g2 >= 0.0 && s.g2 < 1.0, at + "gamma outside [0, 1)");
            PREQ(s.flip >= 0 && s.flip <= 2, at + "flip must be 0, 1 or 2");
            PREQ(s.out % 8 == 0, at + "uint8 output not 8-byte aligned");
        } else {
            PREQ(s.out % 16 == 0, at + "float32 output not 16-byte aligned");
        }
        p.src = (const void*)s.src;
        p.out = (void*)s.out;
        p.resc = in->kind == 0 ? (const float*)s.resc : nullptr;
        p.ws = (uint32_t*)(in->workspace + WS_HEAD) + (uint64_t)i * stack_words(img);
        if (in->kind == 0 && !resize_only) {
            // compact: the slices [k0, k1) of the stacks back to back; sc is offset so that slice kk
            // is at sc + kk img img
            p.sc = (float*)in->scratch + (int64_t)sc_off - (int64_t)s.k0 * img * img;
            sc_off += (int64_t)(s.k1 - s.k0) * img * img;
        }
        p.K = s.K;
        p.k0 = s.k0;
        p.k1 = s.k1;
        p.flip = resize_only ? 0 : s.flip;
        p.r1 = s.r1;
        p.r2 = s.r2;
        p.g1 = s.g1;
        p.g2 = s.g2;
        if (in->kind == 1) {
            PREQ(s.src % 16 == 0, at + "float32 input not 16-byte aligned");
            p.mode = M_FLOAT;
            p.rb = rb_want;
        } else {
            PREQ(s.hr >= 1 && s.wr >= 1, at + "empty region");
            PREQ(s.y0 >= 0 && s.y0 < s.y1 && s.y1 <= s.hr && s.x0 >= 0 && s.x0 < s.x1 && s.x1 <= s.wr,
                 at + "box outside the region");
            PREQ((int64_t)s.K * s.hr * s.wr < (1ll << 31) - 2, at + "region of 2^31 or more values");
            p.hr = s.hr;
            p.wr = s.wr;
            p.y0 = s.y0;
            p.x0 = s.x0;
            p.h = s.y1 - s.y0;
            p.w = s.x1 - s.x0;
            // LDS per block: ns_max resized rows of img floats + ns_max raw rows of rp dwords
            p.rp = (p.w + 2) / 2;
            p.inv_rp = 1.0f / (float)p.rp;
            p.dpl = (p.rp + 63) / 64;
            // the LDS holds ns_max rows of img floats and one or two buffers of ns_max rows of
            // dpl * 64 raw dwords: two when that still gives blocks of rb_want rows
            const double sc_h = p.h > img ? (double)p.h / img : 1.0;
            const int need = (int)ceil(rb_want * sc_h) + 2;
            p.dbuf = need * (img + 128 * p.dpl) <= STAGE ? 1 : 0;
            const int cap = STAGE / (img + (p.dbuf ? 128 : 64) * p.dpl);
            if (p.h == img && p.w == img) {
                p.mode = M_IDENT;
                PREQ(cap >= 1, at + "crop too wide for this img");
                p.rb = rb_want < cap ? rb_want : cap;
                p.ns_max = p.rb;
            } else if (p.h > img) {
                p.mode = M_AREA;
                p.Tx = p.w != img ? area_taps_max(p.w, img) : 0;
                p.Ty = area_taps_max(p.h, img);
                PREQ(p.Tx <= MAX_T && p.Ty <= MAX_T, at + "area table longer than 16 taps");
                // rb output rows read at most rb * h / img + 2 source rows
                const double scale = (double)p.h / img;
                PREQ(scale + 2.0 <= cap, at + "area downscale factor too large for this img and width");
                const int fit = (int)((cap - 2) / scale);
                p.rb = rb_want < fit ? rb_want : fit;
                p.ns_max = (int)ceil(p.rb * scale) + 2;
            } else {
                p.mode = M_BILIN;
                p.rh = (float)p.h / (float)img;
                p.rw = (float)p.w / (float)img;
                PREQ(cap >= 2, at + "crop too wide for this img");
                p.rb = rb_want < cap - 1 ? rb_want : cap - 1;   // rb + 1 source rows
                p.ns_max = p.rb + 1;
            }
        }
        p.bps = (img + p.rb - 1) / p.rb;
        p.nblk = (s.k1 - s.k0) * p.bps;
    }
    int outside = 0;
    for (int i = 0; i < a.n; ++i) {
        const PStack& p = a.s[i];
        const int o = (p.K - (p.k1 - p.k0)) * (img * img / 8);
        outside = o > outside ? o : outside;
    }
    const int wn = assign_grids(a);
    PREQ(wn < (1 << 30), "too many workgroups");
    int sb = (img + NT - 1) / NT;
    const int sc = (W_CLEAR + NT * 4 - 1) / (NT * 4), so = (outside + NT * 4 - 1) / (NT * 4);
    sb = sb > sc ? sb : sc;
    sb = sb > so ? sb : so;
    setup_blocks = sb < 1024 ? sb : 1024;
    return 0;
}

int grid_of(const PArgs& a, int grid) {
    const PStack& l = a.s[a.n - 1];
    return grid == 0 ? l.wg_hist + (l.nblk + l.hb - 1) / l.hb
         : grid == 1 ? l.wg_hist2 + (l.nblk + l.hb2 - 1) / l.hb2
                     : l.wg_norm + (l.nblk + l.nb - 1) / l.nb;
}

}  // namespace

extern "C" int d8s_prep_workspace(int32_t n_stacks, int32_t img, uint64_t* bytes) {
    const char* what = "d8s_prep_workspace";
    PREQ(bytes != nullptr, "null output");
    PREQ(n_stacks >= 1 && n_stacks <= MAX_S, "n_stacks must be 1 .. 16");
    PREQ(img >= 8 && img <= 4096 && img % 8 == 0, "img must be a multiple of 8 in 8 .. 4096");
    *bytes = WS_HEAD + 4ull * stack_words(img) * (uint64_t)n_stacks;
    return 0;
}

extern "C" int d8s_prep(const D8sPrepArgs* in, void* stream) {
    PArgs a;
    int sb = 0;
    if (const int rc = prepare(in, "d8s_prep", false, a, sb)) return rc;
    hipStream_t st = (hipStream_t)stream;
    const dim3 gs(sb, a.n);
    k_prep_setup<<<gs, NT, 0, st>>>(a, 1);
    // kind 0: the resize once (with the level-1 count) into the scratch stacks, then the float32 passes
    const PArgs f = in->kind == 0 ? float_view(a) : a, w = wide_view(f);
    const int gw = grid_of(w, 1), gn = grid_of(f, 2);
    if (in->kind == 0)
        k_prep_hist<1, 1, true><<<grid_of(a, 0), NT, 0, st>>>(a);
    else
        k_prep_hist<1, 0><<<gw, WIDE, 0, st>>>(w);
    k_prep_select<1><<<a.n, NT, 0, st>>>(a);
    k_prep_hist<2, 0><<<gw, WIDE, 0, st>>>(w);
    k_prep_select<2><<<a.n, NT, 0, st>>>(a);
    k_prep_hist<3, 0><<<gw, WIDE, 0, st>>>(w);
    k_prep_select<3><<<a.n, NT, 0, st>>>(a);
    k_prep_norm<0><<<gn, NT, 0, st>>>(f);
    return d8s_host_launched("d8s_prep");
}

extern "C" int d8s_prep_resize(const D8sPrepArgs* in, void* stream) {
    PArgs a;
    int sb = 0;
    if (const int rc = prepare(in, "d8s_prep_resize", true, a, sb)) return rc;
    hipStream_t st = (hipStream_t)stream;
    k_prep_setup<<<dim3(sb, a.n), NT, 0, st>>>(a, 0);
    k_prep_resize<<<grid_of(a, 2), NT, 0, st>>>(a);
    return d8s_host_launched("d8s_prep_resize");
}

extern "C" int d8s_grid_sample(const D8sGridArgs* a, void* stream) {
    const char* what = "d8s_grid_sample";
    PREQ(a != nullptr, "null arguments");
    PREQ(a->kind == 0 || a->kind == 1, "kind must be 0 (fp16 images) or 1 (uint8 volume gather)");
    PREQ(a->src && a->out && (a->grid || a->kind == 1), "null pointer");
    PREQ(a->H >= 1 && a->W >= 1 && (int64_t)a->H * a->W < (1ll << 31), "bad image size");
    PREQ(a->grid % 4 == 0, "grid not 4-byte aligned");
    if (a->kind == 1) {
        PREQ(a->slice_idx && a->lut, "null slice_idx or lut");
        PREQ(a->B >= 1 && a->M >= 1 && a->SK >= 1, "bad B, M or SK");
        PREQ((int64_t)a->B * a->M == a->N, "N must be B * M");
    }
    PREQ(a->N >= 1 && a->N < 65536 * GIMG, "N must be 1 .. 524287");
    const int64_t HW = (int64_t)a->H * a->W;
    const dim3 grid((unsigned)((HW + NT - 1) / NT), (unsigned)((a->N + GIMG - 1) / GIMG));
    hipStream_t st = (hipStream_t)stream;
    if (a->grid == 0) {
        k_grid_gather<<<dim3((unsigned)((HW + 8 * NT - 1) / (8 * NT)), grid.y), NT, 0, st>>>(*a);
    } else if (a->W % 4 == 0 && a->grid % 16 == 0 && a->out % 8 == 0 && a->src % 4 == 0) {
        // four pixels a thread: rows of whole dwords (uint8 and fp16 alike), the grid's and output's quads
        // aligned
        const unsigned gx = (unsigned)((HW / 4 + NT - 1) / NT + 7) / 8 * 8;
        // (a grid has at most 65535 y blocks: more images take further launches)
        const int ni = a->kind == 1 ? G4IMG<1> : G4IMG<0>;
        for (int n0 = 0; n0 < a->N; n0 += 65535 * ni) {
            const dim3 g4(gx, (unsigned)std::min(65535, (a->N - n0 + ni - 1) / ni));
            if (a->kind == 1)
                k_grid_sample4<1><<<g4, NT, 0, st>>>(*a, n0);
            else
                k_grid_sample4<0><<<g4, NT, 0, st>>>(*a, n0);
        }
    } else if (a->kind == 1) {
        k_grid_sample<1><<<grid, NT, 0, st>>>(*a);
    } else {
        k_grid_sample<0><<<grid, NT, 0, st>>>(*a);
    }
    return d8s_host_launched("d8s_grid_sample");
}

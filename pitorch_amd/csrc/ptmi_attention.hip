// Causal attention over many positions at once, forward and backward, on
// v_mfma_f32_16x16x4_f32: the training step's attention (pt_train.c:224-255
// forward, :780-811 backward) and the prompt's in ptmi_model_generate.
//
// One block holds a tile of 16*QT rows of one head; its waves take the other
// side's 16-position blocks in turn (wave w: blocks w, w + NW, ...), each
// with sums of its own, and meet once, through LDS, at the end: no barrier
// and no LDS in the loop.  Every score tile is computed transposed to what
// its consumer contracts over, so the result registers of one product are
// the operand registers of the next:
//   lane l supplies A[l%16][l/16] and B[l/16][l%16]; result register r of
//   lane l is C[4*(l/16)+r][l%16].  A contraction may take its index in any
//   order that A and B share, so step s over a 16-position block takes
//   position 4*(l/16) + s, which is result register s.
// With S^T = K.Q^T a lane's four results are keys 4g..4g+3 of query l%16:
// the softmax statistics of a query are lane-local but for two cross-lane
// moves, and O^T += V^T.P^T takes P^T from those registers.
//
// The scores are recomputed in the backward from the forward's row maximum
// and 1/sum (the reference's P = e^(s - max) * (1/sum)), so no T x T array
// is written or read: with P and dS in memory a layer of 12 heads x 1024
// positions moves 250 MB, 40 us by itself.
// Blocks of the same rows of all heads are neighbours in the grid and the
// rows with the most work come first, so the long blocks start together and
// the short ones fill in (head by head, as (tile, head): 55, 82 and 100 us).
// 12 heads x 1024 positions x 64 (us; one block per row and head on the
// vector units before): forward 136 -> 33, row half 140 -> 47, column half
// 172 -> 52.  Bound by the latency of a wave's own products, exps and loads
// (the fp32 matrix units alone would need 11, 16 and 21 us); four waves per
// block instead of eight: 44, 61 and 67 us.
#include "ptmi_model.h"

#include <cmath>

namespace ptmi {

namespace {

typedef float f4v __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f4v mfma4(float a, float b, f4v c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// e^x for arguments that a row maximum was subtracted from (at most a
// rounding above 0), without branches: 2^n * Taylor(r) to r^7, |r| <= ln2/2,
// n*ln2 taken off in two parts.  d_expf stops at r^5 (2.4e-6 off); here
// running sums are rescaled by further factors of it, which would add up.
// As there, arguments below -87.3 give 0; NaN stays NaN.
__device__ __forceinline__ float exp_le0(float x) {
    const float n = __builtin_rintf(x * 1.4426950408889634f);
    const float r = fmaf(-n, -1.9046542e-9f, fmaf(-n, 0.69314718246459961f, x));
    float p = fmaf(r, 1.9841270e-4f, 1.3888889e-3f);
    p = fmaf(r, p, 8.3333333e-3f);
    p = fmaf(r, p, 4.1666667e-2f);
    p = fmaf(r, p, 1.6666667e-1f);
    p = fmaf(r, p, 0.5f);
    p = fmaf(r, p, 1.0f);
    p = fmaf(r, p, 1.0f);
    p = ldexpf(p, (int)n);
    return x < -87.3f ? 0.0f : p;
}

// The rows' float4s [g*HQ, (g+1)*HQ) of a head row at p (head_dim = 4*n4
// floats; PAD: slots past it are zero).  Lane group g = lane/16 holds one
// quarter of the contraction over head_dim.
template <int HQ, bool PAD>
__device__ __forceinline__ void load_row(float4 (&r)[HQ], const float *p, int g, int n4) {
    const float4 *p4 = reinterpret_cast<const float4 *>(p);
#pragma unroll
    for (int q = 0; q < HQ; q++) {
        const int i = g * HQ + q;
        if constexpr (PAD) {
            const float4 x = p4[min(i, n4 - 1)];
            const bool in = i < n4;
            r[q] = make_float4(in ? x.x : 0.f, in ? x.y : 0.f, in ? x.z : 0.f, in ? x.w : 0.f);
        } else {
            r[q] = p4[i];
        }
    }
}

// Rows t0 + 4g + s (clamped to `last`), columns 16*cb + li (clamped to the
// head: results past it are never stored).
template <int HQ, bool PAD>
__device__ __forceinline__ void load_cols(float (&v)[4][HQ], const float *p, long ld, int t0, int last, int g, int li,
                                          int hd) {
#pragma unroll
    for (int s = 0; s < 4; s++) {
        const float *row = p + (long)min(t0 + 4 * g + s, last) * ld;
#pragma unroll
        for (int cb = 0; cb < HQ; cb++) v[s][cb] = row[PAD ? min(cb * 16 + li, hd - 1) : cb * 16 + li];
    }
}

// Two sums side by side: half the chain of dependent products, and of roundings.
template <int HQ>
__device__ __forceinline__ f4v dots(const float4 (&a)[HQ], const float4 (&b)[HQ]) {
    f4v c = {0.f, 0.f, 0.f, 0.f}, d = c;
#pragma unroll
    for (int q = 0; q < HQ; q++) {
        c = mfma4(a[q].x, b[q].x, c);
        d = mfma4(a[q].y, b[q].y, d);
        c = mfma4(a[q].z, b[q].z, c);
        d = mfma4(a[q].w, b[q].w, d);
    }
    return c + d;
}

// acc[cb] (rows: columns 16*cb.. of v, columns: this tile's rows) += v^T . w
template <int HQ>
__device__ __forceinline__ void wsum(f4v (&acc)[HQ], const float (&v)[4][HQ], const float (&w)[4]) {
#pragma unroll
    for (int s = 0; s < 4; s++)
#pragma unroll
        for (int cb = 0; cb < HQ; cb++) acc[cb] = mfma4(v[s][cb], w[s], acc[cb]);
}

// The waves' 16-row tiles, summed in wave order: store this wave's (row li,
// columns 16*cb + 4g + r), then out(row, float4 index, sum) for every float4.
template <int HQ, int NW, typename F>
__device__ __forceinline__ void merge(const f4v (&acc)[HQ], float *red, int n4, F &&out) {
    constexpr int P = 16 * HQ + 4;                         // pitch in floats
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, li = lane & 15, g = lane >> 4;
    __syncthreads();                                       // earlier readers of red are done
#pragma unroll
    for (int cb = 0; cb < HQ; cb++)
        *reinterpret_cast<f4v *>(red + (wave * 16 + li) * P + cb * 16 + 4 * g) = acc[cb];
    __syncthreads();
    for (int e = threadIdx.x; e < 16 * n4; e += 64 * NW) {
        const int i = e / n4, c = e - i * n4;
        f4v v = *reinterpret_cast<const f4v *>(red + i * P + 4 * c);
#pragma unroll
        for (int w = 1; w < NW; w++) v += *reinterpret_cast<const f4v *>(red + (w * 16 + i) * P + 4 * c);
        out(i, c, v);
    }
}

// rope_backward (pt_backward_ops.c:52-69) of a float4 (two pairs) at
// columns 4*c4.. of a head, position t.
__device__ __forceinline__ f4v rope_bwd4(f4v v, int c4, int hd, int t) {
    float c, s;
    f4v o;
    d_rope_cs(4 * c4, hd, t, &c, &s);
    o.x = v.x * c + v.y * s;
    o.y = -v.x * s + v.y * c;
    d_rope_cs(4 * c4 + 2, hd, t, &c, &s);
    o.z = v.z * c + v.w * s;
    o.w = -v.z * s + v.w * c;
    return o;
}

__device__ __forceinline__ float xmax_groups(float v) {   // over lanes l, l^16, l^32, l^48
    LanePair p = pl16(v);
    v = fmaxf(p.lo, p.hi);
    p = pl32(v);
    return fmaxf(p.lo, p.hi);
}
__device__ __forceinline__ float xsum_groups(float v) { return xsum32(xsum16(v)); }

// Forward: query rows [16*QT*tile, ...) of head blockIdx.x, at positions
// pos0 + row, over keys 0..position.  The last rows (the most keys) go out
// first, so that short blocks fill in behind the long ones.
template <int HQ, int QT, int NW, bool PAD>
__global__ __launch_bounds__(64 * NW) void k_attn_rows_fwd(AttnFwdArgs a) {
    __shared__ __align__(16) float red[NW * 16 * (16 * HQ + 4)];
    __shared__ float st_m[NW][16 * QT], st_l[NW][16 * QT];
    const int h = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6, li = lane & 15, g = lane >> 4;
    const int hd = PAD ? a.head_dim : 16 * HQ, n4 = hd >> 2;
    const int r0 = (int)(gridDim.y - 1 - blockIdx.y) * 16 * QT;
    const int last = a.pos0 + min(r0 + 16 * QT, a.rows) - 1;   // the tile's last position: its last key
    const int nkb = last / 16 + 1;
    const float *q = a.q + h * hd, *k = a.k + h * hd, *v = a.v + h * hd;
    float4 qf[QT][HQ];
#pragma unroll
    for (int t = 0; t < QT; t++)
        load_row<HQ, PAD>(qf[t], q + (long)min(r0 + 16 * t + li, a.rows - 1) * a.ldq, g, n4);
    f4v acc[QT][HQ];
    float m[QT], l[QT];
#pragma unroll
    for (int t = 0; t < QT; t++) {
        m[t] = -INFINITY;
        l[t] = 0.0f;
#pragma unroll
        for (int cb = 0; cb < HQ; cb++) acc[t][cb] = f4v{0.f, 0.f, 0.f, 0.f};
    }
    float4 kf[HQ];
    float vt[4][HQ];
    if (wave < nkb) {                                       // wave-uniform
        load_row<HQ, PAD>(kf, k + (long)min(wave * 16 + li, last) * a.ldkv, g, n4);
        load_cols<HQ, PAD>(vt, v, a.ldkv, wave * 16, last, g, li, hd);
    }
    for (int kb = wave; kb < nkb; kb += NW) {
        // the next block's rows (the last block again at the end) are in flight during this one's products
        float4 kn[HQ];
        float vn[4][HQ];
        const int nx = min(kb + NW, nkb - 1) * 16;
        load_row<HQ, PAD>(kn, k + (long)min(nx + li, last) * a.ldkv, g, n4);
        load_cols<HQ, PAD>(vn, v, a.ldkv, nx, last, g, li, hd);
#pragma unroll
        for (int t = 0; t < QT; t++) {
            const f4v s = dots<HQ>(kf, qf[t]);
            const int pos = a.pos0 + r0 + 16 * t + li, key = kb * 16 + 4 * g;
            float p[4], bm = -INFINITY;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                p[r] = s[r] * a.scale;
                bm = key + r <= pos ? fmaxf(bm, p[r]) : bm;
            }
            const float mn = fmaxf(m[t], xmax_groups(bm));
            if (__any(mn > m[t])) {                          // uniform; rare after a row's first blocks
                const float f = exp_le0(m[t] - (mn == -INFINITY ? 0.0f : mn));
                l[t] *= f;
                m[t] = mn;
#pragma unroll
                for (int cb = 0; cb < HQ; cb++) acc[t][cb] *= f;
            }
            const float ref = mn == -INFINITY ? 0.0f : mn;  // no key yet: e^(-inf) = 0
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const float e = exp_le0(p[r] - ref);
                p[r] = key + r <= pos ? e : 0.0f;
                l[t] += p[r];
            }
            wsum<HQ>(acc[t], vt, p);
        }
#pragma unroll
        for (int i = 0; i < HQ; i++) kf[i] = kn[i];
#pragma unroll
        for (int s = 0; s < 4; s++)
#pragma unroll
            for (int cb = 0; cb < HQ; cb++) vt[s][cb] = vn[s][cb];
    }
#pragma unroll
    for (int t = 0; t < QT; t++) {
        l[t] = xsum_groups(l[t]);
        if (g == 0) { st_m[wave][16 * t + li] = m[t]; st_l[wave][16 * t + li] = l[t]; }
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < QT; t++) {
        float gm = -INFINITY;
#pragma unroll
        for (int w = 0; w < NW; w++) gm = fmaxf(gm, st_m[w][16 * t + li]);
        const float ref = gm == -INFINITY ? 0.0f : gm;
        float gl = 0.0f;
#pragma unroll
        for (int w = 0; w < NW; w++) gl += st_l[w][16 * t + li] * exp_le0(st_m[w][16 * t + li] - ref);
        const float inv = 1.0f / gl, f = exp_le0(m[t] - ref) * inv;
#pragma unroll
        for (int cb = 0; cb < HQ; cb++) acc[t][cb] *= f;
        const int row = r0 + 16 * t + li;
        if (a.row_max && wave == 0 && g == 0 && row < a.rows) {
            a.row_max[(long)h * a.stat_ld + row] = gm;
            a.row_inv[(long)h * a.stat_ld + row] = inv;
        }
        merge<HQ, NW>(acc[t], red, n4, [&](int i, int c, f4v o) {
            const int r = r0 + 16 * t + i;
            if (r < a.rows) *reinterpret_cast<f4v *>(a.out + (long)r * a.ldo + h * hd + 4 * c) = o;
        });
    }
}

// Backward, row half (pt_train.c:780-811): for the query rows of a tile,
// delta = sum(d_out * out) (the softmax backward's dot product, kept for the
// column half), dS^T = P^T * (V.d_out^T - delta) * scale and
// dQ^T += K^T.dS^T; dq is stored after rope_backward.
template <int HQ, int QT, int NW, bool PAD>
__global__ __launch_bounds__(64 * NW) void k_attn_rows_bwd(AttnBwdArgs a) {
    __shared__ __align__(16) float red[NW * 16 * (16 * HQ + 4)];
    const int h = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6, li = lane & 15, g = lane >> 4;
    const int hd = PAD ? a.head_dim : 16 * HQ, n4 = hd >> 2;
    const int r0 = (int)(gridDim.y - 1 - blockIdx.y) * 16 * QT;
    const int last = min(r0 + 16 * QT, a.rows) - 1, nkb = last / 16 + 1;
    const float *q = a.qkv + h * hd, *k = q + a.dim, *v = k + a.dim;
    float4 qf[QT][HQ], gf[QT][HQ];
    float m[QT], inv[QT], de[QT];
#pragma unroll
    for (int t = 0; t < QT; t++) {
        const int row = min(r0 + 16 * t + li, a.rows - 1);
        float4 of[HQ];
        load_row<HQ, PAD>(qf[t], q + (long)row * a.ldqkv, g, n4);
        load_row<HQ, PAD>(gf[t], a.d_out + (long)row * a.dim + h * hd, g, n4);
        load_row<HQ, PAD>(of, a.out + (long)row * a.dim + h * hd, g, n4);
        m[t] = a.row_max[(long)h * a.stat_ld + row];
        inv[t] = a.row_inv[(long)h * a.stat_ld + row];
        // in the order of the products V.d_out^T: a row of one key (out = v) then has dS = 0, as in the reference
        const f4v d = dots<HQ>(of, gf[t]);
        const float dl = li & 2 ? (li & 1 ? d.w : d.z) : (li & 1 ? d.y : d.x);
        de[t] = xsum_groups(li >> 2 == g ? dl : 0.0f);
        if (wave == 0 && g == 0 && r0 + 16 * t + li < a.rows) a.delta[(long)h * a.stat_ld + row] = de[t];
    }
    f4v acc[QT][HQ];
#pragma unroll
    for (int t = 0; t < QT; t++)
#pragma unroll
        for (int cb = 0; cb < HQ; cb++) acc[t][cb] = f4v{0.f, 0.f, 0.f, 0.f};
    for (int kb = wave; kb < nkb; kb += NW) {
        float4 kf[HQ], vf[HQ];
        float kt[4][HQ];
        const long key_row = min(kb * 16 + li, last);
        load_row<HQ, PAD>(kf, k + key_row * a.ldqkv, g, n4);
        load_row<HQ, PAD>(vf, v + key_row * a.ldqkv, g, n4);
        load_cols<HQ, PAD>(kt, k, a.ldqkv, kb * 16, last, g, li, hd);
#pragma unroll
        for (int t = 0; t < QT; t++) {
            const f4v s = dots<HQ>(kf, qf[t]), dp = dots<HQ>(vf, gf[t]);
            const int pos = r0 + 16 * t + li, key = kb * 16 + 4 * g;
            float ds[4];
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const float p = exp_le0(s[r] * a.scale - m[t]) * inv[t];
                ds[r] = key + r <= pos ? p * (dp[r] - de[t]) * a.scale : 0.0f;
            }
            wsum<HQ>(acc[t], kt, ds);
        }
    }
#pragma unroll
    for (int t = 0; t < QT; t++)
        merge<HQ, NW>(acc[t], red, n4, [&](int i, int c, f4v o) {
            const int r = r0 + 16 * t + i;
            if (r < a.rows)
                *reinterpret_cast<f4v *>(a.d_qkv + (long)r * a.ldqkv + h * hd + 4 * c) = rope_bwd4(o, c, hd, r);
        });
}

// Backward, column half: for the keys of a tile, over the query rows at or
// after them, dV^T += d_out^T.P and dK^T += Q^T.dS; dk is stored after
// rope_backward.
template <int HQ, int KT, int NW, bool PAD>
__global__ __launch_bounds__(64 * NW) void k_attn_cols_bwd(AttnBwdArgs a) {
    __shared__ __align__(16) float red[NW * 16 * (16 * HQ + 4)];
    const int h = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6, li = lane & 15, g = lane >> 4;
    const int hd = PAD ? a.head_dim : 16 * HQ, n4 = hd >> 2;
    const int k0 = (int)blockIdx.y * 16 * KT, last = a.rows - 1, nqb = last / 16 + 1;
    const float *q = a.qkv + h * hd, *k = q + a.dim, *v = k + a.dim, *go = a.d_out + h * hd;
    const float *mp = a.row_max + (long)h * a.stat_ld, *ip = a.row_inv + (long)h * a.stat_ld;
    const float *dp_ = a.delta + (long)h * a.stat_ld;
    float4 kf[KT][HQ], vf[KT][HQ];
#pragma unroll
    for (int t = 0; t < KT; t++) {
        const long row = min(k0 + 16 * t + li, last);
        load_row<HQ, PAD>(kf[t], k + row * a.ldqkv, g, n4);
        load_row<HQ, PAD>(vf[t], v + row * a.ldqkv, g, n4);
    }
    f4v av[KT][HQ], ak[KT][HQ];
#pragma unroll
    for (int t = 0; t < KT; t++)
#pragma unroll
        for (int cb = 0; cb < HQ; cb++) av[t][cb] = ak[t][cb] = f4v{0.f, 0.f, 0.f, 0.f};
    for (int qb = k0 / 16 + wave; qb < nqb; qb += NW) {
        float4 qf[HQ], gf[HQ];
        float qt[4][HQ], gt[4][HQ];
        const long row = min(qb * 16 + li, last);
        load_row<HQ, PAD>(qf, q + row * a.ldqkv, g, n4);
        load_row<HQ, PAD>(gf, go + row * a.dim, g, n4);
        // statistics are kept for multiples of 16 rows (those past the last are not used)
        const int q4 = qb * 16 + 4 * g;
        const f4v m = *reinterpret_cast<const f4v *>(mp + q4), inv = *reinterpret_cast<const f4v *>(ip + q4);
        const f4v de = *reinterpret_cast<const f4v *>(dp_ + q4);
        load_cols<HQ, PAD>(qt, q, a.ldqkv, qb * 16, last, g, li, hd);
        load_cols<HQ, PAD>(gt, go, a.dim, qb * 16, last, g, li, hd);
#pragma unroll
        for (int t = 0; t < KT; t++) {
            const f4v s = dots<HQ>(qf, kf[t]), dp = dots<HQ>(gf, vf[t]);
            const int key = k0 + 16 * t + li;
            float p[4], ds[4];
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const bool use = q4 + r <= last && q4 + r >= key;
                const float e = exp_le0(s[r] * a.scale - m[r]) * inv[r];
                p[r] = use ? e : 0.0f;
                ds[r] = use ? e * (dp[r] - de[r]) * a.scale : 0.0f;
            }
            wsum<HQ>(av[t], gt, p);
            wsum<HQ>(ak[t], qt, ds);
        }
    }
#pragma unroll
    for (int t = 0; t < KT; t++) {
        merge<HQ, NW>(av[t], red, n4, [&](int i, int c, f4v o) {
            const int r = k0 + 16 * t + i;
            if (r <= last) *reinterpret_cast<f4v *>(a.d_qkv + (long)r * a.ldqkv + 2 * a.dim + h * hd + 4 * c) = o;
        });
        merge<HQ, NW>(ak[t], red, n4, [&](int i, int c, f4v o) {
            const int r = k0 + 16 * t + i;
            if (r <= last)
                *reinterpret_cast<f4v *>(a.d_qkv + (long)r * a.ldqkv + a.dim + h * hd + 4 * c) = rope_bwd4(o, c, hd, r);
        });
    }
}

// Waves per block and 16-row tiles per block: what the registers hold.
constexpr int waves_for(int hq) { return hq <= 4 ? 8 : 4; }

// Two 16-row tiles per block where even half as many blocks keep every CU
// busy (two fill 256 CUs less evenly but load K and V half as often).
// Backward of a layer, us, one / two tiles: 12 heads x 1024 rows of 64
// 57.9 + 54.8 / 46.6 + 51.9; whole steps of two layers: 12 x 512 738 / 757,
// 8 x 1024 729 / 748, 12 x 1000 1272 / 1255.  The forward is level.
inline bool two_tiles(int rows, int heads, int head_dim) {
    return head_dim % 16 == 0 && head_dim <= 64 && (long)rows * heads >= 11000;
}

using FwdFn = void (*)(AttnFwdArgs);
using BwdFn = void (*)(AttnBwdArgs);

#define PER_HQ(K, T, PAD_)                                                                         \
    {K<1, T, waves_for(1), PAD_>, K<2, T, waves_for(2), PAD_>, K<3, T, waves_for(3), PAD_>,        \
     K<4, T, waves_for(4), PAD_>, K<5, T, waves_for(5), PAD_>, K<6, T, waves_for(6), PAD_>,        \
     K<7, T, waves_for(7), PAD_>, K<8, T, waves_for(8), PAD_>}

}  // namespace

int launch_attn_fwd(const AttnFwdArgs &a, int heads, hipStream_t s) {
    static const FwdFn one[2][8] = {PER_HQ(k_attn_rows_fwd, 1, false), PER_HQ(k_attn_rows_fwd, 1, true)};
    static const FwdFn two[4] = {k_attn_rows_fwd<1, 2, 8, false>, k_attn_rows_fwd<2, 2, 8, false>,
                                 k_attn_rows_fwd<3, 2, 8, false>, k_attn_rows_fwd<4, 2, 8, false>};
    const int hq = (a.head_dim + 15) / 16, pad = a.head_dim % 16 != 0;
    const bool pair = two_tiles(a.rows, heads, a.head_dim);
    const int tile = pair ? 32 : 16;
    hipLaunchKernelGGL(pair ? two[hq - 1] : one[pad][hq - 1], dim3(heads, (a.rows + tile - 1) / tile),
                       dim3(64 * waves_for(hq)), 0, s, a);
    PTMI_HIP(hipGetLastError());
    return PTMI_OK;
}

int launch_attn_bwd(const AttnBwdArgs &a, int heads, hipStream_t s) {
    static const BwdFn rows1[2][8] = {PER_HQ(k_attn_rows_bwd, 1, false), PER_HQ(k_attn_rows_bwd, 1, true)};
    static const BwdFn cols1[2][8] = {PER_HQ(k_attn_cols_bwd, 1, false), PER_HQ(k_attn_cols_bwd, 1, true)};
    static const BwdFn rows2[4] = {k_attn_rows_bwd<1, 2, 8, false>, k_attn_rows_bwd<2, 2, 8, false>,
                                   k_attn_rows_bwd<3, 2, 8, false>, k_attn_rows_bwd<4, 2, 8, false>};
    static const BwdFn cols2[4] = {k_attn_cols_bwd<1, 2, 8, false>, k_attn_cols_bwd<2, 2, 8, false>,
                                   k_attn_cols_bwd<3, 2, 8, false>, k_attn_cols_bwd<4, 2, 8, false>};
    const int hq = (a.head_dim + 15) / 16, pad = a.head_dim % 16 != 0;
    const bool pair = two_tiles(a.rows, heads, a.head_dim);
    const int tile = pair ? 32 : 16;
    const dim3 grid(heads, (a.rows + tile - 1) / tile), threads(64 * waves_for(hq));
    hipLaunchKernelGGL(pair ? rows2[hq - 1] : rows1[pad][hq - 1], grid, threads, 0, s, a);
    hipLaunchKernelGGL(pair ? cols2[hq - 1] : cols1[pad][hq - 1], grid, threads, 0, s, a);
    PTMI_HIP(hipGetLastError());
    return PTMI_OK;
}

}  // namespace ptmi

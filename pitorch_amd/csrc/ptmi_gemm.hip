// fp32 GEMMs on the CDNA4 matrix cores: C[M,N] (+)= op(A)[M,K] . op(B)[K,N],
// small ones with v_mfma_f32_16x16x4_f32, the others as products of three-way bf16
// splits with v_mfma_f32_32x32x16_bf16 (gemm_choice).  These replace the training backward's
// per-position matvecs / CPU outer products:
//   dW = dY^T X  (TN) — matmul_backward_weight_batched, pt_train.c:475-492
//   dX = dY W    (NN) — backward_input_pretrans, pt_train.c:442-453
//   Y  = X W^T   (NT) — the batched form of the training forward's matvecs
//
// The small tile: 32x32, K step 32, 256 threads = 4 waves in a 2x2 grid, each
// wave a 16x16 MFMA block.  Tiles are staged in LDS k-major (As[k][m],
// Bs[k][n], columns XOR-swizzled so no LDS access has bank conflicts).  Two K
// tiles are in flight in registers while a third feeds the matrix cores
// from LDS (double-buffered), so each tile's global latency is covered by
// two K steps of MFMAs.  Operand layout of the 16x16x4 f32 MFMA (CDNA3/4):
// lane l supplies A[l%16][l/16] and B[l/16][l%16]; result register r of lane
// l is C[4*(l/16)+r][l%16].
// Long-K GEMMs with small output grids split K over blockIdx.z into a
// workspace and reduce in split order afterwards (deterministic, no
// atomics).
#include "ptmi_internal.h"

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <utility>

namespace ptmi {

namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

constexpr int BK = 32;
constexpr int kXcdGrid = 768;             // grids this large take their tiles in XCD order
constexpr int kRing32 = 2;                // K tiles in flight in the 32x32 register ring

struct GemmArgs {
    const float *A; long lda;
    const float *B; long ldb;
    float *C; long ldc;
    const float *Cin;      // accumulate: C = Cin + op(A).op(B) (Cin == C in place), same ldc
    int M, N, K;
    int accumulate;
    float *partial;        // split-K workspace [splits][M][N] or null
    int k_per_split;
    GemmEpi epi;           // fused element-wise epilogue (whole-K launches only)
    GemmNorm nrm;          // fused RMSNorm of the A rows (NT, whole K)
    float *upd;            // fused SGD step of the weight C is the gradient of (TnGemm), or null
    const float *lr;
    const unsigned *keep;
};

// One GEMM of a grouped launch: its arguments and its range of tiles.
struct GemmGroupDesc {
    GemmArgs g;
    int tiles_n;           // tiles along N
    int tile0;             // first block of this GEMM in the grouped grid
};

// Read by loads whose element lies outside the operand (ragged edges and
// the K tail), so every load is unconditional and needs no select after it.
__device__ __align__(16) float g_gemm_zero[16] = {};

// One operand tile (R = 32 or 64 rows of the M or N side x 32 k) per K step;
// each of the 256 threads moves E = R*32/256 floats (4 or 8).  KMAJOR (R = 32): the operand
// is stored with k as the row index (A^T for TN, B for NN/TN); otherwise k
// is the contiguous index.
//   KMAJOR:  thread -> (k = tid/(R/E),     idx = E*(tid%(R/E)) + c)
//   !KMAJOR: thread -> (idx = tid/(32/E),  k = E*(tid%(32/E)) + c)
// VEC: 16-byte float4 loads; the launcher guarantees aligned rows and a
// contiguous extent (idx_lim for KMAJOR, K otherwise) that is a multiple of
// 4, so a float4 is either wholly inside the operand or wholly outside.
// Elements outside read g_gemm_zero: only the address is selected, before
// the load, so the loads of a tile stay in flight together (a select on the
// loaded value, or a branch, makes the compiler wait for every load issued
// so far).
template <bool KMAJOR, int R, bool VEC>
__device__ __forceinline__ void load_tile(const float *P, long ld, int idx_lim, int i0, int k0, int kend, int tid,
                                          float (&r)[R * BK / 256]) {
    constexpr int E = R * BK / 256;
    const float *zero = g_gemm_zero;
    if (KMAJOR) {
        const int k = k0 + tid / (R / E), i = i0 + E * (tid % (R / E));
        const bool kin = k < kend;
        const float *row = P + (long)(kin ? k : 0) * ld;
        if constexpr (VEC) {
#pragma unroll
            for (int c = 0; c < E; c += 4) {
                const bool in = kin && i + c < idx_lim;
                const float4 v = *reinterpret_cast<const float4 *>(in ? row + i + c : zero + c);
                r[c] = v.x; r[c + 1] = v.y; r[c + 2] = v.z; r[c + 3] = v.w;
            }
        } else {
#pragma unroll
            for (int c = 0; c < E; c++) r[c] = *((kin && i + c < idx_lim) ? row + i + c : zero + c);
        }
    } else {
        const int i = i0 + tid / (BK / E), k = k0 + E * (tid % (BK / E));
        const bool iin = i < idx_lim;
        const float *row = P + (long)(iin ? i : 0) * ld;
        if constexpr (VEC) {
#pragma unroll
            for (int c = 0; c < E; c += 4) {
                const bool in = iin && k + c < kend;
                const float4 v = *reinterpret_cast<const float4 *>(in ? row + k + c : zero + c);
                r[c] = v.x; r[c + 1] = v.y; r[c + 2] = v.z; r[c + 3] = v.w;
            }
        } else {
#pragma unroll
            for (int c = 0; c < E; c++) r[c] = *((iin && k + c < kend) ? row + k + c : zero + c);
        }
    }
}

// LDS holds each operand tile k-major, S[k][col] with rows of R floats, the
// column XOR-swizzled by row so that, with LDS's 32 banks and a wave64 b32 access served as two
// half-waves (b128 as four 8-lane groups), every access below is
// conflict-free:
//  * the MFMA operand reads (a half-wave reads rows k, k+1 at 16 columns):
//    bit 4 of the swizzle differs between rows k and k+1;
//  * the transposing b32 stores of !KMAJOR operands (a half-wave writes one
//    row per k group at 8 or 4 consecutive columns): the swizzle's bits
//    3..4 (R = 64) or 2..4 (R = 32) take a different value per k group;
//  * the b128 stores of KMAJOR operands (8 lanes write one row, 4 floats each).
// Bits 0..1 are never swizzled, so float4 chunks stay whole.
template <bool KMAJOR, int R>
__device__ __forceinline__ int lds_col(int r, int c) {
    if constexpr (KMAJOR) {
        static_assert(R == 32, "k-major tiles are 32 wide");
        return c ^ ((r & 1) << 4);
    } else if constexpr (R == 64) {
        return c ^ ((((r & 1) ^ ((r >> 3) & 1)) << 4) | (((r >> 4) & 1) << 3));
    } else {
        return c ^ ((((r & 1) ^ ((r >> 2) & 1)) << 4) | (((r >> 3) & 1) << 3) | (((r >> 4) & 1) << 2));
    }
}

template <bool KMAJOR, int R>
__device__ __forceinline__ void store_tile(float (*S)[R], int tid, const float (&r)[R * BK / 256]) {
    constexpr int E = R * BK / 256;
    if (KMAJOR) {
        const int k = tid / (R / E), i = E * (tid % (R / E));
#pragma unroll
        for (int c = 0; c < E; c += 4)
            *reinterpret_cast<float4 *>(&S[k][lds_col<KMAJOR, R>(k, i + c)]) =
                make_float4(r[c], r[c + 1], r[c + 2], r[c + 3]);
    } else {
        const int i = tid / (BK / E), k = E * (tid % (BK / E));
#pragma unroll
        for (int c = 0; c < E; c++) S[k + c][lds_col<KMAJOR, R>(k + c, i)] = r[c];
    }
}

// Epilogue of output element (m, n) with sum v (already scaled by a fused
// RMSNorm's 1/rms).  Columns n and n^1 of a row sit in lanes l and l^1, which
// the fused epilogues pair with a DPP swap: every lane of a wave calls this,
// and bounds are checked after the swap.
template <int EPI>
__device__ __forceinline__ void store_elem(const GemmArgs &g, float v, int m, int n, int z, float lrv) {
    if constexpr (EPI == GEMM_EPI_ROPE) {
        // RoPE of the q and k columns at the row's position (pt_ops.c:33-49;
        // training forward pt_train.c:217)
        const float pv = dpp_xor1(v);
        const int D = g.epi.rope_dim, col = n + g.epi.col0;
        if (col < 2 * D) {
            const int ip = (col < D ? col : col - D) & ~1;
            float c, sn;
            d_rope_cs(ip, g.epi.head_dim, g.epi.pos0 + m, &c, &sn);
            v = (n & 1) ? pv * sn + v * c : v * c - pv * sn;
        }
        if (g.epi.out && col >= D) {                             // k and v to the caches
            if (n < g.N && m < g.M) {
                if (col < 2 * D) g.epi.out[(long)m * g.epi.ld + (col - D)] = v;
                else g.epi.out2[(long)m * g.epi.ld + (col - 2 * D)] = v;
            }
            return;
        }
    } else if constexpr (EPI == GEMM_EPI_SWIGLU) {
        // columns (2i, 2i+1) = (h1, h3): out[m][i] = (h1*sigmoid(h1))*h3,
        // the training form of silu (pt_train.c:280-284)
        const float pv = dpp_xor1(v);
        if (!(n & 1) && n < g.N && m < g.M) {
            const float sig = 1.0f / (1.0f + d_expf(-v));
            g.epi.out[(long)m * g.epi.ld + (n >> 1)] = (v * sig) * pv;
        }
        if (g.epi.only_out) return;
    }
    if (n >= g.N || m >= g.M) return;
    if constexpr (EPI == GEMM_EPI_SWIGLU_BWD) {
        // silu*gate backward (pt_train.c:696-721) into the interleaved
        // (d_h1, d_h3) columns, plus silu(h1)*h3 for dW2; d_sh itself is not kept
        const float *hp = g.epi.aux + (long)m * g.epi.aux_ld + 2 * n;
        const float h1 = hp[0], h3 = hp[1];
        const float sig = 1.0f / (1.0f + d_expf(-h1));
        const float silu_val = h1 * sig;
        g.epi.out2[(long)m * g.epi.ld2 + n] = silu_val * h3;
        const float d_silu = v * h3;
        float *dp = g.epi.out + (long)m * g.epi.ld + 2 * n;
        dp[1] = v * silu_val;
        dp[0] = d_silu * sig * (1.0f + h1 * (1.0f - sig));
    } else if (g.partial) {
        g.partial[((long)z * g.M + m) * g.N + n] = v;
    } else {
        const long o = (long)m * g.ldc + n;
        const float cv = g.accumulate ? g.Cin[o] + v : v;
        g.C[o] = cv;
        // sgd_step (pt_train.c:870-873) on the weight this gradient belongs to
        if (g.upd && !(g.keep && ((g.keep[m >> 5] >> (m & 31)) & 1u))) g.upd[o] -= lrv * cv;
    }
}

// Epilogue of one wave's FM x FN 16x16 blocks: block (i, j) of the wave
// covers rows mb + 16i .. and columns nb + 16j ..; lane l holds rows
// 4*(l/16) + r, column l%16 of it (the 16x16x4 MFMA result layout).
template <int EPI, int FM, int FN>
__device__ __forceinline__ void gemm_store(const GemmArgs &g, const floatx4 (&acc)[FM][FN], int mb, int nb, int z,
                                           int li, int lk, const float *rs = nullptr, int rs_m0 = 0) {
    const float lrv = g.upd ? *g.lr : 0.0f;
#pragma unroll
    for (int i = 0; i < FM; i++) {
#pragma unroll
        for (int j = 0; j < FN; j++) {
            const int n = nb + j * 16 + li;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int m = mb + i * 16 + 4 * lk + r;
                float v = acc[i][j][r];
                if (rs) v *= rs[m - rs_m0];                     // fused RMSNorm: the row's 1/rms
                store_elem<EPI>(g, v, m, n, z, lrv);
            }
        }
    }
}

// Fused RMSNorm: the block of N tile j stores its share of rows m0 ..
// m0+R-1 (float4 columns [j*c4, (j+1)*c4) of K/4, c4 = ceil(K/4 / tiles))
// of X (to x_out when completed here) and of X * inv * w (to xn_out), all
// loads of a pass in flight together; the block of tile 0 also marks the
// rows' tokens (EMBED, rows < M-1) in tok_bits.
template <int NORM, int R>
__device__ __forceinline__ void norm_rows_out(const GemmArgs &g, int m0, int j, int tiles, const float *inv) {
    const GemmNorm &nm = g.nrm;
    const int K4 = g.K / 4, c4 = (K4 + tiles - 1) / tiles, c_lo = j * c4, c_n = min(c4, K4 - c_lo);
    const int tid = threadIdx.x;
    const float *zero = g_gemm_zero;
    for (int e = tid; e < R * c_n; e += 256) {
        const int r = e / c_n, m = m0 + r;
        const bool in = m < g.M;
        const long col = 4L * (c_lo + (e - r * c_n));
        const long o = (long)min(m, g.M - 1) * g.K + col;
        float4 x;
        if constexpr (NORM == GEMM_NORM_SPLITS) {
            float4 p[kNormSplits];
#pragma unroll
            for (int zz = 0; zz < kNormSplits; zz++)
                p[zz] = *reinterpret_cast<const float4 *>(zz < nm.pk.splits ? nm.pk.parts + zz * nm.pk.stride + o : zero);
            const float4 c = *reinterpret_cast<const float4 *>(nm.cin ? nm.cin + o : zero);
            float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
            for (int zz = 0; zz < kNormSplits; zz++) {
                const bool use = zz < nm.pk.splits;
                v.x = use ? v.x + p[zz].x : v.x;
                v.y = use ? v.y + p[zz].y : v.y;
                v.z = use ? v.z + p[zz].z : v.z;
                v.w = use ? v.w + p[zz].w : v.w;
            }
            x = nm.cin ? make_float4(c.x + v.x, c.y + v.y, c.z + v.z, c.w + v.w) : v;
        } else if constexpr (NORM == GEMM_NORM_EMBED) {
            x = *reinterpret_cast<const float4 *>(nm.emb + (long)nm.tok[min(m, g.M - 1)] * g.K + col);
        } else {
            x = *reinterpret_cast<const float4 *>(g.A + o);
        }
        const float4 w = *reinterpret_cast<const float4 *>(nm.w + col);
        if (!in) continue;
        if constexpr (NORM != GEMM_NORM_PLAIN) *reinterpret_cast<float4 *>(nm.x_out + o) = x;
        const float iv = inv[r];
        *reinterpret_cast<float4 *>(nm.xn_out + o) = make_float4(x.x * iv * w.x, x.y * iv * w.y, x.z * iv * w.z, x.w * iv * w.w);
    }
    if constexpr (NORM == GEMM_NORM_EMBED) {
        const int m = m0 + tid;
        if (j == 0 && tid < R && m < g.M - 1) {
            const int tk = nm.tok[m];
            atomicOr(&nm.tok_bits[tk >> 5], 1u << (tk & 31));
        }
    }
}

constexpr int kChains = BK / 4;
// acc[0] = the sum of the NC partial sums, pairwise
template <int NC, int FM, int FN>
__device__ __forceinline__ void sum_chains(floatx4 (&acc)[NC][FM][FN]) {
#pragma unroll
    for (int h = NC / 2; h > 0; h /= 2)
#pragma unroll
        for (int c = 0; c < h; c++)
#pragma unroll
            for (int i = 0; i < FM; i++)
#pragma unroll
                for (int j = 0; j < FN; j++) acc[c][i][j] += acc[c + h][i][j];
}

// One TMxTN output tile of g at (m0, n0) over K range split z.  The LDS
// tiles use the swizzled layout of lds_col.
template <bool AT, bool BT, int TM, int TN, int P, bool VEC, int EPI = GEMM_EPI_NONE, int NORM = 0>
__device__ __forceinline__ void gemm_tile(const GemmArgs &g, int m0, int n0, int z) {
    constexpr int FM = TM / 32, FN = TN / 32;          // 16x16 MFMA blocks per wave
    constexpr int EA = TM * BK / 256, EB = TN * BK / 256;
    static_assert(NORM == 0 || (!AT && TM == 32 && VEC && EA == 4), "fused norm: NT, 32-row float4 A tiles");
    __shared__ float As[2][BK][TM];
    __shared__ float Bs[2][BK][TN];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    const int li = lane & 15, lk = lane >> 4;
    const int kb = z * g.k_per_split;
    const int kend = min(g.K, kb + g.k_per_split);
    const int nk = kb < kend ? (kend - kb + BK - 1) / BK : 0;

    // One 16x16 block per wave: the 8 MFMAs of a K step go to 8 sums, added
    // pairwise at the end, so each is rounded an eighth as often (64x768x288
    // and its gradients: 3.0e-7 -> 1.2e-7 from 64-bit sums).
    // Not TN: the 32 registers cost the grouped weight gradients occupancy
    // (64 steps of stories15M, T=256: 50.0 -> 52.8 ms).
    // The 64x64 tile's four blocks per wave have four chains each.
    constexpr int NC = AT ? 1 : FM * FN == 1 ? kChains : 4;
    floatx4 acc[NC][FM][FN];
#pragma unroll
    for (int c = 0; c < NC; c++)
#pragma unroll
        for (int i = 0; i < FM; i++)
#pragma unroll
            for (int j = 0; j < FN; j++) acc[c][i][j] = floatx4{0.f, 0.f, 0.f, 0.f};

    // P K tiles in flight in a register ring (tile t in slot t % P); the
    // loop is unrolled by P so every slot index is a compile-time constant.
    float ra[P][EA], rb[P][EB];
    // Fused RMSNorm: thread tid owns A row na_i and k offset na_k of every K
    // step (the load_tile mapping); the ring holds the raw row values (the
    // split-K partials and the addend, summed at the LDS store) and the norm
    // weights; the A tile takes x * w, and the row's sum of squares builds up.
    constexpr int NL = NORM == GEMM_NORM_SPLITS ? kNormSplits + 1 : 1;
    const int na_i = m0 + tid / (BK / EA), na_k = EA * (tid % (BK / EA));
    float4 nr[P][NL], ng[P];
    float nss = 0.0f;
    const float *na_row = g.A + (long)min(na_i, g.M - 1) * g.lda;
    if constexpr (NORM == GEMM_NORM_EMBED) na_row = g.nrm.emb + (long)g.nrm.tok[min(na_i, g.M - 1)] * g.K;
    auto load = [&](int s, int slot, float (&xa)[EA], float (&xb)[EB]) {
        if constexpr (NORM != 0) {
            const float *zero = g_gemm_zero;
            const int k = kb + s * BK + na_k;
            const bool in = na_i < g.M && k < kend;
            if constexpr (NORM == GEMM_NORM_SPLITS) {
                const long o = (long)min(na_i, g.M - 1) * g.K + k;
#pragma unroll
                for (int zz = 0; zz < kNormSplits; zz++)
                    nr[slot][zz] = *reinterpret_cast<const float4 *>(
                        in && zz < g.nrm.pk.splits ? g.nrm.pk.parts + zz * g.nrm.pk.stride + o : zero);
                nr[slot][kNormSplits] = *reinterpret_cast<const float4 *>(in && g.nrm.cin ? g.nrm.cin + o : zero);
            } else {
                nr[slot][0] = *reinterpret_cast<const float4 *>(in ? na_row + k : zero);
            }
            ng[slot] = *reinterpret_cast<const float4 *>(in ? g.nrm.w + k : zero);
        } else {
            load_tile<AT, TM, VEC>(g.A, g.lda, g.M, m0, kb + s * BK, kend, tid, xa);
        }
        load_tile<!BT, TN, VEC>(g.B, g.ldb, g.N, n0, kb + s * BK, kend, tid, xb);
    };
    auto store = [&](int s, int slot, const float (&xa)[EA], const float (&xb)[EB]) {
        if constexpr (NORM != 0) {
            float4 x = nr[slot][0];
            if constexpr (NORM == GEMM_NORM_SPLITS) {
                // the standalone kernel's order: ((0 + p0) + p1) + ..., then cin + sum
                float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
                for (int zz = 0; zz < kNormSplits; zz++) {
                    const bool use = zz < g.nrm.pk.splits;
                    v.x = use ? v.x + nr[slot][zz].x : v.x;
                    v.y = use ? v.y + nr[slot][zz].y : v.y;
                    v.z = use ? v.z + nr[slot][zz].z : v.z;
                    v.w = use ? v.w + nr[slot][zz].w : v.w;
                }
                const float4 c = nr[slot][kNormSplits];
                x = g.nrm.cin ? make_float4(c.x + v.x, c.y + v.y, c.z + v.z, c.w + v.w) : v;
            }
            nss += x.x * x.x + x.y * x.y + x.z * x.z + x.w * x.w;
            const float4 w = ng[slot];
            const float xw[EA] = {x.x * w.x, x.y * w.y, x.z * w.z, x.w * w.w};
            store_tile<AT, TM>(As[s & 1], tid, xw);
        } else {
            store_tile<AT, TM>(As[s & 1], tid, xa);
        }
        store_tile<!BT, TN>(Bs[s & 1], tid, xb);
    };
    // The operands of k group kk+4*RA are read from LDS before the MFMAs of
    // group kk issue, so their latency overlaps RA groups of MFMAs (RA = 2
    // and 3 measured no faster).
    constexpr int RA = 1;
    auto compute = [&](int s) {
        const int buf = s & 1;
        float a[RA + 1][FM], b[RA + 1][FN];
        auto read = [&](int kk, float (&ar)[FM], float (&br)[FN]) {
#pragma unroll
            for (int i = 0; i < FM; i++) ar[i] = As[buf][kk + lk][lds_col<AT, TM>(kk + lk, wm * (TM / 2) + i * 16 + li)];
#pragma unroll
            for (int j = 0; j < FN; j++) br[j] = Bs[buf][kk + lk][lds_col<!BT, TN>(kk + lk, wn * (TN / 2) + j * 16 + li)];
        };
#pragma unroll
        for (int r = 0; r < RA; r++) read(4 * r, a[r], b[r]);
#pragma unroll
        for (int kk = 0; kk < BK; kk += 4) {
            const int c = (kk / 4) % (RA + 1);
            if (kk + 4 * RA < BK) read(kk + 4 * RA, a[(kk / 4 + RA) % (RA + 1)], b[(kk / 4 + RA) % (RA + 1)]);
            __builtin_amdgcn_sched_barrier(0);              // keep the reads ahead of the MFMAs
#pragma unroll
            for (int i = 0; i < FM; i++)
#pragma unroll
                for (int j = 0; j < FN; j++)
                    acc[kk / 4 % NC][i][j] =
                        __builtin_amdgcn_mfma_f32_16x16x4f32(a[c][i], b[c][j], acc[kk / 4 % NC][i][j], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
    };

#pragma unroll
    // Loads are unconditional (tiles past the K range read zeros): a load
    // under a branch leaves the compiler unsure how many loads are in flight,
    // and it then waits for all of them, which empties the ring.
    for (int t = 0; t < P; t++) load(t, t, ra[t], rb[t]);
    store(0, 0, ra[0], rb[0]);
    __syncthreads();
    // Step s: tile s is in LDS; its register slot (s % P) is free, so tile
    // s+P is fetched into it; tile s+1 goes to the other LDS buffer.  Full
    // groups of P steps run without branches; the last nk % P steps follow.
    int s0 = 0;
    for (; s0 + P <= nk; s0 += P) {
#pragma unroll
        for (int u = 0; u < P; u++) {
            load(s0 + u + P, u, ra[u], rb[u]);
            __builtin_amdgcn_sched_barrier(0);              // issue the loads before the MFMAs
            compute(s0 + u);
            store(s0 + u + 1, (u + 1) % P, ra[(u + 1) % P], rb[(u + 1) % P]);
            __syncthreads();
        }
    }
#pragma unroll
    for (int u = 0; u + 1 < P; u++) {
        if (s0 + u < nk) {                                  // uniform
            compute(s0 + u);
            store(s0 + u + 1, (u + 1) % P, ra[(u + 1) % P], rb[(u + 1) % P]);
            __syncthreads();
        }
    }

    if constexpr (NC > 1) sum_chains(acc);
    if constexpr (NORM != 0) {
        // 1/rms of the block's rows (the standalone kernel's formula); every
        // N tile's block stores its share of the rows and normalized rows
        __shared__ float n_inv[TM];
        nss = group_sum<BK / EA>(nss);
        if (tid % (BK / EA) == 0) n_inv[tid / (BK / EA)] = 1.0f / d_sqrtf(nss / (float)g.K + 1e-5f);
        __syncthreads();
        norm_rows_out<NORM, TM>(g, m0, n0 / TN, (g.N + TN - 1) / TN, n_inv);
        gemm_store<EPI, FM, FN>(g, acc[0], m0 + wm * (TM / 2), n0 + wn * (TN / 2), z, li, lk, n_inv, m0);
    } else {
        gemm_store<EPI, FM, FN>(g, acc[0], m0 + wm * (TM / 2), n0 + wn * (TN / 2), z, li, lk);
    }
}

// ── Direct-to-LDS tiles ──────────────────────────────────────────────────
// gfx950's global_load_lds_dwordx4 moves a 16-byte chunk per lane from
// global memory straight into LDS, at the wave's LDS base + 16*lane (lane
// layout checked on the MI355X): no staging registers and no LDS store
// instructions.  Each operand tile keeps its global layout in LDS, permuted in whole
// 16-byte chunks (the only granularity a DMA load can place):
//  * k-contiguous operands ([i][k]: A of NN/NT, B^T of NT): rows of BK=32
//    floats (128 bytes), chunk c of row i at slot c ^ kc_swz(i).  A lane
//    reads the 4 k of its row for 4 MFMA steps as one b128 (lane group g
//    takes k = 4g..4g+3 of each 16-k group).  A b128 read serves 16 lanes
//    (16 rows) at a time across the 64 banks, where rows i and i+8 start on
//    the same bank; kc_swz gives the 16 rows 16 distinct bank groups;
//  * k-major operands ([k][i]: A^T of TN, B of NN/TN): rows of TI floats,
//    the column XOR-ed with 16 in rows whose bit 2 of k is set; the two k
//    rows a half-wave reads (g = 0, 1) then sit 16 banks apart.
// Both operands use the same order of k inside a 16-k group (lane group g,
// step s -> k = 4g + s), so every product pairs the same k.
// The 128x96 tile below is for weight gradients (TN) of one K step (gemm_choice);
// it has two LDS stages: the loads of tile s+1 are issued before the MFMAs of tile
// s and waited for (vmcnt, in order) at the next step's barrier.
constexpr int kDlStages = 2;

// Chunk-slot swizzle of row i of a k-contiguous tile: i & 7 spreads 8
// consecutive rows over the 8 slots; bit 3 of i moves rows i and i+8 to
// different slots.
__device__ __forceinline__ int kc_swz(int i) { return (i & 7) ^ ((i >> 3) & 1); }

template <int N>
__device__ __forceinline__ void wait_vmcnt() {                   // s_waitcnt vmcnt(N), other counters untouched
    static_assert(N >= 0 && N < 64, "vmcnt");
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}

// This thread's DMA loads of one operand tile (TI rows of the M or N side x
// BK k, k0 = first k) into `lds`; 64-chunk regions are dealt to the NW
// waves round-robin, and a wave with no region left loads zeros into `junk`
// so that every wave issues the same number of loads.
template <bool KMAJOR, int TI, int NW>
__device__ __forceinline__ void dl_issue(const float *P, long ld, int ilim, int i0, int k0, int kend, float *lds,
                                         float *junk, int wave, int lane) {
    constexpr int CPI = BK / 4;                          // chunks per row, k-contiguous layout
    constexpr int R = TI * CPI / 64;
#pragma unroll
    for (int j = 0; j < (R + NW - 1) / NW; j++) {
        const int rgn = j * NW + wave;
        const bool real = rgn < R;                       // wave-uniform
        const int S = (real ? rgn : 0) * 64 + lane;      // chunk slot in the tile
        const float *src = g_gemm_zero;
        if constexpr (KMAJOR) {
            constexpr int CPR = TI / 4;                  // chunks per LDS row
            const int k = S / CPR, t = S % CPR;
            const int i = i0 + 4 * (t ^ (((k >> 2) & 1) << 2)), kk = k0 + k;
            if (real && kk < kend && i < ilim) src = P + (long)kk * ld + i;
        } else {
            const int i = S / CPI, t = S % CPI;
            const int ii = i0 + i, kk = k0 + 4 * (t ^ kc_swz(i));
            if (real && ii < ilim && kk < kend) src = P + (long)ii * ld + kk;
        }
        typedef const void __attribute__((address_space(1))) *gptr;
        typedef void __attribute__((address_space(3))) *lptr;
        __builtin_amdgcn_global_load_lds((gptr)src, (lptr)(real ? lds + rgn * 256 : junk), 16, 0, 0);
    }
}

// One TMxTN output tile on WM x WN waves (each (TM/WM) x (TN/WN)), both
// operands k-major (TN).
template <int TM, int TN, int WM, int WN>
__device__ __forceinline__ void gemm_tile_dl(const GemmArgs &g, int m0, int n0, int z) {
    constexpr int NW = WM * WN, NS = kDlStages;
    constexpr int FM = TM / WM / 16, FN = TN / WN / 16;
    static_assert(FM * WM * 16 == TM && FN * WN * 16 == TN, "tile");
    constexpr int STAGE = (TM + TN) * BK;
    __shared__ __align__(16) float smem[NS * STAGE + 256];
    float *junk = smem + NS * STAGE;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave / WN, wn = wave % WN;
    const int li = lane & 15, lk = lane >> 4;
    const int kb = z * g.k_per_split;
    const int kend = min(g.K, kb + g.k_per_split);
    const int nk = kb < kend ? (kend - kb + BK - 1) / BK : 0;

    floatx4 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};

    auto issue = [&](int t) {
        float *st = smem + (t % NS) * STAGE;
        const int k0 = kb + t * BK;
        dl_issue<true, TM, NW>(g.A, g.lda, g.M, m0, k0, kend, st, junk, wave, lane);
        dl_issue<true, TN, NW>(g.B, g.ldb, g.N, n0, k0, kend, st + TM * BK, junk, wave, lane);
    };
    // MFMA operands of 16-k group q: lane group lk takes k = 16q + 4lk + s
    // in step s (a float4 per fragment, one k per component).
    auto read_a = [&](const float *st, int q, floatx4 (&a)[FM]) {
#pragma unroll
        for (int f = 0; f < FM; f++)
#pragma unroll
            for (int s = 0; s < 4; s++) {
                const int k = 16 * q + 4 * lk + s, i = wm * (TM / WM) + f * 16 + li;
                a[f][s] = st[k * TM + (i ^ (((k >> 2) & 1) << 4))];
            }
    };
    auto read_b = [&](const float *st, int q, floatx4 (&b)[FN]) {
#pragma unroll
        for (int h = 0; h < FN; h++)
#pragma unroll
            for (int s = 0; s < 4; s++) {
                const int k = 16 * q + 4 * lk + s, i = wn * (TN / WN) + h * 16 + li;
                b[h][s] = st[TM * BK + k * TN + (i ^ (((k >> 2) & 1) << 4))];
            }
    };

    if (nk > 0) issue(0);
    for (int s = 0; s < nk; s++) {
        // tile s has landed in every wave's share once each wave's own
        // loads are done (vmcnt) and all waves passed the barrier; the
        // barrier also ends every read of the stage tile s+1 overwrites
        wait_vmcnt<0>();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (s + 1 < nk) issue(s + 1);
        const float *st = smem + (s % NS) * STAGE;
        floatx4 a[2][FM], b[2][FN];
        read_a(st, 0, a[0]);
        read_b(st, 0, b[0]);
        read_a(st, 1, a[1]);
        read_b(st, 1, b[1]);
#pragma unroll
        for (int q = 0; q < 2; q++)
#pragma unroll
            for (int ss = 0; ss < 4; ss++)
#pragma unroll
                for (int f = 0; f < FM; f++)
#pragma unroll
                    for (int h = 0; h < FN; h++)
                        acc[f][h] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[q][f][ss], b[q][h][ss], acc[f][h], 0, 0, 0);
    }
    gemm_store<GEMM_EPI_NONE, FM, FN>(g, acc, m0 + wm * (TM / WM), n0 + wn * (TN / WN), z, li, lk);
}

// f(integral_constant<int, s>) for s = S...
template <typename F, int... S>
__device__ __forceinline__ void unrolled(F &f, std::integer_sequence<int, S...>) {
    (f(std::integral_constant<int, S>{}), ...);
}

// The per-layer GEMMs' 32x32 tile with every K tile of its split in flight
// at once: the block issues the DMA loads of all NSK tiles (each into its
// own LDS stage; tiles past the split's K range load zeros) before its first
// MFMA, and starts tile s once the loads behind it are the only ones left
// (vmcnt counts them).  The register ring holds one or two tiles ahead, so
// each of its K steps waits about one load latency; here the block waits
// for about one.  Operand layout, MFMA k order and epilogue as
// gemm_tile_dl with 2 x 2 waves of 16 x 16.  NT (B^T k-contiguous) or NN
// (BKM: B stored [K][N]).
template <bool BKM, int NSK, int EPI>
__device__ __forceinline__ void gemm_tile_panel(const GemmArgs &g, int m0, int n0, int z) {
    constexpr int TM = 32, TN = 32, WN = 2, NW = 4, CPI = BK / 4;
    constexpr int STAGE = (TM + TN) * BK;
    constexpr int LPT = (TM * CPI / 64 + NW - 1) / NW + (TN * CPI / 64 + NW - 1) / NW;
    static_assert((NSK - 1) * LPT < 64, "vmcnt");
    __shared__ __align__(16) float smem[NSK * STAGE + 256];
    float *junk = smem + NSK * STAGE;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave / WN, wn = wave % WN;
    const int li = lane & 15, lk = lane >> 4;
    const int kb = z * g.k_per_split;
    const int kend = min(g.K, kb + g.k_per_split);
    const int nk = kb < kend ? (kend - kb + BK - 1) / BK : 0;
#pragma unroll
    for (int t = 0; t < NSK; t++) {
        float *st = smem + t * STAGE;
        dl_issue<false, TM, NW>(g.A, g.lda, g.M, m0, kb + t * BK, kend, st, junk, wave, lane);
        dl_issue<BKM, TN, NW>(g.B, g.ldb, g.N, n0, kb + t * BK, kend, st + TM * BK, junk, wave, lane);
    }
    floatx4 acc[kChains][1][1];                                     // as gemm_tile's
#pragma unroll
    for (int c = 0; c < kChains; c++) acc[c][0][0] = floatx4{0.f, 0.f, 0.f, 0.f};
    const int ia = wm * 16 + li, ib = wn * 16 + li;
    // step s, unrolled (each wait takes a constant count)
    auto step = [&](auto sc) {
        constexpr int s = decltype(sc)::value;
        wait_vmcnt<(NSK - 1 - s) * LPT>();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (s < nk) {                                               // uniform
            const float *st = smem + s * STAGE, *sb = st + TM * BK;
            floatx4 a[2], b[2];
#pragma unroll
            for (int q = 0; q < 2; q++) {
                a[q] = *reinterpret_cast<const floatx4 *>(st + (ia * CPI + ((4 * q + lk) ^ kc_swz(ia))) * 4);
                if constexpr (BKM) {
#pragma unroll
                    for (int u = 0; u < 4; u++) {
                        const int k = 16 * q + 4 * lk + u;
                        b[q][u] = sb[k * TN + (ib ^ (((k >> 2) & 1) << 4))];
                    }
                } else {
                    b[q] = *reinterpret_cast<const floatx4 *>(sb + (ib * CPI + ((4 * q + lk) ^ kc_swz(ib))) * 4);
                }
            }
#pragma unroll
            for (int q = 0; q < 2; q++)
#pragma unroll
                for (int u = 0; u < 4; u++)
                    acc[4 * q + u][0][0] =
                        __builtin_amdgcn_mfma_f32_16x16x4f32(a[q][u], b[q][u], acc[4 * q + u][0][0], 0, 0, 0);
        }
    };
    unrolled(step, std::make_integer_sequence<int, NSK>{});
    sum_chains(acc);
    gemm_store<EPI, 1, 1>(g, acc[0], m0 + wm * 16, n0 + wn * 16, z, li, lk);
}

// ── fp32 products on the bf16 matrix cores ───────────────────────────────
// The large and middle GEMMs.  v_mfma_f32_32x32x16_bf16 runs 16x the
// multiply-adds per cycle of v_mfma_f32_32x32x2_f32, and an fp32 number is
// exactly the sum of three bf16: x = h + m + l, h the nearest bf16, m the
// nearest to x - h, l the rest (24 significant bits in all).  a*b is taken as
// the six largest of the nine partial products, smallest first into one fp32
// accumulator: al*bh, ah*bl, am*bm, am*bh, ah*bm, ah*bh.  The three dropped are
// together below 2^-24 of |a*b| (+ 2^-33) and of either sign (h and m are rounded,
// not cut), and the accumulator rounds 6 times per 16 k instead of 16 times, so
// results are nearer to 64-bit sums than the fp32 MFMA tiles' (relative error at K = 768
// and 2048: 5.0e-7 and 8.1e-7 before, 4.2e-7 and 6.9e-7 in 128x128 tiles,
// 2.1e-7 and 3.4e-7 in 64x64 tiles, whose four waves each sum a quarter of
// K).  A single product among zeros is up to 3 x 2^-24 off, where fp32 MFMAs
// round it to nearest (2^-24): sums of fewer than 16 terms are left to them.
// A tile is computed again with fp32 MFMAs, and so comes out as the fp32 tiles
// give it, where a sum is not finite (infinities, NaNs, numbers that round past
// the bf16 range) or subnormal, or where an operand has bits below bf16's
// smallest number, 2^-133, as operands below 2^-109 can.  Rounding m and
// watching for such bits cost 1 to 6% (NN 1024x768x32000 283 -> 299 us, NT 1024x32000x768
// 271 -> 289).
// What bounds it: the MFMAs (32 cycles each) and the splits (8 VALU
// instructions per MFMA) issue side by side; with the splits taken out the same
// kernels reach 180-195 TFLOP/s, the bf16 matrix rate under the card's power limit.
//
// Operand tiles reach LDS as fp32 by DMA, KD = 16 or 32 k at a time, in whole
// 16-byte chunks: k-contiguous operands as rows of KD floats with the chunks
// of row i permuted so that 16 rows' same chunk spread over all banks;
// k-major operands as rows of TI floats with bit 5 of the column flipped
// where bit 3 of k is set (a lane half reads 8 k, the other half the next 8).
// The loads are buffer loads with a per-lane offset: elements outside the
// operand get an offset past the descriptor's range and come back as zeros,
// so addresses are worked out once per tile (again for a ragged K step) and
// no load is under a branch.  E floats per lane and load: 4, or 1 where rows
// are not 16-byte aligned (the same tile with four times the load
// instructions: NT 1024x2048x768 24.9 -> 28.3 us).
constexpr int kOutside = (int)0x80000000;     // past every descriptor's range

// 16 or 4 bytes per lane to lds + lane * size.
typedef void __attribute__((address_space(3))) *lds_ptr;
__device__ __forceinline__ void dma16(__amdgpu_buffer_rsrc_t rs, float *lds, int off) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr)lds, 16, off, 0, 0, 0);
}
__device__ __forceinline__ void dma4(__amdgpu_buffer_rsrc_t rs, float *lds, int off) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr)lds, 4, off, 0, 0, 0);
}

template <bool KMAJOR, int TI, int KD, int E, int NW>
struct TileDma {
    static constexpr int N = TI * KD / (64 * E * NW);           // loads per wave
    static_assert(N * 64 * E * NW == TI * KD && (KD == 16 || KD == 32), "whole loads");
    int off[N];
    static __device__ __forceinline__ int swz(int i) { return KD == 32 ? kc_swz(i) : (i >> 2) & 3; }
    // This lane's byte offsets from the tile's first element; krem: the k
    // left from there.  ld < kMaxSplitLd keeps them below 2^31.
    __device__ __forceinline__ void init(long ld, int ilim, int i0, int wave, int lane, int krem) {
#pragma unroll
        for (int j = 0; j < N; j++) {
            const int S = E * ((j * NW + wave) * 64 + lane);    // position in the tile
            int i, k;
            if constexpr (KMAJOR) {
                k = S / TI;
                i = (S % TI) ^ (((k >> 3) & 1) << 5);
            } else {
                i = S / KD;
                k = 4 * (((S % KD) >> 2) ^ swz(i)) + (S & 3);
            }
            const long o = KMAJOR ? (long)k * ld + i : (long)i * ld + k;
            off[j] = i0 + i < ilim && k < krem ? (int)(4 * o) : kOutside;
        }
    }
    // records: 0x7fffffff, or 0 to load zeros only
    __device__ __forceinline__ void issue(const float *base, int records, float *lds, int wave) const {
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void *)base, (short)0, records, 0x00020000);
#pragma unroll
        for (int j = 0; j < N; j++) {
            float *dst = lds + (j * NW + wave) * 64 * E;
            if constexpr (E == 4) dma16(rs, dst, off[j]);
            else dma4(rs, dst, off[j]);
        }
    }
    // x[e] = element (i, k = 16q + 8*lh + e) of the tile in LDS
    static __device__ __forceinline__ void read(const float *t, int i, int q, int lh, float (&x)[8]) {
        if constexpr (KMAJOR) {
#pragma unroll
            for (int e = 0; e < 8; e++) x[e] = t[(16 * q + 8 * lh + e) * TI + (i ^ (lh << 5))];
        } else {
#pragma unroll
            for (int c = 0; c < 2; c++) {
                const floatx4 v = *reinterpret_cast<const floatx4 *>(t + i * KD + 4 * ((4 * q + 2 * lh + c) ^ swz(i)));
#pragma unroll
                for (int e = 0; e < 4; e++) x[4 * c + e] = v[e];
            }
        }
    }
};
constexpr int kShortK = 16;                   // fewer terms are left to fp32 MFMAs
constexpr long kMaxSplitLd = 1L << 22;        // 128 rows of it take at most 2^31 bytes

typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned uintx4 __attribute__((ext_vector_type(4)));

// x[e] = o[0][e] + o[1][e] + o[2][e] (see above).  h and m are rounded to nearest, so
// |m| <= 2^-8 and |l| <= 2^-17 of x's leading power of two (m cut instead: 2^-16).  The
// low halves of `lost` collect what l's bf16 cannot hold (x below 2^-109).
__device__ __forceinline__ void split_bf16(const float (&x)[8], bf16x8 (&o)[3], unsigned &lost) {
    constexpr unsigned kTop = 0xffff0000u, kHighHalves = 0x07060302u;
    uintx4 h, m, l;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const floatx2 v = {x[2 * e], x[2 * e + 1]};
        h[e] = __builtin_bit_cast(unsigned, __builtin_convertvector(v, bf16x2));
        const floatx2 r = {v.x - __uint_as_float(h[e] << 16), v.y - __uint_as_float(h[e] & kTop)};
        m[e] = __builtin_bit_cast(unsigned, __builtin_convertvector(r, bf16x2));
        const unsigned l0 = __float_as_uint(r.x - __uint_as_float(m[e] << 16)), l1 = __float_as_uint(r.y - __uint_as_float(m[e] & kTop));
        l[e] = __builtin_amdgcn_perm(l1, l0, kHighHalves);
        lost |= l0 | l1;
        asm("" : "+v"(lost));                                   // now: gathered later, the l would be held till then
    }
    o[0] = __builtin_bit_cast(bf16x8, h);
    o[1] = __builtin_bit_cast(bf16x8, m);
    o[2] = __builtin_bit_cast(bf16x8, l);
}

// Two 32-row fragments of each operand: 16 k in fp32, and split.
struct RawFrags { float a[2][8], b[2][8]; };
struct SplitFrags { bf16x8 a[2][3], b[2][3]; };

__device__ __forceinline__ void split_frags(const RawFrags &x, SplitFrags &o, unsigned &lost) {
#pragma unroll
    for (int f = 0; f < 2; f++) split_bf16(x.a[f], o.a[f], lost);
#pragma unroll
    for (int f = 0; f < 2; f++) split_bf16(x.b[f], o.b[f], lost);
}

__device__ __forceinline__ void split_products(const SplitFrags &x, floatx16 (&acc)[2][2]) {
    constexpr int pa[6] = {2, 0, 1, 1, 0, 0}, pb[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
    for (int p = 0; p < 6; p++)
#pragma unroll
        for (int f = 0; f < 2; f++)
#pragma unroll
            for (int h = 0; h < 2; h++)
                acc[f][h] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x.a[f][pa[p]], x.b[h][pb[p]], acc[f][h], 0, 0, 0);
}

// A sum the bf16 products do not vouch for: not finite, or subnormal (its
// products' parts are below what fp32 sums hold).
__device__ __forceinline__ bool unsure(float s) {
    return __builtin_amdgcn_classf(s, 0x297);                   // NaN, infinity, subnormal
}

template <int F>
__device__ __forceinline__ void zero_acc(floatx16 (&acc)[F][F]) {
#pragma unroll
    for (int f = 0; f < F; f++)
#pragma unroll
        for (int h = 0; h < F; h++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[f][h][v] = 0.0f;
}

// This wave's loads have landed (vmcnt) and its LDS reads are done (lgkmcnt:
// their values may be used only later).
__device__ __forceinline__ void wait_loads_and_reads() {
    __builtin_amdgcn_s_waitcnt(7 << 4);                         // vmcnt(0) lgkmcnt(0)
    asm volatile("" ::: "memory");
}
__device__ __forceinline__ void wait_reads() {
    __builtin_amdgcn_s_waitcnt(15 | (3 << 14) | (7 << 4));      // lgkmcnt(0)
    asm volatile("" ::: "memory");
}
// The same for every wave of the block.
__device__ __forceinline__ void block_loads_and_reads() {
    wait_loads_and_reads();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// The T x T tile at (m0, n0) over k in [kb, kend) with fp32 MFMAs, on 2 x 2
// waves of T/2 x T/2: the cases above that bf16 products do not cover.  smem:
// 4*T*BK floats.
template <bool AK, bool BKM, int T, int E>
__device__ __forceinline__ void fp32_mma(const GemmArgs &g, int m0, int n0, int kb, int kend, float *smem,
                                         floatx16 (&acc)[T / 64][T / 64]) {
    constexpr int F = T / 64, STAGE = 2 * T * BK;
    using DA = TileDma<AK, T, BK, E, 4>;
    using DB = TileDma<BKM, T, BK, E, 4>;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave >> 1, wn = wave & 1, li = lane & 31, lh = lane >> 5;
    zero_acc<F>(acc);
    for (int k0 = kb; k0 < kend; k0 += BK) {
        DA da;
        DB db;
        da.init(g.lda, g.M, m0, wave, lane, kend - k0);
        db.init(g.ldb, g.N, n0, wave, lane, kend - k0);
        da.issue(g.A + (AK ? (long)k0 * g.lda + m0 : (long)m0 * g.lda + k0), 0x7fffffff, smem, wave);
        db.issue(g.B + (BKM ? (long)k0 * g.ldb + n0 : (long)n0 * g.ldb + k0), 0x7fffffff, smem + T * BK, wave);
        block_loads_and_reads();
        for (int q = 0; q < 2 && k0 + 16 * q < kend; q++) {     // uniform
            float xa[F][8], xb[F][8];
#pragma unroll
            for (int f = 0; f < F; f++) {
                DA::read(smem, wm * (T / 2) + f * 32 + li, q, lh, xa[f]);
                DB::read(smem + T * BK, wn * (T / 2) + f * 32 + li, q, lh, xb[f]);
            }
#pragma unroll
            for (int e = 0; e < 8; e++)
#pragma unroll
                for (int f = 0; f < F; f++)
#pragma unroll
                    for (int h = 0; h < F; h++)
                        acc[f][h] = __builtin_amdgcn_mfma_f32_32x32x2f32(xa[f][e], xb[h][e], acc[f][h], 0, 0, 0);
        }
        block_loads_and_reads();
    }
    static_assert(STAGE <= 4 * T * BK, "one stage");
}

// A bf16-product tile's output rows: C, or this split's partial product.  Plain
// sums are added and stored by buffer operations whose elements outside the
// output have an offset past the descriptor's range: no branch and no 64-bit
// address per element, and all of a lane's loads of C in flight together (one
// by one, each load, add and store waited for the one before).  Rows shorter
// than kMaxSplitLd keep the offsets below 2^31.  TN 32000x768x1024 with
// accumulate 342 -> 285 us, 17248x669x64 63 -> 31 (47 in 32x32 tiles), NT
// 1024x8192x64 17.5 -> 15.0 (fp32 128-wide tiles 16.7).
struct TileOut {
    __amdgpu_buffer_rsrc_t out, cin;
    bool add;
    int ld, rows, cols;                     // rows and columns left from the tile's first
    __device__ __forceinline__ TileOut(const GemmArgs &g, int m0, int n0, int z) {
        const bool part = g.partial != nullptr;
        add = !part && g.accumulate;
        ld = (int)(part ? g.N : g.ldc);
        rows = g.M - m0;
        cols = g.N - n0;
        const long at = (long)m0 * ld + n0;
        out = __builtin_amdgcn_make_buffer_rsrc((part ? g.partial + (long)z * g.M * g.N : g.C) + at, (short)0, 0x7fffffff, 0x00020000);
        cin = __builtin_amdgcn_make_buffer_rsrc((void *)((add ? g.Cin : g.C) + at), (short)0, 0x7fffffff, 0x00020000);
    }
    __device__ __forceinline__ int at(int r, int c) const { return r < rows && c < cols ? 4 * (r * ld + c) : kOutside; }
    // v[i] at offsets off[i]
    template <int N>
    __device__ __forceinline__ void put(const float (&v)[N], const int (&off)[N]) const {
        float c[N];
        if (add)                                                // uniform
#pragma unroll
            for (int i = 0; i < N; i++) c[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(cin, off[i], 0, 0));
#pragma unroll
        for (int i = 0; i < N; i++)
            __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, add ? c[i] + v[i] : v[i]), out, off[i], 0, 0);
    }
};

// 128x128 output tile at (m0, n0) over K range split z: 2 x 2 waves of
// 64x64, K steps of 32 in two LDS stages.  A wave's splits of one 16-k block
// go between its MFMAs of the block before; the next tile's loads are in
// flight meanwhile.  For outputs of many tiles and short K (gemm_split_tile), where
// the 64x64 tile's start and sum cost more than its lighter splits save: NT
// 1024x32000x768 474 -> 340 us (64x64 tiles 396), TN 32000x768x1024 528 -> 340.
template <bool AK, bool BKM, int E, int EPI>
__device__ __forceinline__ void gemm_tile_split128(const GemmArgs &g, int m0, int n0, int z) {
    constexpr int T = 128, STAGE = 2 * T * BK;
    using DA = TileDma<AK, T, BK, E, 4>;
    using DB = TileDma<BKM, T, BK, E, 4>;
    __shared__ __align__(16) float smem[2 * STAGE];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave >> 1, wn = wave & 1, li = lane & 31, lh = lane >> 5;
    const int kb = z * g.k_per_split, kend = min(g.K, kb + g.k_per_split);
    const int nk = kb < kend ? (kend - kb + BK - 1) / BK : 0;
    const float *A0 = g.A + (AK ? (long)kb * g.lda + m0 : (long)m0 * g.lda + kb);
    const float *B0 = g.B + (BKM ? (long)kb * g.ldb + n0 : (long)n0 * g.ldb + kb);
    const long stepA = AK ? BK * g.lda : BK, stepB = BKM ? BK * g.ldb : BK;
    DA da;
    DB db;
    auto place = [&](int krem) {
        da.init(g.lda, g.M, m0, wave, lane, krem);
        db.init(g.ldb, g.N, n0, wave, lane, krem);
    };
    auto issue = [&](int s) {
        if (s == nk - 1 && s > 0) place(kend - kb - s * BK);    // the last K step may be ragged
        float *st = smem + (s & 1) * STAGE;
        da.issue(A0 + s * stepA, 0x7fffffff, st, wave);
        db.issue(B0 + s * stepB, 0x7fffffff, st + T * BK, wave);
    };
    RawFrags x;
    auto read = [&](int s, int q) {
        const float *st = smem + (s & 1) * STAGE;
#pragma unroll
        for (int f = 0; f < 2; f++) DA::read(st, wm * 64 + f * 32 + li, q, lh, x.a[f]);
#pragma unroll
        for (int f = 0; f < 2; f++) DB::read(st + T * BK, wn * 64 + f * 32 + li, q, lh, x.b[f]);
    };
    floatx16 acc[2][2];
    zero_acc<2>(acc);
    unsigned lost = 0;
    if (nk > 0 && g.K >= kShortK) {                             // uniform
        SplitFrags s0, s1;
        place(min(BK, kend - kb));
        issue(0);
        block_loads_and_reads();
        if (nk > 1) issue(1);
        read(0, 0);
        split_frags(x, s0, lost);
        for (int s = 0; s < nk; s++) {
            read(s, 1);
            __builtin_amdgcn_sched_barrier(0);
            split_products(s0, acc);
            split_frags(x, s1, lost);
            __builtin_amdgcn_sched_barrier(0);
            if (s + 1 < nk) {
                // tile s+1 is in, and every wave has read tile s, whose
                // stage tile s+2 overwrites
                block_loads_and_reads();
                if (s + 2 < nk) issue(s + 2);
                read(s + 1, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
            split_products(s1, acc);
            split_frags(x, s0, lost);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    bool again = g.K < kShortK || (lost & 0xffffu) != 0;
#pragma unroll
    for (int f = 0; f < 2; f++)
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int v = 0; v < 16; v++) again |= unsure(acc[f][h][v]);
    if (__syncthreads_or(again)) fp32_mma<AK, BKM, T, E>(g, m0, n0, kb, kend, smem, acc);     // uniform
    // C[(v/4)*8 + 4*(l/32) + v%4][l%32] is component v of lane l
    const int rb = wm * 64 + 4 * lh, cb = wn * 64 + li;
    if constexpr (EPI == GEMM_EPI_NONE) {
        const TileOut o(g, m0, n0, z);
#pragma unroll
        for (int f = 0; f < 2; f++)
#pragma unroll
            for (int h = 0; h < 2; h++) {
                float s[16];
                int off[16];
#pragma unroll
                for (int v = 0; v < 16; v++) {
                    s[v] = acc[f][h][v];
                    off[v] = o.at(rb + f * 32 + (v >> 2) * 8 + (v & 3), cb + h * 32);
                }
                o.put(s, off);
            }
    } else {
#pragma unroll
        for (int f = 0; f < 2; f++)
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
                for (int v = 0; v < 16; v++)
                    store_elem<EPI>(g, acc[f][h][v], m0 + rb + f * 32 + (v >> 2) * 8 + (v & 3), n0 + cb + h * 32, z, 0.0f);
    }
}

// 64x64 output tile at (m0, n0) over K range split z, K dealt to the four waves:
// wave w takes the 16-k blocks w, w+4, ... of the whole tile, through two LDS
// stages of its own, and the four sums meet in LDS at the end.  So no barrier
// lies in the main loop, every element is split once per block (2 x 2 waves
// of 32x32 split each twice), and a lone block per CU keeps all four SIMDs
// on MFMAs with independent accumulators (as 2 x 2 waves a K step of 32
// takes 0.65-0.85 us there, here about 0.25).  A ragged last block comes first in
// its wave's order, so its offsets cost one more init and no extra wait.
// Measured (launches back to back; the 32x32 and 64x64 fp32 tiles before):
// NT 1024x2048x768 41.6 -> 24.9 us, NN 1024x768x2048 45.7 -> 27.1, TN
// 2048x768x1024 43.2 -> 27.0, NN 1024x768x32000 562 -> 291.  Three or four
// stages (one block per CU) and eight waves were slower except for a lone
// block per CU (27.1 -> 25.4 with eight waves).
template <bool AK, bool BKM, int E, int EPI>
__device__ __forceinline__ void gemm_tile_slice64(const GemmArgs &g, int m0, int n0, int z) {
    constexpr int T = 64, KD = 16, NS = 2, NW = 4, STAGE = 2 * T * KD;
    using DA = TileDma<AK, T, KD, E, 1>;
    using DB = TileDma<BKM, T, KD, E, 1>;
    constexpr int LPT = DA::N + DB::N;
    static_assert((NS - 1) * LPT < 64, "vmcnt");
    __shared__ __align__(16) float smem[NW * NS * STAGE];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int li = lane & 31, lh = lane >> 5;
    const int kb = z * g.k_per_split, kend = min(g.K, kb + g.k_per_split);
    const int nf = max(0, kend - kb) / KD, tail = max(0, kend - kb) % KD;     // whole blocks, ragged k
    const int first = tail > 0 && nf % NW == wave;               // 1: the ragged block is this wave's block 0
    const int n = first + (nf - wave + NW - 1) / NW;
    const float *A0 = g.A + (AK ? (long)kb * g.lda + m0 : (long)m0 * g.lda + kb);
    const float *B0 = g.B + (BKM ? (long)kb * g.ldb + n0 : (long)n0 * g.ldb + kb);
    const long stepA = AK ? KD * g.lda : KD, stepB = BKM ? KD * g.ldb : KD;
    float *ring = smem + wave * NS * STAGE;
    DA da;
    DB db;
    auto place = [&](int krem) {
        da.init(g.lda, g.M, m0, 0, lane, krem);
        db.init(g.ldb, g.N, n0, 0, lane, krem);
    };
    // this wave's block j (past its last: zeros) into its stage `st`
    auto issue = [&](int j, int st) {
        const bool in = j < n;
        const long c = !in ? 0 : first && j == 0 ? nf : (long)(j - first) * NW + wave;
        float *d = ring + st * STAGE;
        da.issue(A0 + c * stepA, in ? 0x7fffffff : 0, d, 0);
        db.issue(B0 + c * stepB, in ? 0x7fffffff : 0, d + T * KD, 0);
    };
    RawFrags x;
    auto read = [&](int st) {
        const float *p = ring + st * STAGE;
#pragma unroll
        for (int f = 0; f < 2; f++) DA::read(p, f * 32 + li, 0, lh, x.a[f]);
#pragma unroll
        for (int f = 0; f < 2; f++) DB::read(p + T * KD, f * 32 + li, 0, lh, x.b[f]);
    };
    floatx16 acc[2][2];
    zero_acc<2>(acc);
    unsigned lost = 0;
    if (n > 0 && g.K >= kShortK) {                              // wave-uniform
        SplitFrags s0, s1;
        if (first) place(tail);
        else place(KD);
        issue(0, 0);
        if (first) place(KD);
        issue(1, 1);
        wait_vmcnt<LPT>();
        asm volatile("" ::: "memory");
        read(0);
        split_frags(x, s0, lost);
        wait_reads();
        issue(2, 0);
        for (int j = 0; j < n; j += 2) {
            // blocks j+1 and j+2 are in flight, s0 holds block j's parts
            wait_vmcnt<LPT>();
            asm volatile("" ::: "memory");
            read(1);
            __builtin_amdgcn_sched_barrier(0);
            split_products(s0, acc);
            split_frags(x, s1, lost);
            __builtin_amdgcn_sched_barrier(0);
            wait_reads();
            issue(j + 3, 1);
            wait_vmcnt<LPT>();
            asm volatile("" ::: "memory");
            read(0);
            __builtin_amdgcn_sched_barrier(0);
            split_products(s1, acc);
            split_frags(x, s0, lost);
            __builtin_amdgcn_sched_barrier(0);
            wait_reads();
            issue(j + 4, 0);
        }
    }
    block_loads_and_reads();                                    // the rings are free
    // C[(v/4)*8 + 4*lh + v%4][l%32] is component v; columns of rows with bit
    // 2 set are flipped by 32 (the two lane halves then use different banks)
    float *const red = smem;
#pragma unroll
    for (int f = 0; f < 2; f++)
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int v = 0; v < 16; v++)
                red[(wave * T + f * 32 + (v >> 2) * 8 + 4 * lh + (v & 3)) * T + ((h * 32 + li) ^ (lh << 5))] = acc[f][h][v];
    __syncthreads();
    // wave w sums rows w, w+4, ...; lane = column
    float sum[T / NW];
    bool again = g.K < kShortK || (lost & 0xffffu) != 0;
#pragma unroll
    for (int e = 0; e < T / NW; e++) {
        const float *p = red + (e * NW + wave) * T + (lane ^ ((e & 1) << 5));      // row bit 2 = bit 0 of e
        sum[e] = ((p[0] + p[T * T]) + p[2 * T * T]) + p[3 * T * T];
        again |= unsure(sum[e]);
    }
    if (__syncthreads_or(again)) {                            // uniform
        floatx16 fa[1][1];
        fp32_mma<AK, BKM, T, E>(g, m0, n0, kb, kend, smem, fa);
#pragma unroll
        for (int v = 0; v < 16; v++)
            red[((wave >> 1) * 32 + (v >> 2) * 8 + 4 * lh + (v & 3)) * T + (wave & 1) * 32 + li] = fa[0][0][v];
        __syncthreads();
#pragma unroll
        for (int e = 0; e < T / NW; e++) sum[e] = red[(e * NW + wave) * T + lane];
    }
    if constexpr (EPI == GEMM_EPI_NONE) {
        const TileOut o(g, m0, n0, z);
        int off[T / NW];
#pragma unroll
        for (int e = 0; e < T / NW; e++) off[e] = o.at(e * NW + wave, lane);
        o.put(sum, off);
        if (!g.upd) return;                                     // uniform
        // sgd_step (pt_train.c:870-873) on the weight this gradient belongs to, rows not kept
        const float lrv = *g.lr;
        const __amdgpu_buffer_rsrc_t upd = __builtin_amdgcn_make_buffer_rsrc(g.upd + (long)m0 * g.ldc + n0, (short)0, 0x7fffffff, 0x00020000);
        float w[T / NW];
#pragma unroll
        for (int e = 0; e < T / NW; e++) {
            const int m = min(m0 + e * NW + wave, g.M - 1);
            if (g.keep && ((g.keep[m >> 5] >> (m & 31)) & 1u)) off[e] = kOutside;
            w[e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(upd, off[e], 0, 0));
        }
#pragma unroll
        for (int e = 0; e < T / NW; e++)
            __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, w[e] - lrv * sum[e]), upd, off[e], 0, 0);
    } else {
#pragma unroll
        for (int e = 0; e < T / NW; e++) store_elem<EPI>(g, sum[e], m0 + e * NW + wave, n0 + lane, z, 0.0f);
    }
}

// Workgroups go to the 8 XCDs round-robin by linear id, and each XCD has its
// own L2.  Block b runs tile xcd_tile(b): XCD c gets the c-th contiguous
// range of the tiles, in order, so tiles that read the same operand tile
// run together on one XCD and fetch it into that L2 once.
__device__ __forceinline__ int xcd_tile(int b, int total) {
    const int q = total >> 3, r = total & 7, c = b & 7;
    return c * q + min(c, r) + (b >> 3);
}

// Grids of kXcdGrid blocks and more take tiles in xcd_tile order: split
// index slowest; within a split, neighbouring tiles share the tile of the
// larger operand (A's rows when M > N, else B's columns).  Smaller grids
// (at most a few blocks per CU, no reuse to gain) keep the grid's order.
// The bound of two waves per SIMD keeps the chains (NN and NT) in VGPRs: in
// AGPRs the register allocator moved all eight of them on every K step
// (36 moves and 9 waits per two steps; NT 77x496x448 7.45 -> 6.56 us, 6.46 with
// one chain; 77 NN and NT shapes on these tiles 0.940 -> 0.990 of one chain's
// speed, the rest is the chains' sum).  TN, with one chain, is level in either.
template <bool AT, bool BT, int TM, int TN, int P, bool VEC, int EPI = GEMM_EPI_NONE, int NORM = 0>
__global__ __launch_bounds__(256, AT ? 1 : 2) void k_gemm(GemmArgs g) {
    const int gx = gridDim.x, gy = gridDim.y, per_z = gx * gy, total = per_z * gridDim.z;
    int m = blockIdx.y, n = blockIdx.x, z = blockIdx.z;
    if (total >= kXcdGrid) {                                        // uniform
        const int t = xcd_tile(blockIdx.x + gx * (blockIdx.y + gy * blockIdx.z), total);
        z = t / per_z;
        const int u = t - z * per_z;
        if (g.M > g.N) m = u / gx, n = u - m * gx;
        else n = u / gy, m = u - n * gy;
    }
    gemm_tile<AT, BT, TM, TN, P, VEC, EPI, NORM>(g, m * TM, n * TN, z);
}

// The direct-to-LDS GEMM (grid and tile order as k_gemm).
template <int TM, int TN, int WM, int WN>
__global__ __launch_bounds__(64 * WM * WN) void k_gemm_dl(GemmArgs g) {
    const int gx = gridDim.x, gy = gridDim.y, per_z = gx * gy, total = per_z * gridDim.z;
    int m = blockIdx.y, n = blockIdx.x, z = blockIdx.z;
    if (total >= kXcdGrid) {                                        // uniform
        const int t = xcd_tile(blockIdx.x + gx * (blockIdx.y + gy * blockIdx.z), total);
        z = t / per_z;
        const int u = t - z * per_z;
        if (g.M > g.N) m = u / gx, n = u - m * gx;
        else n = u / gy, m = u - n * gy;
    }
    gemm_tile_dl<TM, TN, WM, WN>(g, m * TM, n * TN, z);
}

// The per-layer panel GEMM (grid, tile order and register bound as k_gemm).
template <bool BKM, int NSK, int EPI>
__global__ __launch_bounds__(256, 2) void k_gemm_panel(GemmArgs g) {
    const int gx = gridDim.x, gy = gridDim.y, per_z = gx * gy, total = per_z * gridDim.z;
    int m = blockIdx.y, n = blockIdx.x, z = blockIdx.z;
    if (total >= kXcdGrid) {                                        // uniform
        const int t = xcd_tile(blockIdx.x + gx * (blockIdx.y + gy * blockIdx.z), total);
        z = t / per_z;
        const int u = t - z * per_z;
        if (g.M > g.N) m = u / gx, n = u - m * gx;
        else n = u / gy, m = u - n * gy;
    }
    gemm_tile_panel<BKM, NSK, EPI>(g, m * 32, n * 32, z);
}

// The bf16-product GEMMs (grid of T x T tiles, T = 64 or 128; tile order as k_gemm).
template <bool AK, bool BKM, int T, int E, int EPI>
__global__ __launch_bounds__(256, 2) void k_gemm_split(GemmArgs g) {
    const int gx = gridDim.x, gy = gridDim.y, per_z = gx * gy, total = per_z * gridDim.z;
    const int t = xcd_tile(blockIdx.x + gx * (blockIdx.y + gy * blockIdx.z), total);
    const int z = t / per_z, u = t - z * per_z;
    int m, n;
    if (g.M > g.N) m = u / gx, n = u - m * gx;
    else n = u / gy, m = u - n * gy;
    if constexpr (T == 128) gemm_tile_split128<AK, BKM, E, EPI>(g, m * T, n * T, z);
    else gemm_tile_slice64<AK, BKM, E, EPI>(g, m * T, n * T, z);
}

// Grouped TN GEMMs (whole K): block b runs tile t = xcd_tile(b) - d.tile0 of
// the descriptor d whose tile range holds it.  The launch covers entries
// [i0, i1) of the table, whose tiles start at d[i0].tile0 (a tile's result
// does not depend on the block that computes it, so a launch of a sub-range
// gives the same bits as the whole table).
__device__ __forceinline__ const GemmGroupDesc &group_tile(const GemmGroupDesc *d, int i0, int i1, int &t) {
    const int b = d[i0].tile0 + xcd_tile(blockIdx.x, gridDim.x);
    int i = i0;
    while (i + 1 < i1 && d[i + 1].tile0 <= b) i++;
    t = b - d[i].tile0;
    return d[i];
}
// 32x32 fp32 tiles; they run along N first, so neighbours share the A^T tile.
template <int TM, int TN, bool VEC>
__global__ __launch_bounds__(256) void k_gemm_tn_group(const GemmGroupDesc *d, int i0, int i1) {
    int t;
    const GemmGroupDesc &e = group_tile(d, i0, i1, t);
    gemm_tile<true, false, TM, TN, kRing32, VEC>(e.g, (t / e.tiles_n) * TM, (t % e.tiles_n) * TN, 0);
}
// 64x64 tiles of bf16 products; neighbours share the tile of the larger operand.
template <int E>
__global__ __launch_bounds__(256, 2) void k_gemm_tn_group_split(const GemmGroupDesc *d, int i0, int i1) {
    int t;
    const GemmGroupDesc &e = group_tile(d, i0, i1, t);
    const int gx = e.tiles_n, gy = (e.g.M + 63) / 64;
    int m, n;
    if (e.g.M > e.g.N) m = t / gx, n = t - m * gx;
    else n = t / gy, m = t - n * gy;
    gemm_tile_slice64<true, true, E, GEMM_EPI_NONE>(e.g, m * 64, n * 64, 0);
}

// C = (Cin +) sum_z partial[z], z ascending.
__global__ __launch_bounds__(256) void k_splitk_reduce(const float *partial, int splits, float *C, const float *Cin,
                                                       long ldc, int M, int N, int accumulate) {
    const long idx = (long)blockIdx.x * 256 + threadIdx.x;
    if (idx >= (long)M * N) return;
    const int m = (int)(idx / N), n = (int)(idx % N);
    const float s = sum_splits(partial, splits, (long)M * N, idx);
    const long o = (long)m * ldc + n;
    C[o] = accumulate ? Cin[o] + s : s;
}

inline bool al16(const void *p) { return ((uintptr_t)p & 15u) == 0; }

constexpr size_t kScratchFloats = (size_t)4 << 20;      // split-K partials of ptmi_gemm_dev_noalloc

// How many splits the fp32 tiles take: 32x32 tiles with K cut into whole
// steps of at least eight per split where the grid is small.  K >= 4096 counts
// 64x64 tiles and splits to 1024 blocks (the count ptmi_gemm_dev_noalloc
// admits calls by, and the one split sums are held against).  `chosen` splits
// fit the workspace; cutting K into whole steps gives `splits` (<= chosen).
struct SplitPlan { int chosen, splits, k_per_split; };
SplitPlan split_plan(int op, int M, int N, int K, size_t ws_floats, int ek) {
    if (ek != GEMM_EPI_NONE) return SplitPlan{1, 1, K};          // the epilogue needs whole-K sums
    const bool big = K >= 4096 || (op == 2 && (long)M * N >= (4L << 20));
    const int T = big ? 64 : 32;
    const long blocks = (long)((N + T - 1) / T) * ((M + T - 1) / T);
    const int nk = (K + BK - 1) / BK;
    int splits = 1;
    if (big && K >= 4096 && blocks < 512) splits = (int)std::min<long>((1024 + blocks - 1) / blocks, nk / 8);
    else if (!big && blocks < 128 && nk > 9) splits = std::min(8, nk / 8);
    while (splits > 1 && (size_t)splits * M * N > ws_floats) splits--;
    const int chosen = std::max(1, splits);
    const int kps = ((K + chosen - 1) / chosen + BK - 1) / BK * BK;
    return SplitPlan{chosen, (K + kps - 1) / kps, kps};
}

// Kernel and K split of a GEMM.  GEMM_32: 32x32 fp32 MFMA tiles, K split by
// split_plan; GEMM_64 and GEMM_128: bf16 products, the smaller estimate of a launch's
// time in us, fitted to 1850 launches back to back on the MI355X (256 CUs;
// n = blocks per CU; measured -> estimated; over those the choice takes 0.4%
// longer than the fastest of the three would):
//   GEMM_32:  3.2 + i * (n - 1) + steps * (0.1 + s * n), n >= 1, steps of 32 k; i, s =
//        0.4, 0.18 NT, 0.3, 0.19 NN, 0.2, 0.19 TN: NT 827x1600x376 16.9 -> 16.9,
//        NN 1024x4096x64 13.7 -> 14.0, TN 1184x2000x176 15.1 -> 15.7, 36x160x6725 10.1 -> 10.3
//   GEMM_64:  3.6 + ceil(n) * (1.85 + 0.65 * steps), at least two steps of 64 k:
//        131x960x896 10.8 -> 11.3 (split), 1024x2048x768 25.1 -> 22.9, 423x3808x1408 34.5 -> 35.9
//   GEMM_128: 3.2 + ceil(n) * (2.8 + 1.3 * steps), n >= 1, steps of 32 k, 2.0 each at
//        n = 1 (a lone block per CU): 1024x8192x64 15.0 -> 14.0, 1024x32000x768 265 -> 275,
//        1024x4096x96 12.3 -> 12.0
//   split K: + 3 and the partials' traffic at 3.5 TB/s.
// Without 16-byte rows the 32 tiles' loads cost 1.5x per step, the others' 1.2x
// (501x517x1003: 24.6 against 16.1 us with three splits).  The bf16 tiles keep
// their partial sums at most as long as the fp32 tiles' would be (the 64
// tile sums four of its own), so no result is summed in fewer pieces.
// Two fp32 tiles stay where they are faster than all three:
//   GEMM_DL (128x96, direct to LDS): TN outputs of 4 Mi elements and more, one
//        K step and no accumulate: 32000x288x16 14.4 us against 15.6 (GEMM_128); with
//        accumulate 4096x1100x16 16.8 against 11.5, at K = 48 20.6 against 19.4.
//   GEMM_64F (64x64): NT outputs of that size from at most 64 rows, which leave half
//        of a 128 tile empty, K <= 96: 64x65600x20 10.3 against 13.9 (14.2, GEMM_32),
//        at K = 96 16.9 against 18.0, at K = 128 19.4 against 19.3 (GEMM_64).
enum GemmKind { GEMM_32, GEMM_64F, GEMM_DL, GEMM_64, GEMM_128 };
struct GemmChoice {
    GemmKind kind;
    int tm, tn, splits, k_per_split;
    float us, us32;                                             // its estimate and the 32 tiles'
};
GemmChoice gemm_choice(int op, int M, int N, int K, long lda, long ldb, long ldc, bool vec, bool accumulate,
                       size_t ws_floats, int ek) {
    const SplitPlan p = split_plan(op, M, N, K, ws_floats, ek);
    const double mn = (double)M * N, cus = 256.0;
    auto blocks = [&](int T) { return (double)((N + T - 1) / T) * ((M + T - 1) / T); };
    auto reduce = [&](int s) { return s > 1 ? 3.0 + (s + 1) * mn * 4.0 / 3.5e6 : 0.0; };
    auto steps = [&](int k, int per) { return (double)((k + per - 1) / per); };
    const double fill[3] = {0.3, 0.2, 0.4}, per_step[3] = {0.19, 0.19, 0.18};
    const double n32 = std::max(1.0, blocks(32) * p.splits / cus);
    const double us32 = 3.2 + fill[op] * (n32 - 1) + reduce(p.splits) +
                        (vec ? 1.0 : 1.5) * steps(p.k_per_split, BK) * (0.1 + per_step[op] * n32);
    GemmChoice best = {GEMM_32, 32, 32, p.splits, p.k_per_split, (float)us32, (float)us32};
    const bool large = mn >= (4L << 20), split_ok = std::max({lda, ldb, ldc}) < kMaxSplitLd;
    if (ek == GEMM_EPI_NONE && op == 1 && vec && p.splits == 1 && large && (!split_ok || (K < 48 && !accumulate)))
        return GemmChoice{GEMM_DL, 128, 96, 1, K, (float)us32, (float)us32};
    if (ek == GEMM_EPI_NONE && op == 2 && large && M <= 64 && K <= 96)
        return GemmChoice{GEMM_64F, 64, 64, 1, K, (float)us32, (float)us32};
    if (!split_ok || (ek != GEMM_EPI_NONE && !vec)) return best;
    if (us32 < 7.0) return best;                                 // below any of the others
    const int max_s = ek != GEMM_EPI_NONE ? 1 : std::max(1, std::min(64, K / 128));
    for (int s = 1; s <= max_s; s += 1 + s / 8) {
        const double red = reduce(s);
        if (s > 1 && ((size_t)s * M * N > std::min(ws_floats, kScratchFloats) || 6.7 + red > best.us)) break;
        const int kps = ((K + s - 1) / s + BK - 1) / BK * BK, splits = (K + kps - 1) / kps;
        for (int T = 64; T <= 128; T += 64) {
            if (kps > (T == 64 ? 4 : 1) * p.k_per_split) continue;
            const double n = blocks(T) * splits / cus;
            // (RoPE's N is 3K: there 128x128 would lead, by 5%, only from 2048 rows of 2048-wide models)
            if (T == 128 && (n < 1.0 || ek == GEMM_EPI_ROPE)) continue;
            const double per = T == 64 ? 1.85 + 0.65 * std::max(2.0, steps(kps, 64)) : 2.8 + (n > 1.0 ? 1.3 : 2.0) * steps(kps, BK);
            const double us = (T == 64 ? 3.6 : 3.2) + (vec ? 1.0 : 1.2) * std::ceil(n) * per + red;
            if (us < best.us)
                best = GemmChoice{T == 64 ? GEMM_64 : GEMM_128, T, T, splits, splits > 1 ? kps : K, (float)us, (float)us32};
        }
    }
    return best;
}

}  // namespace

bool gemm_norm_fusable(int M, int N, int K, const float *A, long lda, const float *B, long ldb, int epi_kind,
                       const GemmNorm &nm) {
    if (nm.kind < GEMM_NORM_PLAIN || nm.kind > GEMM_NORM_EMBED || !nm.w || !nm.xn_out) return false;
    if (epi_kind != GEMM_EPI_ROPE && epi_kind != GEMM_EPI_SWIGLU) return false;
    if (M <= 0 || N <= 0 || K <= 0 || K % 4 || lda != K || ldb % 4 || ldb < K) return false;
    if (!A || !B || !al16(A) || !al16(B) || !al16(nm.w) || !al16(nm.xn_out)) return false;
    // the fused norm runs on the 32x32 tiles only, and spares a launch (about 5 us)
    const GemmChoice ch = gemm_choice(2, M, N, K, lda, ldb, N, true, false, 0, epi_kind);
    if (ch.kind != GEMM_32 && ch.us + 5.0f < ch.us32) return false;
    if (nm.kind != GEMM_NORM_PLAIN && (!nm.x_out || !al16(nm.x_out))) return false;
    if (nm.kind == GEMM_NORM_SPLITS &&
        (nm.pk.splits < 1 || nm.pk.splits > kNormSplits || !nm.pk.parts || !al16(nm.pk.parts) || nm.pk.stride % 4 ||
         nm.pk.stride < (long)M * K || (nm.cin && !al16(nm.cin))))
        return false;
    if (nm.kind == GEMM_NORM_EMBED && (!nm.tok || !nm.emb || !nm.tok_bits || !al16(nm.emb))) return false;
    return true;
}

size_t gemm_workspace_floats(int op, int M, int N, int K, size_t ws_floats) {
    if (M <= 0 || N <= 0 || K <= 0) return 0;
    const SplitPlan p = split_plan(op, M, N, K, ws_floats, GEMM_EPI_NONE);
    return p.chosen > 1 ? (size_t)p.chosen * M * N : 0;
}

// Launch op(A).op(B) with shapes validated; `ws` (optional) is a split-K
// workspace of ws_floats floats.
int launch_gemm(int op, const float *A, long lda, const float *B, long ldb, float *C, long ldc, int M, int N,
                int K, int accumulate, float *ws, size_t ws_floats, hipStream_t s, const float *Cin, SplitK *defer,
                const GemmEpi *epi, const GemmNorm *norm) {
    if (defer) *defer = SplitK{nullptr, 0, 0};
    const int ek = epi ? epi->kind : GEMM_EPI_NONE;
    const int nk_kind = norm ? norm->kind : 0;
    if (nk_kind && (op != 2 || accumulate || !gemm_norm_fusable(M, N, K, A, lda, B, ldb, ek, *norm)))
        return set_error(PTMI_ERR_ARG, "gemm: the fused norm does not fit this GEMM");
    if (ek == GEMM_EPI_SWIGLU_BWD ? (op != 0 || !epi->out || !epi->out2 || !epi->aux)
                                  : ek != GEMM_EPI_NONE && (op != 2 || N % 2 || (ek == GEMM_EPI_SWIGLU && !epi->out) ||
                                                            (ek == GEMM_EPI_ROPE &&
                                                             (epi->rope_dim % 2 || epi->head_dim <= 0 || epi->col0 % 2 ||
                                                              (epi->out && (!epi->out2 || N + epi->col0 != 3 * epi->rope_dim))))))
        return set_error(PTMI_ERR_ARG, "gemm: fused epilogue %d does not fit this GEMM", ek);
    if (M <= 0 || N <= 0 || K <= 0) return set_error(PTMI_ERR_ARG, "gemm: M=%d N=%d K=%d", M, N, K);
    if (!A || !B || !C) return set_error(PTMI_ERR_ARG, "gemm: null operand");
    if (op < 0 || op > 2) return set_error(PTMI_ERR_ARG, "gemm: op %d", op);
    const bool AT = op == 1, BT = op == 2;
    // minimum leading dimensions
    if ((AT ? lda < M : lda < K) || (BT ? ldb < K : ldb < N) || ldc < N)
        return set_error(PTMI_ERR_ARG, "gemm: leading dimension too small");
    GemmArgs g;
    g.A = A; g.lda = lda; g.B = B; g.ldb = ldb; g.C = C; g.ldc = ldc;
    g.M = M; g.N = N; g.K = K; g.accumulate = accumulate;
    g.Cin = Cin ? Cin : C;
    g.upd = nullptr; g.lr = nullptr; g.keep = nullptr;
    // float4 loads when both operands have aligned rows and a contiguous
    // extent that is a multiple of 4 (M for A^T, K for A; K for B^T, N for B)
    const bool vec = al16(A) && lda % 4 == 0 && (AT ? M : K) % 4 == 0 && al16(B) && ldb % 4 == 0 &&
                     (BT ? K : N) % 4 == 0;
    // Kernel choice.  Small GEMMs are bound by the latency of their K steps
    // and stay on 32x32 tiles (split_plan cuts K at about eight K steps per split:
    // K=768: 3 splits, K=1536: 6; with the panel kernel taking up to 9 K
    // steps at once, eight per split ran the stories15M T=256 step in
    // 0.769-0.771 ms against 0.778-0.783 with six, and nine and ten were no
    // faster); larger ones take the bf16-product tiles (gemm_choice).  The
    // fused norm runs on the 32x32 tiles.
    GemmChoice ch = gemm_choice(op, M, N, K, lda, ldb, ldc, vec, accumulate, ws_floats, ek);
    if (nk_kind && ch.kind != GEMM_32) ch = GemmChoice{GEMM_32, 32, 32, 1, K, ch.us32, ch.us32};
    const int gx = (N + ch.tn - 1) / ch.tn, gy = (M + ch.tm - 1) / ch.tm;
    const int splits = ch.splits;
    g.k_per_split = ch.k_per_split;
    g.partial = splits > 1 ? ws : nullptr;
    g.epi = epi ? *epi : GemmEpi{};
    g.nrm = norm ? *norm : GemmNorm{};
    // The grid holds 65535 tiles along M.  More rows than 65535 tiles of split_plan's are
    // refused; where its tiles are 64 rows and the choice's 32, they go in two parts.
    const int plan_rows = K >= 4096 || (op == 2 && (long)M * N >= (4L << 20)) ? 64 : 32;
    if ((M + plan_rows - 1) / plan_rows > 65535) return set_error(PTMI_ERR_ARG, "gemm: M too large");
    if (gy > 65535) {
        if (ek != GEMM_EPI_NONE || defer) return set_error(PTMI_ERR_ARG, "gemm: M too large");
        const int rows = 65535 * ch.tm;
        const int st = launch_gemm(op, A, lda, B, ldb, C, ldc, rows, N, K, accumulate, ws, ws_floats, s, Cin);
        if (st) return st;
        return launch_gemm(op, A + (AT ? (long)rows : (long)rows * lda), lda, B, ldb, C + (long)rows * ldc, ldc, M - rows, N, K,
                           accumulate, ws, ws_floats, s, Cin ? Cin + (long)rows * ldc : nullptr);
    }
    dim3 grid(gx, gy, splits);
    using KFn = void (*)(GemmArgs);
    static const KFn kernels[2][3] = {
        {k_gemm<false, false, 32, 32, kRing32, false>, k_gemm<true, false, 32, 32, kRing32, false>,
         k_gemm<false, true, 32, 32, kRing32, false>},
        {k_gemm<false, false, 32, 32, kRing32, true>, k_gemm<true, false, 32, 32, kRing32, true>,
         k_gemm<false, true, 32, 32, kRing32, true>}};
    KFn fn = kernels[vec][op];
    if (ek != GEMM_EPI_NONE) {
        static const KFn fused[2][2] = {
            {k_gemm<false, true, 32, 32, kRing32, false, GEMM_EPI_ROPE>, k_gemm<false, true, 32, 32, kRing32, true, GEMM_EPI_ROPE>},
            {k_gemm<false, true, 32, 32, kRing32, false, GEMM_EPI_SWIGLU>, k_gemm<false, true, 32, 32, kRing32, true, GEMM_EPI_SWIGLU>}};
        static const KFn fused_nn[2] = {k_gemm<false, false, 32, 32, kRing32, false, GEMM_EPI_SWIGLU_BWD>,
                                        k_gemm<false, false, 32, 32, kRing32, true, GEMM_EPI_SWIGLU_BWD>};
        fn = ek == GEMM_EPI_SWIGLU_BWD ? fused_nn[vec] : fused[ek == GEMM_EPI_SWIGLU][vec];
    }
    if (nk_kind) {                                       // fusable: 32x32 float4 tiles, whole K
        static const KFn fused_norm[2][3] = {
            {k_gemm<false, true, 32, 32, kRing32, true, GEMM_EPI_ROPE, GEMM_NORM_PLAIN>,
             k_gemm<false, true, 32, 32, kRing32, true, GEMM_EPI_ROPE, GEMM_NORM_SPLITS>,
             k_gemm<false, true, 32, 32, kRing32, true, GEMM_EPI_ROPE, GEMM_NORM_EMBED>},
            {k_gemm<false, true, 32, 32, kRing32, true, GEMM_EPI_SWIGLU, GEMM_NORM_PLAIN>,
             k_gemm<false, true, 32, 32, kRing32, true, GEMM_EPI_SWIGLU, GEMM_NORM_SPLITS>,
             k_gemm<false, true, 32, 32, kRing32, true, GEMM_EPI_SWIGLU, GEMM_NORM_EMBED>}};
        if (!vec || splits != 1) return set_error(PTMI_ERR_STATE, "gemm: fused norm without whole-K float4 tiles");
        fn = fused_norm[ek == GEMM_EPI_SWIGLU][nk_kind - 1];
    }
    const bool split = ch.kind == GEMM_64 || ch.kind == GEMM_128;
    if (split) {
#define PTMI_SPLIT_KERNELS(T_)                                                                                        \
    {{k_gemm_split<false, true, T_, 1, 0>, k_gemm_split<true, true, T_, 1, 0>, k_gemm_split<false, false, T_, 1, 0>}, \
     {k_gemm_split<false, true, T_, 4, 0>, k_gemm_split<true, true, T_, 4, 0>, k_gemm_split<false, false, T_, 4, 0>}}
        static const KFn plain[2][2][3] = {PTMI_SPLIT_KERNELS(64), PTMI_SPLIT_KERNELS(128)};
#undef PTMI_SPLIT_KERNELS
        static const KFn fused[2][3] = {                 // by epilogue kind - 1
            {k_gemm_split<false, false, 64, 4, GEMM_EPI_ROPE>, k_gemm_split<false, false, 64, 4, GEMM_EPI_SWIGLU>,
             k_gemm_split<false, true, 64, 4, GEMM_EPI_SWIGLU_BWD>},
            {nullptr, k_gemm_split<false, false, 128, 4, GEMM_EPI_SWIGLU>,
             k_gemm_split<false, true, 128, 4, GEMM_EPI_SWIGLU_BWD>}};
        const int big = ch.kind == GEMM_128;
        fn = ek != GEMM_EPI_NONE ? fused[big][ek - 1] : plain[big][vec][op];
    }
    // Per-layer 32x32 GEMMs with at most 9 K tiles per split: the panel
    // kernel, every K tile in flight at once.  PTMI_GEMM_PANEL is a bit mask
    // of the GEMMs that take it: 1 NT, 2 NN with the SwiGLU backward
    // epilogue, 4 the other NN (default 3).  Measured in the stories15M T=256
    // training step (kernel µs per step, eager trace): NT Wo + w2 72.8 ->
    // 70.4, QKV 37.8 -> 37.0, d_sh 45.2 -> 40.2; the split-K NN (w1|w3 and
    // QKV dX) 82.0 -> 90.9, so those keep the ring.  Graph-mode step
    // 0.780-0.785 ms against 0.787-0.796 (mask 0) and 0.790-0.795 (mask 7).
    static const int use_panel = [] { const char *e = getenv("PTMI_GEMM_PANEL"); return e ? atoi(e) & 7 : 3; }();
    const int nk_split = (ch.k_per_split + BK - 1) / BK;
    const int panel_bit = op == 2 ? 1 : ek == GEMM_EPI_SWIGLU_BWD ? 2 : 4;
    if ((use_panel & panel_bit) && ch.kind == GEMM_32 && vec && !nk_kind && op != 1 && nk_split <= 9) {
        using PFn = void (*)(GemmArgs);
        static const PFn panel[2][2][4] = {
            {{k_gemm_panel<false, 6, GEMM_EPI_NONE>, k_gemm_panel<false, 6, GEMM_EPI_ROPE>,
              k_gemm_panel<false, 6, GEMM_EPI_SWIGLU>, nullptr},
             {k_gemm_panel<false, 9, GEMM_EPI_NONE>, k_gemm_panel<false, 9, GEMM_EPI_ROPE>,
              k_gemm_panel<false, 9, GEMM_EPI_SWIGLU>, nullptr}},
            {{k_gemm_panel<true, 6, GEMM_EPI_NONE>, nullptr, nullptr, k_gemm_panel<true, 6, GEMM_EPI_SWIGLU_BWD>},
             {k_gemm_panel<true, 9, GEMM_EPI_NONE>, nullptr, nullptr, k_gemm_panel<true, 9, GEMM_EPI_SWIGLU_BWD>}}};
        const int ei = ek == GEMM_EPI_NONE ? 0 : ek == GEMM_EPI_ROPE ? 1 : ek == GEMM_EPI_SWIGLU ? 2 : 3;
        const PFn pf = panel[op == 0][nk_split > 6][ei];
        if (pf) fn = pf;
    }
    if (ch.kind == GEMM_64F) fn = vec ? k_gemm<false, true, 64, 64, kRing32, true> : k_gemm<false, true, 64, 64, kRing32, false>;
    if (ch.kind == GEMM_DL) fn = k_gemm_dl<128, 96, 4, 2>;
    hipLaunchKernelGGL(fn, grid, dim3(ch.kind == GEMM_DL ? 512 : 256), 0, s, g);
    PTMI_HIP(hipGetLastError());
    if (splits > 1 && defer) {
        *defer = SplitK{ws, splits, (long)M * N};
    } else if (splits > 1) {
        const long n = (long)M * N;
        hipLaunchKernelGGL(k_splitk_reduce, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, ws, splits, C, g.Cin,
                           ldc, M, N, accumulate);
        PTMI_HIP(hipGetLastError());
    }
    return PTMI_OK;
}

size_t gemm_group_desc_bytes(int n) { return sizeof(GemmGroupDesc) * (size_t)n; }

int gemm_tn_group_prepare(const TnGemm *list, int n, const float *lr, void *host_desc, TnGroupPlan *plan) {
    GemmGroupDesc *d = static_cast<GemmGroupDesc *>(host_desc);
    int vec = 1;
    // Tile: the smaller estimate over all entries.  The 64 tiles' counts 3.4 us more per
    // tile than gemm_choice's for the weights' update, which the many 32x32 blocks hide
    // behind each other's products.  Whole training steps with 32 / 64 tiles, us:
    // stories110M T=256 3315 / 3536, T=384 4206 / 4231, T=512 5079 / 4917, T=1024 8784 /
    // 7870; stories42M T=512 2322 / 2307; 252-wide, 7 layers, T=400 829 / 827, T=700 1070 / 1043.
    double us32 = 3.2, us64 = 3.6;
    bool fits = true;
    for (int i = 0; i < n; i++) {
        const TnGemm &e = list[i];
        auto blocks = [&](int T) { return (double)((e.M + T - 1) / T) * ((e.N + T - 1) / T); };
        us32 += (e.K + BK - 1) / BK * 0.19 * blocks(32) / 256.0;
        us64 += (6.0 + 0.65 * ((e.K + 63) / 64)) * blocks(64) / 256.0;
        fits = fits && std::max({e.lda, e.ldb, e.ldc}) < kMaxSplitLd;
    }
    const int tile = fits && us64 < us32 ? 64 : 32;
    int t = 0;
    for (int i = 0; i < n; i++) {
        const TnGemm &e = list[i];
        if (e.M <= 0 || e.N <= 0 || e.K <= 0 || !e.A || !e.B || !e.C || e.lda < e.M || e.ldb < e.N || e.ldc < e.N)
            return set_error(PTMI_ERR_ARG, "grouped gemm %d: bad shape", i);
        GemmArgs &g = d[i].g;
        g = GemmArgs{};
        g.A = e.A; g.lda = e.lda; g.B = e.B; g.ldb = e.ldb; g.C = e.C; g.ldc = e.ldc; g.Cin = e.C;
        g.M = e.M; g.N = e.N; g.K = e.K; g.accumulate = 0; g.partial = nullptr; g.k_per_split = e.K;
        if (e.upd && !lr) return set_error(PTMI_ERR_ARG, "grouped gemm %d: update without a learning rate", i);
        g.upd = e.upd; g.lr = lr; g.keep = e.keep;
        if (!(al16(e.A) && e.lda % 4 == 0 && e.M % 4 == 0 && al16(e.B) && e.ldb % 4 == 0 && e.N % 4 == 0)) vec = 0;
        d[i].tiles_n = (e.N + tile - 1) / tile;
        d[i].tile0 = t;
        t += d[i].tiles_n * ((e.M + tile - 1) / tile);
        if (i == 0) plan->first_tiles = t;
    }
    plan->tiles = t;
    plan->vec = vec;
    plan->tile = tile;
    return PTMI_OK;
}

int launch_gemm_tn_group(const void *dev_desc, int i0, int i1, int tiles, const TnGroupPlan &plan, hipStream_t s) {
    if (i1 <= i0 || tiles <= 0) return PTMI_OK;
    using Fn = void (*)(const GemmGroupDesc *, int, int);
    static const Fn fns[2][2] = {{k_gemm_tn_group<32, 32, false>, k_gemm_tn_group<32, 32, true>},
                                 {k_gemm_tn_group_split<1>, k_gemm_tn_group_split<4>}};
    hipLaunchKernelGGL(fns[plan.tile == 64][plan.vec], dim3((unsigned)tiles), dim3(256), 0, s,
                       static_cast<const GemmGroupDesc *>(dev_desc), i0, i1);
    PTMI_HIP(hipGetLastError());
    return PTMI_OK;
}

}  // namespace ptmi

using namespace ptmi;

namespace {

// Host-pointer GEMM: upload, run, download (the drop-in replacements for
// the reference's host-memory GEMM calls).
int host_gemm(int op, const float *A, size_t a_n, long lda, const float *B, size_t b_n, long ldb, float *C, int M,
              int N, int K, int accumulate) {
    int st = ensure_init();
    if (st) return st;
    hipStream_t s = lib_stream();
    const size_t c_n = (size_t)M * N;
    const size_t ws_n = std::min<size_t>(c_n * 64, (size_t)64 << 20);
    float *dA = scratch_buf(0, a_n + b_n + c_n);
    float *ws = scratch_buf(3, ws_n);
    if (!dA || !ws) return ptmi_last_status();
    float *dB = dA + a_n, *dC = dB + b_n;
    PTMI_HIP(hipMemcpyAsync(dA, A, a_n * sizeof(float), hipMemcpyHostToDevice, s));
    PTMI_HIP(hipMemcpyAsync(dB, B, b_n * sizeof(float), hipMemcpyHostToDevice, s));
    if (accumulate) PTMI_HIP(hipMemcpyAsync(dC, C, c_n * sizeof(float), hipMemcpyHostToDevice, s));
    if ((st = launch_gemm(op, dA, lda, dB, ldb, dC, N, M, N, K, accumulate, ws, ws_n, s))) return st;
    PTMI_HIP(hipMemcpyAsync(C, dC, c_n * sizeof(float), hipMemcpyDeviceToHost, s));
    PTMI_HIP(hipStreamSynchronize(s));
    return PTMI_OK;
}

}  // namespace

namespace ptmi {

// Split-K workspace of ptmi_gemm_dev: up to 64 partial products, at most
// 256 MiB.
size_t gemm_dev_ws_floats(int M, int N) {
    if (M <= 0 || N <= 0) return 0;
    return std::min<size_t>((size_t)M * N * 64, (size_t)64 << 20);
}

// Calls on the library's stream follow one another and may all split K through
// one workspace.  Those on streams of the caller may overlap, so they split only
// where the fp32 tiles would (split_plan; few blocks, long K), through a
// workspace of their own: a GEMM that those tiles run whole shares nothing
// with a call on another stream.
static bool callers_stream(const void *stream) { return stream && stream != (const void *)lib_stream(); }
static size_t split_ws_floats(int op, int M, int N, int K, bool callers) {
    const size_t n = gemm_dev_ws_floats(M, N);
    return callers && gemm_workspace_floats(op, M, N, K, n) == 0 ? 0 : n;
}

// ── the entry point that allocates nothing ───────────────────────────────
// ptmi_gemm_dev_noalloc keeps its split-K partials in this file-scope
// device array (16 MiB; each GPU the library runs on holds it until the
// process ends).  In host code `scratch` names a host-side stand-in, not
// device memory: the device address comes from hipGetSymbolAddress, once
// per device at ptmi_init, and only that address is handed to kernels.
constexpr size_t kNoAllocScratchFloats = kScratchFloats;
constexpr int kMaxDevices = 64;
static __device__ __align__(256) float scratch[kNoAllocScratchFloats];
static float *g_scratch_dev[kMaxDevices] = {};

int gemm_scratch_setup(int device) {
    if (device < 0 || device >= kMaxDevices)
        return set_error(PTMI_ERR_ARG, "device %d: no GEMM scratch slot", device);
    if (g_scratch_dev[device]) return PTMI_OK;
    void *p = nullptr;
    hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return hip_check(e, "hipGetSymbolAddress(scratch)");
    if (!p) return set_error(PTMI_ERR_HIP, "hipGetSymbolAddress(scratch) gave no address");
    g_scratch_dev[device] = static_cast<float *>(p);
    return PTMI_OK;
}

}  // namespace ptmi

extern "C" {

int ptmi_gemm_dev_noalloc(int op, const float *dA, long lda, const float *dB, long ldb, float *dC, long ldc, int M,
                          int N, int K, int accumulate, void *stream) {
    if (!lib_initialised())
        return set_error(PTMI_ERR_STATE, "ptmi_gemm_dev_noalloc: call ptmi_init first (it locates the scratch)");
    float *ws = g_scratch_dev[lib_device()];
    if (!ws) return set_error(PTMI_ERR_STATE, "ptmi_gemm_dev_noalloc: no scratch on device %d", lib_device());
    // The K split of the fp32 tiles must fit the fixed scratch, also where
    // the bf16-product tiles (whose split always fits) take the call.
    const size_t need = gemm_workspace_floats(op, M, N, K, gemm_dev_ws_floats(M, N));
    if (need > kNoAllocScratchFloats)
        return set_error(PTMI_ERR_ARG,
                         "ptmi_gemm_dev_noalloc: %dx%dx%d counts %zu floats of split-K partials (fp32 tiles); the fixed "
                         "scratch holds %zu",
                         M, N, K, need, kNoAllocScratchFloats);
    // the split is chosen from ptmi_gemm_dev's workspace size, not the
    // scratch's, so that both take the same number of splits
    return launch_gemm(op, dA, lda, dB, ldb, dC, ldc, M, N, K, accumulate, ws,
                       std::min(kNoAllocScratchFloats, split_ws_floats(op, M, N, K, callers_stream(stream))),
                       stream ? (hipStream_t)stream : lib_stream());
}

int ptmi_gemm_dev(int op, const float *dA, long lda, const float *dB, long ldb, float *dC, long ldc, int M, int N,
                  int K, int accumulate, void *stream) {
    int st = ensure_init();
    if (st) return st;
    const bool callers = callers_stream(stream);
    const size_t ws_n = split_ws_floats(op, M, N, K, callers);
    float *ws = ws_n ? scratch_buf(callers ? 4 : 3, ws_n) : nullptr;
    if (ws_n && !ws) return ptmi_last_status();
    return launch_gemm(op, dA, lda, dB, ldb, dC, ldc, M, N, K, accumulate, ws, ws_n,
                       stream ? (hipStream_t)stream : lib_stream());
}

int ptmi_gemm_plan(int op, int M, int N, int K, long lda, long ldb, long ldc, int aligned, int accumulate, int epilogue,
                   int callers, int plan[4]) {
    if (!plan || op < 0 || op > 2 || M <= 0 || N <= 0 || K <= 0 || epilogue < GEMM_EPI_NONE || epilogue > GEMM_EPI_SWIGLU_BWD)
        return set_error(PTMI_ERR_ARG, "ptmi_gemm_plan: bad arguments");
    const GemmChoice c = gemm_choice(op, M, N, K, lda, ldb, ldc, aligned != 0, accumulate != 0,
                                     split_ws_floats(op, M, N, K, callers != 0), epilogue);
    plan[0] = c.tm;
    plan[1] = c.tn;
    plan[2] = c.kind != GEMM_64 && c.kind != GEMM_128;
    plan[3] = c.splits;
    return PTMI_OK;
}

int ptmi_sgemm_rect(const float *A, const float *B, float *C, int M, int K, int N, int accumulate) {
    if (!A || !B || !C || M <= 0 || N <= 0 || K <= 0)
        return set_error(PTMI_ERR_ARG, "ptmi_sgemm_rect: bad arguments (M=%d K=%d N=%d)", M, K, N);
    return host_gemm(0, A, (size_t)M * K, K, B, (size_t)K * N, N, C, M, N, K, accumulate);
}

int ptmi_matmul_backward_weight_batched_checked(float *d_W, const float *d_y_all, const float *x_all, int out_dim,
                                                int in_dim, int T) {
    if (!d_W || !d_y_all || !x_all || out_dim <= 0 || in_dim <= 0 || T < 0)
        return set_error(PTMI_ERR_ARG, "ptmi_matmul_backward_weight_batched: bad arguments");
    if (T == 0) return PTMI_OK;
    // dW[out,in] += dY[T,out]^T . X[T,in]   (TN: A stored [K=T][M=out])
    return host_gemm(1, d_y_all, (size_t)T * out_dim, out_dim, x_all, (size_t)T * in_dim, in_dim, d_W, out_dim, in_dim,
                     T, 1);
}

int ptmi_matmul_backward_input_batched(float *d_x_all, const float *W, const float *d_y_all, int out_dim, int in_dim,
                                       int T, int accumulate) {
    if (!d_x_all || !W || !d_y_all || out_dim <= 0 || in_dim <= 0 || T < 0)
        return set_error(PTMI_ERR_ARG, "ptmi_matmul_backward_input_batched: bad arguments");
    if (T == 0) return PTMI_OK;
    // dX[T,in] (+)= dY[T,out] . W[out,in]   (NN)
    return host_gemm(0, d_y_all, (size_t)T * out_dim, out_dim, W, (size_t)out_dim * in_dim, in_dim, d_x_all, T, in_dim,
                     out_dim, accumulate);
}

// The reference's void entries report failure by panicking
// (libpi/libc/demand.h:20-60): message on stderr, then abort().
static void panic_on(int st, const char *what) {
    if (st == PTMI_OK) return;
    fprintf(stderr, "%s: %s\n", what, ptmi_last_error());
    abort();
}

void ptmi_sgemm_rect_tmu(const float *A, const float *B, float *C, int M, int K, int N, int num_qpus,
                         int accumulate) {
    // num_qpus selects no resource here, but keeps the reference's range
    // check (gemm_rect.c:34: 1..12); N needs no multiple of 16 (:33).
    if (num_qpus < 1 || num_qpus > 12)
        panic_on(set_error(PTMI_ERR_ARG, "num_qpus %d outside 1..12", num_qpus), "ptmi_sgemm_rect_tmu");
    panic_on(ptmi_sgemm_rect(A, B, C, M, K, N, accumulate), "ptmi_sgemm_rect_tmu");
}

void ptmi_sgemm_cpu(const float *A, const float *B, float *C, int M, int K, int N) {
    panic_on(ptmi_sgemm_rect(A, B, C, M, K, N, 0), "ptmi_sgemm_cpu");
}

void ptmi_matmul_backward_weight_batched(float *d_W, const float *d_y_all, const float *x_all, int out_dim,
                                         int in_dim, int T) {
    panic_on(ptmi_matmul_backward_weight_batched_checked(d_W, d_y_all, x_all, out_dim, in_dim, T),
             "ptmi_matmul_backward_weight_batched");
}

}  // extern "C"

// The prompt of ptmi_model_generate (the prefill half of pt_text.c:344-350),
// all positions at once.
//
// A position whose next token the prompt forces is needed only for its keys
// and values: its logits are never looked at.  Token by token each of them
// streams every weight from memory (stories110M: 440 MB, 162 us); here they
// are the rows of GEMMs, so the weights are read once per kPrefillRows
// positions, the classifier not at all, and the last layer stops at its keys
// and values.  K and V go from the QKV product's epilogue straight into the
// decode caches, which the attention then reads.  700 positions of stories110M
// and 32 decoded: 117.6 -> 7.3 ms.  Long prompts are bound by their GEMMs
// (0.12 TFLOP in 2 ms for 700 positions), short ones by the latency of each
// of the seven kernels of a layer (4 to 13 us).
#include "ptmi_model.h"

#include <algorithm>

namespace ptmi {

namespace {

// Positions per pass: what fills the chip with GEMM tiles, and the bound of
// the buffers (a 4096-position prompt runs as four passes).
constexpr int kPrefillRows = 1024;
constexpr size_t kPrefillWs = (size_t)8 << 20;     // split-K partials, floats (as the training step's)
// Fewer forced positions than this go token by token: the pass takes as long
// for one as for 32, seven launches per layer.  Prompt pass and decode steps
// of n forced positions plus the last, us: stories110M n = 3 758 / 679, n = 4
// 767 / 831, n = 32 772 / 4993, n = 999 2431; stories15M n = 2 288 / 280, n = 4
// 293 / 428, n = 128 322 / 9585; 432-wide, 9 layers, n = 3 489 / 498.
constexpr int kMinPrefill = 4;

inline size_t align_up(size_t v, size_t a) { return (v + a - 1) / a * a; }

}  // namespace

// The pass's buffers (stories110M: 59 MB), once per model: at creation for a
// model that does not train, else with the first prompt that needs them.
// Without room for them the prompt runs token by token.
bool prefill_reserve(ptmi_model *m) {
    if (m->pre_mem) return true;
    const Config &c = m->c;
    const size_t R = std::min(c.seq_len, kPrefillRows), D = c.dim, H = c.hidden;
    size_t sizes[] = {R * D, R * D, R * 3 * D, R * D, R * H, kPrefillWs};
    float **dst[] = {&m->pre_x, &m->pre_xn, &m->pre_q, &m->pre_ao, &m->pre_sh, &m->pre_ws};
    size_t total = 0;
    for (size_t n : sizes) total += align_up(n, 64);
    if (hipMalloc(&m->pre_mem, total * sizeof(float)) != hipSuccess) {
        (void)hipGetLastError();
        m->pre_mem = nullptr;
        return false;
    }
    size_t o = 0;
    for (int i = 0; i < 6; i++) { *dst[i] = m->pre_mem + o; o += align_up(sizes[i], 64); }
    m->pre_rows = (int)R;
    m->pre_ws_floats = kPrefillWs;
    return true;
}

int prefill_positions(ptmi_model *m, int n_prompt, int max_tokens) {
    // the last position run is a decode step: its logits are the call's
    const int n = std::min(n_prompt, max_tokens) - 1;
    return n >= kMinPrefill && prefill_reserve(m) ? n : 0;
}

void prefill_destroy(ptmi_model *m) {
    if (m->pre_mem) (void)hipFree(m->pre_mem);
    m->pre_mem = nullptr;
}

// Keys and values of positions [0, n) from the tokens in m->prompt.
int enqueue_prefill(ptmi_model *m, int n, hipStream_t s) {
    const Resident *r = m->res;
    const Config &c = m->c;
    const int D = c.dim, H = c.hidden, L = c.n_layers, QS = 3 * D;
    const long KV = c.kv_dim, S = c.seq_len;
    const SplitK none = {};
    int st;
    for (int p0 = 0; p0 < n; p0 += m->pre_rows) {
        const int T = std::min(m->pre_rows, n - p0);
        // C = epi(rmsnorm(x) . W^T); x is first completed from the pending
        // split-K sums, or gathered from the embedding table (tok)
        auto norm_gemm = [&](const float *w, const SplitK &pk, const int *tok, const float *W, int N, float *C,
                             const GemmEpi &epi) -> int {
            GemmNorm nm = {};
            nm.kind = GEMM_NORM_PLAIN;
            nm.w = w;
            nm.xn_out = m->pre_xn;
            if (!tok && pk.splits == 0 && gemm_norm_fusable(T, N, D, m->pre_x, D, W, D, epi.kind, nm))
                return launch_gemm(2, m->pre_x, D, W, D, C, N, T, N, D, 0, nullptr, 0, s, nullptr, nullptr, &epi, &nm);
            launch_rmsnorm_rows(m->pre_x, w, m->pre_xn, T, D, pk, m->pre_x, tok, r->emb, nullptr, s);
            PTMI_HIP(hipGetLastError());
            return launch_gemm(2, m->pre_xn, D, W, D, C, N, T, N, D, 0, m->pre_ws, m->pre_ws_floats, s, nullptr,
                               nullptr, &epi);
        };
        SplitK pend = none;
        for (int l = 0; l < L; l++) {
            float *kc = m->kc + l * S * KV, *vc = m->vc + l * S * KV;
            const bool last = l == L - 1;
            GemmEpi rope = {GEMM_EPI_ROPE, kc + p0 * KV, KV, D, c.head_dim, vc + p0 * KV};
            rope.pos0 = p0;
            rope.col0 = last ? D : 0;                            // the last layer: k and v only
            if ((st = norm_gemm(r->rms_att + (long)l * D, pend, l == 0 ? m->prompt + p0 : nullptr,
                                r->wqkv + (long)l * QS * D + (long)rope.col0 * D, QS - rope.col0, m->pre_q, rope)))
                return st;
            if (last) break;
            AttnFwdArgs fa = {m->pre_q, QS, kc, vc, KV, m->pre_ao, D, nullptr, nullptr, 0, T, p0, c.head_dim,
                              host_att_scale(c.head_dim)};
            if ((st = launch_attn_fwd(fa, c.n_heads, s))) return st;
            if ((st = launch_gemm(2, m->pre_ao, D, r->wo + (long)l * D * D, D, m->pre_x, D, T, D, D, 1, m->pre_ws,
                                  m->pre_ws_floats, s, m->pre_x, &pend)))
                return st;
            GemmEpi swiglu = {GEMM_EPI_SWIGLU, m->pre_sh, H, 0, 0};
            swiglu.only_out = 1;                                 // (C stands for the unstored h1 and h3)
            if ((st = norm_gemm(r->rms_ffn + (long)l * D, pend, nullptr, r->w13 + (long)l * 2 * H * D, 2 * H, m->pre_sh,
                                swiglu)))
                return st;
            if ((st = launch_gemm(2, m->pre_sh, H, r->w2 + (long)l * D * H, H, m->pre_x, D, T, D, H, 1, m->pre_ws,
                                  m->pre_ws_floats, s, m->pre_x, &pend)))
                return st;
        }
    }
    return PTMI_OK;
}

}  // namespace ptmi

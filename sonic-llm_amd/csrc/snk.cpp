// The kernel-level C ABI (include/sn_kernels.h) over the launchers the engine uses.
#include <hip/hip_runtime.h>
#include <string.h>

#include <algorithm>
#include <vector>

#include "../../include/sn_kernels.h"
#include "sn_kernels_internal.h"

extern "C" size_t snk_q4_stripes_bytes(int N, int K) { return q4t_bytes(N, K); }

extern "C" int snk_q4_repack(const void* d_q4, int N, int K, void* d_stripes, void* stream) {
    if (N <= 0 || K <= 0 || K % 32) return -1;
    q4_repack((const uint8_t*) d_q4, N, K, (uint8_t*) d_stripes, 1, 0, (hipStream_t) stream);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

extern "C" size_t snk_q8_tiles_bytes(int N, int K) { return wt_bytes(WT_Q8_0, N, K); }

extern "C" int snk_q8_repack(const void* d_q8, int N, int K, void* d_tiles, void* stream) {
    if (N <= 0 || K <= 0 || K % 32) return -1;
    q4_repack((const uint8_t*) d_q8, N, K, (uint8_t*) d_tiles, 1, 0, (hipStream_t) stream, WT_Q8_0);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

extern "C" int snk_moe_router(const float* d_hn, int R, int E, const float* d_router, int NE, float* d_lg,
                              void* stream) {
    if (R < 0 || E <= 0 || E % 4 || NE <= 0) return -1;
    moe_router(d_hn, d_router, R, E, NE, d_lg, (hipStream_t) stream);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

extern "C" int snk_moe_tile_rows(int R, int NE, int k) {
    if (R < 0 || NE <= 0 || k <= 0) return -1;
    return 16 * (std::min(NE, R * k) + (R * k + 15) / 16);
}

extern "C" int snk_moe_select(const float* d_lg, int R, int NE, int k, int32_t* d_ids, float* d_w, int32_t* d_prow,
                              int32_t* d_rsrc, int32_t* d_items, int32_t* d_count, void* stream) {
    if (R < 0 || NE <= 0 || k <= 0) return -1;
    const int rc = moe_select(d_lg, R, NE, k, snk_moe_tile_rows(R, NE, k), d_ids, d_w, d_prow, d_rsrc, d_items,
                              d_count, (hipStream_t) stream);
    return rc == 0 && hipGetLastError() == hipSuccess ? 0 : -1;
}

// moe_route through a throwaway set of counters: the one-launch routing (same results as snk_moe_router +
// snk_moe_select); *xerr (optional) receives the XCD check
extern "C" int snk_moe_route(const float* d_hn, int R, int E, const float* d_router, int NE, int k, float* d_lg,
                             int32_t* d_ids, float* d_w, int32_t* d_prow, int32_t* d_rsrc, int32_t* d_items,
                             int32_t* d_count, int* xerr, void* stream) {
    hipStream_t st = (hipStream_t) stream;
    int nxcd = 1;
    if (!xcd_round_robin(st, &nxcd)) return -1;
    const int cnt_len = 1 << 14;
    uint64_t* cnt = nullptr;
    int32_t* gx = nullptr;  // [0] the global counter, [1] the XCD check
    if (hipMalloc(&cnt, cnt_len * 8) != hipSuccess) return -1;
    if (hipMalloc(&gx, 8) != hipSuccess) {
        hipFree(cnt);
        return -1;
    }
    int rc = hipMemsetAsync(cnt, 0, cnt_len * 8, st) == hipSuccess && hipMemsetAsync(gx, 0, 8, st) == hipSuccess ? 0 : -1;
    if (rc == 0)
        rc = moe_route(d_hn, d_router, R, E, NE, k, snk_moe_tile_rows(R, NE, k), d_lg, d_ids, d_w, d_prow, d_rsrc,
                       d_items, d_count, cnt, cnt_len, gx, gx + 1, nxcd, st);
    int32_t h[2] = {0, 0};
    if (hipStreamSynchronize(st) != hipSuccess || hipMemcpy(h, gx, 8, hipMemcpyDeviceToHost) != hipSuccess) rc = -1;
    if (xerr) *xerr = h[1];
    hipFree(cnt);
    hipFree(gx);
    return rc == 0 && hipGetLastError() == hipSuccess ? 0 : -1;
}

extern "C" int snk_gemm_grouped(int wt, const void* d_w, size_t wstride, const int32_t* d_items,
                                const int32_t* d_count, int max_items, const void* d_xa, int P, int N, int K,
                                float* d_part, size_t part_bytes, const int32_t* d_rmask, void* stream) {
    if ((wt != WT_Q4_0 && wt != WT_Q8_0) || P <= 0 || N <= 0 || K <= 0 || K % 32 || max_items <= 0 ||
        max_items > (P + 15) / 16)
        return -1;
    const int rc = q4_gemm_grouped((const uint8_t*) d_w, wstride, d_items, d_count, max_items, (const uint8_t*) d_xa, P,
                                   N, K, d_part, part_bytes, (hipStream_t) stream, wt, d_rmask);
    return rc >= 0 && hipGetLastError() == hipSuccess ? 0 : -1;
}

extern "C" size_t snk_argmax_workspace_bytes(int n, int V) { return n > 0 && V > 0 ? argmax_workspace_bytes(n, V) : 0; }

extern "C" int snk_argmax(const float* d_logits, int V, int n, const int32_t* d_ban, int nban, const uint8_t* d_skip,
                          int32_t* d_out, float* d_rec, void* d_ws, size_t ws_bytes, void* stream) {
    if (n < 0 || V <= 0 || nban < 0 || nban > 8 || (nban > 0 && !d_ban)) return -1;
    const int rc = argmax_rows(d_logits, V, n, d_ban, nban, d_skip, d_out, d_rec, d_ws, ws_bytes, (hipStream_t) stream);
    return rc == 0 && hipGetLastError() == hipSuccess ? 0 : -1;
}

extern "C" size_t snk_xa_bytes(int M, int K) { return xa_bytes(M, K); }

extern "C" size_t snk_q6k_tiles_bytes(int N, int K) { return N > 0 && K > 0 && K % 256 == 0 ? q6t_bytes(N, K) : 0; }

extern "C" int snk_q6k_repack(const void* d_q6k, int N, int K, void* d_tiles, void* stream) {
    if (N <= 0 || K <= 0 || K % 256) return -1;
    q6k_repack((const uint8_t*) d_q6k, N, K, (uint8_t*) d_tiles, (hipStream_t) stream);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

extern "C" int snk_q6k_dequant(const void* d_tiles, int N, int K, float* d_w, void* stream) {
    if (N <= 0 || K <= 0 || K % 256) return -1;
    q6k_dequant((const uint8_t*) d_tiles, N, K, d_w, (hipStream_t) stream);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

extern "C" size_t snk_xk_bytes(int M, int K) { return M > 0 && K > 0 && K % 256 == 0 ? xk_bytes(M, K) : 0; }

extern "C" int snk_quant_q8k(const float* d_x, int M, int K, int ldx, const float* d_norm_w, float eps, void* d_xk,
                             void* stream) {
    if (M <= 0 || K <= 0 || K % 256 || ldx < K) return -1;
    quant_q8k(d_x, nullptr, M, K, ldx, d_norm_w, eps, (uint8_t*) d_xk, (hipStream_t) stream);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

extern "C" int snk_q6k_gemm(const void* d_tiles, const void* d_xk, int M, int N, int K, float* d_y, int ldy,
                            void* stream) {
    if (M <= 0 || N <= 0 || K <= 0 || K % 256 || ldy < N) return -1;
    const int rc = q6k_gemm((const uint8_t*) d_tiles, (const uint8_t*) d_xk, M, N, K, d_y, ldy, (hipStream_t) stream);
    return rc == 0 && hipGetLastError() == hipSuccess ? 0 : -1;
}

extern "C" int snk_quant_act(const float* d_x, int M, int K, int ldx, const float* d_norm_w, float eps, void* d_xa,
                             void* stream) {
    if (M <= 0 || K <= 0 || K % 32 || ldx < K || ldx % 4) return -1;
    quant_act(d_x, nullptr, M, K, ldx, d_norm_w, eps, (uint8_t*) d_xa, nullptr, 0, (hipStream_t) stream);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

extern "C" size_t snk_q4_workspace_bytes(int M, int N, int K) { return q4_workspace_bytes(M, N, K); }

extern "C" int snk_q4_plan(int N, int K, int wt, int* spw, int* ks) {
    if (N <= 0 || K <= 0 || K % 32 || (wt != WT_Q4_0 && wt != WT_Q8_0)) return -1;
    const GemmPlan p = q4_plan(N, K, wt);
    if (spw) *spw = p.spw;
    if (ks) *ks = p.ks;
    return 0;
}

extern "C" int snk_q4_gemm(const void* d_stripes, const void* d_xa, int M, int N, int K, float* d_y, int ldy, int epi,
                           void* d_ws, size_t ws_bytes, void* stream) {
    if (M <= 0 || N <= 0 || K <= 0 || K % 32 || epi < 0 || epi > 2) return -1;
    if (epi == SNK_EPI_SWIGLU ? (N % 32 != 0 || ldy < N / 2) : ldy < N) return -1;
    const int rc = q4_gemm((const uint8_t*) d_stripes, (const uint8_t*) d_xa, M, N, K, d_y, ldy, epi, (float*) d_ws,
                           ws_bytes, (hipStream_t) stream);
    return rc == 0 && hipGetLastError() == hipSuccess ? 0 : -1;
}

extern "C" int snk_q4_gemm_swiglu(const void* d_stripes, const void* d_xa, int M, int N, int K, float* d_h,
                                  void* d_xo, void* stream) {
    if (M <= 0 || N <= 0 || K <= 0 || K % 32 || !d_h || !d_xo || d_xo == d_xa) return -1;
    if (M < 256 || !q4_gemm_swiglu_fits(M, N, K, WT_Q4_0)) return 1;  // (prompt rows, as the header says)
    const int rc = q4_gemm_swiglu((const uint8_t*) d_stripes, (const uint8_t*) d_xa, M, N, K, d_h, (uint8_t*) d_xo,
                                  (hipStream_t) stream, WT_Q4_0);
    return rc == 1 && hipGetLastError() == hipSuccess ? 0 : -1;
}

extern "C" size_t snk_q8_workspace_bytes(int M, int N, int K) { return q4_workspace_bytes(M, N, K, WT_Q8_0); }

extern "C" int snk_q8_gemm(const void* d_tiles, const void* d_xa, int M, int N, int K, float* d_y, int ldy, int epi,
                           void* d_ws, size_t ws_bytes, void* stream) {
    if (M <= 0 || N <= 0 || K <= 0 || K % 32 || epi < 0 || epi > 2) return -1;
    if (epi == SNK_EPI_SWIGLU ? (N % 32 != 0 || ldy < N / 2) : ldy < N) return -1;
    const int rc = q4_gemm((const uint8_t*) d_tiles, (const uint8_t*) d_xa, M, N, K, d_y, ldy, epi, (float*) d_ws,
                           ws_bytes, (hipStream_t) stream, WT_Q8_0);
    return rc == 0 && hipGetLastError() == hipSuccess ? 0 : -1;
}

extern "C" double snk_q4_gemm_time(const void* const* d_stripes, int n_copies, const void* d_xa, int M, int N, int K,
                                   float* d_y, int ldy, void* d_ws, size_t ws_bytes, int iters, void* stream) {
    hipStream_t st = (hipStream_t) stream;
    hipEvent_t a, b;
    if (hipEventCreate(&a) != hipSuccess || hipEventCreate(&b) != hipSuccess) return -1.0;
    // the raw matmul (the k-slice sums), as a step runs it; one untimed launch per copy
    (void) d_y;
    (void) ldy;
    for (int c = 0; c < n_copies; ++c)
        if (q4_gemm_raw((const uint8_t*) d_stripes[c], (const uint8_t*) d_xa, M, N, K, (float*) d_ws, ws_bytes, st) < 0)
            return -1.0;
    hipEventRecord(a, st);
    for (int i = 0; i < iters; ++i)
        q4_gemm_raw((const uint8_t*) d_stripes[i % n_copies], (const uint8_t*) d_xa, M, N, K, (float*) d_ws, ws_bytes,
                    st);
    hipEventRecord(b, st);
    hipEventSynchronize(b);
    float ms = 0.0f;
    hipEventElapsedTime(&ms, a, b);
    hipEventDestroy(a);
    hipEventDestroy(b);
    return hipGetLastError() == hipSuccess ? 1000.0 * ms / iters : -1.0;
}

extern "C" double snk_read_time(const void* const* d_bufs, int n_copies, size_t bytes, float* d_sink, int iters,
                                void* stream) {
    if (n_copies <= 0 || bytes < 16 || bytes % 16 || iters <= 0 || !d_sink) return -1.0;
    hipStream_t st = (hipStream_t) stream;
    hipEvent_t a, b;
    if (hipEventCreate(&a) != hipSuccess || hipEventCreate(&b) != hipSuccess) return -1.0;
    for (int c = 0; c < n_copies; ++c) read_floor(d_bufs[c], bytes, d_sink, st);
    hipEventRecord(a, st);
    for (int i = 0; i < iters; ++i) read_floor(d_bufs[i % n_copies], bytes, d_sink, st);
    hipEventRecord(b, st);
    hipEventSynchronize(b);
    float ms = 0.0f;
    hipEventElapsedTime(&ms, a, b);
    hipEventDestroy(a);
    hipEventDestroy(b);
    return hipGetLastError() == hipSuccess ? 1000.0 * ms / iters : -1.0;
}

extern "C" double snk_q4_gemm_plan_time(const void* const* d_stripes, int n_copies, const void* d_xa, int M, int N,
                                        int K, void* d_ws, size_t ws_bytes, int mt, int spw, int G, int iters,
                                        void* stream) {
    hipStream_t st = (hipStream_t) stream;
    hipEvent_t a, b;
    if (hipEventCreate(&a) != hipSuccess || hipEventCreate(&b) != hipSuccess) return -1.0;
    for (int c = 0; c < n_copies; ++c)
        if (q4_gemm_raw_plan((const uint8_t*) d_stripes[c], (const uint8_t*) d_xa, M, N, K, (float*) d_ws, ws_bytes,
                             st, WT_Q4_0, mt, spw, G) < 0)
            return -1.0;
    hipEventRecord(a, st);
    for (int i = 0; i < iters; ++i)
        q4_gemm_raw_plan((const uint8_t*) d_stripes[i % n_copies], (const uint8_t*) d_xa, M, N, K, (float*) d_ws,
                         ws_bytes, st, WT_Q4_0, mt, spw, G);
    hipEventRecord(b, st);
    hipEventSynchronize(b);
    float ms = 0.0f;
    hipEventElapsedTime(&ms, a, b);
    hipEventDestroy(a);
    hipEventDestroy(b);
    return hipGetLastError() == hipSuccess ? 1000.0 * ms / iters : -1.0;
}

extern "C" int snk_q4_gemm_plan_sums(const void* d_stripes, const void* d_xa, int M, int N, int K, float* d_y,
                                     void* d_ws, size_t ws_bytes, int mt, int spw, int G, void* stream) {
    // the plan's slices added in order into y [M][N] (for checking a plan against the default one)
    const int ks = q4_gemm_raw_plan((const uint8_t*) d_stripes, (const uint8_t*) d_xa, M, N, K, (float*) d_ws,
                                    ws_bytes, (hipStream_t) stream, WT_Q4_0, mt, spw, G);
    if (ks < 0) return -1;
    q4_reduce_slices((const float*) d_ws, ks, M, N, d_y, (hipStream_t) stream);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

// ---- attention work lists
struct snk_attn {
    int n_rows, H, KVH, max_pages, page_cells, max_chunks, n_items, n_mrows, n_runs;
    bool whole;
    // the fold (chunk items and merge in one launch, k_attn_fold): plain chunk lists only; its counters and XCD check
    bool plain = false, fold = false;
    int n_groups = 0, max_nc = 0, nxcd = 0;
    uint64_t* d_cnt = nullptr;
    int32_t* d_xerr = nullptr;
    AttnGroup* d_groups = nullptr;
    AttnItem* d_items = nullptr;
    AttnItem* d_runs = nullptr;
    int32_t* d_mrows = nullptr;
    int32_t* d_pos = nullptr;
    float* d_part = nullptr;
};

extern "C" snk_attn* snk_attn_new_pt(int n_rows, const int32_t* seq, const int32_t* pos, int H, int KVH,
                                     int max_pages, int page_cells, int mode, const int32_t* pt, char* err,
                                     int err_len);
extern "C" snk_attn* snk_attn_new_mode(int n_rows, const int32_t* seq, const int32_t* pos, int H, int KVH,
                                       int max_pages, int page_cells, int mode, char* err, int err_len) {
    return snk_attn_new_pt(n_rows, seq, pos, H, KVH, max_pages, page_cells, mode, nullptr, err, err_len);
}

extern "C" snk_attn* snk_attn_new_pt(int n_rows, const int32_t* seq, const int32_t* pos, int H, int KVH,
                                     int max_pages, int page_cells, int mode, const int32_t* pt, char* err,
                                     int err_len) {
    if (n_rows <= 0 || H <= 0 || KVH <= 0 || H % KVH || 16 % (H / KVH) || (page_cells != 32 && page_cells != 64) ||
        mode < -1 || mode > 2) {
        sn_set_err(err, err_len, "snk_attn_new: bad shape");
        return nullptr;
    }
    for (int r = 0; r < n_rows; ++r)
        if (pos[r] < 0 || pos[r] >= max_pages * page_cells) {
            sn_set_err(err, err_len, "snk_attn_new: a position is outside the page table");
            return nullptr;
        }
    AttnPlan pl;
    attn_plan(n_rows, seq, pos, H, KVH, page_cells, pl, mode, pt, max_pages);
    snk_attn* p = new snk_attn();
    p->n_rows = n_rows;
    p->H = H;
    p->KVH = KVH;
    p->max_pages = max_pages;
    p->page_cells = page_cells;
    p->max_chunks = pl.max_chunk;
    p->n_items = (int) pl.items.size();
    p->n_mrows = (int) pl.mrows.size();
    p->n_runs = (int) pl.runs.size();
    p->whole = pl.whole;
    bool ok = hipMalloc(&p->d_groups, pl.groups.size() * sizeof(AttnGroup)) == hipSuccess &&
              hipMalloc(&p->d_items, std::max<size_t>(1, pl.items.size()) * sizeof(AttnItem)) == hipSuccess &&
              hipMalloc(&p->d_runs, std::max<size_t>(1, pl.runs.size()) * sizeof(AttnItem)) == hipSuccess &&
              hipMalloc(&p->d_mrows, std::max<size_t>(1, pl.mrows.size()) * 4) == hipSuccess &&
              hipMalloc(&p->d_pos, (size_t) n_rows * 4) == hipSuccess &&
              hipMalloc(&p->d_part, (size_t) n_rows * H * p->max_chunks * 130 * 4) == hipSuccess;
    ok = ok && hipMemcpy(p->d_groups, pl.groups.data(), pl.groups.size() * sizeof(AttnGroup), hipMemcpyHostToDevice) == hipSuccess &&
         (pl.items.empty() || hipMemcpy(p->d_items, pl.items.data(), pl.items.size() * sizeof(AttnItem), hipMemcpyHostToDevice) == hipSuccess) &&
         (pl.runs.empty() || hipMemcpy(p->d_runs, pl.runs.data(), pl.runs.size() * sizeof(AttnItem), hipMemcpyHostToDevice) == hipSuccess) &&
         (pl.mrows.empty() || hipMemcpy(p->d_mrows, pl.mrows.data(), pl.mrows.size() * 4, hipMemcpyHostToDevice) == hipSuccess) &&
         hipMemcpy(p->d_pos, pos, (size_t) n_rows * 4, hipMemcpyHostToDevice) == hipSuccess;
    if (!ok) {
        sn_set_err(err, err_len, "snk_attn_new: device allocation failed");
        snk_attn_free(p);
        return nullptr;
    }
    // plain chunk items (every group's chunks, one item each, none shared): the fold's form, available where the device
    // deals launches to its XCDs in turn (off until snk_attn_fold turns it on: measured slower than the two launches)
    p->n_groups = (int) pl.groups.size();
    int nct = 0;
    for (const AttnGroup& g : pl.groups) {
        const int nc = (g.pos0 + g.nrows - 1) / ATT_CHUNK + 1;
        p->max_nc = std::max(p->max_nc, nc);
        nct += nc;
    }
    p->plain = !pl.whole && pl.runs.empty() && nct == p->n_items && p->max_nc <= 127;
    for (const AttnItem& it : pl.items) p->plain = p->plain && it.share[0] < 0;
    if (p->plain && xcd_round_robin(nullptr, &p->nxcd)) {
        const size_t nc8 = (size_t) p->n_groups * KVH * CNT_STRIDE * 8;
        if (!(hipMalloc(&p->d_cnt, nc8) == hipSuccess && hipMalloc(&p->d_xerr, 4) == hipSuccess &&
              hipMemset(p->d_cnt, 0, nc8) == hipSuccess && hipMemset(p->d_xerr, 0, 4) == hipSuccess &&
              hipDeviceSynchronize() == hipSuccess)) {
            hipFree(p->d_cnt);
            hipFree(p->d_xerr);
            p->d_cnt = nullptr, p->d_xerr = nullptr;  // (no fold for this list)
        }
    }
    return p;
}

extern "C" int snk_attn_fold(snk_attn* p, int on) {
    // withdrawn: one run of the fold's bitwise test against the two launches differed on one MI355X (no cause found
    // by reading the handoff, 45 repeats on another box equal), so the form is never taken and `on` is refused
    (void) on;
    if (p) p->fold = false;
    return 0;
}

extern "C" int snk_attn_xcd_faults(const snk_attn* p) {
    int32_t v = 0;
    if (!p || !p->d_xerr || hipMemcpy(&v, p->d_xerr, 4, hipMemcpyDeviceToHost) != hipSuccess) return -1;
    return v;
}

extern "C" snk_attn* snk_attn_new(int n_rows, const int32_t* seq, const int32_t* pos, int H, int KVH, int max_pages,
                                  int page_cells, char* err, int err_len) {
    return snk_attn_new_mode(n_rows, seq, pos, H, KVH, max_pages, page_cells, -1, err, err_len);
}

static AttnArgs attn_args(snk_attn* p, const float* d_q, int ldq, const void* d_kpool, const void* d_vpool,
                          const int32_t* d_pt, float scale, float* d_out, int ldo) {
    AttnArgs a{};
    a.q = d_q;
    a.ldq = ldq;
    a.kpool = (const uint16_t*) d_kpool;
    a.vpool = (const uint16_t*) d_vpool;
    a.pt = d_pt;
    a.max_pages = p->max_pages;
    a.page_cells = p->page_cells;
    a.groups = p->d_groups;
    a.items = p->d_items;
    a.n_items = p->n_items;
    a.runs = p->d_runs;
    a.n_runs = p->n_runs;
    a.part = p->d_part;
    a.max_chunks = p->max_chunks;
    a.out = d_out;
    a.ldo = ldo;
    a.H = p->H;
    a.KVH = p->KVH;
    a.scale = scale;
    a.n_rows = p->n_rows;
    a.row_pos = p->d_pos;
    a.whole = p->whole ? 1 : 0;
    a.mrows = p->d_mrows;
    a.n_mrows = p->n_mrows;
    if (p->fold) {
        a.fold = 1, a.n_groups = p->n_groups, a.fold_chunks = p->max_nc, a.nxcd = p->nxcd;
        a.cnt = p->d_cnt, a.xerr = p->d_xerr;
    }
    return a;
}

extern "C" int snk_attn_run(snk_attn* p, const float* d_q, int ldq, const void* d_kpool, const void* d_vpool,
                            const int32_t* d_pt, float scale, float* d_out, int ldo, void* stream) {
    if (!p || ldq < p->H * 128 || ldo < p->H * 128) return -1;
    const AttnArgs a = attn_args(p, d_q, ldq, d_kpool, d_vpool, d_pt, scale, d_out, ldo);
    if (paged_attention(a, (hipStream_t) stream) != 0) return -1;
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

extern "C" double snk_attn_time(snk_attn* p, const float* d_q, int ldq, const void* d_kpool, const void* d_vpool,
                                const int32_t* d_pt, float scale, float* d_out, int ldo, int iters, void* stream) {
    hipStream_t st = (hipStream_t) stream;
    const AttnArgs a = attn_args(p, d_q, ldq, d_kpool, d_vpool, d_pt, scale, d_out, ldo);
    hipEvent_t e0, e1;
    if (hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess) return -1.0;
    paged_attention(a, st);
    hipEventRecord(e0, st);
    for (int i = 0; i < iters; ++i) paged_attention(a, st);
    hipEventRecord(e1, st);
    hipEventSynchronize(e1);
    float ms = 0.0f;
    hipEventElapsedTime(&ms, e0, e1);
    hipEventDestroy(e0);
    hipEventDestroy(e1);
    return hipGetLastError() == hipSuccess ? 1000.0 * ms / iters : -1.0;
}

extern "C" int snk_attn_whole(const snk_attn* p) { return p && p->whole ? 1 : 0; }

extern "C" int snk_attn_runs(const snk_attn* p) { return p ? p->n_runs : 0; }

extern "C" void snk_attn_free(snk_attn* p) {
    if (!p) return;
    hipFree(p->d_groups);
    hipFree(p->d_items);
    hipFree(p->d_runs);
    hipFree(p->d_mrows);
    hipFree(p->d_pos);
    hipFree(p->d_part);
    hipFree(p->d_cnt);
    hipFree(p->d_xerr);
    delete p;
}

extern "C" int snk_qk_rope(float* d_qkv, int ldqkv, int R, int H, int KVH, const float* d_qw, const float* d_kw,
                           float eps, float theta_scale, const int32_t* d_seq, const int32_t* d_pos, const int32_t* d_pt,
                           int max_pages, int page_cells, void* d_kpool, void* d_vpool, void* stream) {
    if (R <= 0 || H <= 0 || KVH <= 0 || ldqkv < (H + 2 * KVH) * 128 || (page_cells != 32 && page_cells != 64)) return -1;
    const int rc = qk_norm_rope_kv(d_qkv, ldqkv, nullptr, 1, R, H, KVH, d_qw, d_kw, eps, theta_scale, d_seq, d_pos, d_pt,
                                   max_pages, page_cells, (uint16_t*) d_kpool, (uint16_t*) d_vpool, (hipStream_t) stream);
    return rc == 0 && hipGetLastError() == hipSuccess ? 0 : -1;
}

// The extern "C" surface of libferric_hip (declared in include/ferric_hip.h): argument checks with
// the reference's error behaviour, weight handles, and thin dispatch into the kernel launchers.
#include "f16x2.hpp"
#include "hostmem.hpp"
#include "prompt.hpp"

#include <stdarg.h>
#include <stdio.h>
#include <string.h>

#include <mutex>
#include <vector>

namespace {

// The intermediate of fhip_ffn_noalloc: [rows_x, n_ff] f32 between the gate|up and the down mat-vec. It lives in the code
// object, so each device the library runs on holds its own copy (512 KiB) from load to process exit and no call has to
// allocate. Host code never uses the array's name as an address: fhip_init asks the runtime for the device address of the
// current device's copy and keeps it per device.
constexpr size_t NOALLOC_FLOATS = 131072;
static __device__ __align__(256) float scratch[NOALLOC_FLOATS];
constexpr int MAX_DEVICES = 64;
float* g_scratch_ptr[MAX_DEVICES] = {};

thread_local char g_err[512] = "";
int g_device = -1;
// What a new weight handle starts with (fhip_matvec_precision, fhip_batch_policy); read when a handle is made, never at a launch.
int g_default_planes = 3;
int g_default_batch_policy = FHIP_BATCH_ORDERED;
int g_cus = 0;
size_t g_lds = 64 * 1024;

bool block_info(uint32_t ty, size_t& vals, size_t& bytes) {
    switch (ty) {
        case FHIP_Q8_0: vals = 32; bytes = 34; return true;
        case FHIP_Q4_K: vals = 256; bytes = 144; return true;
        case FHIP_Q6_K: vals = 256; bytes = 210; return true;
        case FHIP_Q4_0: vals = 32; bytes = 18; return true;
        case FHIP_Q4_1: vals = 32; bytes = 20; return true;
        case FHIP_Q5_0: vals = 32; bytes = 22; return true;
        case FHIP_Q5_1: vals = 32; bytes = 24; return true;
        case FHIP_Q5_K: vals = 256; bytes = 176; return true;
        case FHIP_IQ4_NL: vals = 32; bytes = 18; return true;
        case FHIP_IQ4_XS: vals = 256; bytes = 136; return true;
        case FHIP_MXFP4: vals = 32; bytes = 17; return true;
        default: return false;
    }
}

const char* type_name(uint32_t ty) {
    switch (ty) {
        case FHIP_Q8_0: return "Q8_0";
        case FHIP_Q4_K: return "Q4_K";
        case FHIP_Q6_K: return "Q6_K";
        case FHIP_Q4_0: return "Q4_0";
        case FHIP_Q4_1: return "Q4_1";
        case FHIP_Q5_0: return "Q5_0";
        case FHIP_Q5_1: return "Q5_1";
        case FHIP_Q5_K: return "Q5_K";
        case FHIP_IQ4_NL: return "IQ4_NL";
        case FHIP_IQ4_XS: return "IQ4_XS";
        case FHIP_MXFP4: return "MXFP4";
        default: return "?";
    }
}

int need_init() {
    if (g_device < 0) return fhip::set_error(FHIP_ERR_ARG, "fhip_init has not been called");
    return FHIP_OK;
}

// Shape checks of the per-format constructors: crates/ferric-tensor/src/dtype.rs:1271-1272 (Q8_0),
// :1389-1390 (Q4_K), :1148-1149 (Q6_K) -- `assert_eq!(cols % blk, 0)` and exact byte length.
int make_weight(uint32_t ty, size_t nbytes, size_t rows, size_t cols, fhip_weight& w) {
    size_t vals, bytes;
    if (!block_info(ty, vals, bytes)) return fhip::set_error(FHIP_ERR_UNSUPPORTED_TYPE, "QMatrix: no native matmul for ggml type %u", ty);
    if (cols % vals != 0) return fhip::set_error(FHIP_ERR_SHAPE, "%s cols must be a multiple of %zu", type_name(ty), vals);
    size_t row_bytes = cols / vals * bytes;
    if (nbytes != rows * row_bytes) return fhip::set_error(FHIP_ERR_SHAPE, "unexpected %s byte length", type_name(ty));
    if (rows > 0x7FFFFFFFull || cols > 0x7FFFFFFFull) return fhip::set_error(FHIP_ERR_SHAPE, "weight dimensions exceed 2^31");
    w.type = ty; w.rows = rows; w.cols = cols; w.row_bytes = row_bytes; w.nbytes = nbytes; w.d_raw = nullptr; w.owns = false;
    w.planes = g_default_planes; w.batch_policy = g_default_batch_policy;
    fhip::gemm_f16x2_lay_out(&w);
    return FHIP_OK;
}

}  // namespace

namespace fhip {

int set_error(int code, const char* fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
    return code;
}

int check_hip(hipError_t e, const char* what) {
    if (e == hipSuccess) return FHIP_OK;
    return set_error(FHIP_ERR_HIP, "%s: %s", what, hipGetErrorString(e));
}

int device_cus() { return g_cus; }
size_t device_lds_bytes() { return g_lds; }

// The streaming mat-vec exists in two copies, one per activation precision; these forward to the one the weight names.
// From three rows on (Q8_0: four), Q4_K, Q5_K, Q6_K and Q8_0 batches go four rows at a time through the kernel that multiplies on the 4 x 4 x 4 int8
// matrix instruction (gemv_quad.hip: the same arithmetic and the same bits per row, one pass over the weight for four rows);
// what is left of a batch, one or two rows, takes the dot-product kernel.
// Batches of the 32-value formats from here on go up to sixteen rows at a time through the kernel that multiplies on the 16 x 16 x 32
// int8 matrix instruction (gemv_wide.hip: the same bits per row); what is left of a batch goes on as a batch of its own. Its cost is the quantiser's, per activation row and workgroup,
// plus the weight once; the dot-product kernel's is a launch and the weight per pass, of one to four rows by how many of them its registers hold at that width. us, dot-product |
// wide, each by itself and the weights in the Infinity Cache, three rows at 24 bits: IQ4_NL 1024 x 5120 7.4 | 9.0, 1024 x 16384 20.3 | 22.0, 2000 x 8192 16.6 | 12.2, 3000 x 5632
// 10.7 | 9.5, 4096 x 4096 8.7 | 8.3, 8000 x 1600 7.7 | 7.1, 12000 x 1600 10.1 | 8.2 (at 16 bits 2048 x 8192 9.1 | 11.3, 9000 x 2048 7.8 | 8.1; Q5_0
// 4124 x 5024 11.1 | 14.4, 2579 x 7296 11.6 | 13.5, 12677 x 1920 10.1 | 10.9: the dot-product kernel's up to 24 M weights). Four, of small weights, ahead is: this kernel
// over a whole number of its groups of 512 columns, Q5_0 2706 x 1536 6.8 | 5.6, Q4_0 1432 x 1024 at 16 bits 4.9 | 4.3; with two passes of the dot-product kernel, Q4_0 560 x 1792 9.2 | 6.4,
// MXFP4 258 x 3520 10.7 | 7.8, IQ4_XS 1498 x 2048 at 16 bits 8.6 | 5.6 (but Q5_0, whose fifth bits cost this one's items more, 412 x 14336 19.6 | 21.8); with one pass of it, up to 256 rows, which leave its CUs a row each
// or none, 0.7 .. 0.95, and from 4097 on, where a CU has its second tile, 0.83 .. 1.0 (Q5_0 at 16 bits 1.03); between these at 24 bits, IQ4_NL 300 x 1056 0.84, Q4_0 1024 x 7168 11.1 | 9.5, and at 16 over 1568 .. 3072 columns, 0.95. The
// dot-product kernel is: of Q5_0, 793 x 928 5.3 | 6.2, 696 x 4896 8.9 | 10.7; of 513 .. 1024 rows to 1536 columns, 842 x 1376 Q5_1 5.6 | 6.2; of formats with a minimum a block to 1024, 900 x 800 1.08; at 16 bits to 1536, MXFP4 1.03, and over
// the longer rows, MXFP4 399 x 4256 7.1 | 8.3; and of rows short of a group, Q4_0 900 x 352 4.5 | 5.1, unless very many, 26545 x 288 at 24 bits 0.83 (MXFP4 of up to 256 is level at 24 bits, 20 x 352 5.07 | 5.01,
// and behind at 16, 4.40 | 4.78). Over 3640 drawn products, both precisions, 0.88 of the dot-product kernel's time, 46 of them longer by more than 3 %, at most 1.08 times (this kernel for all of them 0.89, and 927
// longer, up to 1.42 times; the better of both each time 0.865).
// At 16 bits and more than 6144 columns two passes
// are ahead too: 1024 x 7168 9.2 | 10.3, 500 x 16000 15.6 | 17.4. Cold: Q4_0 34816 x 5120 at four rows 42.3 | 32.6, at five 62.9 | 38.9; sixteen: IQ4_NL 1467 x 1760 37.1 | 12.1, Q4_0
// 34816 x 5120 169 | 64. Q8_0 has the others at three and four rows of up to 5120 columns: three, dot-product |
// wide, 4096 x 4096 9.6 | 10.7; four, four-row | wide, 34816 x 5120 48.4 | 57.5, 5120 x 5120 15.1 | 17.5, 2048 x 4096 10.1 | 10.8 (but 4096 x 4096 12.5 | 11.0, 12288 x 4096 22.8 | 19.6).
static bool wide_for_four(const fhip_weight* w, bool whole) {      // of up to 8 M weights
    const size_t rows = w->rows, cols = w->cols;
    const bool q5 = w->type == FHIP_Q5_0;
    if (cols < 512) return cols >= 256 && (rows > 20480 || (whole && !q5 && rows > 10240) || (w->type == FHIP_MXFP4 && cols > 256 && rows <= 256));
    if (cols % 512 == 0 && cols <= 3072) return true;
    const bool one_pass = (w->planes == 3 ? gemv_pass_rows_p3(w, 4, 0) : gemv_pass_rows_p2(w, 4, 0)) == 4;
    if (one_pass && cols <= 3072) {
        if (rows <= 256) return !q5 || cols <= 1536;
        if (rows > 4096) return whole || !q5;
        if (q5) return whole && cols > 1536 && rows > 1536;
        if (rows > 512 && rows <= 1024 && cols <= 1536) return false;
        return cols > 1536 || w->type == FHIP_IQ4_XS || (whole && (cols > 1024 || (w->type != FHIP_Q4_1 && w->type != FHIP_Q5_1)));
    }
    if (!whole) return cols <= 6144 && !one_pass;
    return !q5 || (cols <= 12288 && !one_pass);
}
bool takes_wide(const fhip_weight* w, size_t t) {
    const size_t weights = w->rows * w->cols;
    if (w->type == FHIP_Q8_0 && t < 5 && w->cols <= 5120) return false;
    if (t < 3) return false;
    const bool q8 = w->type == FHIP_Q8_0, whole = w->planes == 3 && !q8;     // 24 bits
    if (t == 3 && weights < ((size_t)(whole && w->cols <= 8192 && w->type != FHIP_Q5_0 ? 12 : 24) << 20)) return false;
    if (t == 4 && weights < ((size_t)8 << 20) && (q8 || !wide_for_four(w, whole))) return false;
    return w->planes == 3 ? gemv_wide_supports_p3(w, t < 16 ? t : 16) : gemv_wide_supports_p2(w, t < 16 ? t : 16);
}
bool g_quad_matvec = true, g_generic_forced = false;
// What the first rows of a mat-vec batch of `left` rows take: the kernel and how many rows. Three rows of Q8_0 are one pass of the dot-product kernel
// and four one pass of the four-row one, us, dot-product | four-row, three rows: 1024 x 1024 4.8 | 5.7, 1024 x 5120 7.7 | 9.6, 2048 x 2048 6.1 | 7.3, 4096 x 4096
// 9.6 | 12.1, 12288 x 4096 16.7 | 22.0, 34816 x 5120 45.8 | 48.6; four: 1024 x 5120 9.1 | 9.9, 2048 x 2048 9.7 | 7.5, 4096 x 4096 14.3 | 12.4, 34816 x 5120 54.8 | 48.3.
struct MatvecPass { int kernel; size_t rows; };
MatvecPass matvec_pass(const fhip_weight* w, size_t left, size_t n_ff) {
    if (left >= 3 && g_quad_matvec && !g_generic_forced) {
        if (!n_ff && takes_wide(w, left)) return {FHIP_ROUTE_WIDE, left < 16 ? left : 16};
        if (w->type == FHIP_Q8_0 && left == 3) return {FHIP_ROUTE_DOT, left};
        if (w->planes == 3 ? gemv_quad_supports_p3(w, 4, n_ff) : gemv_quad_supports_p2(w, 4, n_ff)) return {FHIP_ROUTE_QUAD, left < 4 ? left : 4};
    }
    return {FHIP_ROUTE_DOT, left};
}
int launch_gemv(const fhip_weight* w, const float* d_x, size_t rows_x, float* d_y, size_t n_ff, hipStream_t s) {
    const bool p3 = w->planes == 3;
    if (rows_x < 3 || !d_x || !d_y) return p3 ? launch_gemv_p3(w, d_x, rows_x, d_y, n_ff, s) : launch_gemv_p2(w, d_x, rows_x, d_y, n_ff, s);
    const size_t out_rows = n_ff ? n_ff : w->rows;
    for (size_t m0 = 0; m0 < rows_x;) {
        const MatvecPass pass = matvec_pass(w, rows_x - m0, n_ff);
        const float* x = d_x + m0 * w->cols;
        float* y = d_y + m0 * out_rows;
        int rc;
        switch (pass.kernel) {
            case FHIP_ROUTE_WIDE: rc = p3 ? launch_gemv_wide_p3(w, x, pass.rows, y, s) : launch_gemv_wide_p2(w, x, pass.rows, y, s); break;
            case FHIP_ROUTE_QUAD: rc = p3 ? launch_gemv_quad_p3(w, x, pass.rows, y, n_ff, s) : launch_gemv_quad_p2(w, x, pass.rows, y, n_ff, s); break;
            default: rc = p3 ? launch_gemv_p3(w, x, pass.rows, y, n_ff, s) : launch_gemv_p2(w, x, pass.rows, y, n_ff, s);
        }
        if (rc) return rc;
        m0 += pass.rows;
    }
    return FHIP_OK;
}
bool gemv_quad_matvec(bool on) {
    const bool before = g_quad_matvec;
    g_quad_matvec = on;
    return before;
}
int launch_gemv_norm(const fhip_weight* w, const float* d_x, float* d_y, size_t n_ff, const NormParams& norm, hipStream_t s) {
    return w->planes == 3 ? launch_gemv_norm_p3(w, d_x, d_y, n_ff, norm, s) : launch_gemv_norm_p2(w, d_x, d_y, n_ff, norm, s);
}
int launch_gemv_sel(const fhip_weight* w, const float* d_x, float* d_y, size_t out_rows, bool swiglu, const SelParams& sel, hipStream_t s) {
    return w->planes == 3 ? launch_gemv_sel_p3(w, d_x, d_y, out_rows, swiglu, sel, s) : launch_gemv_sel_p2(w, d_x, d_y, out_rows, swiglu, sel, s);
}
void gemv_force_generic(bool on) {
    g_generic_forced = on;
    gemv_force_generic_p2(on);
    gemv_force_generic_p3(on);
}

}  // namespace fhip

using fhip::check_hip;
using fhip::set_error;

namespace {

size_t align256(size_t n) { return (n + 255) & ~(size_t)255; }

// ---- the library's own workspace, one per stream -------------------------------------------------------------------------
// The one-pass small-batch kernels need a few megabytes of device memory beside their operands (prepared activation rows,
// the gate|up intermediate). The drop-in entry points (fhip_matmul_q, fhip_matmul_q_swiglu, fhip_ffn) have no argument for
// it, so the library keeps a buffer per stream: work on one stream is ordered, so calls there can share it. It only ever
// grows, to the next power of two, and a buffer that was outgrown stays allocated until fhip_workspace_release: a graph
// captured earlier may still name it. Growing means hipMalloc, which a capturing stream does not allow.
struct StreamWs { hipStream_t s; void* cur; size_t n; std::vector<void*> retired; };
std::mutex g_ws_mu;
std::vector<StreamWs> g_ws;

// optional: *out is null where the stream has not got it and cannot be given it now (it is capturing, or no memory is left); other captures of the thread stay as they are
int lib_workspace(hipStream_t s, size_t need, void** out, const char* who, bool optional = false) {
    *out = nullptr;
    std::lock_guard<std::mutex> lock(g_ws_mu);
    StreamWs* e = nullptr;
    for (auto& w : g_ws) if (w.s == s) e = &w;
    if (e && e->n >= need) { *out = e->cur; return FHIP_OK; }
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(s, &st) != hipSuccess) (void)hipGetLastError();
    if (st != hipStreamCaptureStatusNone && optional) return FHIP_OK;
    if (st != hipStreamCaptureStatusNone)
        return set_error(FHIP_ERR_ARG, "%s: the library workspace of this stream has to grow to %zu bytes, which a capturing stream does not "
                         "allow: call fhip_workspace_reserve(stream, %zu) before the capture begins", who, need, need);
    size_t n = 1 << 20;
    while (n < need) n <<= 1;
    void* p = nullptr;
    if (optional) {
        if (!(p = fhip::device_malloc_beside_captures(n))) return FHIP_OK;
    } else if (const int rc = fhip::device_malloc(&p, n, "hipMalloc (library workspace)")) return rc;
    if (!e) { g_ws.push_back(StreamWs{s, nullptr, 0, {}}); e = &g_ws.back(); }
    if (e->cur) e->retired.push_back(e->cur);
    e->cur = p; e->n = n;
    *out = p;
    return FHIP_OK;
}

void release_workspace(hipStream_t s) {
    std::lock_guard<std::mutex> lock(g_ws_mu);
    for (size_t i = 0; i < g_ws.size(); i++) {
        if (g_ws[i].s != s) continue;
        (void)hipStreamSynchronize(s);
        if (g_ws[i].cur) (void)hipFree(g_ws[i].cur);
        for (void* p : g_ws[i].retired) (void)hipFree(p);
        g_ws.erase(g_ws.begin() + i);
        return;
    }
}

// The matrix-core GEMM with its K-split scratch (partial tiles of the tiles that several workgroups share) taken from the
// stream's library workspace.
static int gemm_bf16_lib_ws(const fhip_weight* w, const uint16_t* d_x, size_t t, float* d_y, hipStream_t s, const char* who, bool run_sums = false) {
    const size_t need = fhip::gemm_bf16_ws_bytes(w, t, run_sums);
    void* ws = nullptr;
    if (need) {
        int rc = lib_workspace(s, need, &ws, who);
        if (rc) return rc;
    }
    return fhip::launch_gemm_bf16(w, d_x, t, d_y, s, (float*)ws, need, run_sums);
}

// ---- which kernel a batch takes ---------------------------------------------------------------------------------------------
// One or two activation rows go through the streaming mat-vec (one pass over the weights serves two rows). From three rows on
// (five for Q8_0) the f16 hi/lo matrix-core kernels multiply groups of up to 32 rows (Q8_0 with sums by atomics: 16); longer batches are cut
// into such groups. FHIP_BATCH_F32_MATVEC keeps every batch on the mat-vec's arithmetic (launch_gemv: four rows a pass for Q4_K /
// Q5_K / Q6_K, up to sixteen for the 32-value formats, on the int8 matrix instructions, a few rows on the dot-product kernel): a row then has the same
// bits whatever batch it is part of.

size_t f16x2_group(const fhip_weight* w) { return w->type == FHIP_Q8_0 && w->batch_policy != FHIP_BATCH_ORDERED ? 16 : 32; }
// Three and four rows of a Q4_K / Q5_K / Q6_K weight whose rows the four-row mat-vec (gemv_quad.hip) covers in one pass (up to 10240
// columns) take that kernel under every policy: one launch, no workspace, and the bits of a batch of one, which callers are promised. The f16 kernels are the faster
// ones where sums are in order (4 rows, us, this kernel | held or resident: 1024 x 5120 Q4_K 10.9 | 7.1, 5120 x 5120 12.3 | 10.3, 34816 x 5120 29.5 | 26.2, Q6_K 151936 x 5120
// 162 | 136); with atomic sums they were level (12.5 | 12.6, 7168 x 5120 14.1 | 14.5, the last 164 | 178). Longer rows take two passes (5120 x 17408 43.8 | 18.4) and stay on the f16 kernels.
bool matmul_takes_quad(const fhip_weight* w, size_t t) {
    if (t < 3 || t > 4 || w->cols > 10240) return false;      // (Q8_0: 5120, gemv_quad_supports)
    return w->planes == 3 ? fhip::gemv_quad_supports_p3(w, t, 0) : fhip::gemv_quad_supports_p2(w, t, 0);
}
bool takes_f16x2(const fhip_weight* w, size_t rows_x) {
    if (w->batch_policy == FHIP_BATCH_F32_MATVEC) return false;
    if (w->type != FHIP_Q4_K && w->type != FHIP_Q5_K && w->type != FHIP_Q6_K && w->type != FHIP_Q8_0) return false;
    if (rows_x < (w->type == FHIP_Q8_0 ? 5u : 3u)) return false;
    if (matmul_takes_quad(w, rows_x)) return false;
    return fhip::gemm_f16x2_takes(w, rows_x < f16x2_group(w) ? rows_x : f16x2_group(w));
}

// Fused gate|up + SwiGLU at three or four rows: one pass of the int8 matrix-instruction mat-vec (gemv_quad.hip, 32 us on
// 34816 x 5120), whose rows carry the bits they have in a batch of one; the f16 kernel and the SwiGLU launch behind it take 24 + 4
// with sums in order, 31 + 5 by atomics. The down projection of such batches stays on the f16 kernels (5120 x 17408: 21 us against 43).
bool swiglu_takes_quad(const fhip_weight* gu, size_t t) {
    if (t < 3 || t > 4 || gu->rows % 2 != 0 || gu->cols > 10240) return false;   // (one pass of the kernel, as matmul_takes_quad)
    return gu->planes == 3 ? fhip::gemv_quad_supports_p3(gu, t, gu->rows / 2) : fhip::gemv_quad_supports_p2(gu, t, gu->rows / 2);
}

// fhip_ffn on a group of t rows needs no library workspace when the down projection does not take the f16 kernels, or when
// gate|up takes neither them nor the four-row mat-vec: both matmuls then go through the mat-vec launcher.
bool ffn_direct(const fhip_weight* gu, const fhip_weight* down, size_t t) {
    return !takes_f16x2(down, t) || (!takes_f16x2(gu, t) && !swiglu_takes_quad(gu, t));
}

// y [t, rows] = 0 on the stream, by the mat-vec launcher's fill kernel (what a weight without columns gives)
int zero_outputs(size_t t, size_t rows, float* d_y, hipStream_t s) {
    fhip_weight z{};
    z.type = FHIP_Q8_0; z.rows = rows; z.cols = 0; z.planes = 2;
    return fhip::launch_gemv(&z, d_y, t, d_y, 0, s);
}

// y [t, w->rows] = x [t, cols] W^T for t rows of one group; ws: f16x2_matmul_ws(w, t) bytes
// (FHIP_BATCH_ORDERED: behind the prepared activations, the partial outputs of the ranges that K is cut into)
size_t f16x2_matmul_ws(const fhip_weight* w, size_t t) {
    return align256(fhip::gemm_f16x2_xp_bytes(w, t)) + (w->batch_policy == FHIP_BATCH_ORDERED ? align256(fhip::gemm_f16x2_parts_bytes(w, t)) : 0);
}
// What such a product takes: the held kernel, or one whose operand rows are made by itself or prepared (own: the rows come as they are)
int f16x2_route(const fhip_weight* w, const float* d_x, size_t t, bool own, const float* d_y) {
    if (own && fhip::gemm_f16x2_held(w, d_x, t, d_y)) return FHIP_ROUTE_HELD;
    if (w->batch_policy == FHIP_BATCH_ORDERED)
        return (own && fhip::gemm_f16x2_resident_own_x(w, d_x, t, d_y) ? FHIP_ROUTE_OWN_ROWS : FHIP_ROUTE_PREPARED) | (fhip::gemm_f16x2_parts(w, t) > 1 ? FHIP_ROUTE_CUT : 0);
    const bool cut = fhip::gemm_f16x2_adds_into_y(w, t);   // along K
    return (own && !cut && fhip::gemm_f16x2_own_x(w, d_x, t) ? FHIP_ROUTE_OWN_ROWS : FHIP_ROUTE_PREPARED) | (cut ? FHIP_ROUTE_CUT : 0);
}
// deferred: the sum of partial outputs is left to the reader of y, which gets *deferred as its `src`
int f16x2_launch(int route, const fhip_weight* w, const float* d_x, size_t t, bool swiglu_in, float* d_y, void* d_ws, hipStream_t s,
                 fhip::F16Parts* deferred, const fhip::F16Parts* src) {
    if (deferred) *deferred = fhip::F16Parts{nullptr, 0, 0, 0};
    if (route == FHIP_ROUTE_HELD) return fhip::launch_gemm_f16x2_held(w, d_x, t, d_y, s);
    uint16_t* xp = (route & ~FHIP_ROUTE_CUT) == FHIP_ROUTE_OWN_ROWS ? nullptr : (uint16_t*)d_ws;
    const bool cut = (route & FHIP_ROUTE_CUT) != 0, ordered = w->batch_policy == FHIP_BATCH_ORDERED;
    const bool clr = cut && !ordered;   // then the split clears y on the side
    int rc = xp ? fhip::launch_xsplit_f16(w, d_x, t, swiglu_in, xp, s, clr ? d_y : nullptr, clr ? t * w->rows : 0, src) : FHIP_OK;
    if (rc) return rc;
    float* part = cut && d_ws ? (float*)((uint8_t*)d_ws + align256(fhip::gemm_f16x2_xp_bytes(w, t))) : nullptr;
    if (ordered) return fhip::launch_gemm_f16x2_resident(w, xp, d_x, t, d_y, part, s, deferred);
    return fhip::launch_gemm_f16x2(w, xp, t, d_y, s, clr, xp ? nullptr : d_x);
}
int f16x2_matmul(const fhip_weight* w, const float* d_x, size_t t, bool swiglu_in, float* d_y, void* d_ws, hipStream_t s,
                 fhip::F16Parts* deferred = nullptr, const fhip::F16Parts* src = nullptr) {
    return f16x2_launch(f16x2_route(w, d_x, t, !swiglu_in && !src, d_y), w, d_x, t, swiglu_in, d_y, d_ws, s, deferred, src);
}

}  // namespace

extern "C" {

int fhip_init(int device) {
    int n = 0;
    int rc = check_hip(hipGetDeviceCount(&n), "hipGetDeviceCount");
    if (rc) return rc;
    if (device < 0 || device >= n) return set_error(FHIP_ERR_ARG, "device %d out of range (%d visible)", device, n);
    if ((rc = check_hip(hipSetDevice(device), "hipSetDevice"))) return rc;
    hipDeviceProp_t prop;
    if ((rc = check_hip(hipGetDeviceProperties(&prop, device), "hipGetDeviceProperties"))) return rc;
    if (strncmp(prop.gcnArchName, "gfx950", 6) != 0)
        return set_error(FHIP_ERR_HIP, "device %d is %s; this library carries gfx950 code only", device, prop.gcnArchName);
    g_cus = prop.multiProcessorCount;
    g_lds = prop.sharedMemPerBlockOptin > prop.sharedMemPerBlock ? prop.sharedMemPerBlockOptin : prop.sharedMemPerBlock;
    if (g_lds < 64 * 1024) g_lds = 64 * 1024;
    if (device < MAX_DEVICES && !g_scratch_ptr[device]) {   // this device's copy of the built-in scratch array
        float* ptr = nullptr;
        if ((rc = check_hip(hipGetSymbolAddress((void**)&ptr, HIP_SYMBOL(scratch)), "hipGetSymbolAddress(scratch)"))) return rc;
        g_scratch_ptr[device] = ptr;
    }
    g_device = device;
    return FHIP_OK;
}

const char* fhip_last_error(void) { return g_err; }
int fhip_device_cus(void) { return g_cus; }

// bytes per element of the unquantized tensor types (crates/ferric-gguf/src/lib.rs:473-475), 0 for anything else
static size_t dense_elem_bytes(uint32_t ty) { return ty == FHIP_F32 ? 4 : (ty == FHIP_F16 || ty == FHIP_BF16 ? 2 : 0); }

size_t fhip_type_size(uint32_t ty, size_t n) {
    if (const size_t eb = dense_elem_bytes(ty)) return n * eb;
    size_t vals, bytes;
    if (!block_info(ty, vals, bytes)) { set_error(FHIP_ERR_UNSUPPORTED_TYPE, "unsupported ggml type %u", ty); return 0; }
    return n / vals * bytes;
}

int fhip_block_bytes(uint32_t ty, size_t* values, size_t* bytes) {
    size_t v, b;
    if (!values || !bytes) return set_error(FHIP_ERR_ARG, "fhip_block_bytes: NULL output");
    if (!block_info(ty, v, b)) return set_error(FHIP_ERR_UNSUPPORTED_TYPE, "unsupported ggml type %u", ty);
    *values = v; *bytes = b;
    return FHIP_OK;
}

// ---- plumbing -------------------------------------------------------------------------------

int fhip_malloc(void** d_ptr, size_t nbytes) {
    if (!d_ptr) return set_error(FHIP_ERR_ARG, "fhip_malloc: NULL output");
    int rc = need_init();
    if (rc) return rc;
    *d_ptr = nullptr;
    // 256 bytes more than asked for: a weight wrapped at the end of such a buffer (fhip_weight_wrap_device) keeps the slack
    // behind its last block that fhip_weight_create gives its own allocations
    return fhip::pool_malloc(d_ptr, nbytes);
}
int fhip_free(void* d_ptr) { return d_ptr ? fhip::pool_free(d_ptr) : FHIP_OK; }
int fhip_memcpy_h2d(void* d, const void* h, size_t n, void* s) {
    if (n == 0) return FHIP_OK;
    if (!d || !h) return set_error(FHIP_ERR_ARG, "fhip_memcpy_h2d: NULL pointer");
    return fhip::copy_h2d(d, h, n, (hipStream_t)s);
}
int fhip_upload(void* d, const void* h, size_t n, void* s) {
    if (n == 0) return FHIP_OK;
    if (!d || !h) return set_error(FHIP_ERR_ARG, "fhip_upload: NULL pointer");
    return fhip::upload(d, h, n, (hipStream_t)s);
}
int fhip_memcpy_d2h(void* h, const void* d, size_t n, void* s) {
    if (n == 0) return FHIP_OK;
    if (!d || !h) return set_error(FHIP_ERR_ARG, "fhip_memcpy_d2h: NULL pointer");
    return fhip::copy_d2h(h, d, n, (hipStream_t)s);
}
int fhip_memcpy_d2d(void* dst, const void* src, size_t n, void* s) {
    if (n == 0) return FHIP_OK;
    if (!dst || !src) return set_error(FHIP_ERR_ARG, "fhip_memcpy_d2d: NULL pointer");
    return check_hip(hipMemcpyAsync(dst, src, n, hipMemcpyDeviceToDevice, (hipStream_t)s), "hipMemcpyAsync D2D");
}
int fhip_memcpy_2d_d2d(void* d, size_t dpitch, const void* src, size_t spitch, size_t width, size_t height, void* s) {
    if (width == 0 || height == 0) return FHIP_OK;
    if (!d || !src) return set_error(FHIP_ERR_ARG, "fhip_memcpy_2d_d2d: NULL pointer");
    if (dpitch < width || spitch < width) return set_error(FHIP_ERR_ARG, "fhip_memcpy_2d_d2d: pitch smaller than the row width");
    return check_hip(hipMemcpy2DAsync(d, dpitch, src, spitch, width, height, hipMemcpyDeviceToDevice, (hipStream_t)s), "hipMemcpy2D D2D");
}
int fhip_memset(void* d, int byte, size_t n, void* s) {
    if (n == 0) return FHIP_OK;
    if (!d) return set_error(FHIP_ERR_ARG, "fhip_memset: NULL pointer");
    return check_hip(hipMemsetAsync(d, byte, n, (hipStream_t)s), "hipMemsetAsync");
}
int fhip_stream_create(void** s) {
    if (!s) return set_error(FHIP_ERR_ARG, "fhip_stream_create: NULL output");
    int rc = need_init();
    if (rc) return rc;
    hipStream_t st;
    rc = check_hip(hipStreamCreateWithFlags(&st, hipStreamNonBlocking), "hipStreamCreate");
    *s = rc ? nullptr : (void*)st;
    return rc;
}
int fhip_stream_destroy(void* s) {
    if (!s) return FHIP_OK;
    release_workspace((hipStream_t)s);   // the library's buffer for this stream goes with it
    fhip::capture_ended((hipStream_t)s, true);
    return check_hip(hipStreamDestroy((hipStream_t)s), "hipStreamDestroy");
}
int fhip_stream_sync(void* s) { return check_hip(hipStreamSynchronize((hipStream_t)s), "hipStreamSynchronize"); }
int fhip_event_create(void** e) {
    if (!e) return set_error(FHIP_ERR_ARG, "fhip_event_create: NULL output");
    int rc = need_init();
    if (rc) return rc;
    hipEvent_t ev;
    rc = check_hip(hipEventCreate(&ev), "hipEventCreate");
    *e = rc ? nullptr : (void*)ev;
    return rc;
}
int fhip_event_destroy(void* e) { return e ? check_hip(hipEventDestroy((hipEvent_t)e), "hipEventDestroy") : FHIP_OK; }
int fhip_event_record(void* e, void* s) { return check_hip(hipEventRecord((hipEvent_t)e, (hipStream_t)s), "hipEventRecord"); }
int fhip_event_sync(void* e) { return check_hip(hipEventSynchronize((hipEvent_t)e), "hipEventSynchronize"); }
int fhip_event_elapsed_ms(void* a, void* b, float* ms) {
    if (!ms) return set_error(FHIP_ERR_ARG, "fhip_event_elapsed_ms: NULL output");
    return check_hip(hipEventElapsedTime(ms, (hipEvent_t)a, (hipEvent_t)b), "hipEventElapsedTime");
}

int fhip_graph_capture_begin(void* s) {
    int rc = need_init();
    if (rc) return rc;
    if (!s) return set_error(FHIP_ERR_ARG, "fhip_graph_capture_begin: needs a stream from fhip_stream_create");
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing((hipStream_t)s, &st) != hipSuccess) (void)hipGetLastError();
    if (st != hipStreamCaptureStatusActive) fhip::capture_begun((hipStream_t)s);   // (begun twice: the runtime says so, and the first one stays)
    rc = check_hip(hipStreamBeginCapture((hipStream_t)s, hipStreamCaptureModeThreadLocal), "hipStreamBeginCapture");
    if (rc && st != hipStreamCaptureStatusActive) fhip::capture_ended((hipStream_t)s, false);
    return rc;
}
int fhip_graph_capture_end(void* s, void** graph_exec) {
    if (!s || !graph_exec) return set_error(FHIP_ERR_ARG, "fhip_graph_capture_end: NULL argument");
    *graph_exec = nullptr;
    hipGraph_t g = nullptr;
    int rc = check_hip(hipStreamEndCapture((hipStream_t)s, &g), "hipStreamEndCapture");
    fhip::capture_ended((hipStream_t)s, false);          // whatever came of it: the thread's capture is over
    if (rc) return rc;
    hipGraphExec_t ge = nullptr;
    rc = check_hip(hipGraphInstantiate(&ge, g, nullptr, nullptr, 0), "hipGraphInstantiate");
    (void)hipGraphDestroy(g);
    if (!rc) *graph_exec = (void*)ge;
    return rc;
}
int fhip_graph_launch(void* ge, void* s) {
    if (!ge) return set_error(FHIP_ERR_ARG, "fhip_graph_launch: NULL graph");
    return check_hip(hipGraphLaunch((hipGraphExec_t)ge, (hipStream_t)s), "hipGraphLaunch");
}
int fhip_graph_destroy(void* ge) { return ge ? check_hip(hipGraphExecDestroy((hipGraphExec_t)ge), "hipGraphExecDestroy") : FHIP_OK; }

// ---- weights --------------------------------------------------------------------------------

int fhip_weight_create(uint32_t ty, const uint8_t* h_raw, size_t nbytes, size_t rows, size_t cols, fhip_weight** out) {
    if (!out) return set_error(FHIP_ERR_ARG, "fhip_weight_create: NULL output");
    *out = nullptr;
    int rc = need_init();
    if (rc) return rc;
    fhip_weight w;
    if ((rc = make_weight(ty, nbytes, rows, cols, w))) return rc;
    if (nbytes && !h_raw) return set_error(FHIP_ERR_ARG, "fhip_weight_create: NULL bytes");
    void* d = nullptr;
    // slack past the stream: a wide load that starts inside the last block may end behind it
    if ((rc = fhip::device_malloc(&d, nbytes + fhip::WEIGHT_SLACK, "hipMalloc(weight)"))) return rc;
    if (nbytes && (rc = check_hip(hipMemcpy(d, h_raw, nbytes, hipMemcpyHostToDevice), "hipMemcpy(weight)"))) { (void)hipFree(d); return rc; }
    if ((rc = check_hip(hipMemset((uint8_t*)d + nbytes, 0, fhip::WEIGHT_SLACK), "hipMemset(weight tail)"))) { (void)hipFree(d); return rc; }
    w.d_raw = (const uint8_t*)d;
    w.owns = true;
    *out = new fhip_weight(w);
    return FHIP_OK;
}

int fhip_weight_create_parts(uint32_t ty, const uint8_t* const* h_parts, const size_t* part_bytes, size_t n_parts, size_t rows, size_t cols,
                             fhip_weight** out) {
    if (!out) return set_error(FHIP_ERR_ARG, "fhip_weight_create_parts: NULL output");
    *out = nullptr;
    int rc = need_init();
    if (rc) return rc;
    if (n_parts && (!h_parts || !part_bytes)) return set_error(FHIP_ERR_ARG, "fhip_weight_create_parts: NULL part list");
    size_t nbytes = 0;
    for (size_t i = 0; i < n_parts; i++) {
        if (part_bytes[i] && !h_parts[i]) return set_error(FHIP_ERR_ARG, "fhip_weight_create_parts: NULL bytes");
        nbytes += part_bytes[i];
    }
    fhip_weight w;
    if ((rc = make_weight(ty, nbytes, rows, cols, w))) return rc;
    void* d = nullptr;
    if ((rc = fhip::device_malloc(&d, nbytes + fhip::WEIGHT_SLACK, "hipMalloc(weight)"))) return rc;
    size_t at = 0;
    for (size_t i = 0; i < n_parts && !rc; i++) {
        if (part_bytes[i]) rc = check_hip(hipMemcpy((uint8_t*)d + at, h_parts[i], part_bytes[i], hipMemcpyHostToDevice), "hipMemcpy(weight)");
        at += part_bytes[i];
    }
    if (!rc) rc = check_hip(hipMemset((uint8_t*)d + nbytes, 0, 256), "hipMemset(weight tail)");
    if (rc) { (void)hipFree(d); return rc; }
    w.d_raw = (const uint8_t*)d;
    w.owns = true;
    *out = new fhip_weight(w);
    return FHIP_OK;
}

int fhip_weight_wrap_device(uint32_t ty, const uint8_t* d_raw, size_t nbytes, size_t rows, size_t cols, fhip_weight** out) {
    if (!out) return set_error(FHIP_ERR_ARG, "fhip_weight_wrap_device: NULL output");
    *out = nullptr;
    int rc = need_init();
    if (rc) return rc;
    fhip_weight w;
    if ((rc = make_weight(ty, nbytes, rows, cols, w))) return rc;
    if (nbytes && !d_raw) return set_error(FHIP_ERR_ARG, "fhip_weight_wrap_device: NULL bytes");
    if (((uintptr_t)d_raw & 15) != 0) return set_error(FHIP_ERR_ARG, "fhip_weight_wrap_device: bytes must be 16-byte aligned");
    if (nbytes) {   // the allocation has to reach fhip::WEIGHT_SLACK bytes past the last block, as the library's own weights do
        uintptr_t start = 0, end = 0;
        if (!fhip::pool_range(d_raw, &start, &end)) {
            hipDeviceptr_t base = nullptr;
            size_t size = 0;
            if (hipMemGetAddressRange(&base, &size, (hipDeviceptr_t)d_raw) != hipSuccess) {
                (void)hipGetLastError();
                return set_error(FHIP_ERR_ARG, "fhip_weight_wrap_device: not a device allocation");
            }
            end = (uintptr_t)base + size;
        }
        const uintptr_t need = (uintptr_t)d_raw + nbytes + fhip::WEIGHT_SLACK;
        if (need > end)
            return set_error(FHIP_ERR_ARG, "fhip_weight_wrap_device: the allocation must extend %zu bytes past the weight's last block "
                             "(it ends %zu bytes behind it); buffers from fhip_malloc always do", fhip::WEIGHT_SLACK, (size_t)(end - ((uintptr_t)d_raw + nbytes)));
    }
    w.d_raw = d_raw;
    w.owns = false;
    *out = new fhip_weight(w);
    return FHIP_OK;
}

void fhip_weight_destroy(fhip_weight* w) {
    if (!w) return;
    if (w->owns && w->d_raw) (void)hipFree((void*)w->d_raw);
    delete w;
}

size_t fhip_weight_rows(const fhip_weight* w) { return w ? w->rows : 0; }
size_t fhip_weight_cols(const fhip_weight* w) { return w ? w->cols : 0; }
size_t fhip_weight_nbytes(const fhip_weight* w) { return w ? w->nbytes : 0; }
uint32_t fhip_weight_type(const fhip_weight* w) { return w ? w->type : 0; }

// ---- unpackers ------------------------------------------------------------------------------

int fhip_f16_to_f32(const uint16_t* d_bits, size_t n, float* d_out, void* stream) {
    int rc = need_init();
    if (rc) return rc;
    if (n && (!d_bits || !d_out)) return set_error(FHIP_ERR_ARG, "fhip_f16_to_f32: NULL pointer");
    return fhip::launch_f16_to_f32(d_bits, n, d_out, (hipStream_t)stream);
}

int fhip_dequant_rows(const fhip_weight* w, size_t row0, size_t nrows, float* d_out, void* stream) {
    int rc = need_init();
    if (rc) return rc;
    if (!w) return set_error(FHIP_ERR_ARG, "fhip_dequant_rows: NULL weight");
    if (row0 > w->rows || nrows > w->rows - row0) return set_error(FHIP_ERR_SHAPE, "fhip_dequant_rows: rows [%zu, %zu) outside [0, %zu)", row0, row0 + nrows, w->rows);
    if (nrows == 0 || w->cols == 0) return FHIP_OK;
    if (!d_out) return set_error(FHIP_ERR_ARG, "fhip_dequant_rows: NULL output");
    size_t vals, bytes;
    block_info(w->type, vals, bytes);
    return fhip::launch_dequant(w->type, w->d_raw + row0 * w->row_bytes, nrows * (w->cols / vals), d_out, (hipStream_t)stream);
}

int fhip_deq_raw(const uint8_t* h_raw, size_t nbytes, size_t n, uint32_t ty, float* h_out, size_t* n_written) {
    int rc = need_init();
    if (rc) return rc;
    if (const size_t eb = dense_elem_bytes(ty)) {
        // lib.rs:499-501: raw[..n * size] first (a panic when the bytes are short), then exactly n values
        if (nbytes / eb < n) return set_error(FHIP_ERR_SHAPE, "range end index %zu out of range for slice of length %zu", n * eb, nbytes);
        if (n_written) *n_written = n;
        if (n == 0) return FHIP_OK;
        if (!h_raw || !h_out) return set_error(FHIP_ERR_ARG, "fhip_deq_raw: NULL pointer");
        if (ty == FHIP_F32) { memcpy(h_out, h_raw, n * 4); return FHIP_OK; }   // the bytes as they are
        void *d_in = nullptr, *d_out = nullptr;
        if ((rc = check_hip(hipMalloc(&d_in, n * 2), "hipMalloc"))) return rc;
        if ((rc = check_hip(hipMalloc(&d_out, n * sizeof(float)), "hipMalloc"))) { (void)hipFree(d_in); return rc; }
        rc = check_hip(hipMemcpy(d_in, h_raw, n * 2, hipMemcpyHostToDevice), "hipMemcpy H2D");
        if (!rc) rc = ty == FHIP_F16 ? fhip::launch_f16_to_f32((const uint16_t*)d_in, n, (float*)d_out, nullptr)
                                     : fhip::launch_bf16_to_f32((const uint16_t*)d_in, n, (float*)d_out, nullptr);
        if (!rc) rc = check_hip(hipMemcpy(h_out, d_out, n * sizeof(float), hipMemcpyDeviceToHost), "hipMemcpy D2H");
        (void)hipFree(d_in);
        (void)hipFree(d_out);
        return rc;
    }
    size_t vals, bytes;
    if (!block_info(ty, vals, bytes)) return set_error(FHIP_ERR_UNSUPPORTED_TYPE, "unsupported ggml type %u", ty);
    if (n && !h_out) return set_error(FHIP_ERR_ARG, "fhip_deq_raw: NULL output");
    size_t nb = n / vals;
    if (nbytes / bytes < nb) nb = nbytes / bytes;  // chunks_exact(..).take(n / blk)
    if (nb && !h_raw) return set_error(FHIP_ERR_ARG, "fhip_deq_raw: NULL bytes");
    // Every dequantizer but Q8_0's pre-sizes the output to n zeros (lib.rs:619, :634, :651, :670, :693, :722, :794); Q8_0
    // pushes whole blocks only and so returns a shorter vector (lib.rs:609-614).
    size_t produced = ty == FHIP_Q8_0 ? nb * vals : n;
    if (n_written) *n_written = produced;
    if (nb && (rc = fhip::dequant_host(ty, h_raw, nb, vals, bytes, h_out))) return rc;
    for (size_t i = nb * vals; i < produced; i++) h_out[i] = 0.0f;
    return FHIP_OK;
}

// ---- matmuls --------------------------------------------------------------------------------

int fhip_matmul_q(const fhip_weight* w, const float* d_x, size_t rows_x, float* d_y, void* stream) {
    int rc = need_init();
    if (rc) return rc;
    if (!w) return set_error(FHIP_ERR_ARG, "fhip_matmul_q: NULL weight");
    if (rows_x == 0 || w->rows == 0) return FHIP_OK;
    if (!d_x || !d_y) return set_error(FHIP_ERR_ARG, "fhip_matmul_q: NULL pointer");
    if (((uintptr_t)d_x & 15) != 0) return set_error(FHIP_ERR_ARG, "fhip_matmul_q: x must be 16-byte aligned");
    hipStream_t s = (hipStream_t)stream;
    if (!takes_f16x2(w, rows_x)) return fhip::launch_gemv(w, d_x, rows_x, d_y, 0, s);
    const size_t grp = f16x2_group(w);
    void* ws = nullptr;
    if (rows_x <= grp) {   // one group: the held kernel needs no workspace
        int route = f16x2_route(w, d_x, rows_x, true, d_y);
        if (route != FHIP_ROUTE_HELD && route != FHIP_ROUTE_OWN_ROWS) {
            const bool without = fhip::gemm_f16x2_held_takes(w, d_x, rows_x, d_y);
            if ((rc = lib_workspace(s, f16x2_matmul_ws(w, rows_x), &ws, "fhip_matmul_q", without))) return rc;
            // No workspace, mostly a capture on a stream that has none. Sums in order: the ranges of K one after the other, the same bits, in the
            // time of as many launches (us with the workspace | without, replayed: Q4_K 8 rows, 2048 x 5120 8.5 | 40, 34816 x 5120 27.5 | 44, 32 rows 2048 x 5120 15 | 80). By atomics:
            // the held kernel's one launch, whose order is as good as any.
            if (!ws) route = w->batch_policy == FHIP_BATCH_ORDERED ? FHIP_ROUTE_OWN_ROWS | FHIP_ROUTE_CUT : FHIP_ROUTE_HELD;
        }
        return f16x2_launch(route, w, d_x, rows_x, false, d_y, ws, s, nullptr, nullptr);
    }
    if ((rc = lib_workspace(s, f16x2_matmul_ws(w, grp), &ws, "fhip_matmul_q"))) return rc;
    for (size_t m0 = 0; m0 < rows_x; m0 += grp) {
        const size_t t = rows_x - m0 < grp ? rows_x - m0 : grp;
        if (takes_f16x2(w, t)) rc = f16x2_matmul(w, d_x + m0 * w->cols, t, false, d_y + m0 * w->rows, ws, s);
        else rc = fhip::launch_gemv(w, d_x + m0 * w->cols, t, d_y + m0 * w->rows, 0, s);   // a last group of one or two rows
        if (rc) return rc;
    }
    return FHIP_OK;
}

int fhip_matmul_q_swiglu(const fhip_weight* gu, const float* d_x, size_t rows_x, float* d_y, void* stream) {
    int rc = need_init();
    if (rc) return rc;
    if (!gu) return set_error(FHIP_ERR_ARG, "fhip_matmul_q_swiglu: NULL weight");
    if (gu->type == FHIP_Q8_0) return set_error(FHIP_ERR_UNSUPPORTED_TYPE, "try_matmul_swiglu: no fused kernel for Q8_0");
    if (gu->rows % 2 != 0) return set_error(FHIP_ERR_SHAPE, "matmul_swiglu: gate_up rows must be even");
    if (rows_x == 0 || gu->rows == 0) return FHIP_OK;
    if (!d_x || !d_y) return set_error(FHIP_ERR_ARG, "fhip_matmul_q_swiglu: NULL pointer");
    if (((uintptr_t)d_x & 15) != 0) return set_error(FHIP_ERR_ARG, "fhip_matmul_q_swiglu: x must be 16-byte aligned");
    hipStream_t s = (hipStream_t)stream;
    const size_t n_ff = gu->rows / 2;
    if (!takes_f16x2(gu, rows_x) || swiglu_takes_quad(gu, rows_x)) return fhip::launch_gemv(gu, d_x, rows_x, d_y, n_ff, s);
    // gate|up for the group in one pass into the workspace, then the reference's un-fused SwiGLU over it
    const size_t grp = f16x2_group(gu), t0 = rows_x < grp ? rows_x : grp;
    const size_t mm = f16x2_matmul_ws(gu, t0);
    void* ws = nullptr;
    if ((rc = lib_workspace(s, mm + align256(t0 * gu->rows * sizeof(float)), &ws, "fhip_matmul_q_swiglu"))) return rc;
    float* g = (float*)((uint8_t*)ws + mm);
    for (size_t m0 = 0; m0 < rows_x; m0 += grp) {
        const size_t t = rows_x - m0 < grp ? rows_x - m0 : grp;
        if (!takes_f16x2(gu, t) || swiglu_takes_quad(gu, t)) { rc = fhip::launch_gemv(gu, d_x + m0 * gu->cols, t, d_y + m0 * n_ff, n_ff, s); }
        else if (!(rc = f16x2_matmul(gu, d_x + m0 * gu->cols, t, false, g, ws, s))) rc = fhip::launch_swiglu(g, t, n_ff, d_y + m0 * n_ff, s);
        if (rc) return rc;
    }
    return FHIP_OK;
}

int fhip_swiglu(const float* d_gu, size_t t, size_t d, float* d_out, void* stream) {
    int rc = need_init();
    if (rc) return rc;
    if (t * d == 0) return FHIP_OK;
    if (!d_gu || !d_out) return set_error(FHIP_ERR_ARG, "fhip_swiglu: NULL pointer");
    return fhip::launch_swiglu(d_gu, t, d, d_out, (hipStream_t)stream);
}

int fhip_ffn(const fhip_weight* gu, const fhip_weight* down, const float* d_x, size_t rows_x, float* d_y, float* d_ws, void* stream) {
    int rc = need_init();
    if (rc) return rc;
    if (!gu || !down) return set_error(FHIP_ERR_ARG, "fhip_ffn: NULL weight");
    if (gu->rows % 2 != 0) return set_error(FHIP_ERR_SHAPE, "ffn: gate_up rows must be even");
    size_t n_ff = gu->rows / 2;
    // crates/ferric-tensor/src/dtype.rs:979-981: down in dim must equal n_ff, down out dim is the model width.
    if (down->cols != n_ff) return set_error(FHIP_ERR_SHAPE, "down in dim must equal n_ff");
    if (rows_x == 0) return FHIP_OK;
    if (!d_x || !d_y || !d_ws) return set_error(FHIP_ERR_ARG, "fhip_ffn: NULL pointer");
    if (gu->type == FHIP_Q8_0) {
        // no fused gate/up kernel for this format: matmul_q then swiglu, as the reference's callers
        // do when try_matmul_swiglu returns None (crates/ferric-llama/src/qwen3.rs:219-227). The
        // [rows_x, 2 n_ff] intermediate then also lives in d_ws, which this path needs 3x larger.
        return set_error(FHIP_ERR_UNSUPPORTED_TYPE, "fhip_ffn: gate_up must be Q4_K or Q6_K");
    }
    hipStream_t s = (hipStream_t)stream;
    size_t grp = f16x2_group(gu) < f16x2_group(down) ? f16x2_group(gu) : f16x2_group(down);
    const size_t t0 = rows_x < grp ? rows_x : grp;
    if (ffn_direct(gu, down, t0)) {
        if ((rc = fhip::launch_gemv(gu, d_x, rows_x, d_ws, n_ff, s))) return rc;
        return fhip::launch_gemv(down, d_ws, rows_x, d_y, 0, s);
    }
    // groups of up to 32 rows, each one pass over gate|up and one over down; SwiGLU happens while the rows are prepared
    // for the down projection. The intermediates live in the library's workspace; d_ws is left alone.
    const size_t mm1 = f16x2_matmul_ws(gu, t0), gb = align256(t0 * gu->rows * sizeof(float));
    void* ws = nullptr;
    if ((rc = lib_workspace(s, mm1 + gb + f16x2_matmul_ws(down, t0), &ws, "fhip_ffn"))) return rc;
    float* g = (float*)((uint8_t*)ws + mm1);
    void* ws2 = (uint8_t*)ws + mm1 + gb;
    for (size_t m0 = 0; m0 < rows_x; m0 += grp) {
        const size_t t = rows_x - m0 < grp ? rows_x - m0 : grp;
        if (ffn_direct(gu, down, t)) {
            if ((rc = fhip::launch_gemv(gu, d_x + m0 * gu->cols, t, d_ws + m0 * n_ff, n_ff, s))) return rc;
            rc = fhip::launch_gemv(down, d_ws + m0 * n_ff, t, d_y + m0 * down->rows, 0, s);
        } else if (swiglu_takes_quad(gu, t)) {
            // three or four rows: silu(gate) * up straight out of the mat-vec, then the down projection's one pass over it
            if (!(rc = fhip::launch_gemv(gu, d_x + m0 * gu->cols, t, g, n_ff, s)))
                rc = f16x2_matmul(down, g, t, false, d_y + m0 * down->rows, ws2, s);
        } else {
            // under the ordered policy gate|up's K-split groups stay partial sums; the split for the down projection adds them
            fhip::F16Parts parts{nullptr, 0, 0, 0};
            if (!(rc = f16x2_matmul(gu, d_x + m0 * gu->cols, t, false, g, ws, s, &parts)))
                rc = f16x2_matmul(down, g, t, true, d_y + m0 * down->rows, ws2, s, nullptr, &parts);
        }
        if (rc) return rc;
    }
    return FHIP_OK;
}

int fhip_ffn_noalloc(const fhip_weight* gu, const fhip_weight* down, const float* d_x, size_t rows_x, float* d_y, void* stream) {
    int rc = need_init();
    if (rc) return rc;
    if (!gu || !down) return set_error(FHIP_ERR_ARG, "fhip_ffn_noalloc: NULL weight");
    if (gu->rows % 2 != 0) return set_error(FHIP_ERR_SHAPE, "ffn: gate_up rows must be even");
    const size_t n_ff = gu->rows / 2;
    if (down->cols != n_ff) return set_error(FHIP_ERR_SHAPE, "down in dim must equal n_ff");
    if (rows_x == 0) return FHIP_OK;
    if (!d_x || !d_y) return set_error(FHIP_ERR_ARG, "fhip_ffn_noalloc: NULL pointer");
    if (gu->type == FHIP_Q8_0) return set_error(FHIP_ERR_UNSUPPORTED_TYPE, "fhip_ffn_noalloc: gate_up must be Q4_K or Q6_K");
    if (rows_x > NOALLOC_FLOATS / (n_ff ? n_ff : 1))
        return set_error(FHIP_ERR_SHAPE, "fhip_ffn_noalloc: rows_x * n_ff = %zu * %zu floats do not fit the built-in scratch of %zu floats; use fhip_ffn",
                         rows_x, n_ff, NOALLOC_FLOATS);
    float* h = g_device < MAX_DEVICES ? g_scratch_ptr[g_device] : nullptr;
    if (!h) return set_error(FHIP_ERR_HIP, "fhip_ffn_noalloc: no scratch address for device %d", g_device);
    // the mat-vec kernels for every batch width (they need nothing beside operands and this intermediate; the one-pass
    // kernels of fhip_ffn would need the library's workspace); every element of h is written before it is read
    hipStream_t s = (hipStream_t)stream;
    if ((rc = fhip::launch_gemv(gu, d_x, rows_x, h, n_ff, s))) return rc;
    return fhip::launch_gemv(down, h, rows_x, d_y, 0, s);
}

static bool known_policy(int policy) { return policy == FHIP_BATCH_AUTO || policy == FHIP_BATCH_F32_MATVEC || policy == FHIP_BATCH_ORDERED; }

int fhip_batch_policy(int policy) {
    const int before = g_default_batch_policy;
    if (known_policy(policy)) g_default_batch_policy = policy;
    return before;
}

int fhip_weight_batch_policy(fhip_weight* w, int policy) {
    if (!w) return set_error(FHIP_ERR_ARG, "fhip_weight_batch_policy: NULL weight");
    const int before = w->batch_policy;
    if (known_policy(policy)) w->batch_policy = policy;
    return before;
}

int fhip_weight_matvec_precision(fhip_weight* w, int bits) {
    if (!w) return set_error(FHIP_ERR_ARG, "fhip_weight_matvec_precision: NULL weight");
    const int before = w->planes == 3 ? 24 : 16;
    if (bits == 0) return before;
    if (bits != 16 && bits != 24) return set_error(FHIP_ERR_ARG, "fhip_weight_matvec_precision: 16 or 24 bits (0 to query), not %d", bits);
    w->planes = bits == 24 ? 3 : 2;
    return before;
}

int fhip_workspace_reserve(void* stream, size_t nbytes) {
    int rc = need_init();
    if (rc) return rc;
    void* p = nullptr;
    return nbytes ? lib_workspace((hipStream_t)stream, nbytes, &p, "fhip_workspace_reserve") : FHIP_OK;
}

size_t fhip_workspace_bytes(const fhip_weight* gu, const fhip_weight* down, size_t rows_x) {
    // what fhip_matmul_q (down == NULL), fhip_matmul_q_swiglu (down == NULL) or fhip_ffn asks of the workspace: the largest
    size_t need = 0;
    if (!gu || rows_x == 0) return 0;
    if (down) {      // fhip_ffn: [gate|up's workspace][the t0 x 2 n_ff intermediate][down's workspace], t0 the widest group
        const size_t grp = f16x2_group(gu) < f16x2_group(down) ? f16x2_group(gu) : f16x2_group(down);
        const size_t t0 = rows_x < grp ? rows_x : grp;
        if (ffn_direct(gu, down, t0)) return 0;
        return f16x2_matmul_ws(gu, t0) + align256(t0 * gu->rows * sizeof(float)) + f16x2_matmul_ws(down, t0);
    }
    if (takes_f16x2(gu, rows_x)) {
        const size_t t0 = rows_x < f16x2_group(gu) ? rows_x : f16x2_group(gu);
        need = f16x2_matmul_ws(gu, t0) + align256(t0 * gu->rows * sizeof(float));
    }
    return need;
}

size_t fhip_workspace_bytes_coop(const fhip_weight* w, const fhip_weight* down, size_t rows_x) {
    // A smaller batch may need more than a larger one, whose tiles fill the chip whole: the most over the batches up to rows_x. A plan
    // follows from the number of 64-row tiles (more than 32 rows) or from the staged rows (8 or 32).
    size_t need = 0;
    auto most = [&](size_t t) {
        for (size_t n : {fhip::gemm_bf16_ws_bytes(w, t), fhip::gemm_bf16_ws_bytes(down, t), fhip::gemm_bf16_swiglu_ws_bytes(w, t), fhip::gemm_bf16_ws_bytes(w, t, true),
                         fhip::gemm_bf16_ws_bytes(down, t, true)}) need = n > need ? n : need;
    };
    auto rows_of = [](const fhip_weight* q) { return q && q->cols ? (((size_t)1 << 31) - 1) / q->cols : (size_t)0; };   // launch_gemm_bf16 refuses more
    const size_t a = rows_of(w), b = rows_of(down), accepted = a > b ? a : b, last = rows_x < accepted ? rows_x : accepted;
    most(last);
    if (last > 8) most(8);
    if (last > 32) most(32);
    for (size_t t = 64; t < last; t += 64) most(t);
    return need;
}

void fhip_workspace_release(void* stream) {
    release_workspace((hipStream_t)stream);
    fhip::pool_trim();
}

static int gemm_q_bf16(const char* who, const fhip_weight* w, const uint16_t* d_x, size_t t, float* d_y, void* stream, bool run_sums) {
    int rc = need_init();
    if (rc) return rc;
    if (!w) return set_error(FHIP_ERR_ARG, "%s: NULL weight", who);
    if (t == 0 || w->rows == 0) return FHIP_OK;
    if (!d_y || (!d_x && w->cols)) return set_error(FHIP_ERR_ARG, "%s: NULL pointer", who);
    if (w->cols == 0) return zero_outputs(t, w->rows, d_y, (hipStream_t)stream);   // empty inner dimension: every dot product is 0
    return gemm_bf16_lib_ws(w, d_x, t, d_y, (hipStream_t)stream, who, run_sums);
}
int fhip_gemm_q_bf16(const fhip_weight* w, const uint16_t* d_x, size_t t, float* d_y, void* stream) {
    return gemm_q_bf16("fhip_gemm_q_bf16", w, d_x, t, d_y, stream, false);
}
int fhip_gemm_q_bf16_run_sums(const fhip_weight* w, const uint16_t* d_x, size_t t, float* d_y, void* stream) {
    return gemm_q_bf16("fhip_gemm_q_bf16_run_sums", w, d_x, t, d_y, stream, true);
}

// ---- mixture-of-experts entry points (crates/ferric-tensor/src/dtype.rs:1582-1780) ----------------------

// ---- decode-layer steps --------------------------------------------------------------------------

int fhip_rmsnorm(const float* d_x, const float* d_weight, size_t rows, size_t d, float eps, float* d_out, void* stream) {
    int rc = need_init();
    if (rc) return rc;
    if (rows == 0 || d == 0) return FHIP_OK;
    if (!d_x || !d_weight || !d_out) return set_error(FHIP_ERR_ARG, "fhip_rmsnorm: NULL pointer");
    return fhip::launch_rmsnorm(d_x, nullptr, d_weight, rows, d, eps, nullptr, d_out, (hipStream_t)stream);
}

int fhip_add_rmsnorm(const float* d_a, const float* d_b, const float* d_weight, size_t rows, size_t d, float eps, float* d_sum,
                     float* d_norm, void* stream) {
    int rc = need_init();
    if (rc) return rc;
    if (rows == 0 || d == 0) return FHIP_OK;
    if (!d_a || !d_b || !d_weight || !d_sum || !d_norm) return set_error(FHIP_ERR_ARG, "fhip_add_rmsnorm: NULL pointer");
    return fhip::launch_rmsnorm(d_a, d_b, d_weight, rows, d, eps, d_sum, d_norm, (hipStream_t)stream);
}

int fhip_add_rmsnorm_bf16(const float* d_a, const float* d_b, const float* d_weight, size_t rows, size_t d, float eps, float* d_sum,
                          uint16_t* d_norm_bf16, void* stream) {
    int rc = need_init();
    if (rc) return rc;
    if (rows == 0 || d == 0) return FHIP_OK;
    if (!d_a || !d_weight || !d_norm_bf16 || (d_b && !d_sum)) return set_error(FHIP_ERR_ARG, "fhip_add_rmsnorm_bf16: NULL pointer");
    return fhip::launch_rmsnorm_bf16(d_a, d_b, d_weight, rows, d, eps, d_b ? d_sum : nullptr, d_norm_bf16, (hipStream_t)stream);
}

int fhip_add(const float* d_a, const float* d_b, size_t n, float* d_out, void* stream) {
    int rc = need_init();
    if (rc) return rc;
    if (n == 0) return FHIP_OK;
    if (!d_a || !d_b || !d_out) return set_error(FHIP_ERR_ARG, "fhip_add: NULL pointer");
    return fhip::launch_add(d_a, d_b, n, d_out, (hipStream_t)stream);
}

int fhip_mul_sigmoid(const float* d_a, const float* d_g, size_t n, float* d_out, void* stream) {
    int rc = need_init();
    if (rc) return rc;
    if (n == 0) return FHIP_OK;
    if (!d_a || !d_g || !d_out) return set_error(FHIP_ERR_ARG, "fhip_mul_sigmoid: NULL pointer");
    return fhip::launch_mul_sigmoid(d_a, d_g, n, d_out, (hipStream_t)stream);
}

int fhip_geglu(const float* d_gu, size_t t, size_t d, float* d_out, void* stream) {
    int rc = need_init();
    if (rc) return rc;
    if (t * d == 0) return FHIP_OK;
    if (!d_gu || !d_out) return set_error(FHIP_ERR_ARG, "fhip_geglu: NULL pointer");
    return fhip::launch_geglu(d_gu, t, d, d_out, (hipStream_t)stream);
}

static int kvq_checks(const char* who, int fmt, size_t width) {
    if (fmt != FHIP_KVQ_Q8_0 && fmt != FHIP_KVQ_Q4_0 && fmt != FHIP_KVQ_Q4_1) return set_error(FHIP_ERR_ARG, "%s: unknown format %d", who, fmt);
    // crates/ferric-tensor/src/kvquant.rs:470
    if (width % 32 != 0) return set_error(FHIP_ERR_SHAPE, "QKvCache row width %zu must be a multiple of 32", width);
    return FHIP_OK;
}

int fhip_kvq_sizes(int fmt, size_t rows, size_t width, size_t* code_words, size_t* scale_words) {
    int rc = kvq_checks("fhip_kvq_sizes", fmt, width);
    if (rc) return rc;
    const size_t nblk = rows * (width / 32);
    if (code_words) *code_words = nblk * (fmt == FHIP_KVQ_Q8_0 ? 8 : 4);
    if (scale_words) *scale_words = fmt == FHIP_KVQ_Q4_1 ? nblk : (nblk + 1) / 2;
    return FHIP_OK;
}

int fhip_kvq_append(int fmt, const float* d_src, size_t src_row_stride, size_t t, size_t width, const uint32_t* d_positions, uint32_t pos_off,
                    int src_at_pos, size_t cap, uint32_t* d_codes, uint32_t* d_scales, void* stream) {
    int rc = need_init();
    if (rc) return rc;
    if ((rc = kvq_checks("fhip_kvq_append", fmt, width))) return rc;
    if (t == 0 || width == 0) return FHIP_OK;
    if (!d_src || !d_codes || !d_scales) return set_error(FHIP_ERR_ARG, "fhip_kvq_append: NULL pointer");
    if (src_row_stride == 0) src_row_stride = width;
    if (src_row_stride < width) return set_error(FHIP_ERR_SHAPE, "fhip_kvq_append: source row stride %zu below the width %zu", src_row_stride, width);
    if (!d_positions && (size_t)pos_off + t > cap)
        return set_error(FHIP_ERR_SHAPE, "fhip_kvq_append: rows %u + %zu exceed the capacity %zu", pos_off, t, cap);
    return fhip::launch_kvq_append(fmt, d_src, src_row_stride, t, width, d_positions, pos_off, src_at_pos != 0, cap, d_codes, (uint16_t*)d_scales,
                                   (hipStream_t)stream);
}

int fhip_kvq_dequantize_rows(int fmt, const uint32_t* d_codes, const uint32_t* d_scales, size_t row0, size_t rows, size_t width,
                             const uint32_t* d_last_pos, float* d_out, void* stream) {
    int rc = need_init();
    if (rc) return rc;
    if ((rc = kvq_checks("fhip_kvq_dequantize_rows", fmt, width))) return rc;
    if (rows == 0 || width == 0) return FHIP_OK;
    if (!d_codes || !d_scales || !d_out) return set_error(FHIP_ERR_ARG, "fhip_kvq_dequantize_rows: NULL pointer");
    if (((uintptr_t)d_out & 15) != 0) return set_error(FHIP_ERR_ARG, "fhip_kvq_dequantize_rows: the output must be 16-byte aligned");
    return fhip::launch_kvq_dequantize(fmt, d_codes, (const uint16_t*)d_scales, row0, rows, width, d_last_pos, d_out, (hipStream_t)stream);
}

static int rope_checks(const char* who, size_t n_heads, size_t head_dim, size_t n_rot) {
    if (n_rot > head_dim || n_rot % 2 != 0) return set_error(FHIP_ERR_SHAPE, "n_rot must be even and <= head_dim");   // lib.rs:437
    if (n_heads > 0xFFFFu || head_dim > 0xFFFFu) return set_error(FHIP_ERR_SHAPE, "%s: n_heads / head_dim exceed 65535", who);
    return FHIP_OK;
}

int fhip_rope(const float* d_x, size_t src_row_stride, size_t t, size_t n_heads, size_t head_dim, size_t n_rot, float base,
              const uint32_t* d_positions, uint32_t pos_off, const float* d_freq_scale, int interleaved, float* d_out, void* stream) {
    int rc = need_init();
    if (rc) return rc;
    if ((rc = rope_checks("fhip_rope", n_heads, head_dim, n_rot))) return rc;
    if (t == 0 || n_heads == 0 || head_dim == 0) return FHIP_OK;
    if (!d_x || !d_out) return set_error(FHIP_ERR_ARG, "fhip_rope: NULL pointer");
    if (src_row_stride == 0) src_row_stride = n_heads * head_dim;
    return fhip::launch_rope(d_x, src_row_stride, t, (int)n_heads, (int)head_dim, (int)n_rot, base, d_positions, pos_off, d_freq_scale,
                             interleaved != 0, d_out, (hipStream_t)stream);
}

int fhip_kv_append2(const float* d_k, const float* d_v, size_t t, size_t width, const uint32_t* d_positions, uint32_t pos_off,
                    float* d_k_cache, float* d_v_cache, size_t cap, void* stream) {
    int rc = need_init();
    if (rc) return rc;
    if (t == 0 || width == 0) return FHIP_OK;
    if (!d_k || !d_v || !d_k_cache || !d_v_cache) return set_error(FHIP_ERR_ARG, "fhip_kv_append2: NULL pointer");
    if (cap > 0xFFFFFFFFull) return set_error(FHIP_ERR_SHAPE, "fhip_kv_append2: capacity exceeds 2^32 rows");
    return fhip::launch_kv_append(d_k, d_v, t, width, d_positions, pos_off, cap, d_k_cache, d_v_cache, (hipStream_t)stream);
}

int fhip_qkv_post(const float* d_qkv, const float* d_bias, const float* d_q_norm, const float* d_k_norm, const uint32_t* d_positions,
                  const float* d_freq_scale, size_t t, size_t n_head, size_t n_kv, size_t head_dim, size_t n_rot, int interleaved,
                  float eps, float base, float* d_q_out, float* d_k_cache, float* d_v_cache, size_t cap, void* stream) {
    int rc = need_init();
    if (rc) return rc;
    if ((rc = rope_checks("fhip_qkv_post", n_head + 2 * n_kv, head_dim, n_rot))) return rc;
    if (t == 0 || head_dim == 0 || n_head + n_kv == 0) return FHIP_OK;
    if (!d_qkv || !d_positions || !d_q_out || !d_k_cache || !d_v_cache) return set_error(FHIP_ERR_ARG, "fhip_qkv_post: NULL pointer");
    if (cap > 0xFFFFFFFFull) return set_error(FHIP_ERR_SHAPE, "fhip_qkv_post: capacity exceeds 2^32 rows");
    return fhip::launch_qkv_post(d_qkv, d_bias, d_q_norm, d_k_norm, d_positions, d_freq_scale, t, (int)n_head, (int)n_kv, (int)head_dim,
                                 (int)n_rot, interleaved != 0, eps, base, d_q_out, d_k_cache, d_v_cache, cap, (hipStream_t)stream);
}

int fhip_qkv_post_packed(const float* d_qkv, const float* d_bias, const float* d_q_norm, const float* d_k_norm, const uint32_t* d_positions,
                         const float* d_freq_scale, size_t t, size_t n_head, size_t n_kv, size_t head_dim, size_t n_rot, int interleaved,
                         float eps, float base, float* d_q_out, float* d_k_out, float* d_v_out, void* stream) {
    int rc = need_init();
    if (rc) return rc;
    if ((rc = rope_checks("fhip_qkv_post_packed", n_head + 2 * n_kv, head_dim, n_rot))) return rc;
    if (t == 0 || head_dim == 0 || n_head + n_kv == 0) return FHIP_OK;
    if (!d_qkv || !d_positions || !d_q_out || !d_k_out || !d_v_out) return set_error(FHIP_ERR_ARG, "fhip_qkv_post_packed: NULL pointer");
    return fhip::launch_qkv_post(d_qkv, d_bias, d_q_norm, d_k_norm, d_positions, d_freq_scale, t, (int)n_head, (int)n_kv, (int)head_dim,
                                 (int)n_rot, interleaved != 0, eps, base, d_q_out, d_k_out, d_v_out, 0, (hipStream_t)stream, true);
}

int fhip_kvq_append2(int fmt, const float* d_k, const float* d_v, size_t src_row_stride, size_t t, size_t width, const uint32_t* d_positions,
                     uint32_t pos_off, size_t cap, uint32_t* d_k_codes, uint32_t* d_k_scales, uint32_t* d_v_codes, uint32_t* d_v_scales,
                     void* stream) {
    int rc = need_init();
    if (rc) return rc;
    if ((rc = kvq_checks("fhip_kvq_append2", fmt, width))) return rc;
    if (t == 0 || width == 0) return FHIP_OK;
    if (!d_k || !d_v || !d_k_codes || !d_k_scales || !d_v_codes || !d_v_scales) return set_error(FHIP_ERR_ARG, "fhip_kvq_append2: NULL pointer");
    if (src_row_stride == 0) src_row_stride = width;
    if (src_row_stride < width) return set_error(FHIP_ERR_SHAPE, "fhip_kvq_append2: source row stride %zu below the width %zu", src_row_stride, width);
    if (!d_positions && (size_t)pos_off + t > cap)
        return set_error(FHIP_ERR_SHAPE, "fhip_kvq_append2: rows %u + %zu exceed the capacity %zu", pos_off, t, cap);
    return fhip::launch_kvq_append(fmt, d_k, src_row_stride, t, width, d_positions, pos_off, false, cap, d_k_codes, (uint16_t*)d_k_scales,
                                   (hipStream_t)stream, d_v, d_v_codes, (uint16_t*)d_v_scales);
}

static int qkv_post_kvq(const char* who, int fmt, const float* d_qkv, const float* d_bias, const float* d_q_norm, const float* d_k_norm, const uint32_t* d_positions,
                        const float* d_freq_scale, size_t t, size_t n_head, size_t n_kv, size_t head_dim, size_t n_rot, int interleaved, float eps, float base, float* d_q_out,
                        uint32_t* d_k_codes, uint32_t* d_k_scales, uint32_t* d_v_codes, uint32_t* d_v_scales, size_t cap, float* d_k_rows, float* d_v_rows, size_t n_rows,
                        size_t past, void* stream) {
    int rc = need_init();
    if (rc) return rc;
    if ((rc = kvq_checks(who, fmt, n_kv * head_dim)) || (rc = rope_checks(who, n_head + 2 * n_kv, head_dim, n_rot))) return rc;
    if (t == 0 || head_dim == 0 || n_head + n_kv == 0) return FHIP_OK;
    if (!fhip::qkv_post_kvq_takes((int)head_dim)) return set_error(FHIP_ERR_SHAPE, "%s: head_dim must be a multiple of 32 up to 256, got %zu", who, head_dim);
    if (!d_qkv || !d_positions || !d_q_out || !d_k_codes || !d_k_scales || !d_v_codes || !d_v_scales) return set_error(FHIP_ERR_ARG, "%s: NULL pointer", who);
    if (cap > 0xFFFFFFFFull) return set_error(FHIP_ERR_SHAPE, "%s: too large for one launch", who);
    return fhip::launch_qkv_post_kvq(fmt, d_qkv, d_bias, d_q_norm, d_k_norm, d_positions, d_freq_scale, t, (int)n_head, (int)n_kv, (int)head_dim, (int)n_rot,
                                     interleaved != 0, eps, base, d_q_out, d_k_codes, (uint16_t*)d_k_scales, d_v_codes, (uint16_t*)d_v_scales, cap,
                                     (hipStream_t)stream, d_k_rows, d_v_rows, n_rows, past);
}
int fhip_qkv_post_kvq(int fmt, const float* d_qkv, const float* d_bias, const float* d_q_norm, const float* d_k_norm, const uint32_t* d_positions,
                      const float* d_freq_scale, size_t t, size_t n_head, size_t n_kv, size_t head_dim, size_t n_rot, int interleaved, float eps,
                      float base, float* d_q_out, uint32_t* d_k_codes, uint32_t* d_k_scales, uint32_t* d_v_codes, uint32_t* d_v_scales, size_t cap,
                      void* stream) {
    return qkv_post_kvq("fhip_qkv_post_kvq", fmt, d_qkv, d_bias, d_q_norm, d_k_norm, d_positions, d_freq_scale, t, n_head, n_kv, head_dim, n_rot, interleaved, eps, base, d_q_out,
                        d_k_codes, d_k_scales, d_v_codes, d_v_scales, cap, nullptr, nullptr, 0, 0, stream);
}
int fhip_qkv_post_kvq_rows(int fmt, const float* d_qkv, const float* d_bias, const float* d_q_norm, const float* d_k_norm, const uint32_t* d_positions,
                           const float* d_freq_scale, size_t t, size_t n_head, size_t n_kv, size_t head_dim, size_t n_rot, int interleaved, float eps,
                           float base, float* d_q_out, uint32_t* d_k_codes, uint32_t* d_k_scales, uint32_t* d_v_codes, uint32_t* d_v_scales, size_t cap,
                           float* d_k_rows, float* d_v_rows, size_t n_rows, size_t past, void* stream) {
    if (!d_k_rows || !d_v_rows || (((uintptr_t)d_k_rows | (uintptr_t)d_v_rows) & 15) != 0)
        return set_error(FHIP_ERR_ARG, "fhip_qkv_post_kvq_rows: the rows' outputs must be there and 16-byte aligned");
    if (past > n_rows || n_rows > cap) return set_error(FHIP_ERR_SHAPE, "fhip_qkv_post_kvq_rows: %zu earlier rows of %zu, a cache of %zu", past, n_rows, cap);
    return qkv_post_kvq("fhip_qkv_post_kvq_rows", fmt, d_qkv, d_bias, d_q_norm, d_k_norm, d_positions, d_freq_scale, t, n_head, n_kv, head_dim, n_rot, interleaved, eps, base,
                        d_q_out, d_k_codes, d_k_scales, d_v_codes, d_v_scales, cap, d_k_rows, d_v_rows, n_rows, past, stream);
}

int fhip_decode_attention_kvq(int fmt, const float* d_q, const uint32_t* d_k_codes, const uint32_t* d_k_scales, const uint32_t* d_v_codes,
                              const uint32_t* d_v_scales, size_t n_head, size_t n_kv, size_t head_dim, size_t len, const uint32_t* d_last_pos,
                              size_t window, float softcap, float* d_ws, float* d_out, void* stream) {
    int rc = need_init();
    if (rc) return rc;
    if ((rc = kvq_checks("fhip_decode_attention_kvq", fmt, n_kv * head_dim))) return rc;
    if (n_head == 0 || head_dim == 0) return FHIP_OK;
    if (!d_q || !d_k_codes || !d_k_scales || !d_v_codes || !d_v_scales || !d_out)
        return set_error(FHIP_ERR_ARG, "fhip_decode_attention_kvq: NULL pointer");
    if (n_head > 0x7FFFFFFFull || n_kv > 0x7FFFFFFFull) return set_error(FHIP_ERR_SHAPE, "fhip_decode_attention_kvq: too many heads");
    return fhip::launch_decode_attention_kvq(fmt, d_q, d_k_codes, (const uint16_t*)d_k_scales, d_v_codes, (const uint16_t*)d_v_scales, (int)n_head,
                                             (int)n_kv, (int)head_dim, len, d_last_pos, window, softcap, d_ws, d_out, (hipStream_t)stream);
}

static int check_causal(const char* who, const void* d_q, const void* d_k, const void* d_v, const void* d_out, size_t n_head, size_t n_kv) {
    if (!d_q || !d_k || !d_v || !d_out) return set_error(FHIP_ERR_ARG, "%s: NULL pointer", who);
    if ((((uintptr_t)d_q | (uintptr_t)d_k | (uintptr_t)d_v | (uintptr_t)d_out) & 15) != 0)
        return set_error(FHIP_ERR_ARG, "%s: pointers must be 16-byte aligned", who);
    if (n_head > 0x7FFFFFFFull || n_kv > 0x7FFFFFFFull) return set_error(FHIP_ERR_SHAPE, "%s: too many heads", who);
    return FHIP_OK;
}

int fhip_causal_attention(const float* d_q, const float* d_k, const float* d_v, size_t t, size_t s, size_t n_head, size_t n_kv, size_t head_dim,
                          size_t window, float softcap, float* d_out, void* stream) {
    int rc = need_init();
    if (rc) return rc;
    if (t == 0 || n_head == 0 || head_dim == 0) return FHIP_OK;
    if ((rc = check_causal("fhip_causal_attention", d_q, d_k, d_v, d_out, n_head, n_kv))) return rc;
    return fhip::launch_causal_attention(d_q, d_k, d_v, t, s, (int)n_head, (int)n_kv, (int)head_dim, window, softcap, true, d_out, nullptr, 0, (hipStream_t)stream);
}

int fhip_causal_attention_bf16(const float* d_q, const float* d_k, const float* d_v, size_t t, size_t s, size_t n_head, size_t n_kv,
                               size_t head_dim, size_t window, float softcap, uint16_t* d_out_bf16, void* stream) {
    int rc = need_init();
    if (rc) return rc;
    if (t == 0 || n_head == 0 || head_dim == 0) return FHIP_OK;
    if ((rc = check_causal("fhip_causal_attention_bf16", d_q, d_k, d_v, d_out_bf16, n_head, n_kv))) return rc;
    return fhip::launch_causal_attention_bf16(d_q, d_k, d_v, t, s, (int)n_head, (int)n_kv, (int)head_dim, window, softcap, true, d_out_bf16, nullptr, 0, (hipStream_t)stream);
}

int fhip_causal_attention_f32_products(const float* d_q, const float* d_k, const float* d_v, size_t t, size_t s, size_t n_head, size_t n_kv, size_t head_dim,
                                       size_t window, float softcap, int out_bf16, void* d_out, void* stream) {
    int rc = need_init();
    if (rc) return rc;
    if (t == 0 || n_head == 0 || head_dim == 0) return FHIP_OK;
    if ((rc = check_causal("fhip_causal_attention_f32_products", d_q, d_k, d_v, d_out, n_head, n_kv))) return rc;
    if (out_bf16)
        return fhip::launch_causal_attention_bf16(d_q, d_k, d_v, t, s, (int)n_head, (int)n_kv, (int)head_dim, window, softcap, false, (uint16_t*)d_out, nullptr, 0,
                                                  (hipStream_t)stream);
    return fhip::launch_causal_attention(d_q, d_k, d_v, t, s, (int)n_head, (int)n_kv, (int)head_dim, window, softcap, false, (float*)d_out, nullptr, 0, (hipStream_t)stream);
}

size_t fhip_causal_attention_ws_bytes(size_t t, size_t s, size_t n_head, size_t head_dim, size_t window) {
    return g_device < 0 || (head_dim != 64 && head_dim != 128) ? 0 : fhip::causal_attention_ws_bytes(t, s, n_head, head_dim, window);
}

int fhip_causal_attention_split(const float* d_q, const float* d_k, const float* d_v, size_t t, size_t s, size_t n_head, size_t n_kv, size_t head_dim,
                                size_t window, float softcap, int out_bf16, void* d_out, float* d_ws, size_t ws_bytes, void* stream) {
    int rc = need_init();
    if (rc) return rc;
    if (t == 0 || n_head == 0 || head_dim == 0) return FHIP_OK;
    if ((rc = check_causal("fhip_causal_attention_split", d_q, d_k, d_v, d_out, n_head, n_kv))) return rc;
    if (((uintptr_t)d_ws & 15) != 0) return set_error(FHIP_ERR_ARG, "fhip_causal_attention_split: pointers must be 16-byte aligned");
    if (out_bf16)
        return fhip::launch_causal_attention_bf16(d_q, d_k, d_v, t, s, (int)n_head, (int)n_kv, (int)head_dim, window, softcap, true, (uint16_t*)d_out, d_ws, ws_bytes,
                                                  (hipStream_t)stream);
    return fhip::launch_causal_attention(d_q, d_k, d_v, t, s, (int)n_head, (int)n_kv, (int)head_dim, window, softcap, true, (float*)d_out, d_ws, ws_bytes, (hipStream_t)stream);
}

size_t fhip_decode_attention_ws_bytes(size_t n_head, size_t n_kv, size_t head_dim, size_t len) {
    if (g_device < 0 || n_kv == 0 || len == 0) return 0;
    int splits = fhip::attn_ws_splits(len, (int)n_head, (int)n_kv, (int)head_dim);
    return splits > 1 ? n_head * (size_t)splits * (head_dim + 2) * sizeof(float) : 0;
}

int fhip_decode_attention_ex(const float* d_q, const float* d_k_cache, const float* d_v_cache, size_t n_head, size_t n_kv, size_t head_dim,
                             size_t len, const uint32_t* d_last_pos, size_t window, float softcap, float* d_ws, float* d_out, void* stream) {
    int rc = need_init();
    if (rc) return rc;
    if (n_head > 0xFFFFu || n_kv > 0xFFFFu || head_dim > 0xFFFFu) return set_error(FHIP_ERR_SHAPE, "fhip_decode_attention: head counts exceed 65535");
    if (n_head == 0 || head_dim == 0) return FHIP_OK;
    if (!d_q || !d_k_cache || !d_v_cache || !d_out) return set_error(FHIP_ERR_ARG, "fhip_decode_attention: NULL pointer");
    if (!(softcap >= 0.f)) return set_error(FHIP_ERR_ARG, "fhip_decode_attention: softcap must be >= 0");
    return fhip::launch_decode_attention(d_q, d_k_cache, d_v_cache, (int)n_head, (int)n_kv, (int)head_dim, len, d_last_pos, window, softcap, d_ws,
                                         d_out, (hipStream_t)stream);
}

int fhip_decode_attention(const float* d_q, const float* d_k_cache, const float* d_v_cache, size_t n_head, size_t n_kv, size_t head_dim,
                          size_t len, const uint32_t* d_last_pos, float* d_ws, float* d_out, void* stream) {
    return fhip_decode_attention_ex(d_q, d_k_cache, d_v_cache, n_head, n_kv, head_dim, len, d_last_pos, 0, 0.f, d_ws, d_out, stream);
}

int fhip_qkv_post_attention(const float* d_qkv, const float* d_bias, const float* d_q_norm, const float* d_k_norm, const uint32_t* d_pos,
                            const float* d_freq_scale, size_t n_head, size_t n_kv, size_t head_dim, size_t n_rot, int interleaved, float eps,
                            float base, float* d_k_cache, float* d_v_cache, size_t cap, size_t len, size_t window, float softcap, float* d_ws,
                            float* d_out, void* stream) {
    int rc = need_init();
    if (rc) return rc;
    if ((rc = rope_checks("fhip_qkv_post_attention", n_head + 2 * n_kv, head_dim, n_rot))) return rc;
    if (n_head == 0 || head_dim == 0) return FHIP_OK;
    if (!d_qkv || !d_pos || !d_k_cache || !d_v_cache || !d_out) return set_error(FHIP_ERR_ARG, "fhip_qkv_post_attention: NULL pointer");
    if (cap > 0xFFFFFFFFull) return set_error(FHIP_ERR_SHAPE, "fhip_qkv_post_attention: capacity exceeds 2^32 rows");
    if (!(softcap >= 0.f)) return set_error(FHIP_ERR_ARG, "fhip_qkv_post_attention: softcap must be >= 0");
    return fhip::launch_qkv_post_attention(d_qkv, d_bias, d_q_norm, d_k_norm, d_pos, d_freq_scale, (int)n_head, (int)n_kv, (int)head_dim, (int)n_rot,
                                           interleaved != 0, eps, base, d_k_cache, d_v_cache, cap, len, window, softcap, d_ws, d_out,
                                           (hipStream_t)stream);
}

int fhip_qkv_post_attention_kvq(int fmt, const float* d_qkv, const float* d_bias, const float* d_q_norm, const float* d_k_norm, const uint32_t* d_pos,
                                const float* d_freq_scale, size_t n_head, size_t n_kv, size_t head_dim, size_t n_rot, int interleaved, float eps,
                                float base, uint32_t* d_k_codes, uint32_t* d_k_scales, uint32_t* d_v_codes, uint32_t* d_v_scales, size_t cap, size_t len,
                                size_t window, float softcap, float* d_ws, float* d_out, void* stream) {
    int rc = need_init();
    if (rc) return rc;
    if ((rc = kvq_checks("fhip_qkv_post_attention_kvq", fmt, n_kv * head_dim)) || (rc = rope_checks("fhip_qkv_post_attention_kvq", n_head + 2 * n_kv, head_dim, n_rot)))
        return rc;
    if (n_head == 0 || head_dim == 0) return FHIP_OK;
    if (!d_qkv || !d_pos || !d_k_codes || !d_k_scales || !d_v_codes || !d_v_scales || !d_out)
        return set_error(FHIP_ERR_ARG, "fhip_qkv_post_attention_kvq: NULL pointer");
    if (n_head > 0x7FFFFFFFull || n_kv > 0x7FFFFFFFull) return set_error(FHIP_ERR_SHAPE, "fhip_qkv_post_attention_kvq: too many heads");
    if (cap > 0xFFFFFFFFull) return set_error(FHIP_ERR_SHAPE, "fhip_qkv_post_attention_kvq: capacity exceeds 2^32 rows");
    if (!(softcap >= 0.f)) return set_error(FHIP_ERR_ARG, "fhip_qkv_post_attention_kvq: softcap must be >= 0");
    return fhip::launch_qkv_post_attention_kvq(fmt, d_qkv, d_bias, d_q_norm, d_k_norm, d_pos, d_freq_scale, (int)n_head, (int)n_kv, (int)head_dim, (int)n_rot, interleaved != 0,
                                               eps, base, d_k_codes, (uint16_t*)d_k_scales, d_v_codes, (uint16_t*)d_v_scales, cap, len, window, softcap, d_ws, d_out,
                                               (hipStream_t)stream);
}

static int norm_matmul_q(const fhip_weight* w, const float* d_x, const float* d_resid, const float* d_norm_w, float eps, float* d_x_out,
                         float* d_h_scratch, int swiglu, float* d_y, uint32_t* d_count, uint32_t by, void* stream) {
    int rc = need_init();
    if (rc) return rc;
    if (!w || !d_x || !d_norm_w || !d_h_scratch || !d_y) return set_error(FHIP_ERR_ARG, "fhip_norm_matmul_q: NULL pointer");
    // every workgroup reads all of x and resid while one of them stores x_out, and all of them store y: none of the outputs
    // may share memory with an input or with each other
    {
        const size_t out_rows = swiglu ? w->rows / 2 : w->rows;
        auto overlap = [](const float* a, size_t na, const float* b, size_t nb) { return a && b && a < b + nb && b < a + na; };
        if (overlap(d_x_out, w->cols, d_x, w->cols) || overlap(d_x_out, w->cols, d_resid, w->cols) || overlap(d_x_out, w->cols, d_norm_w, w->cols))
            return set_error(FHIP_ERR_ARG, "fhip_norm_matmul_q: x_out must not overlap x, resid or norm_w");
        if (overlap(d_y, out_rows, d_x, w->cols) || overlap(d_y, out_rows, d_resid, w->cols) || overlap(d_y, out_rows, d_norm_w, w->cols) ||
            overlap(d_y, out_rows, d_x_out, w->cols))
            return set_error(FHIP_ERR_ARG, "fhip_norm_matmul_q: y must not overlap x, resid, norm_w or x_out");
    }
    if (swiglu && (w->type == FHIP_Q8_0 || w->rows % 2 != 0))
        return set_error(w->type == FHIP_Q8_0 ? FHIP_ERR_UNSUPPORTED_TYPE : FHIP_ERR_SHAPE, "fhip_norm_matmul_q: no fused SwiGLU for this weight");
    if (((uintptr_t)d_x | (uintptr_t)d_resid | (uintptr_t)d_norm_w | (uintptr_t)d_x_out) & 15)
        return set_error(FHIP_ERR_ARG, "fhip_norm_matmul_q: x, resid, norm_w and x_out must be 16-byte aligned");
    const size_t n_ff = swiglu ? w->rows / 2 : 0;
    fhip::NormParams np{d_norm_w, d_resid, d_resid ? d_x_out : nullptr, eps, d_count, by};   // without a residual there is no sum to store
    rc = fhip::launch_gemv_norm(w, d_x, d_y, n_ff, np, (hipStream_t)stream);
    if (rc != fhip::NORM_NOT_FUSED) return rc;
    if ((rc = fhip::launch_rmsnorm(d_x, d_resid, d_norm_w, 1, w->cols, eps, d_resid ? d_x_out : nullptr, d_h_scratch, (hipStream_t)stream, d_count, by))) return rc;
    return fhip::launch_gemv(w, d_h_scratch, 1, d_y, n_ff, (hipStream_t)stream);
}
int fhip_norm_matmul_q(const fhip_weight* w, const float* d_x, const float* d_resid, const float* d_norm_w, float eps, float* d_x_out,
                       float* d_h_scratch, int swiglu, float* d_y, void* stream) {
    return norm_matmul_q(w, d_x, d_resid, d_norm_w, eps, d_x_out, d_h_scratch, swiglu, d_y, nullptr, 0, stream);
}
int fhip_norm_matmul_q_count(const fhip_weight* w, const float* d_x, const float* d_resid, const float* d_norm_w, float eps, float* d_x_out,
                             float* d_h_scratch, int swiglu, float* d_y, uint32_t* d_count, uint32_t by, void* stream) {
    if (!d_count) return set_error(FHIP_ERR_ARG, "fhip_norm_matmul_q_count: NULL pointer");
    return norm_matmul_q(w, d_x, d_resid, d_norm_w, eps, d_x_out, d_h_scratch, swiglu, d_y, d_count, by, stream);
}

int fhip_debug_generic_matvec(int on) {
    fhip::gemv_force_generic(on != 0);
    return FHIP_OK;
}

int fhip_debug_gemm_tile(int tile) { return fhip::gemm_bf16_force_tile(tile); }

int fhip_debug_quad_matvec(int on) { return fhip::gemv_quad_matvec(on != 0) ? 1 : 0; }

int fhip_debug_matmul_route(const fhip_weight* w, const float* d_x, size_t rows_x, const float* d_y, int* kernels, size_t* rows, size_t cap, size_t* n) {
    int rc = need_init();
    if (rc) return rc;
    if (!w || !d_x || !d_y || !kernels || !rows || !n) return set_error(FHIP_ERR_ARG, "fhip_debug_matmul_route: NULL pointer");
    *n = 0;
    auto add = [&](int kernel, size_t r) { if (*n < cap) { kernels[*n] = kernel; rows[*n] = r; } ++*n; };
    const size_t grp = takes_f16x2(w, rows_x) ? f16x2_group(w) : rows_x;
    for (size_t m0 = 0; m0 < rows_x && w->rows; m0 += grp) {
        const size_t t = rows_x - m0 < grp ? rows_x - m0 : grp;
        if (takes_f16x2(w, t)) { add(f16x2_route(w, d_x + m0 * w->cols, t, true, d_y + m0 * w->rows), t); continue; }
        for (size_t r = 0; r < t;) {
            const fhip::MatvecPass pass = fhip::matvec_pass(w, t - r, 0);
            add(pass.kernel, pass.rows);
            r += pass.rows;
        }
    }
    return FHIP_OK;
}

int fhip_debug_matmul_by(const fhip_weight* w, int kernel, const float* d_x, size_t rows_x, float* d_y, void* stream) {
    int rc = need_init();
    if (rc) return rc;
    if (!w || !d_x || !d_y) return set_error(FHIP_ERR_ARG, "fhip_debug_matmul_by: NULL pointer");
    if (rows_x == 0 || rows_x > f16x2_group(w) || w->rows == 0 || !fhip::gemm_f16x2_takes(w, rows_x)) return set_error(FHIP_ERR_ARG, "fhip_debug_matmul_by: not a group of the f16 kernels");
    const bool ordered = w->batch_policy == FHIP_BATCH_ORDERED, cut = ordered ? fhip::gemm_f16x2_parts(w, rows_x) > 1 : fhip::gemm_f16x2_adds_into_y(w, rows_x);
    const bool can = kernel == FHIP_ROUTE_PREPARED || (kernel == FHIP_ROUTE_HELD && fhip::gemm_f16x2_held_takes(w, d_x, rows_x, d_y)) ||
                     (kernel == FHIP_ROUTE_OWN_ROWS && (ordered ? fhip::gemm_f16x2_resident_own_x(w, d_x, rows_x, d_y) : !cut && fhip::gemm_f16x2_own_x(w, d_x, rows_x)));
    if (!can) return set_error(FHIP_ERR_ARG, "fhip_debug_matmul_by: kernel %d cannot do this product", kernel);
    void* ws = nullptr;
    if (kernel != FHIP_ROUTE_HELD && (rc = lib_workspace((hipStream_t)stream, f16x2_matmul_ws(w, rows_x), &ws, "fhip_debug_matmul_by"))) return rc;
    return f16x2_launch(kernel == FHIP_ROUTE_HELD ? kernel : kernel | (cut ? FHIP_ROUTE_CUT : 0), w, d_x, rows_x, false, d_y, ws, (hipStream_t)stream, nullptr, nullptr);
}

int fhip_debug_read_probe(const void* d_src, size_t nbytes, uint32_t* d_sink, void* stream) {
    int rc = need_init();
    if (rc) return rc;
    if (!d_src || !d_sink) return set_error(FHIP_ERR_ARG, "fhip_debug_read_probe: NULL pointer");
    if (((uintptr_t)d_src & 15) != 0) return set_error(FHIP_ERR_ARG, "fhip_debug_read_probe: src must be 16-byte aligned");
    return fhip::launch_read_probe(d_src, nbytes, d_sink, (hipStream_t)stream);
}

int fhip_debug_mfma_probe(int iters, float* d_sink, double* flops, void* stream) {
    int rc = need_init();
    if (rc) return rc;
    if (iters < 1 || !d_sink) return set_error(FHIP_ERR_ARG, "fhip_debug_mfma_probe: iters >= 1 and a sink are needed");
    return fhip::launch_mfma_probe(iters, d_sink, (hipStream_t)stream, flops);
}

int fhip_debug_matmul_q_loop(const fhip_weight* const* ws, size_t n_weights, size_t launches, const float* d_x, int swiglu, float* d_y,
                             void* stream) {
    int rc = need_init();
    if (rc) return rc;
    if (!ws || n_weights == 0 || !d_x || !d_y) return set_error(FHIP_ERR_ARG, "fhip_debug_matmul_q_loop: NULL pointer");
    for (size_t i = 0; i < launches; i++) {
        const fhip_weight* w = ws[i % n_weights];
        rc = swiglu ? fhip_matmul_q_swiglu(w, d_x, 1, d_y, stream) : fhip_matmul_q(w, d_x, 1, d_y, stream);
        if (rc) return rc;
    }
    return FHIP_OK;
}

int fhip_matvec_precision(int bits) {
    const int before = g_default_planes == 3 ? 24 : 16;
    if (bits == 0) return before;
    if (bits != 16 && bits != 24) return set_error(FHIP_ERR_ARG, "fhip_matvec_precision: 16 or 24 bits (0 to query), not %d", bits);
    g_default_planes = bits == 24 ? 3 : 2;
    return before;
}

int fhip_add_count(const float* d_a, const float* d_b, size_t n, float* d_out, uint32_t* d_count, uint32_t by, void* stream) {
    int rc = need_init();
    if (rc) return rc;
    if (!d_count || (n && (!d_a || !d_b || !d_out))) return set_error(FHIP_ERR_ARG, "fhip_add_count: NULL pointer");
    return fhip::launch_add(d_a, d_b, n, d_out, (hipStream_t)stream, d_count, by);
}

int fhip_u32_add(uint32_t* d_words, size_t n, uint32_t delta, void* stream) {
    int rc = need_init();
    if (rc) return rc;
    if (n == 0) return FHIP_OK;
    if (!d_words) return set_error(FHIP_ERR_ARG, "fhip_u32_add: NULL pointer");
    return fhip::launch_u32_add(d_words, n, delta, (hipStream_t)stream);
}

int fhip_moe_topk(const float* d_logits, const float* d_bias, size_t t, size_t n_expert, size_t k, int sigmoid, float scale, int norm,
                  float* d_out, void* stream) {
    int rc = need_init();
    if (rc) return rc;
    if (k < 1 || k > 8) return set_error(FHIP_ERR_SHAPE, "k must be 1..=8");                                   // dtype.rs:1599
    if (n_expert > 1024) return set_error(FHIP_ERR_SHAPE, "moe_topk: n_expert <= 1024 (single-thread scan)");   // dtype.rs:1600
    if (n_expert == 0) return set_error(FHIP_ERR_SHAPE, "moe_topk: n_expert must be positive");
    if (t == 0) return FHIP_OK;
    if (!d_logits || !d_out) return set_error(FHIP_ERR_ARG, "fhip_moe_topk: NULL pointer");
    return fhip::launch_moe_topk(d_logits, d_bias, t, n_expert, (int)k, sigmoid != 0, scale, norm != 0, d_out, (hipStream_t)stream);
}

static int sel_checks(const char* who, const fhip_weight* w, size_t k, size_t expert_rows, fhip::SelParams* sel) {
    if (!w) return set_error(FHIP_ERR_ARG, "%s: NULL weight", who);
    if (k < 1 || k > 8) return set_error(FHIP_ERR_SHAPE, "k must be 1..=8");
    if (expert_rows == 0 || w->rows % expert_rows != 0)
        return set_error(FHIP_ERR_SHAPE, "%s: weight rows %zu are not a whole number of experts of %zu rows", who, w->rows, expert_rows);
    sel->k = (int)k;
    sel->n_expert = (int)(w->rows / expert_rows);
    sel->expert_rows = expert_rows;
    return FHIP_OK;
}

int fhip_matmul_q_swiglu_id(const fhip_weight* w, const float* d_x, size_t t, const float* d_selw, size_t k, size_t eff, float* d_y,
                            void* stream) {
    int rc = need_init();
    if (rc) return rc;
    fhip::SelParams sel{};
    if ((rc = sel_checks("matmul_q_swiglu_id", w, k, 2 * eff, &sel))) return rc;
    if (t == 0) return FHIP_OK;
    if (!d_x || !d_selw || !d_y) return set_error(FHIP_ERR_ARG, "fhip_matmul_q_swiglu_id: NULL pointer");
    if (((uintptr_t)d_x & 15) != 0 || (w->cols * 4) % 16 != 0) return set_error(FHIP_ERR_ARG, "fhip_matmul_q_swiglu_id: x rows must be 16-byte aligned");
    sel.selw = d_selw; sel.x_per_pair = 0; sel.y_stride = eff; sel.npairs = (int)(t * k);
    return fhip::launch_gemv_sel(w, d_x, d_y, eff, true, sel, (hipStream_t)stream);
}

int fhip_matmul_q_relu2_id(const fhip_weight* w, const float* d_x, size_t t, const float* d_selw, size_t k, size_t eff, float* d_y,
                           void* stream) {
    int rc = need_init();
    if (rc) return rc;
    fhip::SelParams sel{};
    if ((rc = sel_checks("matmul_q_relu2_id", w, k, eff, &sel))) return rc;
    if (t == 0) return FHIP_OK;
    if (!d_x || !d_selw || !d_y) return set_error(FHIP_ERR_ARG, "fhip_matmul_q_relu2_id: NULL pointer");
    if (((uintptr_t)d_x & 15) != 0 || (w->cols * 4) % 16 != 0) return set_error(FHIP_ERR_ARG, "fhip_matmul_q_relu2_id: x rows must be 16-byte aligned");
    sel.selw = d_selw; sel.x_per_pair = 0; sel.y_stride = eff; sel.npairs = (int)(t * k); sel.relu2 = 1;
    return fhip::launch_gemv_sel(w, d_x, d_y, eff, false, sel, (hipStream_t)stream);
}

int fhip_matmul_q_id(const fhip_weight* w, const float* d_x, const float* d_selw, size_t k, size_t out_pe, float* d_y, void* stream) {
    int rc = need_init();
    if (rc) return rc;
    fhip::SelParams sel{};
    if ((rc = sel_checks("matmul_q_id", w, k, out_pe, &sel))) return rc;
    if (!d_x || !d_selw || !d_y) return set_error(FHIP_ERR_ARG, "fhip_matmul_q_id: NULL pointer");
    if (((uintptr_t)d_x & 15) != 0 || (w->cols * 4) % 16 != 0) return set_error(FHIP_ERR_ARG, "fhip_matmul_q_id: x rows must be 16-byte aligned");
    sel.selw = d_selw; sel.x_per_pair = 1; sel.y_stride = out_pe; sel.npairs = (int)k;
    return fhip::launch_gemv_sel(w, d_x, d_y, out_pe, false, sel, (hipStream_t)stream);
}

int fhip_matmul_q_id_wsum(const fhip_weight* w, const float* d_x, size_t t, const float* d_selw, size_t k, size_t out_pe, float* d_y,
                          float* d_ws, void* stream) {
    int rc = need_init();
    if (rc) return rc;
    fhip::SelParams sel{};
    if ((rc = sel_checks("matmul_q_id_wsum", w, k, out_pe, &sel))) return rc;
    if (t == 0) return FHIP_OK;
    if (!d_x || !d_selw || !d_y || !d_ws) return set_error(FHIP_ERR_ARG, "fhip_matmul_q_id_wsum: NULL pointer");
    if (((uintptr_t)d_x & 15) != 0 || (w->cols * 4) % 16 != 0) return set_error(FHIP_ERR_ARG, "fhip_matmul_q_id_wsum: x rows must be 16-byte aligned");
    sel.selw = d_selw; sel.x_per_pair = 1; sel.y_stride = out_pe; sel.npairs = (int)(t * k);
    // one launch where the kernel covers the rows; it reads the inputs until its end, so an output laid over one of them takes the two launches,
    // of which only the second writes it
    auto apart = [&](const float* in, size_t n) { return d_y + t * out_pe <= in || in + n <= d_y; };
    if (apart(d_x, t * k * w->cols) && apart(d_selw, t * 2 * k) && out_pe > 0 &&
        (w->planes == 3 ? fhip::launch_gemv_wsum_p3(w, d_x, d_y, out_pe, sel, (hipStream_t)stream, &rc)
                        : fhip::launch_gemv_wsum_p2(w, d_x, d_y, out_pe, sel, (hipStream_t)stream, &rc)))
        return rc;
    if ((rc = fhip::launch_gemv_sel(w, d_x, d_ws, out_pe, false, sel, (hipStream_t)stream))) return rc;
    return fhip::launch_moe_wsum(d_ws, d_selw, t, (int)k, out_pe, d_y, (hipStream_t)stream);
}

int fhip_cvt_f32_bf16(const float* d_x, size_t n, uint16_t* d_out, void* stream) {
    int rc = need_init();
    if (rc) return rc;
    if (n == 0) return FHIP_OK;
    if (!d_x || !d_out) return set_error(FHIP_ERR_ARG, "fhip_cvt_f32_bf16: NULL pointer");
    return fhip::launch_cvt_bf16(d_x, n, d_out, (hipStream_t)stream);
}

int fhip_matmul_q_coop(const fhip_weight* w, const float* d_x, size_t rows_x, float* d_y, uint16_t* d_ws_bf16, void* stream) {
    int rc = need_init();
    if (rc) return rc;
    if (!w) return set_error(FHIP_ERR_ARG, "fhip_matmul_q_coop: NULL weight");
    if (rows_x == 0 || w->rows == 0) return FHIP_OK;
    if (w->cols == 0) return d_y ? zero_outputs(rows_x, w->rows, d_y, (hipStream_t)stream) : set_error(FHIP_ERR_ARG, "fhip_matmul_q_coop: NULL pointer");
    if (!d_x || !d_y || !d_ws_bf16) return set_error(FHIP_ERR_ARG, "fhip_matmul_q_coop: NULL pointer");
    if ((rc = fhip::launch_cvt_bf16(d_x, rows_x * w->cols, d_ws_bf16, (hipStream_t)stream))) return rc;
    return gemm_bf16_lib_ws(w, d_ws_bf16, rows_x, d_y, (hipStream_t)stream, "fhip_matmul_q_coop");
}

// the tiled GEMM applies SwiGLU itself; up to 32 rows the gate|up matrix is small and stays in f32 between two launches
static bool ffn_coop_fused(size_t rows_x) { return rows_x > 32; }

size_t fhip_ffn_coop_ws_bytes(const fhip_weight* gu, const fhip_weight* down, size_t rows_x) {
    if (!gu || !down) return 0;
    return align256(rows_x * gu->cols * 2) + (ffn_coop_fused(rows_x) ? 0 : align256(rows_x * gu->rows * 4)) + align256(rows_x * down->cols * 2);
}

// d_x f32 (converted into the workspace first), or already bf16 in d_xb; d_gu: null, or where gate|up goes in f32 between two launches
static int ffn_coop(const char* who, const fhip_weight* gu, const fhip_weight* down, const float* d_x, const uint16_t* d_xb, float* d_gu, size_t rows_x,
                    float* d_y, void* d_ws, hipStream_t s, bool run_sums = false) {
    int rc = need_init();
    if (rc) return rc;
    if (!gu || !down) return set_error(FHIP_ERR_ARG, "%s: NULL weight", who);
    if (gu->rows % 2 != 0) return set_error(FHIP_ERR_SHAPE, "%s: gate_up rows must be even", who);
    const size_t n_ff = gu->rows / 2;
    if (down->cols != n_ff) return set_error(FHIP_ERR_SHAPE, "down in dim must equal n_ff");
    if (rows_x == 0) return FHIP_OK;
    if ((!d_x && !d_xb) || !d_y || !d_ws) return set_error(FHIP_ERR_ARG, "%s: NULL pointer", who);
    if (((uintptr_t)d_ws & 255) != 0) return set_error(FHIP_ERR_ARG, "%s: workspace must be 256-byte aligned", who);
    // an empty inner dimension on either side: gate and up are 0, silu(0) * 0 = 0, and so is every output
    if (gu->cols == 0 || n_ff == 0) return zero_outputs(rows_x, down->rows, d_y, s);
    const bool in_tile = ffn_coop_fused(rows_x), fused = in_tile && !d_gu;
    uint8_t* ws = (uint8_t*)d_ws;
    uint16_t* xb = (uint16_t*)ws;
    float* g = (float*)(ws + align256(rows_x * gu->cols * 2));
    uint16_t* hb = (uint16_t*)((uint8_t*)g + (in_tile ? 0 : align256(rows_x * gu->rows * 4)));
    if (d_gu) g = d_gu;
    if (!d_xb) {
        if ((rc = fhip::launch_cvt_bf16(d_x, rows_x * gu->cols, xb, s))) return rc;
        d_xb = xb;
    }
    if (fused) {
        const size_t need = fhip::gemm_bf16_swiglu_ws_bytes(gu, rows_x);
        void* split = nullptr;
        if (need && (rc = lib_workspace(s, need, &split, who))) return rc;
        if ((rc = fhip::launch_gemm_bf16_swiglu(gu, d_xb, rows_x, hb, s, (float*)split, need))) return rc;
        return gemm_bf16_lib_ws(down, hb, rows_x, d_y, s, who);
    }
    if ((rc = gemm_bf16_lib_ws(gu, d_xb, rows_x, g, s, who, run_sums))) return rc;
    if ((rc = fhip::launch_swiglu_bf16(g, rows_x, n_ff, hb, s))) return rc;
    return gemm_bf16_lib_ws(down, hb, rows_x, d_y, s, who, run_sums);
}

int fhip_ffn_coop(const fhip_weight* gu, const fhip_weight* down, const float* d_x, size_t rows_x, float* d_y,
                  void* d_ws, void* stream) {
    return ffn_coop("fhip_ffn_coop", gu, down, d_x, nullptr, nullptr, rows_x, d_y, d_ws, (hipStream_t)stream);
}

int fhip_ffn_bf16(const fhip_weight* gu, const fhip_weight* down, const uint16_t* d_x_bf16, float* d_gate_up, size_t rows_x, float* d_y, void* d_ws,
                  void* stream) {
    return ffn_coop("fhip_ffn_bf16", gu, down, nullptr, d_x_bf16, d_gate_up, rows_x, d_y, d_ws, (hipStream_t)stream);
}
int fhip_ffn_bf16_run_sums(const fhip_weight* gu, const fhip_weight* down, const uint16_t* d_x_bf16, float* d_gate_up, size_t rows_x, float* d_y, void* d_ws,
                           void* stream) {
    if (!d_gate_up && need_init() == FHIP_OK && rows_x) return set_error(FHIP_ERR_ARG, "fhip_ffn_bf16_run_sums: NULL pointer");
    return ffn_coop("fhip_ffn_bf16_run_sums", gu, down, nullptr, d_x_bf16, d_gate_up, rows_x, d_y, d_ws, (hipStream_t)stream, true);
}

size_t fhip_matmul_q_f16x2_ws_bytes(const fhip_weight* w, size_t rows_x) {
    if (!fhip::gemm_f16x2_supports(w, rows_x)) return 0;
    return align256(fhip::gemm_f16x2_xp_bytes(w, rows_x));
}

static int f16x2_checks(const char* who, const fhip_weight* w, size_t rows_x) {
    if (rows_x > 32) return set_error(FHIP_ERR_SHAPE, "%s: at most 32 activation rows (got %zu)", who, rows_x);
    if (w->type != FHIP_Q4_K && w->type != FHIP_Q5_K && w->type != FHIP_Q6_K && w->type != FHIP_Q8_0)
        return set_error(FHIP_ERR_UNSUPPORTED_TYPE, "%s: no kernel for ggml type %u (Q4_K, Q5_K, Q6_K and Q8_0 only)", who, w->type);
    if (w->type == FHIP_Q8_0 && rows_x > 16) return set_error(FHIP_ERR_SHAPE, "%s: at most 16 activation rows for Q8_0 (got %zu)", who, rows_x);
    if (rows_x && w->rows && !fhip::gemm_f16x2_supports(w, rows_x))
        return set_error(FHIP_ERR_SHAPE, "%s: weight rows of %zu columns are outside what the kernels take", who, w->cols);
    return FHIP_OK;
}

int fhip_matmul_q_f16x2(const fhip_weight* w, const float* d_x, size_t rows_x, float* d_y, void* d_ws, void* stream) {
    int rc = need_init();
    if (rc) return rc;
    if (!w) return set_error(FHIP_ERR_ARG, "fhip_matmul_q_f16x2: NULL weight");
    if ((rc = f16x2_checks("fhip_matmul_q_f16x2", w, rows_x))) return rc;
    if (rows_x == 0 || w->rows == 0) return FHIP_OK;
    if (!d_x || !d_y || !d_ws) return set_error(FHIP_ERR_ARG, "fhip_matmul_q_f16x2: NULL pointer");
    if (((uintptr_t)d_ws & 255) != 0) return set_error(FHIP_ERR_ARG, "fhip_matmul_q_f16x2: workspace must be 256-byte aligned");
    hipStream_t s = (hipStream_t)stream;
    uint16_t* xp = (uint16_t*)d_ws;
    const bool clr = fhip::gemm_f16x2_adds_into_y(w, rows_x);   // then the split clears y on the side
    if ((rc = fhip::launch_xsplit_f16(w, d_x, rows_x, false, xp, s, clr ? d_y : nullptr, clr ? rows_x * w->rows : 0))) return rc;
    return fhip::launch_gemm_f16x2(w, xp, rows_x, d_y, s, clr);
}

size_t fhip_ffn_f16x2_ws_bytes(const fhip_weight* gu, const fhip_weight* down, size_t rows_x) {
    if (!fhip::gemm_f16x2_supports(gu, rows_x) || !fhip::gemm_f16x2_supports(down, rows_x)) return 0;
    return align256(fhip::gemm_f16x2_xp_bytes(gu, rows_x)) + align256(rows_x * gu->rows * 4) +
           align256(fhip::gemm_f16x2_xp_bytes(down, rows_x));
}

int fhip_ffn_f16x2(const fhip_weight* gu, const fhip_weight* down, const float* d_x, size_t rows_x, float* d_y, void* d_ws,
                   void* stream) {
    int rc = need_init();
    if (rc) return rc;
    if (!gu || !down) return set_error(FHIP_ERR_ARG, "fhip_ffn_f16x2: NULL weight");
    if (gu->rows % 2 != 0) return set_error(FHIP_ERR_SHAPE, "ffn: gate_up rows must be even");
    const size_t n_ff = gu->rows / 2;
    if (down->cols != n_ff) return set_error(FHIP_ERR_SHAPE, "down in dim must equal n_ff");
    if ((rc = f16x2_checks("fhip_ffn_f16x2", gu, rows_x)) || (rc = f16x2_checks("fhip_ffn_f16x2", down, rows_x))) return rc;
    if (rows_x == 0) return FHIP_OK;
    if (!d_x || !d_y || !d_ws) return set_error(FHIP_ERR_ARG, "fhip_ffn_f16x2: NULL pointer");
    if (((uintptr_t)d_ws & 255) != 0) return set_error(FHIP_ERR_ARG, "fhip_ffn_f16x2: workspace must be 256-byte aligned");
    hipStream_t s = (hipStream_t)stream;
    uint8_t* ws = (uint8_t*)d_ws;
    uint16_t* xp1 = (uint16_t*)ws;
    float* g = (float*)(ws + align256(fhip::gemm_f16x2_xp_bytes(gu, rows_x)));
    uint16_t* xp2 = (uint16_t*)((uint8_t*)g + align256(rows_x * gu->rows * 4));
    const bool clr1 = fhip::gemm_f16x2_adds_into_y(gu, rows_x), clr2 = fhip::gemm_f16x2_adds_into_y(down, rows_x);
    if ((rc = fhip::launch_xsplit_f16(gu, d_x, rows_x, false, xp1, s, clr1 ? g : nullptr, clr1 ? rows_x * gu->rows : 0))) return rc;
    if ((rc = fhip::launch_gemm_f16x2(gu, xp1, rows_x, g, s, clr1))) return rc;
    // SwiGLU of [gate | up] is computed while the rows are split for the down projection
    if ((rc = fhip::launch_xsplit_f16(down, g, rows_x, true, xp2, s, clr2 ? d_y : nullptr, clr2 ? rows_x * down->rows : 0))) return rc;
    return fhip::launch_gemm_f16x2(down, xp2, rows_x, d_y, s, clr2);
}

int fhip_matvec_q8_0_host(const float* h_x, const uint8_t* h_w, size_t w_len, size_t rows, size_t cols, float* h_y) {
    int rc = need_init();
    if (rc) return rc;
    // asserts of crates/ferric-tensor/src/cpu_simd.rs:80-83
    if (cols % 32 != 0) return set_error(FHIP_ERR_SHAPE, "Q8_0 cols must be a multiple of 32");
    if (w_len != rows * (cols / 32) * 34) return set_error(FHIP_ERR_SHAPE, "unexpected Q8_0 byte length");
    if (rows == 0) return FHIP_OK;
    if (!h_x || !h_w || !h_y) return set_error(FHIP_ERR_ARG, "fhip_matvec_q8_0_host: NULL pointer");
    fhip_weight* w = nullptr;
    if ((rc = fhip_weight_create(FHIP_Q8_0, h_w, w_len, rows, cols, &w))) return rc;
    void *d_x = nullptr, *d_y = nullptr;
    rc = check_hip(hipMalloc(&d_x, (cols ? cols : 1) * sizeof(float)), "hipMalloc");
    if (!rc) rc = check_hip(hipMalloc(&d_y, rows * sizeof(float)), "hipMalloc");
    if (!rc && cols) rc = check_hip(hipMemcpy(d_x, h_x, cols * sizeof(float), hipMemcpyHostToDevice), "hipMemcpy H2D");
    if (!rc) {
        if (cols == 0) rc = check_hip(hipMemset(d_y, 0, rows * sizeof(float)), "hipMemset");
        else rc = fhip::launch_gemv(w, (const float*)d_x, 1, (float*)d_y, 0, nullptr);
    }
    if (!rc) rc = check_hip(hipMemcpy(h_y, d_y, rows * sizeof(float), hipMemcpyDeviceToHost), "hipMemcpy D2H");
    if (d_x) (void)hipFree(d_x);
    if (d_y) (void)hipFree(d_y);
    fhip_weight_destroy(w);
    return rc;
}

// ---- crates/ferric-tensor/src/cpu_simd.rs:238-331: Pool / matvec_q8_0_pooled --------------------------------
// The reference's pool exists so that a call does not pay its set-up again (thread creation there). What a call of the
// host-buffer mat-vec pays here is the upload of the weight bytes, so the pool keeps those resident: the weight the
// last call used stays in HBM, keyed by the caller's (pointer, length, cols) -- `w` is an immutable Arc<Vec<u8>> in the
// reference -- together with the staging buffers and a stream of its own.
struct fhip_pool {
    size_t threads;
    hipStream_t stream;
    const uint8_t* key;
    size_t key_len, key_cols;
    uint64_t key_print;   // fingerprint of the bytes the key pointed at when they were uploaded
    uint8_t* d_w;
    size_t w_cap;
    float *d_x, *d_y;
    size_t x_cap, y_cap;
    size_t uploads;
};

// FNV-1a over the first and the last 4 KiB and 64 evenly spaced 64-byte samples of the weight: about 12 KiB per call. It catches
// a buffer that was freed and reused, or rewritten, at the same address and length (what pointer + length alone would take for
// the resident weight); it is not a proof of equality -- a caller that edits a few bytes in place still calls fhip_pool_forget.
static uint64_t pool_fingerprint(const uint8_t* w, size_t n) {
    uint64_t h = 1469598103934665603ull;
    auto eat = [&](size_t from, size_t len) {
        for (size_t i = from; i < from + len && i < n; i++) h = (h ^ w[i]) * 1099511628211ull;
    };
    eat(0, 4096);
    if (n > 8192) {
        eat(n - 4096, 4096);
        const size_t step = (n - 8192) / 64;
        for (size_t k = 0; k < 64 && step >= 64; k++) eat(4096 + k * step, 64);
    } else if (n > 4096) {
        eat(4096, n - 4096);
    }
    return h ^ n;
}

int fhip_pool_create(size_t threads, fhip_pool** out) {
    if (!out) return set_error(FHIP_ERR_ARG, "fhip_pool_create: NULL output");
    *out = nullptr;
    int rc = need_init();
    if (rc) return rc;
    fhip_pool* p = new (std::nothrow) fhip_pool();
    if (!p) return set_error(FHIP_ERR_HIP, "fhip_pool_create: out of host memory");
    p->threads = threads ? threads : 1;   // Pool::new: n.max(1)
    if ((rc = check_hip(hipStreamCreate(&p->stream), "hipStreamCreate"))) { delete p; return rc; }
    *out = p;
    return FHIP_OK;
}

size_t fhip_pool_threads(const fhip_pool* p) { return p ? p->threads : 0; }
size_t fhip_pool_uploads(const fhip_pool* p) { return p ? p->uploads : 0; }

void fhip_pool_forget(fhip_pool* p) {
    if (p) { p->key = nullptr; p->key_len = 0; p->key_cols = 0; }
}

void fhip_pool_destroy(fhip_pool* p) {
    if (!p) return;
    (void)hipStreamSynchronize(p->stream);
    if (p->d_w) (void)hipFree(p->d_w);
    if (p->d_x) (void)hipFree(p->d_x);
    if (p->d_y) (void)hipFree(p->d_y);
    (void)hipStreamDestroy(p->stream);
    delete p;
}

static int pool_reserve(void** d, size_t* cap, size_t need, const char* what) {
    if (need <= *cap) return FHIP_OK;
    if (*d) (void)hipFree(*d);
    *d = nullptr; *cap = 0;
    int rc = check_hip(hipMalloc(d, need), what);
    if (!rc) *cap = need;
    return rc;
}

int fhip_matvec_q8_0_pooled(fhip_pool* p, const float* h_x, size_t x_len, const uint8_t* h_w, size_t w_len, size_t cols, size_t lo,
                            size_t hi, float* h_y) {
    int rc = need_init();
    if (rc) return rc;
    if (!p) return set_error(FHIP_ERR_ARG, "fhip_matvec_q8_0_pooled: NULL pool");
    if (lo > hi) return set_error(FHIP_ERR_SHAPE, "empty or inverted span");             // cpu_simd.rs:311
    const size_t rows = hi - lo;
    if (rows == 0) return FHIP_OK;                                                        // :313
    if (!h_y) return set_error(FHIP_ERR_ARG, "fhip_matvec_q8_0_pooled: NULL output");
    const size_t nblk = cols / 32, row_bytes = nblk * 34;                                 // :314; row_q8_0 walks cols / 32 blocks
    if (nblk == 0) { memset(h_y, 0, rows * sizeof(float)); return FHIP_OK; }              // no block: every sum is 0.0
    // the slices of :321 and of row_q8_0 (:62, :64) panic when the row span or the activations run past their arrays
    if (hi > w_len / row_bytes) return set_error(FHIP_ERR_SHAPE, "range end index %zu out of range for slice of length %zu", hi * row_bytes, w_len);
    if (x_len < nblk * 32) return set_error(FHIP_ERR_SHAPE, "range end index %zu out of range for slice of length %zu", nblk * 32, x_len);
    if (!h_x || !h_w) return set_error(FHIP_ERR_ARG, "fhip_matvec_q8_0_pooled: NULL pointer");
    const size_t kcols = nblk * 32, all_rows = w_len / row_bytes;
    const uint64_t print = pool_fingerprint(h_w, all_rows * row_bytes);
    if (p->key != h_w || p->key_len != w_len || p->key_cols != kcols || p->key_print != print) {
        fhip_pool_forget(p);
        if ((rc = pool_reserve((void**)&p->d_w, &p->w_cap, all_rows * row_bytes, "hipMalloc"))) return rc;
        if ((rc = check_hip(hipMemcpyAsync(p->d_w, h_w, all_rows * row_bytes, hipMemcpyHostToDevice, p->stream), "hipMemcpy H2D"))) return rc;
        p->key = h_w; p->key_len = w_len; p->key_cols = kcols; p->key_print = print;
        p->uploads++;
    }
    if ((rc = pool_reserve((void**)&p->d_x, &p->x_cap, kcols * sizeof(float), "hipMalloc"))) return rc;
    if ((rc = pool_reserve((void**)&p->d_y, &p->y_cap, rows * sizeof(float), "hipMalloc"))) return rc;
    if ((rc = check_hip(hipMemcpyAsync(p->d_x, h_x, kcols * sizeof(float), hipMemcpyHostToDevice, p->stream), "hipMemcpy H2D"))) return rc;
    fhip_weight view;
    if ((rc = make_weight(FHIP_Q8_0, rows * row_bytes, rows, kcols, view))) return rc;
    view.d_raw = p->d_w + lo * row_bytes;
    if ((rc = fhip::launch_gemv(&view, p->d_x, 1, p->d_y, 0, p->stream))) return rc;
    if ((rc = check_hip(hipMemcpyAsync(h_y, p->d_y, rows * sizeof(float), hipMemcpyDeviceToHost, p->stream), "hipMemcpy D2H"))) return rc;
    return check_hip(hipStreamSynchronize(p->stream), "hipStreamSynchronize");
}

}  // extern "C"

// Prefill / large-M path: activations are rescaled per row by an exact power of two into fp16,
// weights are dequantized into fp16 (scaled per neuron by an exact power of two), and an
// fp16 x fp16 -> fp32 MFMA GEMM (v_mfma_f32_32x32x16_f16) produces y; the epilogue multiplies
// the two power-of-two scales back.  fp16 (11 significant bits) keeps the weight rounding error
// near 1e-4 relative, which bf16 tiles (8 bits) cannot.
#include <stdlib.h>

#include "common.hpp"
#include "tune.hpp"

namespace mfq {

// ---- core: thread-local error text ---------------------------------------------------
char *error_buffer() {
    static thread_local char buf[512] = {0};
    return buf;
}
int fail(int code, const char *fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(error_buffer(), 512, fmt, ap);
    va_end(ap);
    return code;
}

// ---- activation prep: x16[m, k] = fp16(x[m, k] * 2^-f_m), xscale[m] = 2^f_m ---------------
template <int XF16>
__global__ __launch_bounds__(256) void x_prep_kernel(const uint16_t *__restrict__ x, int64_t ldx, int K, int Kp,
                                                     uint16_t *__restrict__ x16, float *__restrict__ xscale) {
    __shared__ float red[4];
    const int m = blockIdx.x, tid = threadIdx.x;
    const uint16_t *xr = x + static_cast<int64_t>(m) * ldx;
    float amax = 0.f;
    for (int k = tid; k < K; k += 256) {
        const float v = fabsf(x_to_f32<XF16>(xr[k]));
        if (v == v && v <= 3.0e38f) amax = fmaxf(amax, v);
    }
    for (int o = 32; o > 0; o >>= 1) amax = fmaxf(amax, __shfl_xor(amax, o, 64));
    if ((tid & 63) == 0) red[tid >> 6] = amax;
    __syncthreads();
    amax = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    int e = 0;
    if (amax > 0.f) frexpf(amax, &e);  // amax = f * 2^e, f in [0.5, 1)
    e = max(e, kMinRowExp);
    const float inv = ldexpf(1.f, 9 - e);  // row maximum lands in [256, 512)
    if (tid == 0) xscale[m] = ldexpf(1.f, e - 9);
    uint16_t *o16 = x16 + static_cast<int64_t>(m) * Kp;
    for (int k = tid; k < Kp; k += 256) o16[k] = k < K ? f32_to_f16_rne(x_to_f32<XF16>(xr[k]) * inv) : uint16_t(0);
}

// The same for 16-byte aligned rows with K % 8 == 0: 8 values per load and store, the row read once (twice beyond 8192
// values).  Bit-identical results.
template <int XF16>
__global__ __launch_bounds__(256) void x_prep_vec_kernel(const uint16_t *__restrict__ x, int64_t ldx, int K, int Kp,
                                                         uint16_t *__restrict__ x16, float *__restrict__ xscale) {
    __shared__ float red[4];
    constexpr int KEEP = 4;  // chunks of 8 values a thread keeps in registers between the two passes
    const int m = blockIdx.x, tid = threadIdx.x;
    const u32x4_t *xr = reinterpret_cast<const u32x4_t *>(x + static_cast<int64_t>(m) * ldx);
    const int nchunks = K >> 3;
    u32x4_t keep[KEEP];
    float amax = 0.f;
    auto chunk_amax = [&](u32x4_t v) {
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const float a = fabsf(x_to_f32<XF16>(static_cast<uint16_t>(v[t] & 0xffffu)));
            const float b = fabsf(x_to_f32<XF16>(static_cast<uint16_t>(v[t] >> 16)));
            if (a == a && a <= 3.0e38f) amax = fmaxf(amax, a);
            if (b == b && b <= 3.0e38f) amax = fmaxf(amax, b);
        }
    };
#pragma unroll
    for (int i = 0; i < KEEP; ++i) {
        const int c = tid + 256 * i;
        keep[i] = u32x4_t{0u, 0u, 0u, 0u};
        if (c < nchunks) {
            keep[i] = xr[c];
            chunk_amax(keep[i]);
        }
    }
    for (int c = tid + 256 * KEEP; c < nchunks; c += 256) chunk_amax(xr[c]);
    for (int o = 32; o > 0; o >>= 1) amax = fmaxf(amax, __shfl_xor(amax, o, 64));
    if ((tid & 63) == 0) red[tid >> 6] = amax;
    __syncthreads();
    amax = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    int e = 0;
    if (amax > 0.f) frexpf(amax, &e);
    e = max(e, kMinRowExp);
    const float inv = ldexpf(1.f, 9 - e);
    if (tid == 0) xscale[m] = ldexpf(1.f, e - 9);
    u32x4_t *o16 = reinterpret_cast<u32x4_t *>(x16 + static_cast<int64_t>(m) * Kp);
    auto emit = [&](int c, u32x4_t v) {
        u32x4_t h;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const uint32_t lo = f32_to_f16_rne(x_to_f32<XF16>(static_cast<uint16_t>(v[t] & 0xffffu)) * inv);
            const uint32_t hi = f32_to_f16_rne(x_to_f32<XF16>(static_cast<uint16_t>(v[t] >> 16)) * inv);
            h[t] = lo | (hi << 16);
        }
        o16[c] = h;
    };
#pragma unroll
    for (int i = 0; i < KEEP; ++i)
        if (tid + 256 * i < nchunks) emit(tid + 256 * i, keep[i]);
    for (int c = tid + 256 * KEEP; c < nchunks; c += 256) emit(c, xr[c]);
    for (int c = nchunks + tid; c < (Kp >> 3); c += 256) o16[c] = u32x4_t{0u, 0u, 0u, 0u};
}

// ---- fp16 NT GEMM: y[m, n] = sum_k a[m, k] * b[n, k] ----------------------
// 128 x 128 x 32 block tile, 256 threads = 4 waves of 64 x 64 (2 x 2 MFMA 32x32x16 tiles).
constexpr int GBM = 128, GBN = 128, GBK = 32, GLD = GBK + 8;  // LDS row stride in halves (80 bytes)

__global__ __launch_bounds__(256) void gemm_f16_nt_kernel(const uint16_t *__restrict__ a, int64_t lda,
                                                          const uint16_t *__restrict__ b, int64_t ldb, int M, int N,
                                                          int K, float *__restrict__ y, int64_t ldy) {
    __shared__ __attribute__((aligned(16))) uint16_t As[2][GBM * GLD];
    __shared__ __attribute__((aligned(16))) uint16_t Bs[2][GBN * GLD];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int bm = blockIdx.y * GBM, bn = blockIdx.x * GBN;
    const int wm = (wave >> 1) * 64, wn = (wave & 1) * 64;
    // global -> LDS: each thread moves 16 halves of A and of B per K step (row = tid/2, half-row = tid&1)
    const int lr = tid >> 1, lc = (tid & 1) * 16;
    const bool a_ok = bm + lr < M, b_ok = bn + lr < N;
    const uint16_t *ap = a + static_cast<int64_t>(bm + lr) * lda + lc;
    const uint16_t *bp = b + static_cast<int64_t>(bn + lr) * ldb + lc;
    float16_t acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int t = 0; t < 16; ++t) acc[i][j][t] = 0.f;

    const int nk = K / GBK;
    u32x4_t ra[2], rbv[2];
    auto gload = [&](int kt) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            ra[h] = a_ok ? *reinterpret_cast<const u32x4_t *>(ap + kt * GBK + 8 * h) : u32x4_t{0, 0, 0, 0};
            rbv[h] = b_ok ? *reinterpret_cast<const u32x4_t *>(bp + kt * GBK + 8 * h) : u32x4_t{0, 0, 0, 0};
        }
    };
    auto lstore = [&](int buf) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            *reinterpret_cast<u32x4_t *>(&As[buf][lr * GLD + lc + 8 * h]) = ra[h];
            *reinterpret_cast<u32x4_t *>(&Bs[buf][lr * GLD + lc + 8 * h]) = rbv[h];
        }
    };
    gload(0);
    lstore(0);
    __syncthreads();
    const int fr = lane & 31, fk = (lane >> 5) * 8;
    for (int kt = 0; kt < nk; ++kt) {
        const int buf = kt & 1;
        if (kt + 1 < nk) gload(kt + 1);
#pragma unroll
        for (int kk = 0; kk < GBK; kk += 16) {
            half8_t fa[2], fb[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                fa[i] = *reinterpret_cast<const half8_t *>(&As[buf][(wm + 32 * i + fr) * GLD + kk + fk]);
                fb[i] = *reinterpret_cast<const half8_t *>(&Bs[buf][(wn + 32 * i + fr) * GLD + kk + fk]);
            }
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[i], fb[j], acc[i][j], 0, 0, 0);
        }
        if (kt + 1 < nk) lstore(buf ^ 1);
        __syncthreads();
    }
    // D[row = m, col = n]: lane holds col = lane & 31, rows 8 * (t / 4) + 4 * (lane / 32) + t % 4
#pragma unroll
    for (int i = 0; i < 2; ++i) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int n = bn + wn + 32 * j + (lane & 31);
            if (n >= N) continue;
#pragma unroll
            for (int t = 0; t < 16; ++t) {
                const int m = bm + wm + 32 * i + 8 * (t >> 2) + 4 * (lane >> 5) + (t & 3);
                if (m < M) y[static_cast<int64_t>(m) * ldy + n] = acc[i][j][t];
            }
        }
    }
}

static int gemm_f16_nt(const void *a, int64_t lda, const void *b, int64_t ldb, int M, int N, int K, float *y, int64_t ldy, hipStream_t st) {
    MFQ_REQUIRE(K % GBK == 0 && lda % 8 == 0 && ldb % 8 == 0, MFQ_ERR_INVALID,
                "gemm_f16_nt: K=%d, lda=%lld, ldb=%lld must be multiples of 32 / 8 / 8", K, (long long)lda, (long long)ldb);
    const dim3 grid(static_cast<unsigned>(ceil_div(N, GBN)), static_cast<unsigned>(ceil_div(M, GBM)));
    hipLaunchKernelGGL(gemm_f16_nt_kernel, grid, dim3(256), 0, st, static_cast<const uint16_t *>(a), lda,
                       static_cast<const uint16_t *>(b), ldb, M, N, K, y, ldy);
    return check_launch("gemm_f16_nt");
}

int x_prep(const void *x, int x_dtype, int64_t ldx, int M, int K, int Kp, void *x16, float *xscale, hipStream_t st) {
    const uint16_t *xp = static_cast<const uint16_t *>(x);
    uint16_t *o = static_cast<uint16_t *>(x16);
    const bool vec = K % 8 == 0 && ldx % 8 == 0 && Kp % 8 == 0 && (reinterpret_cast<uintptr_t>(x) & 15) == 0 &&
                     (reinterpret_cast<uintptr_t>(x16) & 15) == 0;
    if (vec) {
        if (x_dtype == MFQ_X_F16) hipLaunchKernelGGL((x_prep_vec_kernel<1>), dim3(M), dim3(256), 0, st, xp, ldx, K, Kp, o, xscale);
        else hipLaunchKernelGGL((x_prep_vec_kernel<0>), dim3(M), dim3(256), 0, st, xp, ldx, K, Kp, o, xscale);
    } else {
        if (x_dtype == MFQ_X_F16) hipLaunchKernelGGL((x_prep_kernel<1>), dim3(M), dim3(256), 0, st, xp, ldx, K, Kp, o, xscale);
        else hipLaunchKernelGGL((x_prep_kernel<0>), dim3(M), dim3(256), 0, st, xp, ldx, K, Kp, o, xscale);
    }
    return check_launch("x_prep");
}

size_t dequant_gemm_workspace(int N, int K, int M);
size_t dequant_gemm_workspace_least(int N, int K, int M);
void dequant_gemm_carve(void *ws, int N, int K, int M, uint16_t *&w16, float *&wscale, int &Kp);
int dequant_gemm(void *ws, size_t ws_bytes, int N, int K, const void *x, int x_dtype, int64_t ldx, int M, float *y, int64_t ldy, hipStream_t st);
int nint_gemv_any(const mfq_nint_desc *d, const void *weight, const void *x, int x_dtype, int64_t ldx, int M, float *y,
                  int64_t ldy, hipStream_t st);
int nint_dequant_f16(const mfq_nint_desc *d, const void *weight, void *w16, int64_t ld, float *rowscale, hipStream_t st);
bool nint_stream_capable(const mfq_nint_desc *d);
bool nint_tile_capable(const mfq_nint_desc *d);
bool nint_tile_glu_pays(const mfq_nint_desc *d, int M);
double nint_tile_us(const mfq_nint_desc *d, int M);
int nint_tile_shape(const mfq_nint_desc *d, int M, bool glu, int *splits);
size_t nint_tile_workspace(const mfq_nint_desc *d, int M);
size_t nint_tile_workspace_least(const mfq_nint_desc *d, int M);
int nint_tile(const mfq_nint_desc *d, const void *weight, const void *x, int x_dtype, int64_t ldx, int M, void *y, int64_t ldy,
              bool glu, int gelu, int f16, void *ws, size_t ws_bytes, hipStream_t st);

}  // namespace mfq

using namespace mfq;

extern "C" const char *mfq_hip_last_error(void) { return error_buffer(); }
extern "C" int mfq_hip_version(void) { return 1; }

extern "C" int mfq_hip_gemm_f16_nt(const void *a, int64_t lda, const void *b, int64_t ldb, int M, int N, int K, float *y,
                                   int64_t ldy, mfq_stream_t stream) {
    MFQ_REQUIRE(a && b && y, MFQ_ERR_INVALID, "gemm_f16_nt: null argument");
    return gemm_f16_nt(a, lda, b, ldb, M, N, K, y, ldy, as_stream(stream));
}

// Up to kGemvMaxM activation rows the weight stream dominates and the GEMV kernels win; tensors with a matrix-core
// streaming kernel (16 rows per pass over the packed weights) stay on it up to kStreamMaxM rows, where re-streaming the
// weights is still cheaper than dequantizing them to fp16 once, or while their passes cost less than the tile kernel.  A
// pass costs a time per weight that follows the unpack of its profile (measured over 3 .. 100 million weights, two passes
// and more: 0.145 / 0.2 / 0.165 / 0.33 / 0.3 / 0.62 us per million for 2- / 3- / 4- / 5- / 6- / 8-bit codes), on top of
// about 4 us (8-bit codes: nothing on top; 1536 x 2048 at 160 rows 18.4 us streaming, 23.3 in tiles).  12288 x 4096 NINT4-32 at 32 / 48 / 64 / 256 rows: 20 / 33 / 33 / 133 us streaming, 25 / 26 / 27 / 44 us in tiles;
// NINT8-48 there at 16 / 64 rows: 34 / 125 against 29 / 30 us.
// The streaming kernels take bf16 rows as they are where the tile kernel scales each row into fp16's range, so they are not
// given more rows for being cheaper than that: the upper limit is 64 * (30 us + 1.9 us per 1024 of K) / (8 us + 0.85 us per
// MB of payload), 2 x the denominator and 1.25 x the numerator for natural-order units.
static constexpr int kGemvMaxM = 8, kStreamMaxM = 256;
static int nint_stream_limit(const mfq_nint_desc *d) {
    static const int env_max = tune_env("MFQ_STREAM_MAX_M", 0);
    if (!nint_stream_capable(d)) return kGemvMaxM;
    if (env_max > 0) return env_max > kGemvMaxM ? env_max : kGemvMaxM;
    if (!nint_tile_capable(d)) return kStreamMaxM;
    if (d->bits == 8) return 160;
    const double t64 = (8.0 + 0.85e-6 * static_cast<double>(d->payload_bytes)) * (d->kind != 1 ? 2.0 : 1.0);
    const double tp = (30.0 + 1.9 * d->neuron_len / 1024.0) * (d->kind != 1 ? 1.25 : 1.0);
    const int m = static_cast<int>(64.0 * tp / t64) / 16 * 16;
    return m < 32 ? 32 : m > 512 ? 512 : m;
}
static bool nint_streams(const mfq_nint_desc *d, int M) {
    static const int env_max = tune_env("MFQ_STREAM_MAX_M", 0);
    if (M <= kGemvMaxM) return true;
    if (M > nint_stream_limit(d)) return false;
    if (env_max > 0 || !nint_tile_capable(d)) return true;
    static const double pass_us[9] = {0, 0, 0.145, 0.2, 0.165, 0.33, 0.3, 0, 0.62};  // per million weights
    const double weights = 1e-6 * d->out * static_cast<double>(d->neuron_len);
    const double stream_us = (d->bits == 8 ? 0.0 : 4.0) + static_cast<double>(ceil_div(M, 16)) * pass_us[d->bits] * weights;
    return stream_us < kTileLeastUs || stream_us < nint_tile_us(d, M);
}

extern "C" size_t mfq_hip_nint_gemm_workspace_bytes(const mfq_nint_desc *d, int M) {
    if (!d || nint_streams(d, M)) return 0;
    if (nint_tile_capable(d)) return nint_tile_workspace(d, M);
    return dequant_gemm_workspace(d->out, d->neuron_len, M);
}

extern "C" int mfq_hip_nint_gemm(const mfq_nint_desc *d, const void *weight, const void *x, int x_dtype, int64_t ldx,
                                 int M, float *y, int64_t ldy, void *workspace, size_t workspace_bytes,
                                 mfq_stream_t stream) {
    MFQ_REQUIRE(d && weight && x && y, MFQ_ERR_INVALID, "nint_gemm: null argument");
    MFQ_REQUIRE(M >= 1, MFQ_ERR_INVALID, "nint_gemm: M=%d", M);
    MFQ_REQUIRE(x_dtype == MFQ_X_BF16 || x_dtype == MFQ_X_F16, MFQ_ERR_INVALID, "nint_gemm: x_dtype=%d", x_dtype);
    MFQ_REQUIRE(ldx >= d->neuron_len && ldy >= d->out, MFQ_ERR_INVALID, "nint_gemm: ldx/ldy smaller than the tensor");
    hipStream_t st = as_stream(stream);
    if (nint_streams(d, M)) return nint_gemv_any(d, weight, x, x_dtype, ldx, M, y, ldy, st);
    if (nint_tile_capable(d)) {
        const size_t need = nint_tile_workspace_least(d, M);
        const bool room = workspace && workspace_bytes >= need;
        // without the workspace the batches the streaming kernels can serve, if more slowly, stay served
        if (!room && M <= nint_stream_limit(d)) return nint_gemv_any(d, weight, x, x_dtype, ldx, M, y, ldy, st);
        MFQ_REQUIRE(room, MFQ_ERR_WORKSPACE, "nint_gemm: workspace %zu < %zu bytes", workspace_bytes, need);
        return nint_tile(d, weight, x, x_dtype, ldx, M, y, ldy, false, 0, 0, workspace, workspace_bytes, st);
    }
    const size_t need = dequant_gemm_workspace_least(d->out, d->neuron_len, M);
    MFQ_REQUIRE(workspace && workspace_bytes >= need, MFQ_ERR_WORKSPACE, "nint_gemm: workspace %zu < %zu bytes",
                workspace_bytes, need);
    uint16_t *w16;
    float *wscale;
    int Kp;
    dequant_gemm_carve(workspace, d->out, d->neuron_len, M, w16, wscale, Kp);
    if (int rc = nint_dequant_f16(d, weight, w16, Kp, wscale, st)) return rc;
    return dequant_gemm(workspace, workspace_bytes, d->out, d->neuron_len, x, x_dtype, ldx, M, y, ldy, st);
}

// The batch sizes at which the fused epilogue runs: those of the tile kernel, where it pays.
static bool nint_gemm_glu_fuses(const mfq_nint_desc *d, int M) { return !nint_streams(d, M) && nint_tile_glu_pays(d, M); }

extern "C" int mfq_hip_nint_gemm_glu(const mfq_nint_desc *d, const void *weight, const void *x, int x_dtype, int64_t ldx,
                                     int M, int activation, void *hidden, int out_dtype, int64_t ldh, void *workspace,
                                     size_t workspace_bytes, mfq_stream_t stream) {
    MFQ_REQUIRE(d && weight && x && hidden, MFQ_ERR_INVALID, "nint_gemm_glu: null argument");
    MFQ_REQUIRE(M >= 1, MFQ_ERR_INVALID, "nint_gemm_glu: M=%d", M);
    MFQ_REQUIRE(x_dtype == MFQ_X_BF16 || x_dtype == MFQ_X_F16, MFQ_ERR_INVALID, "nint_gemm_glu: x_dtype=%d", x_dtype);
    MFQ_REQUIRE(out_dtype == MFQ_X_BF16 || out_dtype == MFQ_X_F16, MFQ_ERR_INVALID, "nint_gemm_glu: out_dtype=%d", out_dtype);
    MFQ_REQUIRE(activation == MFQ_GLU_SILU || activation == MFQ_GLU_GELU, MFQ_ERR_INVALID, "nint_gemm_glu: activation=%d",
                activation);
    MFQ_REQUIRE(d->out % 2 == 0 && ldx >= d->neuron_len && ldh >= d->out / 2, MFQ_ERR_INVALID,
                "nint_gemm_glu: ldx/ldh smaller than the tensor");
    if (!nint_gemm_glu_fuses(d, M))
        return fail(MFQ_ERR_UNSUPPORTED, "nint_gemm_glu: %d rows of this tensor do not take the one-pass tile kernel", M);
    const size_t need = nint_tile_workspace_least(d, M);
    MFQ_REQUIRE(workspace && workspace_bytes >= need, MFQ_ERR_WORKSPACE, "nint_gemm_glu: workspace %zu < %zu bytes",
                workspace_bytes, need);
    return nint_tile(d, weight, x, x_dtype, ldx, M, hidden, ldh, true, activation == MFQ_GLU_GELU, out_dtype == MFQ_X_F16,
                     workspace, workspace_bytes, as_stream(stream));
}

extern "C" int mfq_hip_nint_tile_plan(const mfq_nint_desc *d, int M, int glu, int *splits) {
    if (!d || M < 1 || nint_streams(d, M) || !nint_tile_capable(d) || (glu && !nint_gemm_glu_fuses(d, M))) return -1;
    return nint_tile_shape(d, M, glu != 0, splits);
}

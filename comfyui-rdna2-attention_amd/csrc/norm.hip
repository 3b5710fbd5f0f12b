// RMSNorm for fp16 rows with fp32 math, reading and writing each value once, plus the QK-norm +
// RoPE variant of a Krea 2 block.
//
// norm_row (rms_norm.hip:9-65): TPR threads share a row, thread t owns the 8-value chunks
// t + c TPR. Its sum of squares is accumulated with FMAs chunk by chunk; the partial sums are
// folded by xor butterflies inside each 32-lane half-wave (16, 8, 4, 2, 1; 8, 4, 2, 1 for TPR 16)
// and, for TPR 256, the eight half-wave sums are added in order. rstd = 1 / sqrt(sum / D + eps)
// (correctly rounded, where the reference has rsqrtf), y = fp16(x * rstd * (w + 1)).
// Rows are addressed with (b, h, l) strides, so Q and K are read straight from a linear output;
// the result is written contiguous (B, H, L, D). norm_kernel does a row per TPR threads; norm_rope_kernel, whose
// rows have D = 128, one or two heads of a token per 16 threads.
#include "common.h"

#define NT 256

template <int TPR, int CHUNKS>
__global__ __launch_bounds__(NT) void norm_kernel(const half_t* __restrict__ X, const float* __restrict__ W, half_t* __restrict__ Y, int rows, int D, int L,
                                                  int H, long sb, long sh, long sl, float eps) {
    __shared__ float red[NT / 32];
    const int t = threadIdx.x % TPR, n = blockIdx.x * (NT / TPR) + threadIdx.x / TPR;
    if (TPR < NT && n >= rows) return;
    // Heads go first, so a block reads neighbouring heads of one token.
    const int h = n % H, l = (n / H) % L, b = n / H / L;
    const h8* x = (const h8*)(X + b * sb + h * sh + l * sl);
    // Every load is issued up front, x then the weight, with no load under a branch (chunks past D / 8
    // re-read chunk 0 and are not used), so the weight arrives during the reduction instead of after it;
    // the host picks CHUNKS as the chunks D needs per thread.
    h8 v[CHUNKS];
    f4 wv[CHUNKS][2];
#pragma unroll
    for (int c = 0; c < CHUNKS; c++) {
        const int i = t + c * TPR;
        v[c] = x[i < D / 8 ? i : 0];
    }
#pragma unroll
    for (int c = 0; c < CHUNKS; c++) {
        const int i = t + c * TPR, iw = i < D / 8 ? i : 0;
        wv[c][0] = ((const f4*)W)[iw * 2];
        wv[c][1] = ((const f4*)W)[iw * 2 + 1];
    }
    float sum = 0.f;
#pragma unroll
    for (int c = 0; c < CHUNKS; c++) {
        const int i = t + c * TPR;
        if (i < D / 8) {
#pragma unroll
            for (int j = 0; j < 8; j++) sum = __builtin_fmaf((float)v[c][j], (float)v[c][j], sum);
        }
    }
    sum = xor_butterfly_sum<(TPR < 32 ? TPR : 32)>(sum);
    if (TPR > 32) {
        if ((threadIdx.x & 31) == 0) red[threadIdx.x >> 5] = sum;
        __syncthreads();
        sum = 0.f;
#pragma unroll
        for (int i = 0; i < NT / 32; i++) sum += red[i];
    }
    const float rstd = 1.f / sqrtf(sum / (float)D + eps);
    h8* y = (h8*)(Y + ((size_t)(b * H + h) * L + l) * D);
#pragma unroll
    for (int c = 0; c < CHUNKS; c++) {
        const int i = t + c * TPR;
        if (i < D / 8) {
            const f4 lo = wv[c][0], hi = wv[c][1];
            h8 o;
#pragma unroll
            for (int j = 0; j < 8; j++) o[j] = to_half((float)v[c][j] * rstd * ((j < 4 ? lo[j & 3] : hi[j & 3]) + 1.f));
            y[i] = o;
        }
    }
}

// HPT heads of one token per 16 threads, H / HPT apart so that neighbouring slots still read neighbouring rows. What bounds
// a row of one head is not its 512 bytes of x and y but the 1.5 KiB of weight and frequencies each head's threads load
// again from L2; two heads share them. Replayed on the same tensors: 4096 x 24 heads 12.5 -> 9.7 us, 8192 x 24 20.9 -> 18.1
// (5.6 TB/s of x, y); in a block, after other work, 4096 x 24 takes 11.7. Four heads per 16 threads: 11.3 and 19.5 where two took 11.5 and 19.0.
template <int HPT>
__global__ __launch_bounds__(NT) void norm_rope_kernel(const half_t* __restrict__ X, const float* __restrict__ W, half_t* __restrict__ Y, int units, int L, int H,
                                                       long sb, long sh, long sl, float eps, const f4* __restrict__ F, long fb) {
    constexpr int D = 128, TPR = 16;
    const int t = threadIdx.x % TPR, n = blockIdx.x * (NT / TPR) + threadIdx.x / TPR;
    if (n >= units) return;
    const int G = H / HPT, h0 = n % G, l = (n / G) % L, b = n / G / L;
    const half_t* x = X + b * sb + l * sl + t * 8;
    // Every load up front, as in norm_kernel.
    h8 v[HPT];
    f4 m[4];
#pragma unroll
    for (int c = 0; c < HPT; c++) v[c] = *(const h8*)(x + (h0 + c * G) * sh);
    const f4 lo = ((const f4*)W)[t * 2], hi = ((const f4*)W)[t * 2 + 1];
    const f4* f = F + b * fb + (long)l * (D / 2) + t * 4;
#pragma unroll
    for (int j = 0; j < 4; j++) m[j] = f[j];
#pragma unroll
    for (int c = 0; c < HPT; c++) {
        float sum = 0.f;
#pragma unroll
        for (int j = 0; j < 8; j++) sum = __builtin_fmaf((float)v[c][j], (float)v[c][j], sum);
        sum = xor_butterfly_sum<16>(sum);
        const float rstd = 1.f / sqrtf(sum / (float)D + eps);
        h8 o;
#pragma unroll
        for (int j = 0; j < 8; j++) o[j] = to_half((float)v[c][j] * rstd * ((j < 4 ? lo[j & 3] : hi[j & 3]) + 1.f));
        // rms_norm.hip:48-61: a = fma(m1, x1, fp32(m0 x0)), c = fma(m3, x1, fp32(m2 x0)), each rounded to fp32 and then to
        // fp16 (to_half), like the reference.
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const float x0 = (float)o[j * 2], x1 = (float)o[j * 2 + 1];
            const float a = __builtin_fmaf(m[j][1], x1, m[j][0] * x0), d = __builtin_fmaf(m[j][3], x1, m[j][2] * x0);
            o[j * 2] = to_half(a);
            o[j * 2 + 1] = to_half(d);
        }
        *(h8*)(Y + ((size_t)(b * H + h0 + c * G) * L + l) * D + t * 8) = o;
    }
}

static bool norm_ok(int B, int H, int L, int D) { return B > 0 && H > 0 && L > 0 && D > 0 && D % 8 == 0; }

extern "C" {

// rms_norm_head (rms_norm.hip:67-69): D <= 128, 16 threads per row.
int rda_rms_norm_head(const void* x, const float* w, void* y, int B, int H, int L, int D, long sb, long sh, long sl, float eps, void* stream) {
    if (!norm_ok(B, H, L, D) || D > 128) return RDA_ERR_INVALID;
    const int rows = B * H * L;
    hipLaunchKernelGGL((norm_kernel<16, 1>), dim3((rows + 15) / 16), dim3(NT), 0, (hipStream_t)stream, (const half_t*)x, w, (half_t*)y, rows, D, L,
                       H, sb, sh, sl, eps);
    return (int)hipGetLastError();
}

// rms_norm_row (rms_norm.hip:71-73): 128 < D <= 8192, 256 threads per row.
int rda_rms_norm_row(const void* x, const float* w, void* y, int B, int H, int L, int D, long sb, long sh, long sl, float eps, void* stream) {
    if (!norm_ok(B, H, L, D) || D > 8192) return RDA_ERR_INVALID;
    const int rows = B * H * L;
    // Chunks per thread: as many as D needs (the loads of a thread's unused chunks are not free).
    auto launch = [&](auto kern) {
        hipLaunchKernelGGL(kern, dim3(rows), dim3(NT), 0, (hipStream_t)stream, (const half_t*)x, w, (half_t*)y, rows, D, L, H, sb, sh, sl, eps);
        return (int)hipGetLastError();
    };
    switch ((D / 8 + NT - 1) / NT) {
    case 1: return launch(norm_kernel<NT, 1>);
    case 2: return launch(norm_kernel<NT, 2>);
    case 3: return launch(norm_kernel<NT, 3>);
    default: return launch(norm_kernel<NT, 4>);
    }
}

// rms_norm_rope (rms_norm.hip:75-77): QK-norm over D = 128 then RoPE; freqs [.., L, 64, 2, 2] fp32,
// fb = the batch stride in 2x2 matrices (0 to broadcast one batch).
int rda_rms_norm_rope(const void* x, const float* w, void* y, int B, int H, int L, int D, long sb, long sh, long sl, float eps, const float* freqs,
                      long fb, void* stream) {
    if (!norm_ok(B, H, L, D) || D != 128) return RDA_ERR_INVALID;
    const int rows = B * H * L;
    auto launch = [&](auto kern, int units) {
        hipLaunchKernelGGL(kern, dim3((units + 15) / 16), dim3(NT), 0, (hipStream_t)stream, (const half_t*)x, w, (half_t*)y, units, L, H, sb, sh, sl, eps,
                           (const f4*)freqs, fb);
        return (int)hipGetLastError();
    };
    // Two heads per slot need twice the rows to fill the chip: at 12288 rows both take 3.6 us, at 26424 one head per slot
    // takes 5.35 and two 5.1, at 2100 2.2 and 2.5. An odd number of heads stays with one.
    if (H % 2 == 0 && rows >= 16384) return launch(norm_rope_kernel<2>, rows / 2);
    return launch(norm_rope_kernel<1>, rows);
}

int rda_version(void) { return 1; }

}  // extern "C"

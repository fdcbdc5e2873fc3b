// attention_aux.hip -- the reference-shaped helper kernels around the attention GEMMs:
// Q/K/V bias + head transpose, scale+mask+softmax (in place), transpose back.
// All are pure HBM streaming; 16-byte accesses.
#include "common.hpp"

namespace lg {

// ---- buf[b,head,s,:] = X[b,s,head,:] + bias[head,:]   (attention_kernels.cu:79-224) -----------------
template <typename T>
struct QkvPtrs {
    const T* src[3];
    const T* bias[3];
    T* dst[3];
};

// FUSED = false: three separate [M, n] inputs; true: one packed [M, 3, n] input with bias [3, n].
template <typename T, bool VEC>
__global__ __launch_bounds__(256) void qkv_bias_transpose_kernel(QkvPtrs<T> p, int seq, int head_num, int d,
                                                                 int64_t src_row_stride, int64_t total) {
    constexpr int VN = VEC ? Vec16<T>::N : 1;
    const int t = blockIdx.y;
    const T* __restrict__ src = p.src[t];
    const T* __restrict__ bias = p.bias[t];
    T* dst = p.dst[t];
    const int n = head_num * d;
    const int nv = n / VN;   // vectors per token row
    const int dv = d / VN;   // vectors per head
    for (int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; v < total; v += (int64_t)gridDim.x * blockDim.x) {
        const int64_t tok = v / nv;          // b*seq + s
        const int c = (int)(v % nv);         // vector column inside the row
        const int head = c / dv, e = c % dv;
        const int64_t b = tok / seq;
        const int s = (int)(tok % seq);
        const int64_t si = tok * src_row_stride + (int64_t)c * VN;
        const int64_t di = (((b * head_num + head) * seq + s) * (int64_t)d) + (int64_t)e * VN;
        if (VEC) {
            typedef Vec16<T> V;
            V a = *reinterpret_cast<const V*>(src + si);
            V bb = *reinterpret_cast<const V*>(bias + (int64_t)c * VN);
            V o;
#pragma unroll
            for (int j = 0; j < V::N; ++j) o.set(j, a.get(j) + bb.get(j));
            *reinterpret_cast<V*>(dst + di) = o;
        } else {
            stf(dst + di, ldf(src + si) + ldf(bias + c));
        }
    }
}

template <typename T>
static int launch_qkv(const QkvPtrs<T>& p, int batch, int seq, int head_num, int d, int64_t src_row_stride,
                      hipStream_t stream, const char* what) {
    if (batch < 0 || seq < 0 || head_num <= 0 || d <= 0) { set_error("%s: bad shape", what); return LG_ERR_INVALID; }
    for (int t = 0; t < 3; ++t)
        if (!p.src[t] || !p.bias[t] || !p.dst[t]) { set_error("%s: null pointer", what); return LG_ERR_INVALID; }
    const int64_t M = (int64_t)batch * seq;
    if (M == 0) return LG_OK;
    constexpr int VN = Vec16<T>::N;
    bool vec = (d % VN == 0) && (src_row_stride % VN == 0);
    for (int t = 0; t < 3; ++t) vec = vec && aligned16(p.src[t]) && aligned16(p.bias[t]) && aligned16(p.dst[t]);
    const int64_t total = M * head_num * d / (vec ? VN : 1);
    int64_t grid = (total + 255) / 256;
    if (grid > 32768) grid = 32768;
    if (vec)
        hipLaunchKernelGGL((qkv_bias_transpose_kernel<T, true>), dim3((int)grid, 3), dim3(256), 0, stream, p, seq,
                           head_num, d, src_row_stride, total);
    else
        hipLaunchKernelGGL((qkv_bias_transpose_kernel<T, false>), dim3((int)grid, 3), dim3(256), 0, stream, p, seq,
                           head_num, d, src_row_stride, total);
    return check_launch(what);
}

// ---- dst[b,s,head,:] = src[b,head,s,:]   (attention_kernels.cu:682-742) -----------------------------
template <typename T, bool VEC>
__global__ __launch_bounds__(256) void transpose_back_kernel(T* dst, const T* __restrict__ src, int seq, int head_num,
                                                             int d, int64_t total) {
    constexpr int VN = VEC ? Vec16<T>::N : 1;
    const int dv = d / VN;
    for (int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; v < total; v += (int64_t)gridDim.x * blockDim.x) {
        // v enumerates dst in [b, s, head, e] order
        const int e = (int)(v % dv);
        const int64_t r = v / dv;
        const int head = (int)(r % head_num);
        const int64_t tok = r / head_num;
        const int64_t b = tok / seq;
        const int s = (int)(tok % seq);
        const int64_t si = (((b * head_num + head) * seq + s) * (int64_t)d) + (int64_t)e * VN;
        const int64_t di = v * VN;
        if (VEC) {
            typedef Vec16<T> V;
            *reinterpret_cast<V*>(dst + di) = *reinterpret_cast<const V*>(src + si);
        } else {
            dst[di] = src[si];
        }
    }
}

template <typename T>
static int launch_transpose(T* dst, const T* src, int batch, int seq, int head_num, int d, hipStream_t stream) {
    if (batch < 0 || seq < 0 || head_num <= 0 || d <= 0 || !dst || !src) { set_error("transpose: bad arguments"); return LG_ERR_INVALID; }
    const int64_t n = (int64_t)batch * seq * head_num * d;
    if (n == 0) return LG_OK;
    constexpr int VN = Vec16<T>::N;
    const bool vec = (d % VN == 0) && aligned16(dst) && aligned16(src);
    const int64_t total = n / (vec ? VN : 1);
    int64_t grid = (total + 255) / 256;
    if (grid > 32768) grid = 32768;
    if (vec)
        hipLaunchKernelGGL((transpose_back_kernel<T, true>), dim3((int)grid), dim3(256), 0, stream, dst, src, seq, head_num, d, total);
    else
        hipLaunchKernelGGL((transpose_back_kernel<T, false>), dim3((int)grid), dim3(256), 0, stream, dst, src, seq, head_num, d, total);
    return check_launch("transpose");
}

// ---- softmax (attention_kernels.cu:395-680) -----------------------------------------------------------
//   t = qk*scalar + (1 - mask)*(-10000);  p = exp(t - max t);  out = p / (sum p + 1e-6)
// LPR lanes per row, the row held in registers as NC vectors of 16 bytes per lane, at any alignment (global memory takes such loads and
// stores as whole ones; a last vector that is not whole is read as one too, with elements before it).  What a row costs besides its
// elements -- its place in the mask, two butterflies, a reciprocal -- is a few hundred vector instructions for a wave however many rows it
// holds, and short rows are bound by it: so a wave has as many rows as it has room for, two vectors a lane from 33 vectors on.  One row a
// wave before, us, fp16: 8 x 48 heads, 128 tokens 18.3 -> 6.1, 4 x 16, 200 7.3 -> 4.6, 2 x 48, 333 19.4 -> 13.6, 512 20.6 -> 18.0; fp32
// 8 x 48, 128 15.2 -> 8.3, 4 x 16, 200 6.6 -> 5.1, 2 x 48, 333 20.4 -> 18.8, longer ones level (memory).  Rows longer than 512 vectors take a workgroup
// and three passes each.
// the vector without its first `bytes` bytes (a multiple of the element's size); what comes after its last ones is anything
template <int SIZE, typename V>
__device__ __forceinline__ V vec_from(V v, int bytes) {
    typedef unsigned uint4_t __attribute__((ext_vector_type(4)));
    const uint4_t u = __builtin_bit_cast(uint4_t, v);
    const bool by8 = bytes & 8, by4 = bytes & 4;
    const unsigned a0 = by8 ? u[2] : u[0], a1 = by8 ? u[3] : u[1];
    unsigned b0 = by4 ? a1 : a0, b1 = by4 ? u[2] : a1, b2 = by4 ? u[3] : u[2], b3 = u[3];
    if (SIZE == 2) {
        const unsigned bits = (bytes & 2) * 8;
        b0 = __builtin_amdgcn_alignbit(b1, b0, bits);
        b1 = __builtin_amdgcn_alignbit(b2, b1, bits);
        b2 = __builtin_amdgcn_alignbit(b3, b2, bits);
        b3 = __builtin_amdgcn_alignbit(0, b3, bits);
    }
    return __builtin_bit_cast(V, uint4_t{b0, b1, b2, b3});
}

template <typename T, int NC, int LPR>
__global__ __launch_bounds__(256) void softmax_wave_kernel(T* buf, const T* __restrict__ mask, int seq, int head_num,
                                                           int64_t rows, float scalar) {
    constexpr int VN = Vec16<T>::N;
    typedef T aligned_t __attribute__((ext_vector_type(VN)));
    typedef T vec_t __attribute__((ext_vector_type(VN), aligned(sizeof(T))));
    const int lane = threadIdx.x % LPR;
    const int64_t row = (int64_t)blockIdx.x * (256 / LPR) + threadIdx.x / LPR;
    if (row >= rows) return;
    int64_t b;
    int sq;
    if (rows <= 0x7fffffff) {
        const unsigned head = (unsigned)row / (unsigned)seq;
        b = head / (unsigned)head_num;
        sq = (int)((unsigned)row - head * (unsigned)seq);
    } else {
        b = row / ((int64_t)head_num * seq);
        sq = (int)(row % seq);
    }
    T* p = buf + row * seq;
    const T* mrow = mask + (b * seq + sq) * (int64_t)seq;
    // in a row that is no whole number of vectors, whether the lanes' vectors c are all inside
    auto inside = [&](int c) { return seq % VN == 0 || (c + 1) * LPR * VN <= seq; };
    float t[NC][VN];
    float mx = -1e20f;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        const int i = (lane + c * LPR) * VN;  // this lane's first element of the vector
#pragma unroll
        for (int j = 0; j < VN; ++j) t[c][j] = -1e20f;
        if (inside(c)) {
            if (i < seq) {
                const vec_t a = *reinterpret_cast<const vec_t*>(p + i), m = *reinterpret_cast<const vec_t*>(mrow + i);
#pragma unroll
                for (int j = 0; j < VN; ++j) t[c][j] = (float)a[j] * scalar + (1.0f - (float)m[j]) * -10000.0f;
            }
        } else if (seq >= VN) {
            // the last vector, which is not whole, comes with elements before it, and the lanes beyond read the same one
            const int at = min(i, seq - VN), skip = (i - at) * (int)sizeof(T);
            const aligned_t a = vec_from<sizeof(T)>((aligned_t)*reinterpret_cast<const vec_t*>(p + at), skip);
            const aligned_t m = vec_from<sizeof(T)>((aligned_t)*reinterpret_cast<const vec_t*>(mrow + at), skip);
#pragma unroll
            for (int j = 0; j < VN; ++j)
                if (i + j < seq) t[c][j] = (float)a[j] * scalar + (1.0f - (float)m[j]) * -10000.0f;
        } else {
#pragma unroll
            for (int j = 0; j < VN; ++j)
                if (i + j < seq) t[c][j] = ldf(p + i + j) * scalar + (1.0f - ldf(mrow + i + j)) * -10000.0f;
        }
#pragma unroll
        for (int j = 0; j < VN; ++j) mx = fmaxf(mx, t[c][j]);
    }
    mx = lanes_max<LPR>(mx);
    float sum = 0.f;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        const int i = (lane + c * LPR) * VN;
#pragma unroll
        for (int j = 0; j < VN; ++j) t[c][j] = __expf(t[c][j] - mx);
        if (inside(c)) {
            if (i < seq) {
#pragma unroll
                for (int j = 0; j < VN; ++j) sum += t[c][j];
            }
        } else {
#pragma unroll
            for (int j = 0; j < VN; ++j)
                if (i + j < seq) sum += t[c][j];
        }
    }
    sum = lanes_sum<LPR>(sum);
    const float inv = 1.0f / (sum + 1e-6f);
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        const int i = (lane + c * LPR) * VN;
        if (i + VN <= seq) {
            vec_t o;
#pragma unroll
            for (int j = 0; j < VN; ++j) o[j] = (T)(t[c][j] * inv);
            *reinterpret_cast<vec_t*>(p + i) = o;
        } else if (i < seq) {
#pragma unroll
            for (int j = 0; j < VN; ++j)
                if (i + j < seq) stf(p + i + j, t[c][j] * inv);
        }
    }
}

// rows of any length: one block per row, three passes
template <typename T>
__global__ __launch_bounds__(256) void softmax_scalar_kernel(T* buf, const T* mask, int seq, int head_num, float scalar) {
    __shared__ float scratch[16];
    const int64_t row = blockIdx.x;
    const int64_t b = row / ((int64_t)head_num * seq);
    const int sq = (int)(row % seq);
    T* p = buf + row * seq;
    const T* mrow = mask + (b * seq + sq) * (int64_t)seq;
    float mx = -1e20f;
    for (int i = threadIdx.x; i < seq; i += blockDim.x)
        mx = fmaxf(mx, ldf(p + i) * scalar + (1.0f - ldf(mrow + i)) * -10000.0f);
    mx = block_max(mx, scratch);
    float sum = 0.f;
    for (int i = threadIdx.x; i < seq; i += blockDim.x)
        sum += __expf(ldf(p + i) * scalar + (1.0f - ldf(mrow + i)) * -10000.0f - mx);
    sum = block_sum(sum, scratch);
    const float inv = 1.0f / (sum + 1e-6f);
    for (int i = threadIdx.x; i < seq; i += blockDim.x)
        stf(p + i, __expf(ldf(p + i) * scalar + (1.0f - ldf(mrow + i)) * -10000.0f - mx) * inv);
}

template <typename T>
static int launch_softmax(T* buf, const T* mask, int batch, int seq, int head_num, float scalar, hipStream_t stream) {
    if (batch < 0 || seq < 0 || head_num <= 0 || !buf || !mask) { set_error("attn_softmax: bad arguments"); return LG_ERR_INVALID; }
    const int64_t rows = (int64_t)batch * head_num * seq;
    if (rows == 0) return LG_OK;
    scalar = (float)(T)scalar;  // the reference keeps the scalar as T (bert_layer.h:94)
    constexpr int VN = Vec16<T>::N;
    const int nvec = (seq + VN - 1) / VN;
    if (nvec <= 64 * 8) {
        const int lanes = nvec <= 8 ? 8 : nvec <= 16 ? 16 : nvec <= 64 ? 32 : 64;
        const int64_t grid = (rows + 256 / lanes - 1) / (256 / lanes);
        if (grid > 0x7fffffff) { set_error("attn_softmax: too many rows"); return LG_ERR_INVALID; }
#define LG_SM_LAUNCH(NCC, LANES)                                                                                          \
    hipLaunchKernelGGL((softmax_wave_kernel<T, NCC, LANES>), dim3((unsigned)grid), dim3(256), 0, stream, buf, mask, seq,   \
                       head_num, rows, scalar)
        if (nvec <= 8) LG_SM_LAUNCH(1, 8);
        else if (nvec <= 16) LG_SM_LAUNCH(1, 16);
        else if (nvec <= 32) LG_SM_LAUNCH(1, 32);
        else if (nvec <= 64) LG_SM_LAUNCH(2, 32);
        else if (nvec <= 128) LG_SM_LAUNCH(2, 64);
        else if (nvec <= 256) LG_SM_LAUNCH(4, 64);
        else LG_SM_LAUNCH(8, 64);
#undef LG_SM_LAUNCH
    } else {
        if (rows > 0x7fffffff) { set_error("attn_softmax: too many rows"); return LG_ERR_INVALID; }
        hipLaunchKernelGGL((softmax_scalar_kernel<T>), dim3((unsigned)rows), dim3(256), 0, stream, buf, mask, seq, head_num, scalar);
    }
    return check_launch("attn_softmax");
}

}  // namespace lg

using namespace lg;

extern "C" {

int lg_add_qkv_bias_transpose_f32(float* q_buf, float* k_buf, float* v_buf, const float* Q, const float* bias_Q,
                                  const float* K, const float* bias_K, const float* V, const float* bias_V, int batch,
                                  int seq, int head_num, int size_per_head, void* stream) {
    QkvPtrs<float> p = {{Q, K, V}, {bias_Q, bias_K, bias_V}, {q_buf, k_buf, v_buf}};
    return launch_qkv<float>(p, batch, seq, head_num, size_per_head, (int64_t)head_num * size_per_head,
                             (hipStream_t)stream, "add_qkv_bias_transpose");
}
int lg_add_qkv_bias_transpose_f16(void* q_buf, void* k_buf, void* v_buf, const void* Q, const void* bias_Q,
                                  const void* K, const void* bias_K, const void* V, const void* bias_V, int batch,
                                  int seq, int head_num, int size_per_head, void* stream) {
    QkvPtrs<half_t> p = {{(const half_t*)Q, (const half_t*)K, (const half_t*)V},
                         {(const half_t*)bias_Q, (const half_t*)bias_K, (const half_t*)bias_V},
                         {(half_t*)q_buf, (half_t*)k_buf, (half_t*)v_buf}};
    return launch_qkv<half_t>(p, batch, seq, head_num, size_per_head, (int64_t)head_num * size_per_head,
                              (hipStream_t)stream, "add_qkv_bias_transpose");
}
int lg_add_fused_qkv_bias_transpose_f32(float* q_buf, float* k_buf, float* v_buf, const float* QKV, const float* qkv_bias,
                                        int batch, int seq, int head_num, int size_per_head, void* stream) {
    if (!QKV || !qkv_bias) { set_error("add_fused_qkv_bias_transpose: null pointer"); return LG_ERR_INVALID; }
    const int64_t n = (int64_t)head_num * size_per_head;
    QkvPtrs<float> p = {{QKV, QKV + n, QKV + 2 * n}, {qkv_bias, qkv_bias + n, qkv_bias + 2 * n}, {q_buf, k_buf, v_buf}};
    return launch_qkv<float>(p, batch, seq, head_num, size_per_head, 3 * n, (hipStream_t)stream,
                             "add_fused_qkv_bias_transpose");
}
int lg_add_fused_qkv_bias_transpose_f16(void* q_buf, void* k_buf, void* v_buf, const void* QKV, const void* qkv_bias,
                                        int batch, int seq, int head_num, int size_per_head, void* stream) {
    if (!QKV || !qkv_bias) { set_error("add_fused_qkv_bias_transpose: null pointer"); return LG_ERR_INVALID; }
    const int64_t n = (int64_t)head_num * size_per_head;
    const half_t* x = (const half_t*)QKV;
    const half_t* b = (const half_t*)qkv_bias;
    QkvPtrs<half_t> p = {{x, x + n, x + 2 * n}, {b, b + n, b + 2 * n}, {(half_t*)q_buf, (half_t*)k_buf, (half_t*)v_buf}};
    return launch_qkv<half_t>(p, batch, seq, head_num, size_per_head, 3 * n, (hipStream_t)stream,
                              "add_fused_qkv_bias_transpose");
}
int lg_attn_softmax_f32(float* buffer, const float* attr_mask, int batch, int seq, int head_num, float scalar, void* stream) {
    return launch_softmax<float>(buffer, attr_mask, batch, seq, head_num, scalar, (hipStream_t)stream);
}
int lg_attn_softmax_f16(void* buffer, const void* attr_mask, int batch, int seq, int head_num, float scalar, void* stream) {
    return launch_softmax<half_t>((half_t*)buffer, (const half_t*)attr_mask, batch, seq, head_num, scalar, (hipStream_t)stream);
}
int lg_transpose_f32(float* dst, const float* src, int batch, int seq, int head_num, int size_per_head, void* stream) {
    return launch_transpose<float>(dst, src, batch, seq, head_num, size_per_head, (hipStream_t)stream);
}
int lg_transpose_f16(void* dst, const void* src, int batch, int seq, int head_num, int size_per_head, void* stream) {
    return launch_transpose<half_t>((half_t*)dst, (const half_t*)src, batch, seq, head_num, size_per_head, (hipStream_t)stream);
}

}  // extern "C"

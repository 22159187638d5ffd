// ar_attention.hip -- the C entry points of flash attention (ops.mojo:244-480):
// argument checks, head sizes between the tiled ones, and the choice of the
// fp32 kernels (ar_attn_f32.hip) or the bf16 ones (ar_flash.hip).
#include "ar_internal.hpp"

using namespace ar;

static __host__ __device__ inline bool al16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

#define AR_ATTN_PTRS(...)                                                                   \
    do {                                                                                    \
        const void* ps[] = {__VA_ARGS__};                                                   \
        for (const void* p : ps)                                                            \
            if (!p || !al16(p)) return ar::set_error(AR_EINVAL, "%s: null or unaligned pointer", __func__); \
    } while (0)

// ---- any head_dim <= 128 (ops.mojo:267 accepts every head_dim up to 128) ----
// The tiled kernels exist for head_dim 32, 64 and 128.  Another head_dim runs
// them at the next of those sizes on rows that are zero past head_dim, with
// the softmax scale of the real head_dim: the zero columns add nothing to any
// score or to D, and the output columns past head_dim (O, dQ, dK, dV) are
// exact zeros that are dropped.  The fp32 kernels run on padded copies of
// everything; the bf16 ones pad what they copy anyway (attn_bf16).
namespace {

bool native_hd(int64_t hd) { return hd == 32 || hd == 64 || hd == 128; }
int64_t padded_hd(int64_t hd) { return hd <= 32 ? 32 : (hd <= 64 ? 64 : 128); }
size_t align256(size_t b) { return (b + 255) & ~size_t(255); }

__global__ void pad_rows_k(float* dst, const float* src, int64_t rows, int hd, int hdp) {
    const int64_t n = rows * hdp;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t r = i / hdp;
        const int d = (int)(i - r * hdp);
        dst[i] = d < hd ? src[r * hd + d] : 0.0f;
    }
}
__global__ void unpad_rows_k(float* dst, const float* src, int64_t rows, int hd, int hdp) {
    const int64_t n = rows * hd;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t r = i / hd;
        dst[i] = src[r * hdp + (i - r * hd)];
    }
}

int32_t check_shape(int64_t B, int64_t T, int64_t H, int64_t hd) {
    if (hd <= 0 || B < 0 || T < 0 || H < 0)
        return ar::set_error(AR_EINVAL, "flash attention: bad shape (B %lld, T %lld, H %lld, head_dim %lld)",
                             (long long)B, (long long)T, (long long)H, (long long)hd);
    if (hd > 128)
        return ar::set_error(AR_EUNSUPPORTED, "flash attention: head_dim %lld not in [1, 128]", (long long)hd);
    return AR_OK;
}

// One fp32 attention op at a head_dim outside {32, 64, 128}.  in = {q, k, v[, dO]}.
int32_t attn_padded(ar_stream_t stream, ar::AttnOp op, float* o1, float* o2, const float* const* in,
                    const float* lse, const float* dbuf, int64_t B, int64_t T, int64_t H, int64_t hd,
                    int64_t window) {
    int32_t r = check_shape(B, T, H, hd);
    if (r) return r;
    if (B == 0 || T == 0 || H == 0) return AR_OK;
    const int64_t hdp = padded_hd(hd), rows = B * T * H, n = rows * hdp;
    const int nin = op == ar::AttnOp::FWD ? 3 : 4;
    const int nout = op == ar::AttnOp::DKV ? 2 : 1;
    const size_t each = align256((size_t)n * sizeof(float));
    int32_t st;
    char* w = (char*)ar::workspace(ar::S(stream), (nin + nout) * each, &st);
    if (!w) return st;
    const unsigned g = ar::flat_grid(n, 256);
    float* pin[4] = {nullptr, nullptr, nullptr, nullptr};
    for (int i = 0; i < nin; ++i) {
        pin[i] = (float*)(w + i * each);
        pad_rows_k<<<g, 256, 0, ar::S(stream)>>>(pin[i], in[i], rows, (int)hd, (int)hdp);
    }
    r = ar::check_launch("flash attention: pad head_dim");
    if (r) return r;
    float* p1 = (float*)(w + nin * each);
    float* p2 = op == ar::AttnOp::DKV ? (float*)(w + (nin + 1) * each) : o2;  // FWD: o2 = LSE, unpadded
    const float scale = 1.0f / sqrtf((float)hd);
    r = ar::attn_f32(ar::S(stream), op, p1, p2, pin[0], pin[1], pin[2], pin[3], lse, dbuf, B, T, H, hdp, window,
                     scale);
    if (r) return r;
    const unsigned go = ar::flat_grid(rows * hd, 256);
    unpad_rows_k<<<go, 256, 0, ar::S(stream)>>>(o1, p1, rows, (int)hd, (int)hdp);
    if (op == ar::AttnOp::DKV) unpad_rows_k<<<go, 256, 0, ar::S(stream)>>>(o2, p2, rows, (int)hd, (int)hdp);
    return ar::check_launch("flash attention: unpad head_dim");
}

// One op with bf16 products on fp32 tensors, any head_dim: the two tensors
// that several workgroups stream (in short sequences all of them) are rounded
// and padded into the workspace by one launch, everything else is read and
// written where it is.  The workspace is asked for every operand (and, padded,
// every result): what a call needs does not depend on the sequence's length.
// Against a copy of each operand and of each padded result, the four ops
// together: 708 -> 629 us at 16.8M values a tensor (head_dim 128; 11
// conversions of 18 us became three launches of 28), 189 -> 134 us at a padded
// head_dim (96) and 1.7M.
int32_t attn_bf16(ar_stream_t stream, ar::AttnOp op, float* o1, float* o2, const float* const* in, const float* lse,
                  const float* dbuf, int64_t B, int64_t T, int64_t H, int64_t hd, int64_t window) {
    int32_t r = check_shape(B, T, H, hd);
    if (r) return r;
    if (B == 0 || T == 0 || H == 0) return AR_OK;
    const int64_t n = B * T * H * padded_hd(hd);
    const int nin = op == ar::AttnOp::FWD ? 3 : 4;
    const int nout = native_hd(hd) ? 0 : op == ar::AttnOp::DKV ? 2 : 1;
    const size_t each = align256((size_t)n * sizeof(ar::bf16));
    int32_t st;
    char* w = (char*)ar::workspace(ar::S(stream), nin * each + nout * align256((size_t)n * sizeof(float)), &st);
    if (!w) return st;
    return ar::flash_attn_f32(ar::S(stream), op, o1, o2, in, lse, dbuf, B, T, H, hd, window, (ar::bf16*)w,
                              (int64_t)(each / sizeof(ar::bf16)));
}
}  // namespace

extern "C" int32_t ar_flash_attn_fwd(ar_stream_t stream, float* output, float* lse_out, const float* q, const float* k,
                                     const float* v, int64_t B, int64_t T, int64_t num_heads, int64_t head_dim,
                                     int64_t window_size) {
    AR_ATTN_PTRS(output, q, k, v);
    AR_CHECK_ARG(lse_out != nullptr, "flash_attn_fwd: null lse");
    if (!native_hd(head_dim)) {
        const float* in[3] = {q, k, v};
        return attn_padded(stream, ar::AttnOp::FWD, output, lse_out, in, nullptr, nullptr, B, T, num_heads,
                           head_dim, window_size);
    }
    return ar::attn_f32(S(stream), ar::AttnOp::FWD, output, lse_out, q, k, v, nullptr, nullptr,
                                           nullptr, B, T, num_heads, head_dim, window_size);
}

extern "C" int32_t ar_flash_attn_fwd_bf16(ar_stream_t stream, float* output, float* lse_out, const float* q,
                                          const float* k, const float* v, int64_t B, int64_t T, int64_t num_heads,
                                          int64_t head_dim, int64_t window_size) {
    AR_ATTN_PTRS(output, q, k, v);
    AR_CHECK_ARG(lse_out != nullptr, "flash_attn_fwd_bf16: null lse");
    AR_CHECK_ARG(B >= 0 && T >= 0 && num_heads >= 0, "flash_attn_fwd_bf16: bad shape");
    const float* src[4] = {q, k, v, nullptr};
    return attn_bf16(stream, ar::AttnOp::FWD, output, lse_out, src, nullptr, nullptr, B, T, num_heads, head_dim,
                     window_size);
}
extern "C" int32_t ar_flash_attn_bwd_dq(ar_stream_t stream, float* grad_q, const float* q, const float* k,
                                        const float* v, const float* grad_output, const float* lse, const float* d_buf,
                                        int64_t B, int64_t T, int64_t num_heads, int64_t head_dim,
                                        int64_t window_size) {
    AR_ATTN_PTRS(grad_q, q, k, v, grad_output);
    AR_CHECK_ARG(lse && d_buf, "flash_attn_bwd_dq: null lse / d_buf");
    if (!native_hd(head_dim)) {
        const float* in[4] = {q, k, v, grad_output};
        return attn_padded(stream, ar::AttnOp::DQ, grad_q, nullptr, in, lse, d_buf, B, T, num_heads, head_dim,
                           window_size);
    }
    return ar::attn_f32(S(stream), ar::AttnOp::DQ, grad_q, nullptr, q, k, v, grad_output, lse,
                                           d_buf, B, T, num_heads, head_dim, window_size);
}
extern "C" int32_t ar_flash_attn_bwd_dq_bf16(ar_stream_t stream, float* grad_q, const float* q, const float* k,
                                             const float* v, const float* grad_output, const float* lse,
                                             const float* d_buf, int64_t B, int64_t T, int64_t num_heads,
                                             int64_t head_dim, int64_t window_size) {
    AR_ATTN_PTRS(grad_q, q, k, v, grad_output);
    AR_CHECK_ARG(lse && d_buf, "flash_attn_bwd_dq_bf16: null lse / d_buf");
    AR_CHECK_ARG(B >= 0 && T >= 0 && num_heads >= 0, "flash_attn_bwd_dq_bf16: bad shape");
    const float* src[4] = {q, k, v, grad_output};
    return attn_bf16(stream, ar::AttnOp::DQ, grad_q, nullptr, src, lse, d_buf, B, T, num_heads, head_dim,
                     window_size);
}
extern "C" int32_t ar_flash_attn_bwd_dkv(ar_stream_t stream, float* grad_k, float* grad_v, const float* q,
                                         const float* k, const float* v, const float* grad_output, const float* lse,
                                         const float* d_buf, int64_t B, int64_t T, int64_t num_heads,
                                         int64_t head_dim, int64_t window_size) {
    AR_ATTN_PTRS(grad_k, grad_v, q, k, v, grad_output);
    AR_CHECK_ARG(lse && d_buf, "flash_attn_bwd_dkv: null lse / d_buf");
    if (!native_hd(head_dim)) {
        const float* in[4] = {q, k, v, grad_output};
        return attn_padded(stream, ar::AttnOp::DKV, grad_k, grad_v, in, lse, d_buf, B, T, num_heads, head_dim,
                           window_size);
    }
    return ar::attn_f32(S(stream), ar::AttnOp::DKV, grad_k, grad_v, q, k, v, grad_output, lse,
                                           d_buf, B, T, num_heads, head_dim, window_size);
}
extern "C" int32_t ar_flash_attn_bwd_dkv_bf16(ar_stream_t stream, float* grad_k, float* grad_v, const float* q,
                                              const float* k, const float* v, const float* grad_output,
                                              const float* lse, const float* d_buf, int64_t B, int64_t T,
                                              int64_t num_heads, int64_t head_dim, int64_t window_size) {
    AR_ATTN_PTRS(grad_k, grad_v, q, k, v, grad_output);
    AR_CHECK_ARG(lse && d_buf, "flash_attn_bwd_dkv_bf16: null lse / d_buf");
    AR_CHECK_ARG(B >= 0 && T >= 0 && num_heads >= 0, "flash_attn_bwd_dkv_bf16: bad shape");
    const float* src[4] = {q, k, v, grad_output};
    return attn_bf16(stream, ar::AttnOp::DKV, grad_k, grad_v, src, lse, d_buf, B, T, num_heads, head_dim,
                     window_size);
}

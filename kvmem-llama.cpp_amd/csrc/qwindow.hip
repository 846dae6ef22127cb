// Per-token query window on the device: the query rows the per-token max
// scorer reads, kept where the reference keeps only their sum.
//
// The reference harvests the pre-RoPE, post-q_norm query rows of the query
// span per layer into q_sum_ / q_count_ (harvest_capture('q') and
// harvest_from_host('q'), src/adapter/llama-memory-kvmem.cpp:2157-2172,
// 2206-2219; the strided view is read as ggml lays Qcur out: element (d, h,
// t) at d*nb0 + h*nb1 + t*nb2, bytes_to_f32_token_major :2066-2090).  Here
// the rows themselves are kept, widened to f32 exactly, in a ring of rows
// per layer; at preview they are gathered in token order, either narrowed
// for the MFMA scorer or summed (kvmem_hip_q_accumulate) for the mean-K
// scorer, which then matches the reference's sums bit for bit.
#include "kvmem_internal.hpp"

#include <algorithm>

namespace kvmem_hip {

template <typename QT>
__device__ inline float q_elem(const uint8_t *p) {
    return static_cast<float>(*reinterpret_cast<const QT *>(p));
}

// The (token, row) pairs of a write: packed as token | row << 16 in the
// launch tables when both fit 16 bits, else two words each.
__device__ inline uint2 qwin_pair(const uint8_t *dev, const ArgTables &args, int packed, uint32_t i) {
    if (packed) {
        const uint32_t w = tab_read<uint32_t>(dev, args, 4u * i);
        return make_uint2(w & 0xffffu, w >> 16);
    }
    return make_uint2(tab_read<uint32_t>(dev, args, 8u * i), tab_read<uint32_t>(dev, args, 8u * i + 4u));
}

// grid (n, ceil(E / 256)): pair i = (token in the view, window row).
template <typename QT>
__global__ __launch_bounds__(256) void qwin_write_kernel(const uint8_t *q, uint64_t nb0, uint64_t nb1,
                                                         uint64_t nb2, uint32_t head_dim, uint32_t E,
                                                         const uint8_t *dev, ArgTables args, int packed,
                                                         float *window) {
    const uint32_t i = blockIdx.x;
    const uint32_t e = blockIdx.y * 256u + threadIdx.x;
    if (e >= E) {
        return;
    }
    const uint2 tr = qwin_pair(dev, args, packed, i);
    const uint32_t h = e / head_dim;
    const uint32_t d = e - h * head_dim;
    window[static_cast<uint64_t>(tr.y) * E + e] =
        q_elem<QT>(q + d * nb0 + h * nb1 + static_cast<uint64_t>(tr.x) * nb2);
}

// The same for rows of E contiguous elements, 16 bytes stored per access:
// grid (n, ceil(E / 2048)), two units of 4 elements per thread, both loaded
// before either is stored.  HBM-bound: 512 rows of 6144 f32 move 25 MB in
// 7.3 us (9.9 with one element per thread).
typedef float f32x4_t __attribute__((ext_vector_type(4)));

template <typename QT>
__global__ __launch_bounds__(256) void qwin_write_rows_kernel(const uint8_t *q, uint64_t nb2, uint32_t E,
                                                              const uint8_t *dev, ArgTables args, int packed,
                                                              float *window) {
    typedef QT unit_t __attribute__((ext_vector_type(4)));
    const uint2 tr = qwin_pair(dev, args, packed, blockIdx.x);
    const unit_t *src = reinterpret_cast<const unit_t *>(q + static_cast<uint64_t>(tr.x) * nb2);
    f32x4_t *dst = reinterpret_cast<f32x4_t *>(window + static_cast<uint64_t>(tr.y) * E);
    const uint32_t u0 = blockIdx.y * 512u + threadIdx.x;
    const uint32_t n = E / 4u;
    unit_t v[2];
#pragma unroll
    for (uint32_t j = 0; j < 2u; ++j) {
        if (u0 + j * 256u < n) {
            v[j] = src[u0 + j * 256u];
        }
    }
#pragma unroll
    for (uint32_t j = 0; j < 2u; ++j) {
        if (u0 + j * 256u < n) {
            dst[u0 + j * 256u] = __builtin_convertvector(v[j], f32x4_t);
        }
    }
}

// f32 -> bf16, round to nearest even (NaN stays a quiet NaN).
__device__ inline uint16_t f32_to_bf16_rne(float f) {
    uint32_t u = __float_as_uint(f);
    if ((u & 0x7fffffffu) > 0x7f800000u) {
        return static_cast<uint16_t>((u >> 16) | 0x40u);
    }
    u += 0x7fffu + ((u >> 16) & 1u);
    return static_cast<uint16_t>(u >> 16);
}

template <int OUT>
__device__ inline uint32_t narrow_bits(float v) {
    if constexpr (OUT == KVMEM_TYPE_BF16) {
        return f32_to_bf16_rne(v);
    } else {
        return __builtin_bit_cast(uint16_t, static_cast<_Float16>(v));
    }
}

// grid (n, L): out[l][i][:] = window[l][rows[i]][:] in the output type, one
// element per thread and access (any alignment).
template <int OUT>
__global__ __launch_bounds__(256) void qwin_gather_kernel(const float *window, uint32_t cap, uint32_t E,
                                                          const uint8_t *rows_dev, ArgTables rows_args,
                                                          uint32_t n, uint8_t *out) {
    const uint32_t i = blockIdx.x;
    const uint32_t l = blockIdx.y;
    const uint32_t row = tab_read<uint32_t>(rows_dev, rows_args, 4u * i);
    const float *src = window + (static_cast<uint64_t>(l) * cap + row) * E;
    const uint64_t o = (static_cast<uint64_t>(l) * n + i) * E;
    for (uint32_t e = threadIdx.x; e < E; e += 256u) {
        if constexpr (OUT == KVMEM_TYPE_F32) {
            reinterpret_cast<float *>(out)[o + e] = src[e];
        } else {
            reinterpret_cast<uint16_t *>(out)[o + e] = static_cast<uint16_t>(narrow_bits<OUT>(src[e]));
        }
    }
}

// The same with 16-byte accesses: grid (n, L, ceil(E / 2048)), 8 elements per
// thread, window and out 16-byte aligned and E a multiple of 8.  HBM-bound:
// 64 rows x 16 layers of 6144 f32 to bf16 move 38 MB in 9.0 us (18.2
// with 24 rounds of one element per thread).
template <int OUT>
__global__ __launch_bounds__(256) void qwin_gather_rows_kernel(const float *window, uint32_t cap, uint32_t E,
                                                               const uint8_t *rows_dev, ArgTables rows_args,
                                                               uint32_t n, uint8_t *out) {
    const uint32_t i = blockIdx.x;
    const uint32_t l = blockIdx.y;
    const uint32_t e = (blockIdx.z * 256u + threadIdx.x) * 8u;
    if (e >= E) {
        return;
    }
    const uint32_t row = tab_read<uint32_t>(rows_dev, rows_args, 4u * i);
    const f32x4_t *src = reinterpret_cast<const f32x4_t *>(window + (static_cast<uint64_t>(l) * cap + row) * E + e);
    const uint64_t o = (static_cast<uint64_t>(l) * n + i) * E + e;
    const f32x4_t a = src[0], b = src[1];
    if constexpr (OUT == KVMEM_TYPE_F32) {
        f32x4_t *dst = reinterpret_cast<f32x4_t *>(reinterpret_cast<float *>(out) + o);
        dst[0] = a;
        dst[1] = b;
    } else {
        u32x4_t w;
        w[0] = narrow_bits<OUT>(a[0]) | (narrow_bits<OUT>(a[1]) << 16);
        w[1] = narrow_bits<OUT>(a[2]) | (narrow_bits<OUT>(a[3]) << 16);
        w[2] = narrow_bits<OUT>(b[0]) | (narrow_bits<OUT>(b[1]) << 16);
        w[3] = narrow_bits<OUT>(b[2]) | (narrow_bits<OUT>(b[3]) << 16);
        *reinterpret_cast<u32x4_t *>(reinterpret_cast<uint16_t *>(out) + o) = w;
    }
}

template <int OUT>
static void launch_qwin_gather(hipStream_t stream, const float *window, uint32_t L, uint32_t cap, uint32_t E,
                               const LaunchTables &rows, uint32_t n, uint8_t *out) {
    const uintptr_t both = reinterpret_cast<uintptr_t>(window) | reinterpret_cast<uintptr_t>(out);
    if (E % 8u == 0 && (both & 15u) == 0) {
        qwin_gather_rows_kernel<OUT><<<dim3(n, L, (E + 2047u) / 2048u), 256, 0, stream>>>(window, cap, E, rows.dev,
                                                                                         rows.args, n, out);
    } else {
        qwin_gather_kernel<OUT><<<dim3(n, L), 256, 0, stream>>>(window, cap, E, rows.dev, rows.args, n, out);
    }
}

template <typename QT>
static void launch_qwin_write(hipStream_t stream, const uint8_t *q, size_t nb0, size_t nb1, size_t nb2,
                              uint32_t n_head, uint32_t head_dim, const LaunchTables &pairs, int packed, uint32_t n,
                              float *window) {
    const uint32_t E = n_head * head_dim;
    // rows of contiguous elements whose 4-element units are aligned on both sides
    const bool rows = nb0 == sizeof(QT) && (n_head == 1 || nb1 == head_dim * sizeof(QT)) && E % 4u == 0 &&
                      nb2 % (4u * sizeof(QT)) == 0 && reinterpret_cast<uintptr_t>(q) % (4u * sizeof(QT)) == 0 &&
                      (reinterpret_cast<uintptr_t>(window) & 15u) == 0;
    if (rows) {
        qwin_write_rows_kernel<QT><<<dim3(n, (E + 2047u) / 2048u), 256, 0, stream>>>(q, nb2, E, pairs.dev, pairs.args,
                                                                                    packed, window);
    } else {
        qwin_write_kernel<QT><<<dim3(n, (E + 255u) / 256u), 256, 0, stream>>>(q, nb0, nb1, nb2, head_dim, E,
                                                                             pairs.dev, pairs.args, packed, window);
    }
}

bool load_qwindow_kernels() {
    return load_kernel_object(&qwin_gather_kernel<KVMEM_TYPE_F32>);
}

}  // namespace kvmem_hip

using namespace kvmem_hip;

extern "C" {

int kvmem_hip_q_window_write(kvmem_hip_ctx *ctx, const void *q, int32_t q_type, uint32_t n_head,
                             uint32_t head_dim, size_t nb0, size_t nb1, size_t nb2,
                             const uint32_t *tokens, const uint32_t *rows, uint32_t n, float *window,
                             uint32_t capacity) {
    if (!ctx) {
        return KVMEM_HIP_ERR_INVALID;
    }
    if (n == 0) {
        return KVMEM_HIP_OK;
    }
    if (!q || !tokens || !rows || !window || n_head == 0 || head_dim == 0) {
        return fail(ctx, KVMEM_HIP_ERR_INVALID, "q_window_write: null argument or empty geometry");
    }
    if (q_type != KVMEM_TYPE_F32 && q_type != KVMEM_TYPE_F16 && q_type != KVMEM_TYPE_BF16) {
        return fail(ctx, KVMEM_HIP_ERR_UNSUPPORTED, "q_window_write: query must be F32, F16 or BF16");
    }
    const size_t esz = q_type == KVMEM_TYPE_F32 ? 4 : 2;
    if (nb0 % esz || nb1 % esz || nb2 % esz || (reinterpret_cast<uintptr_t>(q) % esz) ||
        (reinterpret_cast<uintptr_t>(window) & 3u)) {
        return fail(ctx, KVMEM_HIP_ERR_INVALID, "q_window_write: strides must be multiples of the element size");
    }
    std::vector<uint8_t> seen(capacity, 0);
    uint32_t most = 0;
    for (uint32_t i = 0; i < n; ++i) {
        if (rows[i] >= capacity) {
            return fail(ctx, KVMEM_HIP_ERR_INVALID, "q_window_write: row beyond the window's capacity");
        }
        if (seen[rows[i]]) {
            return fail(ctx, KVMEM_HIP_ERR_INVALID, "q_window_write: a row is written twice");
        }
        seen[rows[i]] = 1;
        most = std::max(most, std::max(tokens[i], rows[i]));
    }
    // token | row << 16 where they fit (768 pairs then travel in the kernel
    // arguments), else two words
    const int packed = most <= 0xffffu ? 1 : 0;
    std::vector<uint32_t> pairs;
    pairs.reserve((packed ? 1 : 2) * static_cast<size_t>(n));
    for (uint32_t i = 0; i < n; ++i) {
        if (packed) {
            pairs.push_back(tokens[i] | (rows[i] << 16));
        } else {
            pairs.push_back(tokens[i]);
            pairs.push_back(rows[i]);
        }
    }
    (void) hipSetDevice(ctx->device);
    LaunchTables lt;
    if (!stage_tables(ctx, pairs.data(), pairs.size() * sizeof(uint32_t), lt, "q_window_write list")) {
        return KVMEM_HIP_ERR_RUNTIME;
    }
    if (injected_fail(ctx, KVMEM_HIP_FAIL_LAUNCH, "q_window_write launch")) {
        return KVMEM_HIP_ERR_RUNTIME;
    }
    const uint8_t *qb = static_cast<const uint8_t *>(q);
    if (q_type == KVMEM_TYPE_F32) {
        launch_qwin_write<float>(ctx->stream, qb, nb0, nb1, nb2, n_head, head_dim, lt, packed, n, window);
    } else if (q_type == KVMEM_TYPE_F16) {
        launch_qwin_write<_Float16>(ctx->stream, qb, nb0, nb1, nb2, n_head, head_dim, lt, packed, n, window);
    } else {
        launch_qwin_write<__bf16>(ctx->stream, qb, nb0, nb1, nb2, n_head, head_dim, lt, packed, n, window);
    }
    return hip_ok(ctx, hipGetLastError(), "q_window_write launch") ? KVMEM_HIP_OK : KVMEM_HIP_ERR_RUNTIME;
}

int kvmem_hip_q_window_gather(kvmem_hip_ctx *ctx, const float *window, uint32_t n_layers,
                              uint32_t capacity, uint32_t n_embd_q, const uint32_t *rows, uint32_t n,
                              int32_t out_type, void *out) {
    if (!ctx) {
        return KVMEM_HIP_ERR_INVALID;
    }
    if (n == 0 || n_layers == 0) {
        return KVMEM_HIP_OK;
    }
    if (!window || !rows || !out || n_embd_q == 0) {
        return fail(ctx, KVMEM_HIP_ERR_INVALID, "q_window_gather: null argument");
    }
    if (out_type != KVMEM_TYPE_F32 && out_type != KVMEM_TYPE_F16 && out_type != KVMEM_TYPE_BF16) {
        return fail(ctx, KVMEM_HIP_ERR_UNSUPPORTED, "q_window_gather: output must be F32, F16 or BF16");
    }
    for (uint32_t i = 0; i < n; ++i) {
        if (rows[i] >= capacity) {
            return fail(ctx, KVMEM_HIP_ERR_INVALID, "q_window_gather: row beyond the capacity");
        }
    }
    if (n_layers > 65535u) {
        return fail(ctx, KVMEM_HIP_ERR_INVALID, "q_window_gather: too many layers");
    }
    (void) hipSetDevice(ctx->device);
    // the row list travels in the kernel arguments when it fits (768 rows)
    LaunchTables lt;
    if (!stage_tables(ctx, rows, sizeof(uint32_t) * n, lt, "q_window_gather rows")) {
        return KVMEM_HIP_ERR_RUNTIME;
    }
    if (injected_fail(ctx, KVMEM_HIP_FAIL_LAUNCH, "q_window_gather launch")) {
        return KVMEM_HIP_ERR_RUNTIME;
    }
    uint8_t *o = static_cast<uint8_t *>(out);
    if (out_type == KVMEM_TYPE_F32) {
        launch_qwin_gather<KVMEM_TYPE_F32>(ctx->stream, window, n_layers, capacity, n_embd_q, lt, n, o);
    } else if (out_type == KVMEM_TYPE_F16) {
        launch_qwin_gather<KVMEM_TYPE_F16>(ctx->stream, window, n_layers, capacity, n_embd_q, lt, n, o);
    } else {
        launch_qwin_gather<KVMEM_TYPE_BF16>(ctx->stream, window, n_layers, capacity, n_embd_q, lt, n, o);
    }
    return hip_ok(ctx, hipGetLastError(), "q_window_gather launch") ? KVMEM_HIP_OK : KVMEM_HIP_ERR_RUNTIME;
}

}  // extern "C"

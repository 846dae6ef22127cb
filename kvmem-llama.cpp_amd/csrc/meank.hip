// Mean-K cosine block scorer (the reference's retrieval scorer) and its
// producers: per-block key sums from the F16 history, the decode-time
// running key sum, and the per-layer query sums.
//
// Producer: k_sum[l][b][e] = fp32 sum of the block's F16 keys in token
// order, mean_tokens[l][b] = tokens summed (RawKvStore::capture_mean_f16,
// kvmem/src/host/raw_kv_store.cpp:184-202).  A thread owns four or eight
// consecutive channels and adds token after token, so every channel's sum is the same
// sequence of IEEE additions as the reference's: bit-identical.
//
// Scorer (llama_memory_kvmem::score_retrieval, src/adapter/
// llama-memory-kvmem.cpp:2869-2916):
//   qv[l][h]   = (sum_{gi<g} q_sum[l][h*g+gi]) * (1 / (q_count[l]*g))
//   mk         = k_sum[l][b] * (1 / mean_tokens[l][b])
//   cos[l][b][h] = (qv . mk_h) / (sqrt(|qv|^2) * sqrt(|mk_h|^2) + 1e-6)
//   score[b]   = mean over layers with q_count > 0 of (sum_h cos) / Hkv,
// layer and block sums in double as the reference; blocks with no keys in
// any layer score 0.  Sixteen lanes per (block, layer) compute each head's
// dot products with a lane-then-tree reduction (the reference sums in
// channel order: results agree to ~1e-7 of the norms).  HBM-bound: the
// 16 x 2048-block scorer reads 128 MiB of fp32 sums.
#include "kvmem_internal.hpp"

#include <algorithm>
#include <cmath>
#include <type_traits>
#include <vector>

namespace kvmem_hip {

// acc + the f16 value in the low or high half of w, rounded once: the f16
// operand is widened exactly, so fma(h, 1, acc) is the IEEE sum.
__device__ inline float add_lo(float acc, uint32_t w) {
    float r;
    asm("v_fma_mix_f32 %0, %1, 1.0, %2 op_sel_hi:[1,0,0]" : "=v"(r) : "v"(w), "v"(acc));
    return r;
}
__device__ inline float add_hi(float acc, uint32_t w) {
    float r;
    asm("v_fma_mix_f32 %0, %1, 1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r) : "v"(w), "v"(acc));
    return r;
}

// grid: (items * L) workgroups of E/CH threads; item i = block_ids[i].  The
// keys of (block b, layer l) are T rows of E halves at k + b*block_stride +
// l*layer_stride: a device history [L][cap][T][E] or the K rows of a
// block-major pinned host history.  A thread owns CH consecutive channels
// and adds its rows in token order; the rows of the next batch are loaded
// before the last batch is added, so a wave waits for memory once per batch
// and the additions (one v_fma_mix per element) run under the loads.  16
// blocks x 16 layers of 1024 channels (67 MB of keys): 10.6 us; 44.4 when a
// wave waited for every row.  All of 512 blocks: 361 us = 6.0 TB/s (421).
// Four channels per thread: eight (half the waves, each with twice the
// additions in its chain) take 11.05 and 365 us.  Wide rows of blocks shorter
// than two batches take eight: there a wave costs more than its rows (us, four
// and eight; 16 layers x 1000 blocks of 1024 channels: 4 tokens 51.1 and 45.6,
// 16 tokens 107 and 106, 32 tokens 194 and 195; of 2048 channels: 7 tokens 118
// and 105; of 256 channels: 4 tokens 17.7 and 21.2).
constexpr uint32_t kSumBatch = 16;
constexpr int kSumChannels = 4;
constexpr int kSumChannelsShort = 8;
constexpr uint32_t kSumWide = 1024;

template <int CH>
__global__ __launch_bounds__(2048 / CH) void meank_sum_kernel(const uint8_t *k, uint64_t block_stride,
                                                              uint64_t layer_stride, const uint8_t *ids_dev,
                                                              ArgTables ids_args, uint32_t L, uint32_t cap,
                                                              uint32_t T, uint32_t E, uint32_t last_block,
                                                              uint32_t last_tokens, float *k_sum,
                                                              uint32_t *mean_tokens) {
    typedef uint32_t word_t __attribute__((ext_vector_type(CH / 2)));
    typedef float sums_t __attribute__((ext_vector_type(4)));
    const uint32_t job = blockIdx.x;
    const uint32_t item = job / L;
    const uint32_t l = job - item * L;
    const uint32_t b = tab_read<uint32_t>(ids_dev, ids_args, 4u * item);
    const uint32_t e0 = threadIdx.x * CH;
    if (e0 >= E) {
        return;
    }
    const uint32_t nt = (b == last_block && last_tokens != 0) ? last_tokens : T;
    const uint8_t *base = k + b * block_stride + l * layer_stride + e0 * 2u;
    const uint32_t row = E * 2u;
    auto load = [&](uint32_t t) {
        return __builtin_nontemporal_load(
            reinterpret_cast<const word_t *>(base + static_cast<uint64_t>(t) * row));
    };
    float s[CH];
#pragma unroll
    for (int i = 0; i < CH; ++i) {
        s[i] = 0.0f;
    }
    auto add = [&](word_t w) {
#pragma unroll
        for (int i = 0; i < CH / 2; ++i) {
            s[2 * i] = add_lo(s[2 * i], w[i]);
            s[2 * i + 1] = add_hi(s[2 * i + 1], w[i]);
        }
    };
    word_t cur[kSumBatch];
    uint32_t t = 0;
    if (nt >= kSumBatch) {
#pragma unroll
        for (uint32_t j = 0; j < kSumBatch; ++j) {
            cur[j] = load(j);
        }
        for (; t + 2u * kSumBatch <= nt; t += kSumBatch) {
            word_t next[kSumBatch];
#pragma unroll
            for (uint32_t j = 0; j < kSumBatch; ++j) {
                next[j] = load(t + kSumBatch + j);
            }
#pragma unroll
            for (uint32_t j = 0; j < kSumBatch; ++j) {
                add(cur[j]);
            }
#pragma unroll
            for (uint32_t j = 0; j < kSumBatch; ++j) {
                cur[j] = next[j];
            }
        }
    }
    // the last full batch, with the rows past it already on their way
    const uint32_t tail0 = nt >= kSumBatch ? t + kSumBatch : 0u;
    word_t rest[kSumBatch];
#pragma unroll
    for (uint32_t j = 0; j < kSumBatch; ++j) {
        rest[j] = 0;
        if (tail0 + j < nt) {
            rest[j] = load(tail0 + j);
        }
    }
    if (nt >= kSumBatch) {
#pragma unroll
        for (uint32_t j = 0; j < kSumBatch; ++j) {
            add(cur[j]);
        }
    }
#pragma unroll
    for (uint32_t j = 0; j < kSumBatch; ++j) {
        if (tail0 + j < nt) {
            add(rest[j]);
        }
    }
    float *out = k_sum + (static_cast<uint64_t>(l) * cap + b) * E + e0;
#pragma unroll
    for (int i = 0; i < CH; i += 4) {
        *reinterpret_cast<sums_t *>(out + i) = sums_t{s[i], s[i + 1], s[i + 2], s[i + 3]};
    }
    if (threadIdx.x == 0) {
        mean_tokens[static_cast<uint64_t>(l) * cap + b] = nt;
    }
}

static void launch_meank_sum(hipStream_t stream, uint32_t jobs, const uint8_t *k, uint64_t block_stride,
                             uint64_t layer_stride, const LaunchTables &ids, uint32_t L, uint32_t cap, uint32_t T,
                             uint32_t E, uint32_t last_block, uint32_t last_tokens, float *k_sum,
                             uint32_t *mean_tokens) {
    if (E >= kSumWide && T < 2u * kSumBatch) {
        meank_sum_kernel<kSumChannelsShort><<<jobs, E / kSumChannelsShort, 0, stream>>>(
            k, block_stride, layer_stride, ids.dev, ids.args, L, cap, T, E, last_block, last_tokens, k_sum, mean_tokens);
    } else {
        meank_sum_kernel<kSumChannels><<<jobs, E / kSumChannels, 0, stream>>>(
            k, block_stride, layer_stride, ids.dev, ids.args, L, cap, T, E, last_block, last_tokens, k_sum, mean_tokens);
    }
}

// Query-sum producer: one thread per (layer, channel) adds the listed
// tokens' values in list order onto (or from zero into) q_sum, as the
// reference's harvest loop does per layer (llama-memory-kvmem.cpp:2164-2172).
template <typename QT>
__global__ __launch_bounds__(256) void q_accumulate_kernel(const QT *q, const uint8_t *tok_dev,
                                                           ArgTables tok_args, int listed,
                                                           uint32_t n_list, uint32_t n_tokens,
                                                           uint32_t E, uint32_t L, int reset,
                                                           float *q_sum) {
    const uint32_t e = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t l = blockIdx.y;
    if (e >= E || l >= L) {
        return;
    }
    float *dst = q_sum + static_cast<uint64_t>(l) * E + e;
    float acc = reset ? 0.0f : *dst;
    const QT *src = q + static_cast<uint64_t>(l) * n_tokens * E + e;
    // the rows of a batch are loaded before any is added (one memory latency
    // per batch); they are added in list order as the sequential loop does
    constexpr uint32_t kBatch = 16;
    uint32_t i = 0;
    for (; i + kBatch <= n_list; i += kBatch) {
        float v[kBatch];
#pragma unroll
        for (uint32_t j = 0; j < kBatch; ++j) {
            const uint32_t t = listed ? tab_read<uint32_t>(tok_dev, tok_args, 4u * (i + j)) : i + j;
            v[j] = static_cast<float>(src[static_cast<uint64_t>(t) * E]);
        }
#pragma unroll
        for (uint32_t j = 0; j < kBatch; ++j) {
            acc += v[j];
        }
    }
    for (; i < n_list; ++i) {
        const uint32_t t = listed ? tab_read<uint32_t>(tok_dev, tok_args, 4u * i) : i;
        acc += static_cast<float>(src[static_cast<uint64_t>(t) * E]);
    }
    *dst = acc;
}

// Decode running sum: one lane per channel adds the kept tokens' values in
// token order (strided K view of type KT).  A call has few channels (1024 in
// 16 waves' worth) and a chain of additions, so it is latency-bound: the
// WAVES waves of a workgroup (64 channels) each load a run of 32 tokens at
// once, and the first wave adds all of them in order, its own from registers
// and the others' from LDS.  Up to 32 tokens take one wave.  128 tokens x 1024
// f32 channels: 4.4 us; 52.5 with one token in flight at a time.  (28 tokens of
// f16: 4.2 us per call; 5.2 while each load's branch also widened its value.)
constexpr uint32_t kAddRun = 32;

template <typename KT, int WAVES>
__global__ __launch_bounds__(WAVES * 64) void meank_add_kernel(const uint8_t *k, uint32_t n_embd,
                                                               uint32_t head_dim, uint64_t nb0, uint64_t nb1,
                                                               uint64_t nb2, uint32_t tok0, uint32_t n_keep,
                                                               int reset, float *acc, uint32_t *count) {
    using bits_t = std::conditional_t<sizeof(KT) == 2, uint16_t, uint32_t>;
    auto widen = [](uint32_t bits) { return static_cast<float>(__builtin_bit_cast(KT, static_cast<bits_t>(bits))); };
    __shared__ float rows[WAVES > 1 ? (WAVES - 1) * kAddRun : 1][64];
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = threadIdx.x >> 6;
    const uint32_t e = blockIdx.x * 64u + lane;
    const bool live = e < n_embd;
    if (e == 0 && wave == 0 && count) {
        *count = (reset ? 0u : *count) + n_keep;
    }
    const uint32_t ch = live ? e : 0u;  // (in bounds; not stored)
    const uint32_t head = ch / head_dim;
    const uint32_t dim = ch - head * head_dim;
    const uint8_t *base = k + static_cast<uint64_t>(head) * nb1 + static_cast<uint64_t>(dim) * nb0;
    float s = (reset || wave != 0) ? 0.0f : acc[ch];
    for (uint32_t t0 = 0; t0 < n_keep; t0 += WAVES * kAddRun) {
        const uint32_t mine = t0 + wave * kAddRun;
        // The bits as loaded, each value in a register of its own, widened when
        // it is added: a conversion (or the packing of two 16-bit values) in
        // the branch of a load would wait for that load there.
        uint32_t v[kAddRun];
#pragma unroll
        for (uint32_t j = 0; j < kAddRun; ++j) {
            v[j] = 0u;
            if (mine + j < n_keep) {
                v[j] = *reinterpret_cast<const bits_t *>(base + static_cast<uint64_t>(tok0 + mine + j) * nb2);
            }
        }
        if (wave == 0) {
#pragma unroll
            for (uint32_t j = 0; j < kAddRun; ++j) {
                if (mine + j < n_keep) {
                    s += widen(v[j]);
                }
            }
        }
        if constexpr (WAVES > 1) {
            if (wave != 0) {
#pragma unroll
                for (uint32_t j = 0; j < kAddRun; ++j) {
                    rows[(wave - 1u) * kAddRun + j][lane] = widen(v[j]);
                }
            }
            __syncthreads();
            if (wave == 0) {
                const uint32_t left = n_keep - min(n_keep, t0 + kAddRun);
                const uint32_t n = min(left, (WAVES - 1u) * kAddRun);
                uint32_t j = 0;
                for (; j + 16u <= n; j += 16u) {
                    float x[16];
#pragma unroll
                    for (uint32_t i = 0; i < 16u; ++i) {
                        x[i] = rows[j + i][lane];
                    }
#pragma unroll
                    for (uint32_t i = 0; i < 16u; ++i) {
                        s += x[i];
                    }
                }
                for (; j < n; ++j) {
                    s += rows[j][lane];
                }
            }
            __syncthreads();  // the rows are read before the next run overwrites them
        }
    }
    if (live && wave == 0) {
        acc[e] = s;
    }
}

template <typename KT>
static void launch_meank_add(hipStream_t stream, const uint8_t *k, uint32_t n_embd, uint32_t head_dim, size_t nb0,
                             size_t nb1, size_t nb2, uint32_t tok0, uint32_t n_keep, int reset, float *acc,
                             uint32_t *count) {
    const uint32_t grid = (n_embd + 63u) / 64u;
    if (n_keep <= kAddRun) {
        meank_add_kernel<KT, 1><<<grid, 64, 0, stream>>>(k, n_embd, head_dim, nb0, nb1, nb2, tok0, n_keep, reset,
                                                         acc, count);
    } else {
        meank_add_kernel<KT, 4><<<grid, 256, 0, stream>>>(k, n_embd, head_dim, nb0, nb1, nb2, tok0, n_keep, reset,
                                                          acc, count);
    }
}

// Per-layer 1 / (query rows x group size), 0 for a layer without query
// rows, carried in the kernels' arguments (no upload before them).
constexpr uint32_t kMeankMaxL = 256;
struct LayerScales {
    float v[kMeankMaxL];
};
// The layers with query rows, ascending.
struct ScoredLayers {
    uint32_t n;
    uint32_t l[kMeankMaxL];
};

// One workgroup per (layer, KV head), one thread per channel: the group's
// query sum (heads added in group order, their loads issued eight at a time)
// scaled by invq, and its norm, reduced over the channels.
__global__ __launch_bounds__(256) void meank_query_kernel(const float *q_sum, LayerScales invq, uint32_t L,
                                                          uint32_t Hq, uint32_t Hkv, uint32_t D, float *qv,
                                                          float *nq) {
    __shared__ float part[4];
    const uint32_t i = blockIdx.x;  // l * Hkv + h
    const uint32_t d = threadIdx.x;
    const uint32_t l = i / Hkv;
    const uint32_t h = i - l * Hkv;
    const uint32_t g = Hq / Hkv;
    const float scale = invq.v[l];  // uniform index: read from the argument bytes
    float v = 0.0f;
    if (d < D) {
        constexpr uint32_t kBatch = 8;
        const float *src = q_sum + (static_cast<uint64_t>(l) * Hq + h * g) * D + d;
        float acc = 0.0f;
        for (uint32_t g0 = 0; g0 < g; g0 += kBatch) {
            float x[kBatch];
#pragma unroll
            for (uint32_t j = 0; j < kBatch; ++j) {
                x[j] = g0 + j < g ? src[static_cast<uint64_t>(g0 + j) * D] : 0.0f;
            }
#pragma unroll
            for (uint32_t j = 0; j < kBatch; ++j) {
                if (g0 + j < g) {
                    acc += x[j];
                }
            }
        }
        v = acc * scale;
        qv[static_cast<uint64_t>(i) * D + d] = v;
    }
    float n = v * v;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        n += __shfl_xor(n, off, 64);
    }
    if ((threadIdx.x & 63u) == 0u) {
        part[threadIdx.x >> 6] = n;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        float t = 0.0f;
        for (uint32_t w = 0; w < (blockDim.x + 63u) / 64u; ++w) {
            t += part[w];
        }
        nq[i] = sqrtf(t);
    }
}

// Sum of v over the 16 lanes of a DPP row (quad permutes, bank-masked row
// shifts for distance 4, row rotation by 8); every lane must be active.
__device__ inline float row16_sum(float v) {
    int x = __float_as_int(v);
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, x, 0xB1, 0xF, 0xF, false));  // ^1
    x = __float_as_int(v);
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, x, 0x4E, 0xF, 0xF, false));  // ^2
    x = __float_as_int(v);
    const int t = __builtin_amdgcn_update_dpp(0, x, 0x104, 0xF, 0x5, false);        // +4 (banks 0, 2)
    v += __int_as_float(__builtin_amdgcn_update_dpp(t, x, 0x114, 0xF, 0xA, false));  // -4 (banks 1, 3)
    x = __float_as_int(v);
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, x, 0x128, 0xF, 0xF, false));  // ^8
    return v;
}

// Cosines and their combination over layers: a workgroup of WAVES waves takes
// groups of 4 blocks, every layer of them.  Wave w scores the scored layers w,
// w + WAVES, ..., 16 lanes per block: a lane holds D/16 channels of HS heads as
// float4s (16 KiB per wave with HS = 4 and D = 256), all loaded before the
// first is reduced, and the next step's loads are issued as soon as the last
// head is, before the group's layers meet.  Ahead of a step's key loads its
// wave loads the step's query vectors, 4 KiB, and hands them to its lanes
// through LDS (loads return in order, so a query load behind key loads would
// wait for all of them: 64 layers x 64 blocks 67 us per call so, 27 as it is).
// Every layer's in LDS from the start, where they fit, is no faster: 16 layers
// x 250 blocks 14.0 us per call and 11.6, x 2000 blocks 25.4 and 25.3.  The
// layers' cosine sums meet in LDS, where one thread per block adds them in
// layer order (in double): the mean over scored layers of the cosine sum / Hkv,
// 0 when no layer holds keys of the block.  HBM-bound: every key sum is read
// once.  16 layers x 2048 blocks of 1024 channels (134 MB): 24.1 us = 5.6 TB/s,
// where a kernel for the cosines and one for the combination took 34.0 and 5.0
// with a launch between them.
// Workgroups beyond two per CU would start late and run alone: 2100 blocks take
// 58.3 us per preview with 512 workgroups that go on to the next group, 60.7
// with one workgroup per group.
//  - Launches of at most one workgroup per CU with more than 8 layers have 16
//    waves (the same waves per CU, half the layers one after the other).
//  - With fewer layers than waves and enough blocks, 2^lw_bits waves take the
//    layers and the others further groups of 4 blocks.
typedef float f32x4_t __attribute__((ext_vector_type(4)));
constexpr uint32_t kCosBlocks = 4;
constexpr uint32_t kCosGroups = 512;      // workgroups of a launch, at most: two per CU
extern __shared__ float4 cos_lds[];

// The launch shape of a call: waves of a workgroup, log2 of those that take
// layers side by side, workgroups, heads of a step, and the dynamic LDS: the
// layers' cosine sums of two turns, then each wave's query vectors of a step.
struct CosShape {
    uint32_t waves = 8, lw_bits = 3, grid = 0, heads = 4, lds = 0;
};

static CosShape cos_shape(uint32_t n_scored, uint32_t B, uint32_t Hkv, uint32_t D) {
    CosShape s;
    // steps of four heads, or of two where four would load heads twice
    if (Hkv % 4u != 0 && (Hkv + 1u) / 2u * 2u < (Hkv + 3u) / 4u * 4u) {
        s.heads = 2;
    }
    uint32_t blocks = kCosBlocks;  // of a workgroup's turn
    if (n_scored > 8u && B <= kCosGroups / 2u * blocks) {
        s.waves = 16;
        s.lw_bits = 4;
    }
    while (s.lw_bits > 0u && n_scored <= 1u << (s.lw_bits - 1u) && B >= kCosGroups * 2u * blocks) {
        --s.lw_bits;
        blocks *= 2u;
    }
    s.grid = std::min((B + blocks - 1u) / blocks, kCosGroups);
    s.lds = static_cast<uint32_t>(sizeof(double) * 2u * blocks * n_scored + sizeof(float) * s.waves * s.heads * D);
    return s;
}

template <int D, int HS, int WAVES>
__global__ __launch_bounds__(WAVES * 64) __attribute__((amdgpu_waves_per_eu(4, 4))) void meank_score_kernel(
    const float *k_sum, const uint32_t *mean_tokens, const float *qv, const float *nq, ScoredLayers scored,
    uint32_t lw_bits, uint32_t L, uint32_t B, uint32_t cap, uint32_t Hkv, float *scores) {
    constexpr int P4 = D / 64;             // float4s per lane per head
    constexpr int NQ = HS * (D / 4) / 64;  // float4s per lane of a step's query vectors
    __shared__ uint32_t has_keys[2][WAVES][kCosBlocks];
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t sub = lane & 15u;
    const uint32_t lb = lane >> 4;
    const uint32_t lw = 1u << lw_bits;
    const uint32_t first = wave & (lw - 1u);                // the wave's first scored layer
    const uint32_t in_turn = (wave >> lw_bits) * kCosBlocks + lb;  // the lane's block among the turn's
    const uint32_t per_turn = (WAVES >> lw_bits) * kCosBlocks;
    const uint32_t row4 = Hkv * (D / 4);  // float4s of a key-sum row
    const uint32_t n_groups = (B + per_turn - 1u) / per_turn;
    double *term = reinterpret_cast<double *>(cos_lds);  // [2][per_turn][scored.n]
    f32x4_t *q_lds = reinterpret_cast<f32x4_t *>(term + 2u * per_turn * scored.n) + wave * HS * (D / 4);

    // a step: HS heads of one scored layer, loaded together
    f32x4_t kc[HS][P4];
    float qn[HS];  // query norms
    auto block_of = [&](uint32_t g) { return min(g * per_turn + in_turn, B - 1u); };  // past the end: not stored
    auto load_step = [&](uint32_t g, uint32_t l, uint32_t h0) {
        f32x4_t q[NQ];
#pragma unroll
        for (int hh = 0; hh < HS; ++hh) {
            qn[hh] = nq[l * Hkv + min(h0 + hh, Hkv - 1u)];
        }
#pragma unroll
        for (int j = 0; j < NQ; ++j) {
            const uint32_t at = j * 64 + lane;
            const uint32_t h = min(h0 + at / (D / 4), Hkv - 1u);
            q[j] = reinterpret_cast<const f32x4_t *>(qv)[l * row4 + h * (D / 4) + at % (D / 4)];
        }
        __builtin_amdgcn_sched_barrier(0);  // ahead of the keys
        const f32x4_t *row = reinterpret_cast<const f32x4_t *>(k_sum) +
                             (static_cast<uint64_t>(l) * cap + block_of(g)) * row4 + sub;
#pragma unroll
        for (int hh = 0; hh < HS; ++hh) {
            const f32x4_t *src = row + min(h0 + hh, Hkv - 1u) * (D / 4);  // past the last head: it again, not used
#pragma unroll
            for (int j = 0; j < P4; ++j) {
                // whatever the layer's mean_tokens: every row up to capacity is in bounds
                kc[hh][j] = __builtin_nontemporal_load(src + j * 16);
            }
        }
        __builtin_amdgcn_sched_barrier(0);  // all of them before the first use
#pragma unroll
        for (int j = 0; j < NQ; ++j) {  // (the wave has read the last step's)
            q_lds[j * 64 + lane] = q[j];
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    auto load_tokens = [&](uint32_t g, uint32_t l) { return mean_tokens[static_cast<uint64_t>(l) * cap + block_of(g)]; };
    uint32_t g = blockIdx.x;  // (the grid has at most n_groups workgroups)
    uint32_t mt = 0;          // tokens of the step's layer in the lane's block
    if (first < scored.n) {
        mt = load_tokens(g, scored.l[first]);
        load_step(g, scored.l[first], 0u);
    }
    uint32_t turn = 0;
    for (; g < n_groups; g += gridDim.x, turn ^= 1u) {
        uint32_t has = 0;
        for (uint32_t i = first; i < scored.n; i += lw) {
            const uint32_t l = scored.l[i];
            const float inv = mt ? 1.0f / static_cast<float>(mt) : 0.0f;
            double layer = 0.0;
            for (uint32_t h0 = 0; h0 < Hkv; h0 += HS) {
                if (h0 != 0) {
                    load_step(g, l, h0);
                }
                if (mt == 0u) {  // no keys: whatever the row holds does not count
#pragma unroll
                    for (int hh = 0; hh < HS; ++hh) {
#pragma unroll
                        for (int j = 0; j < P4; ++j) {
                            kc[hh][j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
                        }
                    }
                }
#pragma unroll
                for (int hh = 0; hh < HS; ++hh) {
                    const f32x4_t *qs = q_lds + hh * (D / 4) + sub;
                    float dot = 0.0f, nk = 0.0f;
#pragma unroll
                    for (int j = 0; j < P4; ++j) {
                        const f32x4_t q = qs[j * 16];
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const float m = kc[hh][j][e] * inv;
                            // one rounding per term: 1.373e-8 rms from 64 bits over 35483
                            // scores of 31 shapes, 1.374e-8 with a rounded product
                            dot = __builtin_fmaf(q[e], m, dot);
                            nk = __builtin_fmaf(m, m, nk);
                        }
                    }
                    dot = row16_sum(dot);
                    nk = row16_sum(nk);
                    if (h0 + hh < Hkv) {
                        layer += static_cast<double>(dot / (qn[hh] * sqrtf(nk) + 1e-6f));
                    }
                }
            }
            has |= mt;
            // the wave's next step: its next layer, or its first of the next group
            const bool more = i + lw < scored.n;
            const uint32_t gn = more ? g : g + gridDim.x;
            if (gn < n_groups) {
                const uint32_t ln = scored.l[more ? i + lw : first];
                mt = load_tokens(gn, ln);
                load_step(gn, ln, 0u);
            }
            if (sub == 0u) {
                term[(turn * per_turn + in_turn) * scored.n + i] = layer / static_cast<double>(Hkv);
            }
        }
        if (scored.n != L) {  // the layers without query rows count here too
            for (uint32_t u = first; u < L; u += lw) {
                has |= load_tokens(g, u);
            }
        }
        if (sub == 0u) {
            has_keys[turn][wave][lb] = has;
        }
        __syncthreads();  // (the next group's terms go to the other half)
        const uint32_t t = threadIdx.x;
        const uint32_t b = g * per_turn + t;
        if (t < per_turn && b < B) {
            const uint32_t w0 = (t / kCosBlocks) << lw_bits;
            uint32_t any = 0;
            for (uint32_t w = 0; w < lw; ++w) {
                any |= has_keys[turn][w0 + w][t % kCosBlocks];
            }
            double acc = 0.0;
            for (uint32_t u = 0; u < scored.n; ++u) {
                acc += term[(turn * per_turn + t) * scored.n + u];
            }
            scores[b] = static_cast<float>((any && scored.n) ? acc / scored.n : 0.0);
        }
    }
}

using MeankScoreKernel = void (*)(const float *, const uint32_t *, const float *, const float *, ScoredLayers, uint32_t,
                                  uint32_t, uint32_t, uint32_t, uint32_t, float *);

template <int D>
static MeankScoreKernel meank_score_of(const CosShape &s) {
    if (s.heads == 2u) {
        return s.waves == 16u ? meank_score_kernel<D, 2, 16> : meank_score_kernel<D, 2, 8>;
    }
    return s.waves == 16u ? meank_score_kernel<D, 4, 16> : meank_score_kernel<D, 4, 8>;
}

size_t meank_scratch_bytes(uint32_t L, uint32_t Hkv, uint32_t B, uint32_t D) {
    (void) B;  // the query vectors and their norms; no per-block scratch
    return sizeof(float) * static_cast<size_t>(L) * Hkv * (D + 1);
}

bool load_meank_kernels() {
    return load_kernel_object(&meank_score_kernel<256, 4, 8>);
}

}  // namespace kvmem_hip

using namespace kvmem_hip;

extern "C" {

int kvmem_hip_meank_sums(kvmem_hip_ctx *ctx, const kvmem_hip_history *hist,
                         const uint32_t *block_ids, uint32_t n, float *k_sum,
                         uint32_t *mean_tokens) {
    if (!ctx) {
        return KVMEM_HIP_ERR_INVALID;
    }
    if (n == 0) {
        return KVMEM_HIP_OK;
    }
    if (!hist || !hist->k || !block_ids || !k_sum || !mean_tokens) {
        return fail(ctx, KVMEM_HIP_ERR_INVALID, "meank_sums: null argument");
    }
    const uint32_t E = hist->n_embd_k;
    const uint32_t cap = hist->capacity_blocks ? hist->capacity_blocks : hist->n_blocks;
    if (E == 0 || E % 8 != 0 || E / 8 > 256 || hist->block_tokens == 0 || cap < hist->n_blocks ||
        (reinterpret_cast<uintptr_t>(hist->k) & 15u) || (reinterpret_cast<uintptr_t>(k_sum) & 15u)) {
        return fail(ctx, KVMEM_HIP_ERR_INVALID,
                    "meank_sums: n_embd_k must be a multiple of 8 and at most 2048, 16-byte aligned");
    }
    if (hist->last_block_tokens > hist->block_tokens) {
        // the kernel sums the last block's rows up to this count
        return fail(ctx, KVMEM_HIP_ERR_INVALID, "meank_sums: last_block_tokens above block_tokens");
    }
    for (uint32_t i = 0; i < n; ++i) {
        if (block_ids[i] >= hist->n_blocks) {
            return fail(ctx, KVMEM_HIP_ERR_INVALID, "meank_sums: block id out of range");
        }
    }
    const uint64_t jobs = static_cast<uint64_t>(n) * hist->n_layers;
    if (jobs > 0x7fffffffu) {
        return fail(ctx, KVMEM_HIP_ERR_INVALID, "meank_sums: too many blocks in one call");
    }
    (void) hipSetDevice(ctx->device);
    LaunchTables ids;  // in the kernel arguments up to 768 blocks
    if (!stage_tables(ctx, block_ids, sizeof(uint32_t) * n, ids, "meank_sums ids")) {
        return KVMEM_HIP_ERR_RUNTIME;
    }
    if (injected_fail(ctx, KVMEM_HIP_FAIL_LAUNCH, "meank_sums launch")) {
        return KVMEM_HIP_ERR_RUNTIME;
    }
    const uint64_t block_stride = static_cast<uint64_t>(hist->block_tokens) * E * 2u;
    launch_meank_sum(
        ctx->stream, static_cast<uint32_t>(jobs), static_cast<const uint8_t *>(hist->k), block_stride,
        block_stride * cap, ids, hist->n_layers, cap, hist->block_tokens, E,
        hist->n_blocks - 1, hist->last_block_tokens, k_sum, mean_tokens);
    return hip_ok(ctx, hipGetLastError(), "meank_sums launch") ? KVMEM_HIP_OK : KVMEM_HIP_ERR_RUNTIME;
}

int kvmem_hip_meank_sums_host(kvmem_hip_ctx *ctx, const kvmem_hip_host_history *hist,
                              const uint32_t *block_ids, uint32_t n, uint32_t capacity_blocks,
                              float *k_sum, uint32_t *mean_tokens) {
    if (!ctx) {
        return KVMEM_HIP_ERR_INVALID;
    }
    if (n == 0) {
        return KVMEM_HIP_OK;
    }
    if (!hist || !hist->base || !block_ids || !k_sum || !mean_tokens) {
        return fail(ctx, KVMEM_HIP_ERR_INVALID, "meank_sums_host: null argument");
    }
    const uint32_t E = hist->n_embd_k;
    const uint32_t T = hist->block_tokens;
    const uint32_t cap = capacity_blocks ? capacity_blocks : hist->n_blocks;
    if (E == 0 || E % 8 != 0 || E / 8 > 256 || T == 0 || cap < hist->n_blocks ||
        hist->last_block_tokens > T || (reinterpret_cast<uintptr_t>(hist->base) & 15u) ||
        (reinterpret_cast<uintptr_t>(k_sum) & 15u) || (hist->n_embd_v % 8 != 0)) {
        return fail(ctx, KVMEM_HIP_ERR_INVALID,
                    "meank_sums_host: n_embd_k must be a multiple of 8 and at most 2048, 16-byte aligned");
    }
    for (uint32_t i = 0; i < n; ++i) {
        if (block_ids[i] >= hist->n_blocks) {
            return fail(ctx, KVMEM_HIP_ERR_INVALID, "meank_sums_host: block id out of range");
        }
    }
    const uint64_t jobs = static_cast<uint64_t>(n) * hist->n_layers;
    if (jobs > 0x7fffffffu) {
        return fail(ctx, KVMEM_HIP_ERR_INVALID, "meank_sums_host: too many blocks in one call");
    }
    const uint64_t layer_bytes = static_cast<uint64_t>(T) * (hist->n_embd_k + hist->n_embd_v) * 2u;
    const uint64_t span = layer_bytes * hist->n_layers;
    (void) hipSetDevice(ctx->device);
    // the kernel reads the pinned rows over the link itself
    const uint8_t *view = host_device_view(hist->base, span * hist->n_blocks);
    if (!view) {
        return fail(ctx, KVMEM_HIP_ERR_UNSUPPORTED,
                    "meank_sums_host: the history must lie inside one pinned host allocation");
    }
    LaunchTables ids;
    if (!stage_tables(ctx, block_ids, sizeof(uint32_t) * n, ids, "meank_sums_host ids")) {
        return KVMEM_HIP_ERR_RUNTIME;
    }
    if (injected_fail(ctx, KVMEM_HIP_FAIL_LAUNCH, "meank_sums_host launch")) {
        return KVMEM_HIP_ERR_RUNTIME;
    }
    launch_meank_sum(
        ctx->stream, static_cast<uint32_t>(jobs), view, span, layer_bytes, ids, hist->n_layers, cap, T, E,
        hist->n_blocks - 1, hist->last_block_tokens, k_sum, mean_tokens);
    if (!hip_ok(ctx, hipGetLastError(), "meank_sums_host launch")) {
        return KVMEM_HIP_ERR_RUNTIME;
    }
    // the kernel reads the listed blocks' K rows over the link
    uint64_t rows = 0;
    for (uint32_t i = 0; i < n; ++i) {
        rows += (block_ids[i] + 1 == hist->n_blocks && hist->last_block_tokens) ? hist->last_block_tokens : T;
    }
    note_xfer(ctx, kXferH2D, rows * hist->n_layers * E * 2u);
    return KVMEM_HIP_OK;
}

int kvmem_hip_meank_add(kvmem_hip_ctx *ctx, const void *k, int32_t k_type, uint32_t n_embd,
                        uint32_t head_dim, size_t nb0, size_t nb1, size_t nb2, uint32_t tok0,
                        uint32_t n_keep, int reset, float *acc, uint32_t *count) {
    if (!ctx) {
        return KVMEM_HIP_ERR_INVALID;
    }
    if (!k || !acc || n_embd == 0 || head_dim == 0 || n_embd % head_dim != 0) {
        return fail(ctx, KVMEM_HIP_ERR_INVALID, "meank_add: null pointer or bad geometry");
    }
    const size_t esz = k_type == KVMEM_TYPE_F32 ? 4 : 2;
    if (k_type != KVMEM_TYPE_F32 && k_type != KVMEM_TYPE_F16 && k_type != KVMEM_TYPE_BF16) {
        return fail(ctx, KVMEM_HIP_ERR_UNSUPPORTED, "meank_add: k_type must be F32, F16 or BF16");
    }
    if (nb0 % esz || nb1 % esz || nb2 % esz || (reinterpret_cast<uintptr_t>(k) % esz)) {
        return fail(ctx, KVMEM_HIP_ERR_INVALID, "meank_add: strides must be multiples of the element size");
    }
    if (n_keep == 0 && !reset) {
        return KVMEM_HIP_OK;
    }
    (void) hipSetDevice(ctx->device);
    const uint8_t *kb = static_cast<const uint8_t *>(k);
    if (k_type == KVMEM_TYPE_F32) {
        launch_meank_add<float>(ctx->stream, kb, n_embd, head_dim, nb0, nb1, nb2, tok0, n_keep, reset, acc, count);
    } else if (k_type == KVMEM_TYPE_F16) {
        launch_meank_add<_Float16>(ctx->stream, kb, n_embd, head_dim, nb0, nb1, nb2, tok0, n_keep, reset, acc,
                                   count);
    } else {
        launch_meank_add<__bf16>(ctx->stream, kb, n_embd, head_dim, nb0, nb1, nb2, tok0, n_keep, reset, acc, count);
    }
    return hip_ok(ctx, hipGetLastError(), "meank_add launch") ? KVMEM_HIP_OK : KVMEM_HIP_ERR_RUNTIME;
}

int kvmem_hip_q_accumulate(kvmem_hip_ctx *ctx, const void *q, int32_t q_type, uint32_t n_layers,
                           uint32_t n_tokens, uint32_t n_embd_q, const uint32_t *tokens,
                           uint32_t n_list, int reset, float *q_sum) {
    if (!ctx) {
        return KVMEM_HIP_ERR_INVALID;
    }
    if (!q || !q_sum) {
        return fail(ctx, KVMEM_HIP_ERR_INVALID, "q_accumulate: null argument");
    }
    if (q_type != KVMEM_TYPE_F32 && q_type != KVMEM_TYPE_F16 && q_type != KVMEM_TYPE_BF16) {
        return fail(ctx, KVMEM_HIP_ERR_UNSUPPORTED, "q_accumulate: q_type must be F32, F16 or BF16");
    }
    if (!tokens) {
        n_list = n_tokens;
    }
    for (uint32_t i = 0; tokens && i < n_list; ++i) {
        if (tokens[i] >= n_tokens) {
            return fail(ctx, KVMEM_HIP_ERR_INVALID, "q_accumulate: token index out of range");
        }
    }
    if (n_layers == 0 || n_embd_q == 0 || (n_list == 0 && !reset)) {
        return KVMEM_HIP_OK;
    }
    if (n_layers > 65535) {
        return fail(ctx, KVMEM_HIP_ERR_INVALID, "q_accumulate: too many layers");
    }
    (void) hipSetDevice(ctx->device);
    // the token list travels in the kernel arguments when it fits (768
    // rows), else it is uploaded
    LaunchTables lt;
    const int listed = tokens && n_list ? 1 : 0;
    if (listed && !stage_tables(ctx, tokens, sizeof(uint32_t) * n_list, lt, "q_accumulate tokens")) {
        return KVMEM_HIP_ERR_RUNTIME;
    }
    const dim3 grid((n_embd_q + 255) / 256, n_layers);
    if (q_type == KVMEM_TYPE_F32) {
        q_accumulate_kernel<float><<<grid, 256, 0, ctx->stream>>>(
            static_cast<const float *>(q), lt.dev, lt.args, listed, n_list, n_tokens, n_embd_q, n_layers, reset,
            q_sum);
    } else if (q_type == KVMEM_TYPE_F16) {
        q_accumulate_kernel<_Float16><<<grid, 256, 0, ctx->stream>>>(
            static_cast<const _Float16 *>(q), lt.dev, lt.args, listed, n_list, n_tokens, n_embd_q, n_layers,
            reset, q_sum);
    } else {
        q_accumulate_kernel<__bf16><<<grid, 256, 0, ctx->stream>>>(
            static_cast<const __bf16 *>(q), lt.dev, lt.args, listed, n_list, n_tokens, n_embd_q, n_layers,
            reset, q_sum);
    }
    return hip_ok(ctx, hipGetLastError(), "q_accumulate launch") ? KVMEM_HIP_OK : KVMEM_HIP_ERR_RUNTIME;
}

int kvmem_hip_score_meank(kvmem_hip_ctx *ctx, const kvmem_hip_meank_args *a) {
    if (!ctx) {
        return KVMEM_HIP_ERR_INVALID;
    }
    if (!a || !a->q_sum || !a->q_count || !a->k_sum || !a->mean_tokens || !a->scores) {
        return fail(ctx, KVMEM_HIP_ERR_INVALID, "score_meank: null argument");
    }
    const uint32_t L = a->n_layers, B = a->n_blocks, D = a->head_dim;
    const uint32_t cap = a->capacity_blocks ? a->capacity_blocks : B;
    if (a->n_head_kv == 0 || a->n_head % a->n_head_kv != 0 || (D != 128 && D != 256) || cap < B) {
        return fail(ctx, KVMEM_HIP_ERR_INVALID, "score_meank: bad head geometry");
    }
    if (reinterpret_cast<uintptr_t>(a->k_sum) & 15u) {
        return fail(ctx, KVMEM_HIP_ERR_INVALID, "score_meank: k_sum must be 16-byte aligned");
    }
    if (L > kMeankMaxL) {
        return fail(ctx, KVMEM_HIP_ERR_UNSUPPORTED, "score_meank: more than 256 layers");
    }
    if (L == 0 || B == 0) {
        return KVMEM_HIP_OK;
    }
    const uint32_t g = a->n_head / a->n_head_kv;
    // per-layer 1 / (q_count * g) as the reference computes it in fp32; 0
    // marks a layer without query rows
    LayerScales invq{};
    ScoredLayers scored{};
    for (uint32_t l = 0; l < L; ++l) {
        if (a->q_count[l]) {
            scored.l[scored.n++] = l;
        }
        invq.v[l] = a->q_count[l] ? 1.0f / static_cast<float>(a->q_count[l] * g) : 0.0f;
    }
    (void) hipSetDevice(ctx->device);
    if (!ensure_dev(ctx, ctx->meank_scratch, meank_scratch_bytes(L, a->n_head_kv, B, D),
                    "score_meank scratch")) {
        return KVMEM_HIP_ERR_NOMEM;
    }
    float *qv = static_cast<float *>(ctx->meank_scratch.ptr);  // read as float4
    float *nq = qv + static_cast<size_t>(L) * a->n_head_kv * D;
    if (injected_fail(ctx, KVMEM_HIP_FAIL_LAUNCH, "score_meank launch")) {
        return KVMEM_HIP_ERR_RUNTIME;
    }
    perf_begin(ctx, kPerfScore);
    const uint32_t lh = L * a->n_head_kv;
    meank_query_kernel<<<lh, D, 0, ctx->stream>>>(a->q_sum, invq, L, a->n_head, a->n_head_kv, D, qv, nq);
    const CosShape shape = cos_shape(scored.n, B, a->n_head_kv, D);
    {
        // the kernel which streams the key sums, also timed alone
        PerfLaunchScope timed(ctx, kPerfMeankCos);
        ctx_launch(ctx, D == 256 ? meank_score_of<256>(shape) : meank_score_of<128>(shape), dim3(shape.grid),
                   dim3(shape.waves * 64u), shape.lds, a->k_sum, a->mean_tokens, qv, nq, scored, shape.lw_bits, L, B, cap,
                   a->n_head_kv, a->scores);
        if (hip_ok(ctx, hipGetLastError(), "score_meank launch")) {
            timed.ok();
        } else {
            perf_drop(ctx, kPerfScore);
            return KVMEM_HIP_ERR_RUNTIME;
        }
    }
    perf_end(ctx, kPerfScore);
    return hip_ok(ctx, hipGetLastError(), "score_meank launch") ? KVMEM_HIP_OK : KVMEM_HIP_ERR_RUNTIME;
}

}  // extern "C"

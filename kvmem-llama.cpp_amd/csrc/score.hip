// Per-token max block scorer on the CDNA4 matrix cores.
//
// For layer l, KV head h and block b the scorer needs
//     max_{query rows r of group h, keys j of block b} q_r . k_j
// where the query rows of group h are the (token, head) pairs with head in
// [h*g, (h+1)*g) (GQA, llama-memory-kvmem.cpp:2890-2892).  That is a small
// GEMM (rows x 128 keys x head_dim) whose output is reduced by max at once,
// so no score ever goes to memory.
//
// Mapping.  A workgroup owns one (layer, KV head, row slice) and a contiguous
// range of blocks.  Its 1, 2 or 4 waves hold up to 6 tiles of 16 query rows
// each, resident in VGPRs as f16 A-fragments of v_mfma_f32_16x16x32_f16
// (loaded once; bf16 queries are converted to f16 on the way, exact for
// normal-range values, a wave's rows scaled by a power of two when they would
// overflow f16), so every 16-byte B-fragment read from LDS feeds as many
// MFMAs as the wave has tiles (two reads kept in flight ahead of their
// MFMAs).  The key tile (16 keys per wave of the workgroup) moves HBM -> LDS
// with global_load_lds_dwordx4 (no register staging) into one of two LDS
// buffers while the other's keys are multiplied.
//  - Up to 96 rows fit one wave: it streams its keys alone, without a
//    barrier, the next tile's loads always in flight.  HBM-bound: 14 query
//    tokens of 24 heads over 16 x 2048 blocks read 8.59 GB in 1.22 ms = 7.0
//    TB/s, the rate of a plain read (2.03 ms when every slice was padded to
//    the 384 rows of four waves).
//  - More rows go to two or four waves that share each key tile, one barrier
//    per tile; with four waves of 6 tiles the matrix pipes and the power cap
//    bound it.  384 rows make a slice; more rows make equal slices.
//  - A block's keys are a run of 16-key groups and a tile may hold groups of
//    several blocks, so blocks of 16, 32 or 64 keys cost no padding (16 x
//    4096 blocks of 32 keys, 64-token query: 1.26 ms; 4.35 when every block
//    took two tiles of 64 keys).
//  - A launch of few blocks splits each block's keys over up to four waves'
//    workgroups.
// The per-block max over a wave's lanes uses DPP and the row-swap permutes,
// not LDS.  Inside a tile the 16-byte chunk c of key j sits at chunk position
// c ^ (j mod chunks-per-key), so the 16 keys of a B-fragment read hit 16
// different bank groups; the swizzle is applied on the global side (each lane
// of a direct LDS load fetches the chunk that belongs to its fixed LDS slot).
// Out-of-range query rows and keys (partial last block, a block length or row
// count that is no multiple of 16) are replaced by duplicates of valid ones,
// which leaves the max unchanged and needs no masking.  Each wave writes its
// own per-block max to a partial array; a small kernel folds waves, key parts,
// row slices, KV heads and layers.
//
// The file is built with finite-math semantics (max needs no NaN
// canonicalisation); every identity is -FLT_MAX and inputs are finite F16.
//
// Dispatch order is XCD-aware: consecutive workgroup ids go to different
// XCDs, so the id is decoded such that each XCD works through its own set
// of (layer, head) pairs, keeping their query rows resident in that XCD's
// L2.
#include "kvmem_internal.hpp"

#include <algorithm>
#include <cfloat>
#include <cmath>
#include <mutex>
#include <string>

namespace kvmem_hip {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float float4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void lds_void_t;

constexpr int kMaxTokens = 128;  // keys per block (at most)
// Most row tiles (of 16 query rows) a wave keeps, and waves that share a key
// tile: a row slice is at most 24 tiles = 384 rows.  Six tiles of 256-wide
// rows take 192 of the 256 registers that two waves per SIMD leave a wave.
constexpr int kMaxRowTiles = 6;
constexpr int kMaxRowWaves = 4;
constexpr uint32_t kSliceTiles = kMaxRowTiles * kMaxRowWaves;
constexpr uint32_t kSliceRows = kSliceTiles * 16u;
// Below this many waves in a launch, blocks are split over key parts.  Mean
// time of a call with a line at 256, 384 and 512 waves against none, over 276
// calls of one-wave slices (2 and 4 layers, 4 to 64 blocks), by unsplit waves:
// 96 0.85, 0.84, 0.87; 192 0.90, 0.90, 0.91; 224 0.90, 0.90, 0.97; 256 1.00,
// 0.89, 0.90; 320 1.00, 0.93, 0.93; 384 1.00, 1.00, 0.93; 448 1.00, 1.00, 1.01.
// Each further wave loads the query rows again.
constexpr uint32_t kSplitWaves = 384;
// Cache policy of the tile DMA.  Keys read by one workgroup only stream past
// the caches (nt): L2 stays with the query rows, and the power-capped kernel
// pays less energy (16 x 2048 blocks, 64-token query: 2.404 ms against 2.435
// with the default policy).  Where several row slices read the same keys,
// the default policy keeps a tile in L2 for the slice that comes to it later
// (512-token query over 16 x 8192 blocks: 69.2 ms with nt, 65.3 without).
constexpr int kDmaDefault = 0;
constexpr int kDmaNonTemporal = 2;

struct ScoreParams {
    const uint16_t *q;       // [L][Tq][Hq][D] bf16 or f16 bits
    const uint8_t *k;        // [L][cap][T][Hkv][D] f16
    float *partial;          // [RG * KS * WR][L][Hkv][B]
    uint32_t L, Tq, Hq, Hkv, B, T, last_T, g, R, RG;
    uint32_t KS;             // key parts of a block, a workgroup each
    uint32_t gpb;            // 16-key groups of one key part
    uint32_t cap;            // blocks per layer in memory (>= B)
    uint32_t n_chunks;       // block chunks per (l, h, row slice, key part)
    uint32_t blocks_per_chunk;
    uint32_t slice_rows;     // query rows per slice (RT * 16 * WR)
    uint32_t q_bf16;
    uint32_t xcd_major;      // 1 if (L*Hkv) % 8 == 0
    float scale;             // 1/sqrt(D)
};

// Max over the 64 lanes of a wave without LDS: DPP within each 16-lane row
// (quad permutes, then row rotations by 4 and 8; max is idempotent, so the
// overlapping windows are harmless), then the gfx950 row swaps, which hand
// every lane the value of the other 16-lane row and of the other 32-lane
// half.  Every lane ends with the wave maximum.
__device__ inline float wave_max(float m) {
    int x = __float_as_int(m);
    m = __builtin_fmaxf(m, __int_as_float(__builtin_amdgcn_update_dpp(x, x, 0xB1, 0xF, 0xF, false)));
    x = __float_as_int(m);
    m = __builtin_fmaxf(m, __int_as_float(__builtin_amdgcn_update_dpp(x, x, 0x4E, 0xF, 0xF, false)));
    x = __float_as_int(m);
    m = __builtin_fmaxf(m, __int_as_float(__builtin_amdgcn_update_dpp(x, x, 0x124, 0xF, 0xF, false)));
    x = __float_as_int(m);
    m = __builtin_fmaxf(m, __int_as_float(__builtin_amdgcn_update_dpp(x, x, 0x128, 0xF, 0xF, false)));
    const uint32_t u = __float_as_uint(m);
    const auto s16 = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    m = __builtin_fmaxf(__uint_as_float(s16[0]), __uint_as_float(s16[1]));
    const uint32_t v = __float_as_uint(m);
    const auto s32 = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    return __builtin_fmaxf(__uint_as_float(s32[0]), __uint_as_float(s32[1]));
}

// A wave's query rows as raw 16-bit A fragments (bf16 or f16 bits, not yet
// converted).
template <int RT, int KS, int D>
__device__ __forceinline__ void load_query_bits(const ScoreParams &p, half8_t (&a)[RT][KS], uint32_t l,
                                                uint32_t h, uint32_t row0, uint32_t lrow, uint32_t kgrp) {
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        const uint32_t r = min(row0 + rt * 16u + lrow, p.R - 1u);  // duplicate the last valid row
        const uint32_t t = r / p.g;
        const uint32_t hq = h * p.g + (r - t * p.g);
        const uint16_t *qrow = p.q + ((static_cast<uint64_t>(l) * p.Tq + t) * p.Hq + hq) * D;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            a[rt][ks] = __builtin_bit_cast(half8_t, *reinterpret_cast<const u32x4_t *>(qrow + ks * 32 + kgrp * 8));
        }
    }
}

// Raw bf16 A fragments -> f16 in place, times qscale (a power of two, exact)
// before the rounding.  Returns the largest |q| the lane converted.
template <int RT, int KS, bool SCALED>
__device__ __forceinline__ float convert_query_bits(half8_t (&a)[RT][KS], float qscale) {
    float mx = 0.0f;
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const u32x4_t w = __builtin_bit_cast(u32x4_t, a[rt][ks]);
            half8_t v;
#pragma unroll
            for (int i = 0; i < 4; ++i) {  // two bf16 per word, the low one first
                const float lo = __uint_as_float(w[i] << 16);
                const float hi = __uint_as_float(w[i] & 0xffff0000u);
                mx = __builtin_fmaxf(mx, __builtin_fmaxf(__builtin_fabsf(lo), __builtin_fabsf(hi)));
                v[2 * i] = static_cast<_Float16>(SCALED ? lo * qscale : lo);
                v[2 * i + 1] = static_cast<_Float16>(SCALED ? hi * qscale : hi);
            }
            a[rt][ks] = v;
        }
    }
    return mx;
}

// Waves per SIMD a kernel is built for: its A fragments take RT * D / 8 of
// a wave's registers, about 45 go to the rest.
__host__ __device__ constexpr int score_occupancy(int D, int RT) {
    return RT * D >= 4 * 256 ? 2 : RT * D >= 6 * 128 ? 3 : 4;
}

template <int D, int RT, int WR, bool SEG, bool REUSE>
__global__ __launch_bounds__(WR * 64, score_occupancy(D, RT)) void score_kernel(ScoreParams p) {
    constexpr int KS = D / 32;                       // k-steps of 32
    constexpr int ROW_BYTES = D * 2;                 // one key of one head
    constexpr int CH = D / 8;                        // 16-byte chunks per key
    constexpr int GROUP = 16 * ROW_BYTES;            // 16 keys: 8 KiB (D = 256)
    constexpr int TILE = WR * GROUP;                 // a group per wave
    constexpr int LOADS = GROUP / 1024;              // wave-wide 1 KiB loads of a group
    constexpr int DMA = REUSE ? kDmaDefault : kDmaNonTemporal;

    __shared__ __attribute__((aligned(1024))) uint8_t tiles[2][TILE];

    // ---- decode (layer, head, row slice, key part, chunk) from the workgroup id
    const uint32_t pairs = p.L * p.Hkv;
    const uint32_t n_sub = p.RG * p.KS;
    uint32_t lh, chunk, sub;
    {
        const uint32_t i = blockIdx.x;
        if (p.xcd_major) {
            const uint32_t xcd = i & 7u;
            const uint32_t local = i >> 3;
            sub = local % n_sub;
            const uint32_t rest = local / n_sub;
            chunk = rest % p.n_chunks;
            lh = (rest / p.n_chunks) * 8u + xcd;
        } else {
            sub = i % n_sub;
            const uint32_t rest = i / n_sub;
            chunk = rest % p.n_chunks;
            lh = rest / p.n_chunks;
        }
    }
    if (lh >= pairs) {
        return;
    }
    const uint32_t rg = sub / p.KS;
    const uint32_t part = sub - rg * p.KS;
    const uint32_t l = lh / p.Hkv;
    const uint32_t h = lh - l * p.Hkv;
    const uint32_t b_begin = chunk * p.blocks_per_chunk;
    const uint32_t b_end = min(p.B, b_begin + p.blocks_per_chunk);
    if (b_begin >= b_end) {
        return;
    }

    const uint32_t tid = threadIdx.x;
    const uint32_t wave = WR == 1 ? 0u : __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t lane = tid & 63u;
    const uint32_t lrow = lane & 15u;   // row (A) / key (B) within a 16-tile
    const uint32_t kgrp = lane >> 4;    // which 8 of the 32 k-values

    // ---- K tiles: direct HBM -> LDS, swizzled chunk order.  The keys of the
    // chunk's blocks (of this key part) are a run of 16-key groups; tile `it`
    // holds groups [it*WR, it*WR + WR), and wave w loads group w of it, group
    // `lg` of block `lb` (advanced by WR groups per tile).
    const uint64_t key_stride = static_cast<uint64_t>(p.Hkv) * ROW_BYTES;
    const uint32_t gpb = p.gpb;
    const uint32_t key0 = part * gpb * 16u;  // the key part's first key in a block
    const uint8_t *layer_base =
        p.k + static_cast<uint64_t>(l) * p.cap * p.T * key_stride + static_cast<uint64_t>(h) * ROW_BYTES;
    // A full group has no duplicated keys: the source offset of load `i` (key
    // j = 16*w + KPI*i + lane/CH of the tile, chunk (lane mod CH) ^ (j mod
    // CH)) splits into a uniform part in SGPRs, KPI*i*key_stride, and a
    // per-lane part XOR a per-load constant:
    //   lane_src ^ (((16*w + KPI*i) mod CH) * 16),
    //   lane_src = (lane/CH)*key_stride + ((lane mod CH) ^ (lane/CH))*16
    // (the XORed bits lie below ROW_BYTES, and key_stride is a multiple of
    // it), one VALU per load.  A group past the last key of a partial block
    // (or of a block length that is no multiple of 16) takes the general
    // path, which clamps keys to the last valid one.
    constexpr uint32_t KPI = 1024u / ROW_BYTES;  // keys per wave-wide 1 KiB load
    const uint32_t lane_src = (lane / CH) * static_cast<uint32_t>(key_stride) +
                              (((lane % CH) ^ (lane / CH)) * 16u);
    uint32_t lb = b_begin, lg = wave;
    auto wrap_group = [&]() {
        if constexpr (SEG || WR == 1) {
            while (lg >= gpb) {
                lg -= gpb;
                ++lb;
            }
        } else if (lg >= gpb) {  // a block part is a whole number of tiles
            lg -= gpb;
            ++lb;
        }
    };
    wrap_group();
    auto issue_tile = [&](uint32_t buf) {
        // a group past the chunk's end (the last tile) repeats valid keys;
        // its maxima are never written
        const uint32_t b = SEG ? min(lb, b_end - 1u) : lb;
        const uint32_t k0 = key0 + lg * 16u;
        const uint8_t *base = layer_base + static_cast<uint64_t>(b) * p.T * key_stride;
        const uint32_t nt = (b + 1 == p.B && p.last_T != 0) ? p.last_T : p.T;
        uint8_t *dst = &tiles[buf][wave * GROUP];
        // the lane terms pass through an empty asm so the per-load offsets
        // are recomputed here (a VALU or a few per load) instead of being
        // kept live across the loop next to the registers of query rows
        if (k0 + 16u <= nt) {
            uint32_t ls = lane_src;
            asm volatile("" : "+v"(ls));
            const uint8_t *tbase = base + static_cast<uint64_t>(k0) * key_stride;
#pragma unroll
            for (int i = 0; i < LOADS; ++i) {
                const uint32_t voff = ls ^ (((wave * 16u + KPI * i) & (CH - 1u)) * 16u);
                const uint8_t *src = tbase + static_cast<uint64_t>(KPI * i) * key_stride + voff;
                __builtin_amdgcn_global_load_lds(src, (lds_void_t *) (dst + i * 1024), 16, 0, DMA);
            }
        } else {
            uint32_t ln = lane;
            asm volatile("" : "+v"(ln));
#pragma unroll
            for (int i = 0; i < LOADS; ++i) {
                const uint32_t jg = KPI * i + ln / CH;                      // key within the group
                const uint32_t c = (ln % CH) ^ ((wave * 16u + jg) % CH);    // global chunk held there
                const uint32_t jj = min(k0 + jg, nt - 1u);                  // duplicate the last key
                const uint8_t *src = base + jj * key_stride + c * 16u;
                __builtin_amdgcn_global_load_lds(src, (lds_void_t *) (dst + i * 1024), 16, 0, DMA);
            }
        }
        lg += WR;
        wrap_group();
    };

    const uint32_t n_tiles = ((b_end - b_begin) * gpb + WR - 1u) / WR;
    issue_tile(0u);
    if (WR == 1 && n_tiles > 1u) {
        issue_tile(1u);
    }

    // ---- query rows -> A fragments (resident for the whole workgroup).
    // bf16 rows are converted to f16 as they come.  A bf16 value past f16's
    // range (|q| >= 65536, bf16 exponent >= 143) turns infinite there: then
    // the wave's rows are loaded again and converted times 2^-qexp, which
    // brings its largest |q| below 65536, and its maxima are scaled back on
    // the way out.  Both scalings are exact, so scores do not change.
    // Finding the largest |q| along the way, and only then the scale, takes
    // four VALU instructions per two elements where a pass for the maximum
    // and a scaled conversion took eight: start-up is VALU-bound, and every
    // workgroup pays it.
    half8_t a[RT][KS];
    const uint32_t row0 = rg * p.slice_rows + wave * (RT * 16u);
    load_query_bits<RT, KS, D>(p, a, l, h, row0, lrow, kgrp);
    int qexp = 0;
    if (p.q_bf16 != 0) {
        const float qmax = wave_max(convert_query_bits<RT, KS, false>(a, 1.0f));
        const uint32_t e = __float_as_uint(qmax) >> 23;
        if (e > 142u && e < 255u) {
            qexp = static_cast<int>(e) - 142;
            // loaded anew: the raw bits must not stay live beside the fragments
            uint32_t again = row0;
            asm volatile("" : "+s"(again) :: "memory");
            load_query_bits<RT, KS, D>(p, a, l, h, again, lrow, kgrp);
            (void) convert_query_bits<RT, KS, true>(a, __builtin_ldexpf(1.0f, -qexp));
        }
    }
    const float out_scale = __builtin_ldexpf(p.scale, qexp);

    // LDS byte address of B fragment (kt, ks) in buffer buf, i.e. of the
    // swizzled chunk (ks*4 + kgrp) ^ (key mod CH) of key kt*16 + lrow:
    //   (tiles + buf*TILE + kt*16*ROW_BYTES + lrow*ROW_BYTES + (kgrp ^ lrow)*16)
    //     ^ (ks*64 ^ ((kt*16) mod CH)*16)
    // -- everything at or above the row size is added, the swizzle bits
    // below it XORed in, so one VALU per read and one register per lane.
    const uint32_t lds0 = (uint32_t)(uintptr_t)((const __attribute__((address_space(3))) uint8_t *)(&tiles[0][0]));
    const uint32_t lane_b = lrow * ROW_BYTES + ((kgrp ^ lrow) * 16u);

    float *out = p.partial + ((static_cast<uint64_t>(sub * WR + wave) * p.L + l) * p.Hkv + h) * p.B;
    float m = -FLT_MAX;
    uint32_t cb = b_begin, cg = 0;  // the block and the groups of it in m
    auto flush = [&]() {
        m = wave_max(m);
        if (lane == 0) {
            out[cb] = m * out_scale;
        }
        m = -FLT_MAX;
        cg = 0;
        ++cb;
    };
    for (uint32_t it = 0; it < n_tiles; ++it) {
        const uint32_t buf = it & 1u;
        // this wave's loads of tile `it` have landed.  Alone, a wave keeps
        // the next tile's loads in flight past the wait and refills a buffer
        // as soon as it has read it; waves that share the tile meet at a
        // barrier, after which every wave's loads have landed and every wave
        // is done reading the other buffer.
        if (WR > 1 || it + 1u == n_tiles) {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        } else if (LOADS == 8) {
            asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
        } else {
            static_assert(LOADS == 8 || LOADS == 4, "loads of a group");
            asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
        }
        if constexpr (WR > 1) {
            __syncthreads();
            if (it + 1u < n_tiles) {
                issue_tile(buf ^ 1u);
            }
        }
        // B fragments of the tile: f = kt * KS + ks covers keys kt*16 .. +16
        // and k-slice ks.  The reads are inline asm with explicit
        // lgkmcnt waits that carry the fragment register as an operand:
        // two reads stay in flight ahead of the RT MFMAs that consume a
        // fragment, in three registers.  (Compiler-issued reads ended up
        // with a single register, each read waiting out the MFMAs before
        // it and its own latency after.)  Every read is waited for inside
        // the tile, before the next barrier.
        uint32_t tb = lds0 + buf * TILE + lane_b;
        asm volatile("" : "+v"(tb));  // recompute the read addresses per tile
        auto read_b = [&](int f) {
            const uint32_t kt = static_cast<uint32_t>(f / KS);
            const uint32_t ks = static_cast<uint32_t>(f % KS);
            const uint32_t addr = (tb + kt * (16u * ROW_BYTES)) ^ (ks * 64u ^ ((kt * 16u) & (CH - 1u)) * 16u);
            half8_t r;
            asm volatile("ds_read_b128 %0, %1" : "=v"(r) : "v"(addr) : "memory");
            return r;
        };
        constexpr int NF = WR * KS;
        constexpr int PF = 2;  // reads in flight ahead of the consumed one
        half8_t bq[PF + 1];
#pragma unroll
        for (int f = 0; f < PF; ++f) {
            bq[f] = read_b(f);
        }
        float4_t acc[RT];
#pragma unroll
        for (int f = 0; f < NF; ++f) {
            const int ks = f % KS;
            half8_t &bf = bq[f % (PF + 1)];
            if (f + PF < NF) {
                bq[(f + PF) % (PF + 1)] = read_b(f + PF);
            }
            // LDS reads return in order: wait until only the newer ones
            // (at most PF) are outstanding
            const int newer = (NF - 1 - f) < PF ? (NF - 1 - f) : PF;
            if (newer == 2) {
                asm volatile("s_waitcnt lgkmcnt(2)" : "+v"(bf) :: "memory");
            } else if (newer == 1) {
                asm volatile("s_waitcnt lgkmcnt(1)" : "+v"(bf) :: "memory");
            } else {
                asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(bf) :: "memory");
            }
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                acc[rt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                    a[rt][ks], bf, ks == 0 ? float4_t{0.0f, 0.0f, 0.0f, 0.0f} : acc[rt], 0, 0, 0);
            }
            if (ks == KS - 1) {
#pragma unroll
                for (int rt = 0; rt < RT; ++rt) {
                    m = __builtin_fmaxf(m, __builtin_fmaxf(__builtin_fmaxf(acc[rt][0], acc[rt][1]),
                                                           __builtin_fmaxf(acc[rt][2], acc[rt][3])));
                }
                if constexpr (SEG) {  // a block part may end after any group of the tile
                    if (++cg == gpb && cb < b_end) {
                        flush();
                    }
                }
            }
        }
        if constexpr (WR == 1) {
            // the tile's last fragment was waited for: its buffer is free
            if (it + 2u < n_tiles) {
                issue_tile(buf);
            }
        }
        if constexpr (!SEG) {
            cg += WR;
            if (cg == gpb) {
                flush();
            }
        }
    }
}

// The fold after the scorer, one launch:
//   layer_scores[l][b] = max_{slice, h} partial[slice][l][h][b]
//   scores[b]          = reduce over layers, in layer order, of layer_scores[l][b]
//                        (sum then / L for the mean, or max).
// A workgroup takes 16 blocks; 16 threads per block take the layers l,
// l + 16, ... and issue a layer's partial maxima as one batch of loads.
// After the barrier one thread per block reduces its layers in layer order,
// from LDS (up to kFoldLayers layers; from memory beyond).  The arithmetic is
// the plain loops' (a max chain in (slice, head) order, an ordered float sum),
// so batching changes no bit.  Latency-bound: 2 x 12 blocks 2.1 us, 3.8 with the
// layer scores read back from memory and a division per partial (16 x 2048
// blocks: 5.2 and 6.0).
constexpr uint32_t kFoldBlocks = 16;
constexpr uint32_t kFoldLanes = 256 / kFoldBlocks;
constexpr uint32_t kFoldBatch = 16;
constexpr uint32_t kFoldLayers = 64;
static_assert(kFoldLayers % kFoldBatch == 0, "whole batches from LDS");

__global__ __launch_bounds__(256) void score_fold_kernel(const float *partial, uint32_t S,
                                                         uint32_t L, uint32_t Hkv, uint32_t B,
                                                         float *layer_scores, int mode,
                                                         float *scores) {
    __shared__ float of_layer[kFoldLayers][kFoldBlocks];
    const uint32_t bl = threadIdx.x % kFoldBlocks;
    const uint32_t lane = threadIdx.x / kFoldBlocks;
    const uint32_t b = blockIdx.x * kFoldBlocks + bl;
    const uint32_t per_layer = S * Hkv;
    const uint64_t slice_step = (static_cast<uint64_t>(L) - 1u) * Hkv * B;  // from a slice's last head to the next's first
    if (b < B) {
        for (uint32_t l = lane; l < L; l += kFoldLanes) {
            float best = -FLT_MAX;
            uint32_t h = 0;  // head of the next partial (uniform)
            uint64_t at = static_cast<uint64_t>(l) * Hkv * B + b;
            for (uint32_t i0 = 0; i0 < per_layer; i0 += kFoldBatch) {
                float v[kFoldBatch];
#pragma unroll
                for (uint32_t j = 0; j < kFoldBatch; ++j) {
                    v[j] = i0 + j < per_layer ? partial[at] : -FLT_MAX;
                    at += B;
                    if (++h == Hkv) {
                        h = 0;
                        at += slice_step;
                    }
                }
#pragma unroll
                for (uint32_t j = 0; j < kFoldBatch; ++j) {
                    best = fmaxf(best, v[j]);
                }
            }
            layer_scores[static_cast<uint64_t>(l) * B + b] = best;
            if (l < kFoldLayers) {
                of_layer[l][bl] = best;
            }
        }
    }
    __syncthreads();
    if (lane != 0 || b >= B) {
        return;
    }
    const bool max_mode = mode == KVMEM_LAYER_MAX;
    float acc = max_mode ? -FLT_MAX : 0.0f;
    for (uint32_t l0 = 0; l0 < L; l0 += kFoldBatch) {
        float v[kFoldBatch];
        if (l0 < kFoldLayers) {  // (a whole batch; what lies past L is not used)
#pragma unroll
            for (uint32_t j = 0; j < kFoldBatch; ++j) {
                v[j] = of_layer[l0 + j][bl];
            }
        } else {
#pragma unroll
            for (uint32_t j = 0; j < kFoldBatch; ++j) {
                v[j] = l0 + j < L ? layer_scores[static_cast<uint64_t>(l0 + j) * B + b] : 0.0f;
            }
        }
#pragma unroll
        for (uint32_t j = 0; j < kFoldBatch; ++j) {
            if (l0 + j < L) {
                acc = max_mode ? fmaxf(acc, v[j]) : acc + v[j];
            }
        }
    }
    if (mode == KVMEM_LAYER_MEAN && L > 0) {
        acc = acc / static_cast<float>(L);
    }
    scores[b] = acc;
}

size_t score_partial_bytes(uint32_t L, uint32_t Hkv, uint32_t B, uint32_t n_q_tokens, uint32_t g) {
    // the most any launch shape uses: four partial maxima per row slice and
    // block (waves times key parts), whatever the block count
    const size_t rows = static_cast<size_t>(n_q_tokens) * g;
    const size_t slices = (rows + kSliceRows - 1) / kSliceRows * kMaxRowWaves;
    return sizeof(float) * slices * L * Hkv * B;
}

using ScoreKernel = void (*)(ScoreParams);

// The kernel of a shape: RT row tiles per wave, WR waves on a key tile, SEG
// when a block part is not a whole number of tiles, REUSE when several row
// slices (of four waves then) read the same keys.
template <int D, int WR, bool SEG, bool REUSE>
static ScoreKernel score_kernel_of(uint32_t rt) {
    switch (rt) {
        case 4: return score_kernel<D, 4, WR, SEG, REUSE>;
        case 5: return score_kernel<D, 5, WR, SEG, REUSE>;
        default: return score_kernel<D, 6, WR, SEG, REUSE>;
    }
}
template <int D>
static ScoreKernel score_kernel_of(uint32_t rt, uint32_t wr, bool seg, bool reuse) {
    if (wr == 1) {
        switch (rt) {
            case 1: return score_kernel<D, 1, 1, false, false>;
            case 2: return score_kernel<D, 2, 1, false, false>;
            case 3: return score_kernel<D, 3, 1, false, false>;
            default: return score_kernel_of<D, 1, false, false>(rt);
        }
    }
    if (wr == 2) {
        return seg ? score_kernel_of<D, 2, true, false>(rt) : score_kernel_of<D, 2, false, false>(rt);
    }
    if (reuse) {
        return seg ? score_kernel_of<D, 4, true, true>(rt) : score_kernel_of<D, 4, false, true>(rt);
    }
    return seg ? score_kernel_of<D, 4, true, false>(rt) : score_kernel_of<D, 4, false, false>(rt);
}

bool load_score_kernels() {
    return load_kernel_object(&score_kernel<256, kMaxRowTiles, kMaxRowWaves, false, false>);
}

}  // namespace kvmem_hip

using namespace kvmem_hip;

namespace {

// Validates a scorer call and fills its launch shape (everything but the
// partial-maxima buffer).  Sets *empty when there is nothing to score.
struct ScoreShape {
    uint32_t rt = 0;  // row tiles per wave
    uint32_t wr = 0;  // waves of a workgroup (on one key tile)
    bool seg = false;
    uint64_t grid = 0;
};

int score_setup(kvmem_hip_ctx *ctx, const kvmem_hip_history *hist, const kvmem_hip_score_args *args,
                ScoreParams &p, ScoreShape &shape, bool *empty) {
    *empty = false;
    if (!hist || !args || !hist->k || !args->q || !args->scores) {
        return fail(ctx, KVMEM_HIP_ERR_INVALID, "score: null argument");
    }
    const uint32_t D = args->head_dim;
    if (D != 128 && D != 256) {
        return fail(ctx, KVMEM_HIP_ERR_UNSUPPORTED, "score: head_dim must be 128 or 256");
    }
    if (args->n_head_kv == 0 || args->n_head % args->n_head_kv != 0 || args->n_q_tokens == 0) {
        return fail(ctx, KVMEM_HIP_ERR_INVALID, "score: n_head must be a positive multiple of n_head_kv");
    }
    if (hist->n_embd_k != args->n_head_kv * D) {
        return fail(ctx, KVMEM_HIP_ERR_INVALID, "score: history n_embd_k != n_head_kv*head_dim");
    }
    if (hist->block_tokens == 0 || hist->block_tokens > static_cast<uint32_t>(kMaxTokens) ||
        hist->last_block_tokens > hist->block_tokens) {
        return fail(ctx, KVMEM_HIP_ERR_UNSUPPORTED, "score: block_tokens must be in [1, 128]");
    }
    if (args->q_type != KVMEM_TYPE_BF16 && args->q_type != KVMEM_TYPE_F16) {
        return fail(ctx, KVMEM_HIP_ERR_UNSUPPORTED, "score: query must be bf16 or f16");
    }
    if (args->layer_reduce < KVMEM_LAYER_MEAN || args->layer_reduce > KVMEM_LAYER_SUM) {
        return fail(ctx, KVMEM_HIP_ERR_INVALID, "score: bad layer_reduce");
    }
    if ((reinterpret_cast<uintptr_t>(hist->k) & 15u) || (reinterpret_cast<uintptr_t>(args->q) & 15u)) {
        return fail(ctx, KVMEM_HIP_ERR_INVALID, "score: q and k must be 16-byte aligned");
    }
    const uint32_t L = hist->n_layers;
    const uint32_t B = hist->n_blocks;
    if (L == 0 || B == 0) {
        *empty = true;
        return KVMEM_HIP_OK;
    }
    p = ScoreParams{};
    p.q = static_cast<const uint16_t *>(args->q);
    p.k = static_cast<const uint8_t *>(hist->k);
    p.L = L;
    p.Tq = args->n_q_tokens;
    p.Hq = args->n_head;
    p.Hkv = args->n_head_kv;
    p.B = B;
    p.cap = hist->capacity_blocks ? hist->capacity_blocks : B;
    if (p.cap < B) {
        return fail(ctx, KVMEM_HIP_ERR_INVALID, "score: capacity_blocks below n_blocks");
    }
    p.T = hist->block_tokens;
    p.last_T = hist->last_block_tokens;
    p.g = args->n_head / args->n_head_kv;
    p.R = p.Tq * p.g;
    p.q_bf16 = args->q_type == KVMEM_TYPE_BF16;
    p.scale = 1.0f / std::sqrt(static_cast<float>(D));
    // Row slices of at most 24 tiles, equal but for the last; a slice's tiles
    // go to one wave while they fit its registers, else to two or four waves
    // that share each key tile.
    const uint32_t row_tiles = (p.R + 15u) / 16u;
    p.RG = (row_tiles + kSliceTiles - 1u) / kSliceTiles;
    const uint32_t slice_tiles = (row_tiles + p.RG - 1u) / p.RG;
    shape.wr = slice_tiles <= 6u ? 1u : slice_tiles <= 12u ? 2u : 4u;
    shape.rt = (slice_tiles + shape.wr - 1u) / shape.wr;
    p.slice_rows = shape.rt * shape.wr * 16u;
    const uint32_t pairs = L * p.Hkv;
    // Few blocks: their keys are split over up to four waves' workgroups
    const uint32_t groups = (p.T + 15u) / 16u;  // 16-key groups of a block
    p.KS = 1;
    while (p.KS * shape.wr < kMaxRowWaves && groups % (2u * p.KS) == 0 &&
           static_cast<uint64_t>(pairs) * p.RG * B * p.KS * shape.wr < kSplitWaves) {
        p.KS *= 2u;
    }
    p.gpb = groups / p.KS;
    shape.seg = shape.wr > 1u && p.gpb % shape.wr != 0;
    // Workgroups of a launch: the chip full once, or two or four times where
    // that leaves them chunks of 32 or 64 blocks (of 128 keys).  More rounds
    // even out the end of the launch (16 x 2048 blocks, 64-token query: 2.427
    // ms with four, 2.447 with one); every workgroup loads and converts its
    // query rows first, which short chunks do not repay (16 x 128 blocks:
    // 181 us with four rounds, 163 with one).
    const uint32_t n_sub = p.RG * p.KS;
    // (D = 256: 16 KiB of key tiles per wave hold two waves per SIMD)
    const uint32_t full =
        1024u * (D == 256 ? 2u : static_cast<uint32_t>(score_occupancy(128, static_cast<int>(shape.rt))));
    const uint64_t waves = static_cast<uint64_t>(pairs) * n_sub * shape.wr;  // per chunk
    for (uint32_t rounds = 4; rounds > 0; rounds /= 2u) {
        p.n_chunks = static_cast<uint32_t>(std::min<uint64_t>(B, std::max<uint64_t>(1, full * rounds / waves)));
        p.blocks_per_chunk = (B + p.n_chunks - 1) / p.n_chunks;
        if (static_cast<uint64_t>(p.blocks_per_chunk) * p.T >= 2048u * rounds) {
            break;
        }
    }
    if (p.RG > 1) {
        // Several row slices read the same key tiles.  Their workgroups are
        // consecutive on one XCD, and chunks of at most 64 blocks keep them
        // close enough together for a tile to come from that XCD's L2 (16 x
        // 8192 blocks, 512-token query: 65.3 ms; 67.6 with 16 blocks per
        // chunk, 65.7 with 256).  Up to there the chunk of the least cost: a
        // workgroup's blocks and its start-up, which is worth about 128 keys,
        // by the rounds of workgroups, half as if they ran in step (a short
        // last round leaves the chip idle) and half as if they did not.  16
        // layers x 50 blocks, 384-token query: 343 us (13 blocks per chunk; 394
        // in one round of 50, 371 in 3.75 of 10); 2 x 1454, 512-token query:
        // 1136 us (1256 with 64 blocks per chunk, 1225 with 35).
        const uint32_t chip = full / shape.wr;
        double best = 0.0;
        for (uint32_t bpc = std::min(B, 64u); bpc > 0; --bpc) {
            const double rounds = static_cast<double>(pairs) * p.RG * ((B + bpc - 1) / bpc) / chip;
            const double cost = (rounds + std::ceil(rounds)) * (bpc + 128.0 / p.T);
            if (best == 0.0 || cost < best) {
                best = cost;
                p.blocks_per_chunk = bpc;
            }
        }
    }
    p.n_chunks = (B + p.blocks_per_chunk - 1) / p.blocks_per_chunk;
    p.xcd_major = (pairs % 8u) == 0;
    shape.grid = static_cast<uint64_t>(pairs) * n_sub * p.n_chunks;
    if (shape.grid > 0x7fffffffu) {
        return fail(ctx, KVMEM_HIP_ERR_INVALID, "score: problem too large for one launch");
    }
    return KVMEM_HIP_OK;
}

// The scorer and the fold on the context stream: p.partial receives the
// per-slice maxima, `layers` the per-layer scores.  `timed` brackets the
// scorer with the profiling events of kPerfScore.
int score_launch(kvmem_hip_ctx *ctx, const kvmem_hip_score_args *args, const ScoreParams &p,
                 const ScoreShape &shape, float *layers, bool timed) {
    if (injected_fail(ctx, KVMEM_HIP_FAIL_LAUNCH, "score kernel launch")) {
        return KVMEM_HIP_ERR_RUNTIME;
    }
    if (timed) {
        (void) perf_attach(ctx, kPerfScore);  // the scorer's events ride on its launch
    }
    ctx_launch(ctx,
               args->head_dim == 256 ? score_kernel_of<256>(shape.rt, shape.wr, shape.seg, p.RG > 1)
                                     : score_kernel_of<128>(shape.rt, shape.wr, shape.seg, p.RG > 1),
               dim3(static_cast<uint32_t>(shape.grid)), dim3(shape.wr * 64u), 0, p);
    const bool launched = hip_ok(ctx, hipGetLastError(), "score kernel launch");
    if (timed) {
        perf_detach(ctx, kPerfScore, launched);
    }
    if (!launched) {
        return KVMEM_HIP_ERR_RUNTIME;
    }
    // the fold is not bracketed: a timing event costs the stream a few
    // microseconds, as much as the fold itself
    score_fold_kernel<<<(p.B + kFoldBlocks - 1) / kFoldBlocks, 256, 0, ctx->stream>>>(
        p.partial, p.RG * p.KS * shape.wr, p.L, p.Hkv, p.B, layers, args->layer_reduce, args->scores);
    if (!hip_ok(ctx, hipGetLastError(), "score fold launch")) {
        return KVMEM_HIP_ERR_RUNTIME;
    }
    return KVMEM_HIP_OK;
}

// Scratch of kvmem_hip_score_noalloc, one copy per GPU for the life of the
// process: the per-slice maxima, then (when the caller passes no
// layer_scores) the per-layer scores.  The 256K workload (16 layers x 2048
// blocks, 4 KV heads, a 64-token query of 24 heads) needs 2 MiB + 128 KiB.
constexpr size_t kNoAllocScratchBytes = size_t{8} << 20;
static __device__ __align__(256) uint8_t scratch[kNoAllocScratchBytes];

// Device address of `scratch` on each GPU, looked up once per device, and
// its owner: the context and stream of the last call, whose completion
// event tells when the array is free again.  A call from another context
// while that event is pending would race on the array and is refused
// instead (a context's own calls are ordered: set_stream waits for the old
// stream).
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void *g_scratch_addr[kMaxDevices] = {};
struct ScratchOwner {
    const kvmem_hip_ctx *ctx = nullptr;
    hipStream_t stream = nullptr;
};
ScratchOwner g_scratch_owner[kMaxDevices];

}  // namespace

namespace kvmem_hip {

bool score_scratch_setup(kvmem_hip_ctx *ctx) {
    if (ctx->device < 0 || ctx->device >= kMaxDevices) {
        fail(ctx, KVMEM_HIP_ERR_UNSUPPORTED, "score scratch: device ordinal beyond 63");
        return false;
    }
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_addr[ctx->device]) {
        // the caller made ctx->device current
        void *addr = nullptr;
        if (!hip_ok(ctx, hipGetSymbolAddress(&addr, HIP_SYMBOL(scratch)), "score scratch address")) {
            return false;
        }
        g_scratch_addr[ctx->device] = addr;
    }
    ctx->noalloc_scratch = g_scratch_addr[ctx->device];
    // the owner record's completion event (no timing: cheap to record)
    return hip_ok(ctx, hipEventCreateWithFlags(&ctx->noalloc_done, hipEventDisableTiming), "score scratch event");
}

void score_scratch_release(kvmem_hip_ctx *ctx) {
    if (ctx->device < 0 || ctx->device >= kMaxDevices) {
        return;
    }
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (g_scratch_owner[ctx->device].ctx == ctx) {
        g_scratch_owner[ctx->device] = ScratchOwner{};
    }
}

}  // namespace kvmem_hip

extern "C" int kvmem_hip_score(kvmem_hip_ctx *ctx, const kvmem_hip_history *hist,
                               const kvmem_hip_score_args *args) {
    if (!ctx) {
        return KVMEM_HIP_ERR_INVALID;
    }
    ScoreParams p;
    ScoreShape shape;
    bool empty = false;
    int st = score_setup(ctx, hist, args, p, shape, &empty);
    if (st != KVMEM_HIP_OK || empty) {
        return st;
    }
    (void) hipSetDevice(ctx->device);
    const size_t partial_bytes = score_partial_bytes(p.L, p.Hkv, p.B, p.Tq, p.g);
    if (!ensure_dev(ctx, ctx->score_partial, partial_bytes, "score partial")) {
        return KVMEM_HIP_ERR_NOMEM;
    }
    p.partial = static_cast<float *>(ctx->score_partial.ptr);
    float *layers = args->layer_scores;
    if (!layers) {
        if (!ensure_dev(ctx, ctx->score_layers, sizeof(float) * static_cast<size_t>(p.L) * p.B,
                        "score layer buffer")) {
            return KVMEM_HIP_ERR_NOMEM;
        }
        layers = static_cast<float *>(ctx->score_layers.ptr);
    }
    return score_launch(ctx, args, p, shape, layers, true);
}

extern "C" int kvmem_hip_score_noalloc(kvmem_hip_ctx *ctx, const kvmem_hip_history *hist,
                                       const kvmem_hip_score_args *args) {
    if (!ctx) {
        return KVMEM_HIP_ERR_INVALID;
    }
    ScoreParams p;
    ScoreShape shape;
    bool empty = false;
    int st = score_setup(ctx, hist, args, p, shape, &empty);
    if (st != KVMEM_HIP_OK || empty) {
        return st;
    }
    if (!ctx->noalloc_scratch) {
        return fail(ctx, KVMEM_HIP_ERR_RUNTIME, "score_noalloc: no scratch address for this device");
    }
    const size_t partial_bytes = score_partial_bytes(p.L, p.Hkv, p.B, p.Tq, p.g);
    const size_t layer_off = (partial_bytes + 255) / 256 * 256;
    const size_t need = args->layer_scores ? partial_bytes
                                           : layer_off + sizeof(float) * static_cast<size_t>(p.L) * p.B;
    if (need > kNoAllocScratchBytes) {
        return fail(ctx, KVMEM_HIP_ERR_INVALID,
                    "score_noalloc: " + std::to_string(need) + " bytes of scratch needed, the maximum is " +
                        std::to_string(kNoAllocScratchBytes) + " (use kvmem_hip_score)");
    }
    (void) hipSetDevice(ctx->device);
    // Under graph capture the launches become graph nodes and the call's
    // completion cannot be tracked: its replays run when the caller launches
    // them.  An event recorded in a capture cannot be queried afterwards,
    // so none is recorded and the capturing context stays the owner.
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    if (!hip_ok(ctx, hipStreamIsCapturing(ctx->stream, &capture), "score_noalloc capture status")) {
        return KVMEM_HIP_ERR_RUNTIME;
    }
    const bool capturing = capture != hipStreamCaptureStatusNone;
    // Take the device's array: free when no call is recorded, when the last
    // one came from this context on this stream (queued behind it), or when
    // the last call's completion event has fired.
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    ScratchOwner &own = g_scratch_owner[ctx->device];
    if (own.ctx && !(own.ctx == ctx && own.stream == ctx->stream)) {
        const hipError_t q = hipEventQuery(own.ctx->noalloc_done);
        if (q == hipErrorNotReady) {
            return fail(ctx, KVMEM_HIP_ERR_BUSY,
                        "score_noalloc: another context or stream is still using this GPU's scratch");
        }
        if (q != hipSuccess) {
            return fail(ctx, KVMEM_HIP_ERR_RUNTIME,
                        std::string("score_noalloc: owner event: ") + hipGetErrorString(q));
        }
    }
    uint8_t *base = static_cast<uint8_t *>(ctx->noalloc_scratch);
    p.partial = reinterpret_cast<float *>(base);
    float *layers = args->layer_scores ? args->layer_scores : reinterpret_cast<float *>(base + layer_off);
    st = score_launch(ctx, args, p, shape, layers, false);
    if (st != KVMEM_HIP_OK) {
        // a launch that failed after the scorer kernel was queued leaves that
        // kernel on the array with no owner record: let it drain first (a
        // capture holds nothing that runs)
        if (!capturing) {
            (void) hipStreamSynchronize(ctx->stream);
        }
        return st;
    }
    if (capturing) {
        own.ctx = ctx;
        own.stream = ctx->stream;
        return KVMEM_HIP_OK;
    }
    if (!hip_ok(ctx, hipEventRecord(ctx->noalloc_done, ctx->stream), "score_noalloc completion event")) {
        own = ScratchOwner{};  // nothing tells when the launched work ends: no owner to wait for
        (void) hipStreamSynchronize(ctx->stream);
        return KVMEM_HIP_ERR_RUNTIME;
    }
    own.ctx = ctx;
    own.stream = ctx->stream;
    return KVMEM_HIP_OK;
}

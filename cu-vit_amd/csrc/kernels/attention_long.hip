// Fused attention for sequences beyond the 256 tokens of attention.hip and
// attention_bf16.hip: context = softmax(Q.K^T / 8).V per (image, head) from the
// packed projection, one pass over the keys with a running maximum and sum, so
// neither the [images, heads, tokens, tokens] logits nor a row of them is ever
// stored. It stands in for the reference's three launches
// (src/model/vit.cu:205-245) inside the model; those materialise the logits
// twice, and their rows of tokens elements (577 at 384 pixels) are seldom
// 16-byte aligned, which puts the products on the GEMM's element-wise loads.
//
// What bounds it. 4 * tokens^2 * 64 flops a pair against 4 * tokens * 64
// elements moved: the matrix pipe and the exponentials, never HBM. bf16: a
// wavefront's 64 keys are 16 MFMAs of 32 cycles and about twice that in VALU
// work (scale, exponential, pack: 32 logits a lane). fp32: 128 MFMAs of 32
// cycles per 64 keys, the VALU work a tenth of it and not overlapped.
//
// Split. Two wavefronts share a tile of queries (32 in bf16, 16 in fp32), each
// with its half of every 64-key block, and add up their sums at the end; a
// workgroup is two such tiles and stages the blocks for both (a block's loads
// go out two blocks ahead, two LDS buffers, one barrier a block). Halved keys,
// because a few images have fewer query tiles than the chip has SIMDs (at 577
// tokens 19 (bf16) or 37 (fp32) a head), and one wavefront's walk is then the
// kernel's time; halved whatever the batch, because a row's sums must not
// depend on it. Measured, one part / two / (fp32) four, in us: bf16 at 577
// tokens 1 image x 3 heads 12.2 / 9.5, 8 x 6 13.6 / 13.6, 16 x 12 38.7 / 41.3,
// 32 x 6 at 257 tokens 16.4 / 15.5; fp32 1 x 3 26.7 / 18.1 / 19.1, 8 x 6 48.3 /
// 53.3 / 63.3, 8 x 5 46.9 / 44.3 / 52.5, 4 x 6 at 257 tokens 14.7 / 10.9 / 12.5.
// All of a pair's workgroups go to one XCD, whose L2 then reads the pair's K
// and V from HBM once.
//
// Softmax. With m the running maximum, p = exp2((x - m) c), c = log2 e / 8:
// m is raised only when some query's block maximum exceeds it by more than
// 2^kHeadroom in the exponential, so p stays below 2^kHeadroom and the sums
// and the context accumulators are seldom rescaled; numerator and denominator
// carry the same factor. Logits, sums and context accumulate in fp32 (the
// launches round bf16 logits); bf16 weights are rounded once, as the softmax
// launch stores them. Error against 64 bits at 577 tokens, Q and K of standard
// deviation 1 (0.05): fp32 4.2e-7 (3.1e-7) against the launches' 5.2e-7
// (4.3e-7), bf16 2.3e-3 (2.0e-3) against 4.4e-3 (2.1e-3). A row of -inf logits
// gives NaN, as the launches do; a query whose sums overflow or vanish before
// they are normalised is taken again by itself (attend_normalised).
#include "attention_common.hpp"
#include "launch.hpp"

namespace cuvit::detail {
namespace {

using namespace attention;
using namespace cuvit::device;
using gemm::Mma;

constexpr float kScaledLog2e = 1.4426950408889634F * 0.125F;  // log2 e / sqrt(64)
constexpr float kHeadroom = 8.0F;
constexpr int kWaves = 4;
constexpr int kThreads = kWaves * kWave;
constexpr int kSplit = 2;                        // wavefronts that share a query tile's keys
constexpr int kTilesPerGroup = kWaves / kSplit;  // query tiles of a workgroup

/// Which pair and which group of query tiles a workgroup takes: workgroup b
/// runs on XCD b % 8, and a pair's groups all go to XCD pair % 8.
struct Place {
    int pair;
    int group;
};

__device__ __forceinline__ Place place(int groups) {
    const int slot = static_cast<int>(blockIdx.x) / 8;
    return {static_cast<int>(blockIdx.x) % 8 + 8 * (slot / groups), slot % groups};
}

struct Max2 {
    __device__ __forceinline__ float operator()(float a, float b) const { return fmaxf(a, b); }
};
struct Add2 {
    __device__ __forceinline__ float operator()(float a, float b) const { return a + b; }
};

/// The running maximum and sum of a lane's query, the exponent's shift
/// -(m c), and the factor that what was accumulated so far takes.
struct Running {
    float maximum = -INFINITY;
    float shift = 0.F;
    float sum = 0.F;

    /// Raises the maximum to cover @p block (the block's maximum, alike in
    /// all of the query's lanes) when any query of the wavefront needs it;
    /// true when the accumulated context must take @p factor.
    __device__ __forceinline__ bool raise(float block, float& factor) {
        const bool needed = fmaf(block, kScaledLog2e, shift) > kHeadroom || maximum == -INFINITY;
        if (!__any(needed)) {
            return false;
        }
        const float raised = fmaxf(maximum, block);
        // While every logit so far is -inf the shift stays 0: exp2(-inf) is 0
        // where (-inf) - (-inf) would be NaN.
        const float next = raised == -INFINITY ? 0.F : -(raised * kScaledLog2e);
        // The ratio of the two shifts as the weights see them, roundings included.
        factor = maximum == -INFINITY ? 0.F : __builtin_amdgcn_exp2f(next - shift);
        maximum = raised;
        shift = next;
        sum *= factor;
        return true;
    }

    __device__ __forceinline__ float weight(float logit) const {
        return __builtin_amdgcn_exp2f(fmaf(logit, kScaledLog2e, shift));
    }
};

/// The walk over the keys, shared by both types. Block i sits in LDS buffer
/// i % 2; its loads go out while block i - 2 is worked on (two register sets)
/// and reach LDS while block i - 1 is. One barrier a block: the buffer written
/// in a turn was last read before the barrier that opened it. A block past the
/// tokens loads zeros and is never worked on.
/// A wavefront works on its part of each block only.
template <int Keys, int Edge, int PerThread, typename Prefetch, typename Commit, typename Step>
__device__ __forceinline__ void walk_blocks(int tokens, int part, bool live, Prefetch&& prefetch, Commit&& commit,
                                            Step&& step) {
    Vec16 even[PerThread];
    Vec16 odd[PerThread];
    auto turn = [&](Vec16 (&landed)[PerThread], Vec16 (&freed)[PerThread], int first, int buffer) {
        prefetch(freed, first + 2 * Keys);
        if (live) {
            constexpr int kPart = Keys / kSplit;
            constexpr int kTiles = kPart / Edge;
            const int left = tokens - first - part * kPart;
            static_assert(kTiles <= 2, "a tail is one tile or all of them");
            if (left >= kPart) {
                step(std::integral_constant<int, kTiles>{}, std::false_type{}, buffer, left);
            } else if (kTiles > 1 && left > Edge) {
                step(std::integral_constant<int, kTiles>{}, std::true_type{}, buffer, left);
            } else if (left > 0) {
                step(std::integral_constant<int, 1>{}, std::true_type{}, buffer, left);
            }
        }
        commit(landed, buffer ^ 1);
        __syncthreads();
    };
    prefetch(even, 0);
    prefetch(odd, Keys);
    commit(even, 0);
    __syncthreads();
    for (int first = 0; first < tokens; first += 2 * Keys) {
        turn(odd, even, first, 0);
        if (first + Keys < tokens) {
            turn(even, odd, first + Keys, 1);
        }
    }
}

/// Adds the second part's sum and context accumulators (@p values, Count
/// floats a lane) to the first part's, each scaled to the larger maximum,
/// through @p lds. The parts of a query tile are wavefronts w and w + 1, w
/// even; every wavefront of the workgroup takes part.
template <int Count>
__device__ __forceinline__ void combine_parts(float* lds, int wave, int lane, Running& running, float (&values)[Count]) {
    static_assert(kSplit == 2, "one exchange");
    float* const slot = lds + (wave / kSplit) * (Count + 3) * kWave + lane;
    if (wave % kSplit != 0) {
#pragma unroll
        for (int i = 0; i < Count; ++i) {
            slot[i * kWave] = values[i];
        }
        slot[Count * kWave] = running.maximum;
        slot[(Count + 1) * kWave] = running.shift;
        slot[(Count + 2) * kWave] = running.sum;
    }
    __syncthreads();
    if (wave % kSplit == 0) {
        const float maximum = slot[Count * kWave];
        const float shift = slot[(Count + 1) * kWave];
        const float common = maximum > running.maximum ? shift : running.shift;
        // A part that saw nothing but -inf has sums of 0 and takes factor 0.
        const float mine = running.maximum == -INFINITY ? 0.F : __builtin_amdgcn_exp2f(common - running.shift);
        const float theirs = maximum == -INFINITY ? 0.F : __builtin_amdgcn_exp2f(common - shift);
        running.sum = running.sum * mine + slot[(Count + 2) * kWave] * theirs;
#pragma unroll
        for (int i = 0; i < Count; ++i) {
            values[i] = values[i] * mine + slot[i * kWave] * theirs;
        }
    }
}

/// Whether a query's sums are of no use: its numerators overflowed where the
/// context would not (V within its type, but above 2^128 / (tokens 2^kHeadroom),
/// about 2e33 here), its weights did, or they vanished (logits beyond 2^31,
/// the type's lowest value among them: `shift` is then rounded by more than an
/// exponent's range), or there is an infinity or NaN in it, which stays.
template <int Count> __device__ __forceinline__ bool unusable(float sum, const float (&values)[Count]) {
    float largest[2] = {0.F, 0.F};
#pragma unroll
    for (int i = 0; i < Count; ++i) { // (a NaN stays)
        largest[i / 2 % 2] = __builtin_elementwise_maximum(largest[i / 2 % 2], fabsf(values[i]));
    }
    const float all = __builtin_elementwise_maximum(largest[0], largest[1]);
    return !(all < INFINITY && sum > 0.F && sum < INFINITY);
}

/// The context of one query whose sums were unusable, by a whole wavefront: the
/// exponent is a difference of logits, and what is accumulated stays
/// normalised, so within max |V|, both as in the launches. @p qkv is the pair's
/// Q of token 0. Slow (about 65 us a query at 577 tokens), and seldom run; weights
/// lowered for every query instead would lose as much where V is tiny, and the
/// difference costs an instruction a logit.
template <typename T>
__device__ __forceinline__ void attend_normalised(const T* qkv, T* context_row, int query, int tokens,
                                                  std::int64_t qkv_row, int embed) {
    constexpr int kVec = Elem<T>::kPerVec;
    const int lane = lane_id();
    const T* const q = qkv + query * qkv_row;
    float maximum = -INFINITY;
    float sum = 0.F;
    float value = 0.F; // of dim `lane`
#pragma clang loop unroll(disable)
    for (int first = 0; first < tokens; first += kWave) {
        float logit = -INFINITY; // of key first + lane
        if (first + lane < tokens) {
            const T* const k = qkv + (first + lane) * qkv_row + embed;
            logit = 0.F;
#pragma clang loop unroll(disable)
            for (int d = 0; d < kHeadDim; d += kVec) {
                const Vec16 a = load16(q + d);
                const Vec16 b = load16(k + d);
#pragma unroll
                for (int e = 0; e < kVec; ++e) {
                    logit = fmaf(Elem<T>::get(a, e), Elem<T>::get(b, e), logit);
                }
            }
        }
        const float raised = fmaxf(maximum, wave_allreduce(logit, Max2{}));
        if (raised == -INFINITY) {
            continue;
        }
        const float weight = __builtin_amdgcn_exp2f((logit - raised) * kScaledLog2e);
        const float kept = maximum == -INFINITY ? 0.F : sum * __builtin_amdgcn_exp2f((maximum - raised) * kScaledLog2e);
        maximum = raised;
        sum = kept + wave_allreduce(weight, Add2{});
        if (sum != sum) {
            break; // NaN, whatever follows
        }
        value *= kept / sum;
        const float share = weight / sum;
        const int keys = min(tokens - first, kWave);
        const T* const v = qkv + first * qkv_row + 2 * static_cast<std::int64_t>(embed) + lane;
#pragma clang loop unroll(disable)
        for (int key = 0; key < keys; ++key) {
            const float s = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(share), key));
            value = fmaf(s, Elem<T>::load(v + key * qkv_row), value);
        }
    }
    Elem<T>::store(context_row + lane, sum > 0.F ? value : __builtin_nanf("")); // (no logit above -inf: NaN)
}

// -- bf16 -----------------------------------------------------------------------

constexpr int kEdge = 32;       // queries of a wavefront, keys of an MFMA tile
constexpr int kBlockKeys = 64;  // keys a step
constexpr int kKBlock = 16;     // k of one MFMA

__global__ __launch_bounds__(kThreads, 3) void attention_long_bf16_kernel(
    const std::uint16_t* __restrict__ qkv, std::uint16_t* __restrict__ context, int heads, int tokens,
    int pairs, int groups) {
    using Acc = Mma<std::uint16_t>::Acc;
    constexpr int kBuffer = kBlockKeys * (kHeadDim + kKeyPitch);  // V, then K
    __shared__ Vec16 lds_vectors[2 * kBuffer / 8];
    std::uint16_t* const lds = reinterpret_cast<std::uint16_t*>(lds_vectors);
    const Place at = place(groups);
    if (at.pair >= pairs) {
        return;  // the whole workgroup, before any barrier
    }
    const int t = static_cast<int>(threadIdx.x);
    const int lane = lane_id();
    const int wave = t / kWave;
    const int row = lane % kEdge;
    const int half = lane / kEdge;
    const int image = at.pair / heads;
    const int head = at.pair - image * heads;
    const int embed = heads * kHeadDim;
    const std::int64_t qkv_row = 3 * static_cast<std::int64_t>(embed);
    const std::uint16_t* const q_base = qkv + static_cast<std::int64_t>(image) * tokens * qkv_row + head * kHeadDim;
    const auto q_resource = gemm::buffer_resource(q_base);
    const auto kv_resource = gemm::buffer_resource(q_base + embed);  // V follows K by embed

    const int part = wave % kSplit;
    const int query0 = (at.group * kTilesPerGroup + wave / kSplit) * kEdge;
    const int query = query0 + row;
    const bool live = query0 < tokens;  // the others still stage K and V

    Vec16 q[kHeadDim / kKBlock];
#pragma unroll
    for (int kb = 0; kb < kHeadDim / kKBlock; ++kb) {
        q[kb] = load_or_zero(q_resource, query * qkv_row + kb * kKBlock + 8 * half, query < tokens);
    }

    // A block's K and V: 1024 16-byte chunks, four a thread (V's first).
    constexpr int kChunks = kHeadDim / 8;
    constexpr int kPerThread = 2 * kBlockKeys * kChunks / kThreads;
    static_assert(2 * kBlockKeys * kChunks % kThreads == 0 && kPerThread % 2 == 0, "whole chunks per thread");
    const int chunk_key = t / kChunks;  // plus kThreads / kChunks keys a step
    const int chunk_dim = 8 * (t % kChunks);
    constexpr int kKeyStep = kThreads / kChunks;
    auto prefetch = [&](Vec16 (&ahead)[kPerThread], int first_key) {
#pragma unroll
        for (int i = 0; i < kPerThread; ++i) {
            const int key = first_key + chunk_key + kKeyStep * (i % (kPerThread / 2));
            ahead[i] = load_or_zero(kv_resource, key * qkv_row + chunk_dim + (i < kPerThread / 2 ? embed : 0),
                                    key < tokens);
        }
    };
    auto commit = [&](const Vec16 (&ahead)[kPerThread], int buffer) {
        std::uint16_t* const values = lds + buffer * kBuffer;
        std::uint16_t* const keys = values + kBlockKeys * kHeadDim;
#pragma unroll
        for (int i = 0; i < kPerThread; ++i) {
            const int key = chunk_key + kKeyStep * (i % (kPerThread / 2));
            if (i < kPerThread / 2) {
                store16(values + value_slot(key, chunk_dim), ahead[i]);
            } else {
                store16(keys + key * kKeyPitch + chunk_dim, ahead[i]);
            }
        }
    };

    Running running;
    Acc out[2] = {Acc{}, Acc{}};

    // One block: kTiles 32-key tiles of LDS buffer @p buffer, of which @p valid
    // keys are real when kMasked (otherwise all).
    auto step = [&](auto tiles, auto masked, int buffer, int valid) {
        constexpr int kTiles = decltype(tiles)::value;
        constexpr bool kMasked = decltype(masked)::value;
        const int first_tile = part * (kBlockKeys / kSplit / kEdge);
        const std::uint16_t* const values = lds + buffer * kBuffer + first_tile * kEdge * kHeadDim;
        const std::uint16_t* const keys =
            lds + buffer * kBuffer + kBlockKeys * kHeadDim + first_tile * kEdge * kKeyPitch;
        // Every K fragment of the block, then (behind the logits' MFMAs) every
        // V fragment: one LDS latency each, V's under the softmax. Left alone
        // the compiler reads each fragment right before its MFMA and waits
        // for it, which one or two wavefronts a SIMD do not cover.
        Vec16 kf[kTiles][kHeadDim / kKBlock];
#pragma unroll
        for (int kt = 0; kt < kTiles; ++kt) {
#pragma unroll
            for (int kb = 0; kb < kHeadDim / kKBlock; ++kb) {
                kf[kt][kb] = load16(keys + (kt * kEdge + row) * kKeyPitch + kb * kKBlock + 8 * half);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        Acc x[kTiles];
#pragma unroll
        for (int kb = 0; kb < kHeadDim / kKBlock; ++kb) {
#pragma unroll
            for (int kt = 0; kt < kTiles; ++kt) {
                x[kt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(gemm::bf16x8, kf[kt][kb]),
                                                               __builtin_bit_cast(gemm::bf16x8, q[kb]),
                                                               kb == 0 ? Acc{} : x[kt], 0, 0, 0);
            }
        }
        Vec16 vf[2 * kTiles][2];
#pragma unroll
        for (int kb = 0; kb < 2 * kTiles; ++kb) {
#pragma unroll
            for (int d = 0; d < 2; ++d) {
                vf[kb][d] = value_fragment(values, kb, d * kEdge, lane);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        float block = -INFINITY;
#pragma unroll
        for (int kt = 0; kt < kTiles; ++kt) {
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int key = kt * kEdge + Mma<std::uint16_t>::column(lane, i / 4) + i % 4;
                if (kMasked && key >= valid) {
                    x[kt][i] = -INFINITY;
                }
                block = fmaxf(block, x[kt][i]);
            }
        }
        block = combine_halves(block, Max2{});
        float factor = 1.0F;
        if (running.raise(block, factor)) {
#pragma unroll
            for (int d = 0; d < 2; ++d) {
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    out[d][i] *= factor;
                }
            }
        }
        float sum = 0.F;
#pragma unroll
        for (int kt = 0; kt < kTiles; ++kt) {
            float part[4] = {0.F, 0.F, 0.F, 0.F};
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                x[kt][i] = running.weight(x[kt][i]);
                part[i % 4] += x[kt][i];
            }
            sum += (part[0] + part[1]) + (part[2] + part[3]);
        }
        running.sum += sum;
        // The weights as the second MFMA operand (attention_bf16.hip): runs
        // 2 s and 2 s + 1 traded by halves between lanes l and l ^ 32.
#pragma unroll
        for (int kt = 0; kt < kTiles; ++kt) {
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                Vec16 weights;
#pragma unroll
                for (int w = 0; w < 2; ++w) {
                    const std::uint32_t first = pack_bf16x2(x[kt][8 * s + 2 * w], x[kt][8 * s + 2 * w + 1]);
                    const std::uint32_t second = pack_bf16x2(x[kt][8 * s + 4 + 2 * w], x[kt][8 * s + 4 + 2 * w + 1]);
                    const auto swapped = __builtin_amdgcn_permlane32_swap(first, second, false, false);
                    weights.w[w] = swapped[0];
                    weights.w[2 + w] = swapped[1];
                }
#pragma unroll
                for (int d = 0; d < 2; ++d) {
                    Mma<std::uint16_t>::run(out[d], vf[2 * kt + s][d], weights);
                }
            }
        }
    };

    walk_blocks<kBlockKeys, kEdge, kPerThread>(tokens, part, live, prefetch, commit, step);
    float sums[32];
#pragma unroll
    for (int i = 0; i < 32; ++i) {
        sums[i] = out[i / 16][i % 16];
    }
    combine_parts(reinterpret_cast<float*>(lds), wave, lane, running, sums);
    if (!live || part > 0) {
        return;
    }
    const float total = combine_halves(running.sum, Add2{});
    const float inverse = 1.0F / total;
    std::uint16_t* const rows = context + (static_cast<std::int64_t>(image) * tokens + query0) * embed + head * kHeadDim;
    // The row anew, from the hardware's lane number: kept over the walk it would
    // be the register that costs the third wavefront a SIMD.
    const int out_row = static_cast<int>(__builtin_amdgcn_mbcnt_hi(~0U, __builtin_amdgcn_mbcnt_lo(~0U, 0U))) % kEdge;
    const bool inside = query0 + out_row < tokens;
    const std::uint64_t bad = __ballot(inside && unusable(total, sums));
    std::uint32_t again = static_cast<std::uint32_t>(bad | (bad >> kEdge)); // bit: row of the tile
    if (inside && (again >> out_row & 1U) == 0) {
        std::uint16_t* const destination = rows + static_cast<std::int64_t>(out_row) * embed;
#pragma unroll
        for (int d = 0; d < 2; ++d) {
#pragma unroll
            for (int run = 0; run < 4; ++run) {
                uint2 bits;
                bits.x = pack_bf16x2(sums[16 * d + 4 * run] * inverse, sums[16 * d + 4 * run + 1] * inverse);
                bits.y = pack_bf16x2(sums[16 * d + 4 * run + 2] * inverse, sums[16 * d + 4 * run + 3] * inverse);
                *reinterpret_cast<uint2*>(destination + d * kEdge + Mma<std::uint16_t>::column(lane, run)) = bits;
            }
        }
    }
    for (; __builtin_expect(again != 0, 0); again &= again - 1) {
        const int r = __builtin_ctz(again);
        attend_normalised(q_base, rows + static_cast<std::int64_t>(r) * embed, query0 + r, tokens, qkv_row, embed);
    }
}

// -- fp32 -----------------------------------------------------------------------

constexpr int kEdgeF32 = 16;
constexpr int kBlockKeysF32 = 64;
constexpr int kPitch = kHeadDim + 4;  // floats per LDS row, conflict-free fragment reads
constexpr int kBuffer = 2 * kBlockKeysF32 * kPitch;  // K, then V
constexpr std::size_t kLdsF32 = 2 * kBuffer * sizeof(float);

__global__ __launch_bounds__(kThreads, 2) void attention_long_f32_kernel(const float* __restrict__ qkv,
                                                                      float* __restrict__ context, int heads,
                                                                      int tokens, int pairs, int groups) {
    using gemm::floatx4;
    extern __shared__ Vec16 lds_vectors[];
    float* const lds = reinterpret_cast<float*>(lds_vectors);
    const Place at = place(groups);
    if (at.pair >= pairs) {
        return;  // the whole workgroup, before any barrier
    }
    const int t = static_cast<int>(threadIdx.x);
    const int lane = lane_id();
    const int wave = t / kWave;
    const int row = lane % kEdgeF32;
    const int group = lane / kEdgeF32;
    const int image = at.pair / heads;
    const int head = at.pair - image * heads;
    const int embed = heads * kHeadDim;
    const std::int64_t qkv_row = 3 * static_cast<std::int64_t>(embed);
    const float* const q_base = qkv + static_cast<std::int64_t>(image) * tokens * qkv_row + head * kHeadDim;
    const auto q_resource = gemm::buffer_resource(q_base);
    const auto kv_resource = gemm::buffer_resource(q_base + embed);  // V follows K by embed
    auto load = [&](__amdgpu_buffer_rsrc_t resource, std::int64_t element, bool inside) {
        return gemm::buffer_load16(resource, inside ? static_cast<unsigned int>(element * 4) : gemm::kOutside);
    };

    const int part = wave % kSplit;
    const int query0 = (at.group * kTilesPerGroup + wave / kSplit) * kEdgeF32;
    const int query = query0 + row;
    const bool live = query0 < tokens;  // the others still stage K and V

    Vec16 q[kHeadDim / 16];
#pragma unroll
    for (int kb = 0; kb < kHeadDim / 16; ++kb) {
        q[kb] = load(q_resource, query * qkv_row + 16 * kb + 4 * group, query < tokens);
    }

    // A block's K and V: 1024 16-byte quads, four a thread (K's first).
    constexpr int kQuads = kHeadDim / 4;
    constexpr int kPerThread = 2 * kBlockKeysF32 * kQuads / kThreads;
    constexpr int kKeyStep = kThreads / kQuads;
    static_assert(2 * kBlockKeysF32 * kQuads % kThreads == 0 && kPerThread % 2 == 0, "whole quads per thread");
    const int quad_key = t / kQuads;
    const int quad_dim = 4 * (t % kQuads);
    auto prefetch = [&](Vec16 (&ahead)[kPerThread], int first_key) {
#pragma unroll
        for (int i = 0; i < kPerThread; ++i) {
            const int key = first_key + quad_key + kKeyStep * (i % (kPerThread / 2));
            ahead[i] = load(kv_resource, key * qkv_row + quad_dim + (i < kPerThread / 2 ? 0 : embed), key < tokens);
        }
    };
    auto commit = [&](const Vec16 (&ahead)[kPerThread], int buffer) {
        float* const keys = lds + buffer * kBuffer;
#pragma unroll
        for (int i = 0; i < kPerThread; ++i) {
            const int key = quad_key + kKeyStep * (i % (kPerThread / 2));
            store16(keys + (i < kPerThread / 2 ? 0 : kBlockKeysF32 * kPitch) + key * kPitch + quad_dim, ahead[i]);
        }
    };

    Running running;
    floatx4 out[kHeadDim / 16] = {};

    // One block: kTiles 16-key tiles, of which @p valid keys are real when
    // kMasked. A lane holds its query's keys 4 group .. + 3 of each tile,
    // which is what the weights.V MFMA takes from it.
    auto step = [&](auto tiles, auto masked, int buffer, int valid) {
        constexpr int kTiles = decltype(tiles)::value;
        constexpr bool kMasked = decltype(masked)::value;
        const float* const keys = lds + buffer * kBuffer + part * (kBlockKeysF32 / kSplit) * kPitch;
        const float* const values = keys + kBlockKeysF32 * kPitch;
        // K fragments a tile ahead of their MFMAs, V's likewise below: with one
        // or two wavefronts a SIMD an LDS read that is waited for at once
        // leaves the matrix pipe idle for its latency.
        auto read_keys = [&](Vec16 (&k)[kHeadDim / 16], int jt) {
#pragma unroll
            for (int kb = 0; kb < kHeadDim / 16; ++kb) {
                k[kb] = load16(keys + (16 * jt + row) * kPitch + 16 * kb + 4 * group);
            }
        };
        auto read_values = [&](float (&v)[4][kHeadDim / 16], int jt) {
            const float* const from = values + (16 * jt + 4 * group) * kPitch + row;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
#pragma unroll
                for (int dt = 0; dt < kHeadDim / 16; ++dt) {
                    v[e][dt] = from[e * kPitch + 16 * dt];
                }
            }
        };
        floatx4 x[kTiles];
        Vec16 kf[2][kHeadDim / 16];
        float vf[2][4][kHeadDim / 16];
        read_keys(kf[0], 0);
#pragma unroll
        for (int jt = 0; jt < kTiles; ++jt) {
            if (jt + 1 < kTiles) {
                read_keys(kf[(jt + 1) & 1], jt + 1);
            } else {
                read_values(vf[0], 0);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int kb = 0; kb < kHeadDim / 16; ++kb) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    x[jt] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                        __uint_as_float(kf[jt & 1][kb].w[e]), __uint_as_float(q[kb].w[e]),
                        kb == 0 && e == 0 ? floatx4{0.F, 0.F, 0.F, 0.F} : x[jt], 0, 0, 0);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        float block = -INFINITY;
#pragma unroll
        for (int jt = 0; jt < kTiles; ++jt) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                if (kMasked && 16 * jt + 4 * group + r >= valid) {
                    x[jt][r] = -INFINITY;
                }
                block = fmaxf(block, x[jt][r]);
            }
        }
        block = combine_rows<32>(combine_rows<16>(block, Max2{}), Max2{});
        float factor = 1.0F;
        if (running.raise(block, factor)) {
#pragma unroll
            for (int dt = 0; dt < kHeadDim / 16; ++dt) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    out[dt][r] *= factor;
                }
            }
        }
#pragma unroll
        for (int jt = 0; jt < kTiles; ++jt) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                x[jt][r] = running.weight(x[jt][r]);
            }
            running.sum += (x[jt][0] + x[jt][1]) + (x[jt][2] + x[jt][3]);
        }
#pragma unroll
        for (int jt = 0; jt < kTiles; ++jt) {
            if (jt + 1 < kTiles) {
                read_values(vf[(jt + 1) & 1], jt + 1);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
#pragma unroll
                for (int dt = 0; dt < kHeadDim / 16; ++dt) {
                    out[dt] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[jt & 1][e][dt], x[jt][e], out[dt], 0, 0, 0);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    walk_blocks<kBlockKeysF32, kEdgeF32, kPerThread>(tokens, part, live, prefetch, commit, step);
    float sums[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        sums[i] = out[i / 4][i % 4];
    }
    combine_parts(lds, wave, lane, running, sums);
    if (!live || part > 0) {
        return;
    }
    const float total = combine_rows<32>(combine_rows<16>(running.sum, Add2{}), Add2{});
    const float inverse = 1.0F / total;
    float* const rows = context + (static_cast<std::int64_t>(image) * tokens + query0) * embed + head * kHeadDim;
    std::uint64_t bad = __ballot(query < tokens && unusable(total, sums));
    bad |= bad >> 32;
    std::uint32_t again = static_cast<std::uint32_t>(bad | (bad >> kEdgeF32)) & 0xFFFFU; // bit: row of the tile
    if (query < tokens && (again >> row & 1U) == 0) {
        // Lane holds context[query][16 dt + 4 group .. + 3].
        float* const destination = rows + static_cast<std::int64_t>(row) * embed + 4 * group;
#pragma unroll
        for (int dt = 0; dt < kHeadDim / 16; ++dt) {
            floatx4 value;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                value[r] = sums[4 * dt + r] * inverse;
            }
            *reinterpret_cast<floatx4*>(destination + 16 * dt) = value;
        }
    }
    for (; __builtin_expect(again != 0, 0); again &= again - 1) {
        const int r = __builtin_ctz(again);
        attend_normalised(q_base, rows + static_cast<std::int64_t>(r) * embed, query0 + r, tokens, qkv_row, embed);
    }
}

/// Workgroups: a pair's groups of two query tiles, pairs rounded up to the
/// XCDs (a workgroup past the last pair leaves at once).
unsigned int grid_size(std::int64_t pairs, int groups) {
    return static_cast<unsigned int>((pairs + 7) / 8 * 8 * groups);
}

} // namespace

bool attention_long_supported(std::int64_t pairs, int tokens, int heads, int head_dim, int element_size) {
    // An image's rows within a buffer load's 32-bit offsets, the grid within
    // 31 bits.
    return head_dim == kHeadDim && tokens > 0 && heads > 0 && pairs > 0 &&
           static_cast<std::int64_t>(tokens) * 3 * heads * head_dim * element_size <= 0x7FFFFFF0 &&
           (pairs + 7) / 8 * 8 * ((tokens + 15) / 16) <= 0x7FFFFFFF;
}

hipError_t attention_long_f32(const float* qkv, float* context, int images, int heads, int tokens,
                              hipStream_t stream) {
    const std::int64_t pairs = static_cast<std::int64_t>(images) * heads;
    if (!attention_long_supported(pairs, tokens, heads, kHeadDim, 4)) {
        return hipErrorInvalidValue;
    }
    constexpr int kQueries = kTilesPerGroup * kEdgeF32;
    const int groups = (tokens + kQueries - 1) / kQueries;
    static std::atomic<std::uint64_t> opted_in{0};
    if (const hipError_t opted = allow_lds(reinterpret_cast<const void*>(attention_long_f32_kernel), kLdsF32, opted_in);
        opted != hipSuccess) {
        return opted;
    }
    attention_long_f32_kernel<<<grid_size(pairs, groups), kThreads, kLdsF32, stream>>>(
        qkv, context, heads, tokens, static_cast<int>(pairs), groups);
    return hipGetLastError();
}

hipError_t attention_long_bf16(const std::uint16_t* qkv, std::uint16_t* context, int images, int heads,
                               int tokens, hipStream_t stream) {
    const std::int64_t pairs = static_cast<std::int64_t>(images) * heads;
    if (!attention_long_supported(pairs, tokens, heads, kHeadDim, 2)) {
        return hipErrorInvalidValue;
    }
    constexpr int kQueries = kTilesPerGroup * kEdge;
    const int groups = (tokens + kQueries - 1) / kQueries;
    attention_long_bf16_kernel<<<grid_size(pairs, groups), kThreads, 0, stream>>>(
        qkv, context, heads, tokens, static_cast<int>(pairs), groups);
    return hipGetLastError();
}

} // namespace cuvit::detail

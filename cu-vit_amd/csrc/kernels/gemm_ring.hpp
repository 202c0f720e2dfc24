// The GEMM for products with B given as [N, K] that the persistent bf16 kernel
// (gemm_dma.hpp) and the fp32 panels (gemm_panel.hpp) do not take: in bf16 those
// with too few tiles for the persistent kernel or no whole 256-column tiles. One
// tile per workgroup, operands brought into an LDS ring by direct-to-LDS loads.
//
// What bounds these. Tiles are few and K is short (1 to 48 stages of 64), so
// a tile's time is the latency of its first loads, its waits for a stage and its
// epilogue: at 8224 x 768 x 768 in bf16 with operands from HBM the wavefronts
// wait 63% of their cycles, the MFMAs are busy 15% and the LDS 14%. In fp32 with
// several tiles a CU it is the MFMAs (58% busy at 1576 x 2304 x 768). Loads
// through registers (gemm_kernel.hpp) hold registers and add a write instruction
// per 16 bytes; here the loads land by themselves and two stages per workgroup
// leave room for two (128 x 128) to four (64 x 64) workgroups per CU, which
// cover each other's waits. So two stages are the faster of most tiles, and
// more where little else covers the waits: bf16 three for 64 x 64 tiles alone on
// their CUs or two a CU with a long K and for 128 x 128 tiles alone on their CUs
// (4616 x 768 x 3072: 31 -> 27 us), four for 64 x 32 tiles alone; fp32 three for
// 32 x 16 tiles alone and for 32 x 32 tiles with K above 128 (gemm_choice.hpp has
// the rules). Eight wavefronts of 32 x 64 beat four of 64 x 64 on the 128 x 128
// tile (4616 x 2304 x 768: 24.7 against 25.7 us).
// Before (gemm_kernel.hpp and others since gone) and now, operands in the caches,
// one card, us; bf16:
//   4616 x 1152 x 384          18.4 -> 10.7    197 x 768 x 768 (+=)    8.9 -> 4.9
//   4616 x 384 x 1536 (+=)     18.2 -> 12.5    1576 x 2304 x 768      17.9 -> 10.9
//   4616 x 1536 x 384 (GELU)   18.6 -> 14.9    8224 x 768 x 768       19.0 -> 16.2
//   6304 x 192 x 768 (+=)      11.9 ->  7.4    12608 x 1152 x 384     38.7 -> 20.5
// and fp32:
//   197 x 192 x 768 (+=)        8.7 ->  6.8    577 x 577 x 64 x 24    32.2 -> 21.6
//   788 x 3072 x 768 (GELU)    43.9 -> 40.4    3152 x 768 x 3072      140  -> 128
//
// With kAhead a stage's fragments are read during the stage before, and its
// loads go out between two k-blocks' MFMAs: a wavefront waits about 85 cycles
// to issue one, which its MFMAs in flight then cover. It pays where few
// wavefronts share a SIMD, and costs the registers of a second set. With
// kLoaders as many wavefronts again do nothing but load, for tiles alone on
// their CU.
//
// Stages are rows of 128 bytes (64 bf16 or 32 fp32 of k): chunk c of row r sits
// in 16-byte slot c ^ ((r >> 1) & 7) of its row, conflict-free for the fragment
// reads (bf16 lane l: row l % 32, chunk 2 kb + l / 32; fp32: row l % 16, chunk 4
// kb + l / 16). One buffer_load_dwordx4 ... lds moves eight rows; every loading
// wavefront loads the same number of pieces of A and of B for each stage and
// waits for its own (vmcnt, the newest kSlots - 2 stages
// staying in flight) before the stage's barrier. Loads past the last stage go
// out too, with an offset past the descriptor's range (zeros, no traffic), so
// that the count in flight is the same in every trip.
//
// Epilogue and arithmetic of the bf16 kernel are gemm_dma.hpp's: 32 rows at a
// time through the wavefront's own piece of the drained ring, stored as 16-byte
// pieces (8 bytes or single elements where C's rows are not so aligned); the same
// MFMA over the same K order, then alpha, bias, addend, GELU, old C, one
// rounding, so the results are bitwise those of the other kernels of its type,
// as the fp32 kernel's are. Old C is read before the k loop.
#pragma once

#include "gemm_dma.hpp"

namespace cuvit::detail::gemm {

/// WM x WN wavefronts of TM x TN MFMA tiles of type @p T (bf16 32 x 32, fp32
/// 16 x 16), Slots stages in the ring.
template <typename T, int WM, int WN, int TM, int TN, int Slots, bool Ahead = false, bool Loaders = false>
struct RingShape {
    static constexpr bool kAhead = Ahead;
    static constexpr bool kLoaders = Loaders;
    static_assert(Ahead || !Loaders, "loading wavefronts go with fragments read ahead");
    static constexpr int kEdge = Mma<T>::kEdge;
    static constexpr int kWaves = WM * WN;
    static constexpr int kThreads = kWave * kWaves * (Loaders ? 2 : 1);
    static constexpr int kWN = WN;
    static constexpr int kTM = TM;
    static constexpr int kTN = TN;
    static constexpr int kBM = kEdge * WM * TM;
    static constexpr int kBN = kEdge * WN * TN;
    static constexpr int kSlots = Slots;
    static constexpr int kRowBytes = 128;                    // of a stage, either type
    static constexpr int kBK = kRowBytes / sizeof(T);        // k of a stage
    static constexpr int kChunks = kRowBytes / 16;           // 16-byte chunks per row
    static constexpr int kLoadRows = 1024 / kRowBytes;       // rows of one load instruction
    static constexpr int kLoadsA = kBM / kLoadRows / kWaves; // per wavefront and stage
    static constexpr int kLoadsB = kBN / kLoadRows / kWaves;
    static constexpr int kLoads = kLoadsA + kLoadsB;
    static constexpr int kStageBytes = (kBM + kBN) * kRowBytes;
    static constexpr int kBiasOffset = Slots * kStageBytes;
    static constexpr int kLdsBytes = kBiasOffset + kBN * 4;
    static constexpr int kStagingBytes = kEdge * TN * 64; // bf16: 32 rows of a wavefront's columns
    static_assert(kBM % (kLoadRows * kWaves) == 0 && kBN % (kLoadRows * kWaves) == 0,
                  "every wavefront loads whole pieces of both operands");
    static_assert(kBN <= kThreads, "one thread per bias value");
    static_assert(kWaves * kLoadRows % 16 == 0, "a lane's placement is the same in all its pieces");
    static_assert(Slots >= 2 && (Slots - 1) * kLoads <= 63, "vmcnt");
    static_assert(kBiasOffset >= kWaves * kStagingBytes, "the ring holds every wavefront's staging");
    static_assert(kLdsBytes <= 160 * 1024, "LDS");

    __device__ __forceinline__ static int place(int row, int chunk) { return chunk ^ ((row >> 1) & 7); }
};

/// The batch entry of a workgroup and the number of its tile there. With whole
/// entries to an XCD (TileMap, px < 0) the grid is 8 x tiles x entries / 8, whose
/// x is the XCD, else tiles x entries; nothing is divided.
struct RingSpot {
    int entry;
    int tile;
};

__device__ __forceinline__ RingSpot ring_spot(const TileMap& map, int first_entry) {
    const int x = static_cast<int>(blockIdx.x);
    const int y = static_cast<int>(blockIdx.y);
    return map.px < 0 ? RingSpot{first_entry + 8 * static_cast<int>(blockIdx.z) + x, y} : RingSpot{first_entry + y, x};
}

/// The tile of a workgroup, or false where its XCD's block of the tile grid
/// (TileMap) has fewer tiles, or the batch fewer entries, than the grid allows.
template <typename S>
__device__ __forceinline__ bool ring_tile(const GemmArgs& args, const TileMap& map, const RingSpot& spot, int& row0,
                                          int& col0) {
    const int tiles_n = (args.n + S::kBN - 1) / S::kBN;
    int tile_m = spot.tile / tiles_n;
    int tile_n = spot.tile % tiles_n;
    if (map.px > 0) {
        const int tiles_m = (args.m + S::kBM - 1) / S::kBM;
        // px py = 8, both powers of two: the split points as shifts, since a
        // tile has little time for five integer divisions.
        const int block = static_cast<int>(blockIdx.x & 7U);
        const int index = static_cast<int>(blockIdx.x >> 3);
        const int log_m = 31 - __builtin_clz(static_cast<unsigned int>(map.px));
        const int log_n = 3 - log_m;
        const int part_m = block >> log_n;
        const int part_n = block & (map.py - 1);
        const int m_lo = tiles_m * part_m >> log_m;
        const int m_hi = tiles_m * (part_m + 1) >> log_m;
        const int n_lo = tiles_n * part_n >> log_n;
        const int n_hi = tiles_n * (part_n + 1) >> log_n;
        const int width = n_hi - n_lo;
        if (index >= (m_hi - m_lo) * width) {
            return false;
        }
        tile_m = m_lo + index / width;
        tile_n = n_lo + index % width;
    }
    row0 = __builtin_amdgcn_readfirstlane(tile_m * S::kBM);
    col0 = __builtin_amdgcn_readfirstlane(tile_n * S::kBN);
    return spot.entry < args.count;
}

/// The stage loads of one wavefront: piece p of wavefront w holds stage rows
/// (p kWaves + w) kLoadRows .. + kLoadRows; lane l lands in row l / kChunks,
/// slot l % kChunks of it. Rows past the problem and k past K read as zero.
template <typename T, typename S> struct RingLoads {
    sgpr4 resource_a;
    sgpr4 resource_b;
    unsigned int offset_a;
    unsigned int offset_b;
    unsigned int step_a;
    unsigned int step_b;
    unsigned int lds_base;
    int load_k;
    int depth;

    __device__ __forceinline__ RingLoads(const T* a, const T* b, const GemmArgs& args, int row0, int col0,
                                         int wave, int lane, unsigned int lds) {
        constexpr int kSize = static_cast<int>(sizeof(T));
        const int rows_a = min(args.m - row0, S::kBM);
        const int rows_b = min(args.n - col0, S::kBN);
        resource_a = scalar_resource(a + static_cast<std::int64_t>(row0) * args.lda,
                                     static_cast<unsigned int>(rows_a * args.lda * kSize));
        resource_b = scalar_resource(b + static_cast<std::int64_t>(col0) * args.ldb,
                                     static_cast<unsigned int>(rows_b * args.ldb * kSize));
        const int load_row = wave * S::kLoadRows + lane / S::kChunks;
        load_k = 16 / kSize * S::place(load_row, lane % S::kChunks);
        offset_a = static_cast<unsigned int>((load_row * args.lda + load_k) * kSize);
        offset_b = static_cast<unsigned int>((load_row * args.ldb + load_k) * kSize);
        step_a = static_cast<unsigned int>(__builtin_amdgcn_readfirstlane(S::kWaves * S::kLoadRows * args.lda * kSize));
        step_b = static_cast<unsigned int>(__builtin_amdgcn_readfirstlane(S::kWaves * S::kLoadRows * args.ldb * kSize));
        lds_base = lds + static_cast<unsigned int>(wave * 1024);
        depth = args.k;
    }

    /// Stage @p g into ring slot @p slot.
    __device__ __forceinline__ void issue(int g, int slot) const {
        const int k0 = g * S::kBK;
        const bool inside = load_k + k0 < depth;
        const unsigned int at = static_cast<unsigned int>(k0) * static_cast<unsigned int>(sizeof(T));
        const unsigned int from_a = inside ? offset_a + at : kOutside;
        const unsigned int from_b = inside ? offset_b + at : kOutside;
        const unsigned int m0 = lds_base + static_cast<unsigned int>(slot * S::kStageBytes);
#pragma unroll
        for (int p = 0; p < S::kLoadsA; ++p) {
            load_to_lds(m0 + static_cast<unsigned int>(p * S::kWaves * 1024),
                        from_a + static_cast<unsigned int>(p) * step_a, resource_a);
        }
#pragma unroll
        for (int p = 0; p < S::kLoadsB; ++p) {
            load_to_lds(m0 + static_cast<unsigned int>(S::kBM * S::kRowBytes + p * S::kWaves * 1024),
                        from_b + static_cast<unsigned int>(p) * step_b, resource_b);
        }
    }
};

/// s_waitcnt lgkmcnt(0) as an instruction that the compiler knows, where the
/// barriers' waits are text to it: it then neither waits again for fragments
/// that are there, nor, with a kernel argument's load in flight before the loop
/// (scalar loads share the counter and return in any order), for all of the next
/// stage's before the first MFMA of each (48 x 768 x 3072: 9.2 us, 8.3 without).
/// The barriers' own wait for it stays, and holds whatever the compiler moves.
__device__ __forceinline__ void wait_fragments() { __builtin_amdgcn_s_waitcnt(0xC07F); }

/// The k loop: acc += A.B^T over @p stages stages, the ring kept kSlots - 1
/// stages ahead. On return no load is in flight and no wavefront reads the
/// ring.
template <typename T, typename S>
__device__ __forceinline__ void ring_multiply(const RingLoads<T, S>& loads, const unsigned char* lds, int wave_m,
                                              int wave_n, int lane, bool loading, int stages,
                                              typename Mma<T>::Acc (&acc)[S::kTM][S::kTN]) {
    constexpr int E = S::kEdge;
    constexpr int kBlocks = S::kBK / kKBlock<T>;  // k-blocks per stage
    constexpr int kPerBlock = kWave / E;          // 16-byte chunks of a row per k-block
    const unsigned int a_fragment = static_cast<unsigned int>((wave_m * E * S::kTM + lane % E) * S::kRowBytes);
    const unsigned int b_fragment =
        static_cast<unsigned int>((S::kBM + wave_n * E * S::kTN + lane % E) * S::kRowBytes);
    // E rows further on the placement is the same (its period is 16 rows).
    unsigned int fragment_column[kBlocks];
#pragma unroll
    for (int kb = 0; kb < kBlocks; ++kb) {
        fragment_column[kb] = static_cast<unsigned int>(S::place(lane % E, kPerBlock * kb + lane / E) * 16);
    }
#pragma unroll
    for (int i = 0; i < S::kTM; ++i)
#pragma unroll
        for (int j = 0; j < S::kTN; ++j)
#pragma unroll
            for (int r = 0; r < 4 * Mma<T>::kRuns; ++r)
                acc[i][j][r] = 0.F;
    struct Fragments {
        Vec16 a[kBlocks][S::kTM];
        Vec16 b[kBlocks][S::kTN];
    };
    auto read_block = [&](const unsigned char* base, int kb, Vec16 (&fa)[S::kTM], Vec16 (&fb)[S::kTN]) {
#pragma unroll
        for (int i = 0; i < S::kTM; ++i)
            fa[i] = load16(base + a_fragment + i * E * S::kRowBytes + fragment_column[kb]);
#pragma unroll
        for (int j = 0; j < S::kTN; ++j)
            fb[j] = load16(base + b_fragment + j * E * S::kRowBytes + fragment_column[kb]);
    };
    auto multiply_block = [&](const Vec16 (&fa)[S::kTM], const Vec16 (&fb)[S::kTN]) {
#pragma unroll
        for (int i = 0; i < S::kTM; ++i)
#pragma unroll
            for (int j = 0; j < S::kTN; ++j)
                Mma<T>::run(acc[i][j], fb[j], fa[i]);
    };
    if constexpr (S::kAhead) {
        // A stage's fragments are read during the MFMAs of the stage before it
        // (two register sets), so a stage costs its MFMAs and a barrier, with
        // no LDS latency between them; its slot is free one stage earlier and
        // the ring runs kSlots stages ahead of the registers.
        Fragments set[2];
        auto read = [&](Fragments& f, int slot) {
#pragma unroll
            for (int kb = 0; kb < kBlocks; ++kb)
                read_block(lds + slot * S::kStageBytes, kb, f.a[kb], f.b[kb]);
        };
        if (!S::kLoaders || loading) {
#pragma unroll
            for (int g = 0; g < S::kSlots; ++g) {
                loads.issue(g, g);
            }
        }
        if (S::kLoaders && loading) {
            // Half of the wavefronts only load: what a load costs at issue then
            // delays no MFMA. A stage's slot is free after the barrier that
            // follows its fragment reads.
            asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" : : "n"((S::kSlots - 1) * S::kLoads) : "memory");
            int slot = 0;
            for (int g = 0; g < stages; ++g) {
                asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" : : "n"((S::kSlots - 2) * S::kLoads) : "memory");
                loads.issue(g + S::kSlots, slot);
                slot = slot + 1 == S::kSlots ? 0 : slot + 1;
            }
            stage_barrier(true);
            return;
        }
        wait_fragments(); // (any scalar load)
        if constexpr (S::kLoaders) {
            asm volatile("s_barrier" : : : "memory");
        } else {
            asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" : : "n"((S::kSlots - 1) * S::kLoads) : "memory");
        }
        read(set[0], 0);
        int slot = 0;
        auto step = [&](int g, Fragments& now, Fragments& next) {
            // Stage g + 1 landed, and every wavefront holds stage g in registers.
            wait_fragments();
            if constexpr (S::kLoaders) {
                asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" : : : "memory");
            } else {
                asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier"
                             :
                             : "n"((S::kSlots - 2) * S::kLoads)
                             : "memory");
            }
            const int free_slot = slot;
            slot = slot + 1 == S::kSlots ? 0 : slot + 1;
            read(next, slot);
            __builtin_amdgcn_sched_barrier(0);
            multiply_block(now.a[0], now.b[0]);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (!S::kLoaders) {
                loads.issue(g + S::kSlots, free_slot); // while the MFMAs before run
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int kb = 1; kb < kBlocks; ++kb)
                multiply_block(now.a[kb], now.b[kb]);
            __builtin_amdgcn_sched_barrier(0);
        };
        for (int g = 0; g < stages; g += 2) { // K's spans are whole pairs of stages
            step(g, set[0], set[1]);
            step(g + 1, set[1], set[0]);
        }
    } else {
#pragma unroll
        for (int g = 0; g < S::kSlots - 1; ++g) {
            loads.issue(g, g);
        }
        int slot = 0;
        int free_slot = S::kSlots - 1;
        for (int g = 0; g < stages; ++g) {
            // Stage g landed (each wavefront waits for its own pieces) and every
            // wavefront is done reading stage g - 1, whose slot is refilled.
            wait_fragments();
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"((S::kSlots - 2) * S::kLoads) : "memory");
            loads.issue(g + S::kSlots - 1, free_slot);
#pragma unroll
            for (int kb = 0; kb < kBlocks; ++kb) {
                Vec16 fa[S::kTM];
                Vec16 fb[S::kTN];
                read_block(lds + slot * S::kStageBytes, kb, fa, fb);
                multiply_block(fa, fb);
            }
            free_slot = slot;
            slot = slot + 1 == S::kSlots ? 0 : slot + 1;
        }
    }
    stage_barrier(true);
}

/// The epilogue's parts as in gemm_dma_kernel (alpha is always multiplied in:
/// 1 * x is x, bit for bit). Batch entries from @p first_entry on; with
/// args.rows_per_entry > 0 the rows are entries run as one problem. @p c_run of
/// C's elements are read and written at once: 8, 4 where N and its rows are
/// whole 8-byte pieces only (6304 x 2308 x 768 accumulating 72 -> 41 us against
/// one by one, 196 x 196 x 64 in 96 entries 18.4 -> 9.4), else 1.
template <typename S, bool kBias, bool kGelu, bool kAccumulate, bool kAddend = false>
__global__ __launch_bounds__(S::kThreads) void gemm_ring_kernel(const std::uint16_t* __restrict__ a,
                                                                const std::uint16_t* __restrict__ b,
                                                                const float* __restrict__ bias,
                                                                std::uint16_t* c, GemmArgs args,
                                                                TileMap map, int c_run, int first_entry) {
    constexpr int BM = S::kBM;
    constexpr int BN = S::kBN;
    constexpr int TM = S::kTM;
    constexpr int TN = S::kTN;
    const RingSpot spot = ring_spot(map, first_entry);
    const Offsets entry = entry_offsets(args, spot.entry);
    a += entry.a;
    b += entry.b;
    c += entry.c;
    extern __shared__ Vec16 lds_vectors[];
    unsigned char* const lds = reinterpret_cast<unsigned char*>(lds_vectors);
    const unsigned int lds_base = __builtin_amdgcn_readfirstlane(lds_address(lds));

    const int lane = lane_id();
    const int wavefront = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) / kWave);
    const bool loading = S::kLoaders && wavefront >= S::kWaves;
    const int wave = loading ? wavefront - S::kWaves : wavefront;
    const int wave_m = wave / S::kWN;
    const int wave_n = wave % S::kWN;

    int row0, col0;
    if (!ring_tile<S>(args, map, spot, row0, col0)) {
        return; // the whole workgroup, before any barrier
    }

    // Old C, one 16-byte piece per lane and row group, issued ahead of the
    // stage loads (so older than they are in every wait below).
    constexpr int kRowChunks = 4 * TN;                // 16-byte pieces of a wavefront's row
    constexpr int kRowsPerStore = kWave / kRowChunks; // rows one store instruction covers
    constexpr int kStores = 32 / kRowsPerStore;
    const int store_row = lane / kRowChunks;
    const int store_chunk = lane % kRowChunks;
    const int store_col = col0 + wave_n * 32 * TN + 8 * store_chunk;
    auto group_row = [&](int i, int k) {
        return row0 + (wave_m * TM + i) * 32 + kRowsPerStore * k + store_row;
    };
    // Output row -> its element offset in C (in its entry when entries run as one).
    auto c_offset = [&](int row) -> std::int64_t {
        if (args.rows_per_entry > 0) {
            const int index = row / args.rows_per_entry;
            return index * args.stride_c + static_cast<std::int64_t>(row - index * args.rows_per_entry) * args.ldc;
        }
        return static_cast<std::int64_t>(row) * args.ldc;
    };
    Vec16 old_rows[kAccumulate ? TM : 1][kStores];
    if constexpr (kAccumulate) {
        // One branch on c_run for all of them.
        auto read_old = [&](auto read) {
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int k = 0; k < kStores; ++k) {
                    const int row = group_row(i, k);
                    old_rows[i][k] = Vec16{{0U, 0U, 0U, 0U}};
                    if (row < args.m && store_col < args.n) {
                        old_rows[i][k] = read(c + c_offset(row) + store_col);
                    }
                }
        };
        if (__builtin_expect(c_run == 8, 1)) {
            read_old([](const std::uint16_t* from) { return load16(from); });
        } else if (c_run == 4) {
            read_old([&](const std::uint16_t* from) {
                const uint2 first = *reinterpret_cast<const uint2*>(from);
                const uint2 second =
                    store_col + 4 < args.n ? *reinterpret_cast<const uint2*>(from + 4) : make_uint2(0U, 0U);
                return Vec16{{first.x, first.y, second.x, second.y}};
            });
        } else {
            read_old([&](const std::uint16_t* from) { return load_chunk_scalar(from, 0, 0, 1, 0, args.n - store_col); });
        }
    }
    // The tile's bias into LDS (read by the epilogue, many barriers later).
    float* const bias_slot = reinterpret_cast<float*>(lds + S::kBiasOffset);
    if (kBias && static_cast<int>(threadIdx.x) < BN) {
        const int col = col0 + static_cast<int>(threadIdx.x);
        bias_slot[threadIdx.x] = col < args.n ? bias[col] : 0.F;
    }

    const RingLoads<std::uint16_t, S> loads(a, b, args, row0, col0, wave, lane, lds_base);
    floatx16 acc[TM][TN];
    ring_multiply<std::uint16_t, S>(loads, lds, wave_m, wave_n, lane, loading, (args.k + 127) / 128 * (128 / S::kBK), acc);

    if (loading) {
        return; // no barrier follows
    }

    // The drained ring becomes staging.
    unsigned char* const staging = lds + wave * S::kStagingBytes;
    auto staged = [&](int r, int chunk) {
        return staging + r * (64 * TN) + ((chunk ^ ((r >> (TN == 2 ? 1 : 2)) & (kRowChunks - 1))) * 16);
    };
    const int r = lane & 31;
    static_for<TM>([&](auto tile_i) {
        constexpr int i = decltype(tile_i)::value;
        if constexpr (kAccumulate) {
#pragma unroll
            for (int k = 0; k < kStores; ++k) {
                *reinterpret_cast<Vec16*>(staged(kRowsPerStore * k + store_row, store_chunk)) = old_rows[i][k];
            }
        }
        const int row = row0 + (wave_m * TM + i) * 32 + r;
        Vec16 addend_runs[kAddend ? TN * 4 : 1];
        if constexpr (kAddend) {
            const int local = row >= args.m ? 0 : args.rows_per_entry > 0 ? row % args.rows_per_entry : row;
            const float* const addend_row = args.addend + static_cast<std::int64_t>(local) * args.ld_addend;
            static_for<TN * 4>([&](auto run) {
                constexpr int q = decltype(run)::value;
                const int col = col0 + wave_n * 32 * TN + 32 * (q / 4) + Mma<std::uint16_t>::column(lane, q % 4);
                addend_runs[q] = row < args.m && col < args.n ? load16(addend_row + col) : Vec16{{0U, 0U, 0U, 0U}};
            });
        }
        static_for<TN * 4>([&](auto run) {
            constexpr int j = decltype(run)::value / 4;
            constexpr int q = decltype(run)::value % 4;
            uint2* const at = reinterpret_cast<uint2*>(staged(r, 4 * j + q) + 8 * (lane >> 5));
            Vec16 bias_run{{0U, 0U, 0U, 0U}};
            if constexpr (kBias) {
                bias_run = load16(bias_slot + wave_n * 32 * TN + 32 * j + Mma<std::uint16_t>::column(lane, q));
            }
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
#pragma clang fp contract(off)
                float x = args.alpha * acc[i][j][4 * q + e];
                if constexpr (kBias) {
                    x += __uint_as_float(bias_run.w[e]);
                }
                if constexpr (kAddend) {
                    x += __uint_as_float(addend_runs[4 * j + q].w[e]);
                }
                v[e] = kGelu ? gelu(x) : x;
            }
            if constexpr (kAccumulate) {
                const uint2 old = *at;
                v[0] = add_unfused(bf16_to_float(static_cast<std::uint16_t>(old.x & 0xFFFFU)), v[0]);
                v[1] = add_unfused(bf16_to_float(static_cast<std::uint16_t>(old.x >> 16)), v[1]);
                v[2] = add_unfused(bf16_to_float(static_cast<std::uint16_t>(old.y & 0xFFFFU)), v[2]);
                v[3] = add_unfused(bf16_to_float(static_cast<std::uint16_t>(old.y >> 16)), v[3]);
            }
            *at = make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
        });
        auto write = [&](auto store) {
#pragma unroll
            for (int k = 0; k < kStores; ++k) {
                const int out_row = group_row(i, k);
                const Vec16 v = *reinterpret_cast<const Vec16*>(staged(kRowsPerStore * k + store_row, store_chunk));
                if (out_row < args.m && store_col < args.n) {
                    store(c + c_offset(out_row) + store_col, v);
                }
            }
        };
        if (__builtin_expect(c_run == 8, 1)) {
            write([](std::uint16_t* to, const Vec16& v) { store16(to, v); });
        } else if (c_run == 4) {
            write([&](std::uint16_t* to, const Vec16& v) {
                *reinterpret_cast<uint2*>(to) = make_uint2(v.w[0], v.w[1]);
                if (store_col + 4 < args.n) {
                    *reinterpret_cast<uint2*>(to + 4) = make_uint2(v.w[2], v.w[3]);
                }
            });
        } else {
            write([&](std::uint16_t* to, const Vec16& v) {
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    if (store_col + e < args.n) {
                        Elem<std::uint16_t>::store_bits(to + e, v, e);
                    }
                }
            });
        }
    });
}

/// The fp32 kernel: stages 32 deep (two k-blocks of 16), K rounded up to 64 as
/// in the other fp32 kernels, results stored from the registers (a lane holds
/// four consecutive columns, one store at any alignment; a run that N cuts goes
/// element by element).
template <typename S>
__global__ __launch_bounds__(S::kThreads) void gemm_ring_f32_kernel(const float* __restrict__ a,
                                                                    const float* __restrict__ b,
                                                                    const float* __restrict__ bias, float* c,
                                                                    GemmArgs args, TileMap map, int /* c_run: always 4 */,
                                                                    int first_entry) {
    constexpr int TM = S::kTM;
    constexpr int TN = S::kTN;
    constexpr int E = S::kEdge;
    const RingSpot spot = ring_spot(map, first_entry);
    const Offsets entry = entry_offsets(args, spot.entry);
    extern __shared__ Vec16 lds_vectors[];
    unsigned char* const lds = reinterpret_cast<unsigned char*>(lds_vectors);
    const unsigned int lds_base = __builtin_amdgcn_readfirstlane(lds_address(lds));
    const int lane = lane_id();
    const int wavefront = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) / kWave);
    const bool loading = S::kLoaders && wavefront >= S::kWaves;
    const int wave = loading ? wavefront - S::kWaves : wavefront;
    const int wave_m = wave / S::kWN;
    const int wave_n = wave % S::kWN;
    int row0, col0;
    if (!ring_tile<S>(args, map, spot, row0, col0)) {
        return; // the whole workgroup, before any barrier
    }

    // The epilogue's operands ahead of the stage loads: the bias of this
    // lane's runs and old C.
    const int first_row = row0 + wave_m * E * TM + lane % E;
    const int first_col = col0 + wave_n * E * TN + Mma<float>::column(lane, 0);
    float run_bias[TN][4];
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int col = first_col + E * j + r;
            run_bias[j][r] = bias != nullptr && col < args.n ? bias[col] : 0.F;
        }
    auto local_row = [&](int row) { return args.rows_per_entry > 0 ? row % args.rows_per_entry : row; };
    auto c_row = [&](int row) -> float* {
        const std::int64_t from =
            args.rows_per_entry > 0 ? static_cast<std::int64_t>(row / args.rows_per_entry) * args.stride_c : 0;
        return c + entry.c + from + static_cast<std::int64_t>(local_row(row)) * args.ldc;
    };
    floatx4 old[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int row = first_row + E * i;
            const int col = first_col + E * j;
            old[i][j] = floatx4{0.F, 0.F, 0.F, 0.F};
            if (args.accumulate && row < args.m && col + 3 < args.n) {
                old[i][j] = *reinterpret_cast<const floatx4_unaligned*>(c_row(row) + col);
            }
        }

    const RingLoads<float, S> loads(a + entry.a, b + entry.b, args, row0, col0, wave, lane, lds_base);
    floatx4 acc[TM][TN];
    ring_multiply<float, S>(loads, lds, wave_m, wave_n, lane, loading, (args.k + 63) / 64 * (64 / S::kBK), acc);
    if (loading) {
        return; // no barrier follows
    }

#pragma unroll
    for (int i = 0; i < TM; ++i) {
        const int row = first_row + E * i;
        if (row >= args.m) {
            continue;
        }
        const int local = local_row(row);
        float* const to = c_row(row);
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int col = first_col + E * j;
            float value[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                value[r] = col + r < args.n ? epilogue_value(acc[i][j][r], bias != nullptr, run_bias[j][r], local,
                                                             col + r, args)
                                            : 0.F;
            }
            if (col + 3 < args.n) {
                store4(to + col, value, args.accumulate, old[i][j]);
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    if (col + r < args.n) {
                        to[col + r] = args.accumulate ? add_unfused(to[col + r], value[r]) : value[r];
                    }
                }
            }
        }
    }
}

} // namespace cuvit::detail::gemm

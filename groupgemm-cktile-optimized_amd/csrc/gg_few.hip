// Few-row kernel: forward (x w[g]^T) and dgrad (grad_out w[g]) of groups with few rows, 16-bit and
// fp8, where the time is the reading of w or a problem is too small to fill the GPU with large tiles.
//
// What bounds it: w's bytes from HBM when the problem is large, and the latency of one tile's chain
// (first loads, chunks, sums, stores) when it is small. So tiles are small (16-64 rows, 16-64
// columns: many workgroups, 2-3 per CU) and a tile's contraction is split between the W waves of
// its workgroup: wave i takes the 128-byte chunks i, i + W, .. of the rows (consecutive waves read
// consecutive lines), each with MFMAs of its own, and the sums are added through LDS at the end, in
// wave order.
//
// Operands go from global memory to LDS by DMA (buffer_load ... lds, 16 bytes per lane), into a
// ring of S chunks that belongs to the wave alone: it waits for its own loads by count and no
// barrier stands in the K loop. Registers would need no LDS, but an MFMA operand has lane l hold
// row l % 16, and a load whose 4 consecutive lanes touch 4 lines takes the address unit four times
// as long as the DMA's row-by-row order. Rows are 128 bytes in LDS, their 16-byte pieces stored at
// piece ^ (row % 8), so the 8 rows a read pass covers take 8 different slots. Counters: the LDS is
// active 5-12 % of a launch, 5-8 % of that are bank conflicts forward and 30-38 % with transposed reads.
//
// w stored contraction-major (dgrad, MN): a chunk is 64 (fp8: 128) stored rows of the tile's columns,
// read with ds_read_b64_tr_b16 / _b8, which give each lane consecutive contraction values of its
// column; the order of the values within a lane is the one A's fragments have.
//
// Bounds: A's resource ends at the tile's last valid row, B's at its last valid row (MN: at the
// group's last contraction row), so loads past them read zeros; a piece past K (or an MN piece past
// N), which would read the next row, gets an offset past the resource instead. Stores are masked by
// row and column (N % 8 == 0: four columns are all valid or not).
//
// Measured (MI355X, us per launch back to back, the plans that ran before -> this kernel): bf16
// forward 4 x 256 rows, 512 x 1024 12.3 -> 6.4; 36 x 16, 2048 x 1024 35.9 -> 23.4 (6.4 TB/s of w, part of
// it from the Infinity Cache); 1 x 512, 2880 x 2880 28.5 -> 20.3; 3 x 5 (device sizes), 3328 x 12256 130 -> 38;
// fp8 forward 4 x 3, 9840 x 800 14.7 -> 6.0; dgrad bf16 3 x 14, 1208 x 2048 25.3 ->
// 6.0, fp8 32 x 64, 2512 x 768 26.4 -> 17.3. The ring's depth and the waves were swept (29
// combinations of 1-8 row blocks, 1-4 column blocks, 1-16 waves, 1-4 chunks): what pays is many
// small workgroups per CU, not a deep ring (16 rows: 4 waves x 2 chunks, 2 per CU, 29.1 against
// 34.8 with 4 chunks, 1 per CU, on the second shape, w from HBM). More rows per tile than 64 lose to the 128 x 128 tiles: every
// tile stages its own operands, at a fitted 10-22 TB/s over the chip (kFewStageFwd and its like).
#include "gg_few.h"
#include "gg_kernel_impl.h"

namespace gg {
namespace {

typedef short    tr16x4 __attribute__((ext_vector_type(4)));
typedef __bf16   kbf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 kf16x8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) tr16x4 lds_tr16;
typedef __attribute__((address_space(3))) i32x2  lds_i32x2;

template <int VM> __device__ __forceinline__ void wait_vm() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(VM) : "memory"); }
__device__ __forceinline__ void wait_lds() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// Input formats of one instance (FewFormat in gg_kernel.h) as MFMA operands.
template <int FMT> struct Fmt {
    static constexpr bool f8  = FMT >= kFewE4M3;
    static constexpr bool f16 = FMT == kFewF16;
    static constexpr int  es  = f8 ? 1 : 2;
    static constexpr int  kc  = 128 / es; // contraction values per chunk (128 bytes of a row)
    static constexpr bool a_e5m2 = FMT == kFewE5M2 || FMT == kFewE5M2xE4M3;
    static constexpr bool b_e5m2 = FMT == kFewE5M2;
};

template <bool F16> __device__ __forceinline__ f32x4 mma16(const i32x4 &b, const i32x4 &a, const f32x4 &c) {
    if constexpr (F16)
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(kf16x8, b), __builtin_bit_cast(kf16x8, a), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(kbf16x8, b), __builtin_bit_cast(kbf16x8, a), c, 0, 0, 0);
}

template <int FMT, bool MN, int MB, int NB, int W, int S>
__global__ void __launch_bounds__(W * 64) few_gemm_kernel(const KernelArgs args) {
    using F = Fmt<FMT>;
    constexpr int BM = 16 * MB, BN = 16 * NB;
    constexpr int kARegion = BM * 128, kChunk = (BM + BN) * 128; // bytes of one chunk: A, then B
    constexpr int kRing = W * S * kChunk;
    constexpr int kDmaA = kARegion / 1024, kDmaB = BN * 128 / 1024, kDma = kDmaA + kDmaB;
    constexpr int kSumStride = BN + 4; // floats
    constexpr int kSums = W * BM * kSumStride * 4;
    constexpr int kLds = kSums > kRing ? kSums : kRing;
    static_assert(kLds <= 160 * 1024, "LDS");
    static_assert(S >= 1 && S <= 2 && (S - 1) * kDma <= 63, "vmcnt: one chunk behind the current one at most");
    __shared__ __attribute__((aligned(1024))) unsigned char lds[kLds];
    const int tid = static_cast<int>(threadIdx.x), lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);

    // ---- the group table: lane l holds group l (device sizes), or the table in memory ----
    int       total = args.total_tiles;
    LaneGroup lg{};
    if (args.d_lens != nullptr) {
        int first_bad, overflow;
        if (blockIdx.x == 0) { // the header reports 256 x 256 tiles whatever kernel runs
            lane_group_table(args.d_lens, args.d_offs, args.group_num, args.lens_rows,
                             static_cast<int>(cdiv(args.n, kTileN)), 0, lane, &total, &first_bad, &overflow);
            if (tid == 0) {
                args.d_header->total_tiles = total;
                args.d_header->first_bad   = first_bad;
                args.d_header->overflow    = overflow;
                args.d_header->run_tiles   = 0;
            }
        }
        lg = lane_group_table(args.d_lens, args.d_offs, args.group_num, args.lens_rows, args.n_tiles, 0, lane, &total,
                              &first_bad, &overflow, BM);
    } else if (args.d_total != nullptr) {
        total = *to_const_space(args.d_total);
    }
    const int grid = static_cast<int>(gridDim.x);
    for (int t = static_cast<int>(blockIdx.x); t < total; t += grid) {
        // ---- the tile: group g, row tile tm, column tile tn (row tiles innermost, so that the
        // workgroups that share w rows run next to each other on one XCD) ----
        const int L = xcd_remap(t, total, grid, args.n_xcd);
        // The group is the last one whose first tile is at most L (an empty group shares its successor's).
        // A table of more than 64 groups is narrowed to 64 entries first, by 64 evenly spaced ones at a
        // time: every load waits for the one before, and a scan in steps of 64 took a load per 64 groups
        // for every tile (us per launch, scan -> this: 4096 groups of 8 rows, N = 128, K = 256 191 -> 54;
        // the persistent kernel, which scans once per workgroup, 93).
        int first = 0, span = args.group_num;
        if (args.d_lens == nullptr) {
            while (span > 64) {
                const int      step = (span + 63) / 64;
                const bool     live = lane * step < span;
                const int      t0   = args.groups[live ? first + lane * step : first].tile0;
                const uint64_t mask = __ballot(live && t0 <= L); // bit 0 is set: the range's first entry is at most L
                const int      s    = 63 - __builtin_clzll(mask);
                first += s * step;
                span = min(step, span - s * step);
            }
            const GroupEntry e = args.groups[lane < span ? first + lane : first];
            lg.row0  = e.row0;
            lg.m     = e.m;
            lg.tile0 = e.tile0;
        }
        const int s     = 63 - __builtin_clzll(__ballot(lane < span && lg.tile0 <= L));
        const int g     = first + s;
        const int gm    = __builtin_amdgcn_readlane(lg.m, s);
        const int local = L - __builtin_amdgcn_readlane(lg.tile0, s);
        int64_t   row0  = static_cast<int64_t>(static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(lg.row0), s))) |
                       (static_cast<int64_t>(__builtin_amdgcn_readlane(static_cast<int>(lg.row0 >> 32), s)) << 32);
        const int mts = (gm + BM - 1) / BM;
        const int tn = local / mts, tm = local - tn * mts;
        row0 += static_cast<int64_t>(tm) * BM;
        const int mv = min(BM, gm - tm * BM);
        const int N = args.n, K = args.k;

        // ---- resources, bounded by the tile's valid rows (MN: by the group's w) ----
        const int   lda = args.lda * F::es, ldb = args.ldb * F::es; // bytes
        const char *ap  = static_cast<const char *>(args.x) + row0 * lda;
        const char *bp  = static_cast<const char *>(args.w) +
                         (MN ? static_cast<int64_t>(g) * K * ldb : (static_cast<int64_t>(g) * N + static_cast<int64_t>(tn) * BN) * ldb);
        i32x4 ar = dma_rsrc(ap, static_cast<uint32_t>(mv) * static_cast<uint32_t>(lda));
        i32x4 br = dma_rsrc(bp, MN ? static_cast<uint32_t>(K) * static_cast<uint32_t>(ldb)
                                   : static_cast<uint32_t>(min(BN, N - tn * BN)) * static_cast<uint32_t>(ldb));
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            ar[i] = __builtin_amdgcn_readfirstlane(ar[i]);
            br[i] = __builtin_amdgcn_readfirstlane(br[i]);
        }

        // ---- DMA lane offsets ----
        // K-major rows: DMA d fills rows 8 d .. +7 of 128 bytes; lane l brings row 8 d + l / 8, piece
        // (l % 8) ^ (l / 8) (16 bytes), stored at piece position l % 8.
        constexpr int kBad = static_cast<int>(0x80000000u);
        const int drow = lane >> 3, dpiece = (lane & 7) ^ drow;
        // MN-major B: rows of BN columns (BN * es bytes): contraction row, kBRow lanes of 16 bytes each
        constexpr int kBRow = BN * F::es / 16, kBRowsPerDma = 64 / kBRow;
        const int bkrow = lane / kBRow, bslot = lane % kBRow;
        const int bpiece = MN ? (F::f8 ? bslot ^ ((bkrow >> 1) & (kBRow - 1)) : bslot ^ (bkrow & (kBRow - 1))) : 0;
        const int aoff = drow * lda + dpiece * 16;
        const int boff = MN ? bkrow * ldb + tn * (BN * F::es) + bpiece * 16 : drow * ldb + dpiece * 16;
        const int bcolbad = MN && tn * BN + bpiece * (16 / F::es) >= N ? kBad : 0;
        const int kbytes  = K * F::es;
        const uint32_t ring = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(&lds[0])) + wave * (S * kChunk);
        auto issue = [&](int c, int stage) {
            const uint32_t st  = ring + stage * kChunk;
            const int      bad = (c * 128 + dpiece * 16 >= kbytes) ? kBad : 0; // pieces past K (K-major)
#pragma unroll
            for (int d = 0; d < kDmaA; ++d)
                dma16(st + d * 1024, (aoff + d * 8 * lda + c * 128) | bad, ar, 0);
#pragma unroll
            for (int d = 0; d < kDmaB; ++d)
                dma16(st + kARegion + d * 1024,
                      MN ? (boff + (c * F::kc + d * kBRowsPerDma) * ldb) | bcolbad : (boff + d * 8 * ldb + c * 128) | bad, br, 0);
        };

        f32x4 acc[MB][NB];
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
            for (int j = 0; j < NB; ++j)
                acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

        // ---- the K loop: chunk wave, wave + W, ...; a ring of S chunks per wave, no barrier ----
        const int chunks = (K + F::kc - 1) / F::kc;
        const int mine   = chunks > wave ? (chunks - wave + W - 1) / W : 0;
        const int fr = lane & 15, fq = lane >> 4;
        for (int s = 0; s < min(S, mine); ++s)
            issue(wave + s * W, s);
        for (int c = 0, stage = 0; c < mine; ++c) {
            const int left = mine - 1 - c; // chunks of this wave still behind c, at most S - 1 in flight
            if (left >= S - 1)
                wait_vm<(S - 1) * kDma>();
            else
                wait_vm<0>();
            const unsigned char *sa = lds + wave * (S * kChunk) + stage * kChunk, *sb = sa + kARegion;
            auto a_piece = [&](int i, int piece) {
                return *reinterpret_cast<const i32x4 *>(sa + (16 * i + fr) * 128 + ((piece ^ (fr & 7)) << 4));
            };
            auto b_piece = [&](int j, int piece) {
                return *reinterpret_cast<const i32x4 *>(sb + (16 * j + fr) * 128 + ((piece ^ (fr & 7)) << 4));
            };
            if constexpr (F::f8) {
                const int p0 = 2 * fq + (fq & 1), p1 = 2 * fq + 1 - (fq & 1); // swapped for odd fq: fewer bank conflicts
                i32x8     fb[NB];
#pragma unroll
                for (int j = 0; j < NB; ++j) {
                    if constexpr (MN) {
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            // 8 contraction rows: source lane s of the 16 points at row s / 2, half s % 2
                            const int   row = 32 * fq + 16 * ((r >> 1) ^ (fq & 1)) + 8 * (r & 1) + (fr >> 1);
                            const int   at  = row * BN + ((j ^ ((row >> 1) & (kBRow - 1))) << 4) + (fr & 1) * 8;
                            const i32x2 v   = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_i32x2 *)(sb + at));
                            fb[j][2 * r]     = v[0];
                            fb[j][2 * r + 1] = v[1];
                        }
                    } else {
                        const i32x4 lo = b_piece(j, p0), hi = b_piece(j, p1);
                        fb[j] = i32x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
                    }
                }
#pragma unroll
                for (int i = 0; i < MB; ++i) {
                    const i32x4 lo = a_piece(i, p0), hi = a_piece(i, p1);
                    const i32x8 fa = i32x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
#pragma unroll
                    for (int j = 0; j < NB; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(fb[j], fa, acc[i][j], F::b_e5m2 ? 1 : 0,
                                                                                     F::a_e5m2 ? 1 : 0, 0, 0, 0, 0);
                }
            } else {
#pragma unroll
                for (int kh = 0; kh < 2; ++kh) {
                    i32x4 fb[NB];
#pragma unroll
                    for (int j = 0; j < NB; ++j) {
                        if constexpr (MN) {
#pragma unroll
                            for (int h = 0; h < 2; ++h) {
                                // 4 contraction rows: source lane s of the 16 points at row s / 4, columns 4 (s % 4)
                                const int    row = 32 * kh + 8 * fq + 4 * h + (fr >> 2);
                                const int    at  = row * (BN * 2) + (((2 * j + ((fr & 3) >> 1)) ^ (row & (kBRow - 1))) << 4) + (fr & 1) * 8;
                                const tr16x4 v   = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr16 *)(sb + at));
                                const i32x2  w   = __builtin_bit_cast(i32x2, v);
                                fb[j][2 * h]     = w[0];
                                fb[j][2 * h + 1] = w[1];
                            }
                        } else {
                            fb[j] = b_piece(j, 4 * kh + fq);
                        }
                    }
#pragma unroll
                    for (int i = 0; i < MB; ++i) {
                        const i32x4 fa = a_piece(i, 4 * kh + fq);
#pragma unroll
                        for (int j = 0; j < NB; ++j)
                            acc[i][j] = mma16<F::f16>(fb[j], fa, acc[i][j]);
                    }
                }
            }
            if (c + S < mine) {
                wait_lds(); // this stage's reads are done before its DMAs are issued again
                issue(wave + (c + S) * W, stage);
            }
            stage = stage + 1 == S ? 0 : stage + 1;
        }

        // 20 wait states between the last MFMA and the first read of its accumulators (gfx950 needs
        // up to 19 after a 16-pass MFMA; the build's hazard scan counts each MFMA issue as 4)
        asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 3" ::: "memory");
        // ---- add the waves' sums through LDS (the rings are free: every DMA has landed and been
        // read), in wave order, and store ----
        float *sum = reinterpret_cast<float *>(lds);
        __syncthreads();
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
            for (int j = 0; j < NB; ++j)
                *reinterpret_cast<f32x4 *>(sum + (wave * BM + 16 * i + fr) * kSumStride + 16 * j + 4 * fq) = acc[i][j];
        __syncthreads();
        float scale = 1.f;
        if constexpr (F::f8)
            scale = args.x_scale[0] * args.w_scale[g];
        constexpr int kUnits = BM * BN / 4; // four columns each
        for (int u = tid; u < kUnits; u += W * 64) {
            const int row = u / (BN / 4), col = 4 * (u % (BN / 4));
            f32x4     v   = *reinterpret_cast<const f32x4 *>(sum + row * kSumStride + col);
#pragma unroll
            for (int w = 1; w < W; ++w)
                v += *reinterpret_cast<const f32x4 *>(sum + (w * BM + row) * kSumStride + col);
            if constexpr (F::f8)
                v *= scale;
            if (row < mv && tn * BN + col < N) {
                uint16_t *o = static_cast<uint16_t *>(args.out) + (row0 + row) * static_cast<int64_t>(N) +
                              static_cast<int64_t>(tn) * BN + col;
                *reinterpret_cast<u32x2 *>(o) = pack4<F::f16>(v);
            }
        }
        __syncthreads(); // the sums are read before the next tile's DMAs overwrite them
    }
}

template <int FMT, bool MN, int I> void launch_instance(const KernelArgs &a, int grid, hipStream_t s) {
    constexpr FewInstance f = kFewInstances[I];
    hipLaunchKernelGGL((few_gemm_kernel<FMT, MN, f.tile_m / 16, f.tile_n / 16, f.waves, f.stages>), dim3(static_cast<unsigned>(grid)),
                       dim3(f.waves * 64), 0, s, a);
}

template <int FMT, bool MN> hipError_t launch_format(const KernelArgs &a, int instance, int grid, hipStream_t s) {
    switch (instance) {
    case 0: launch_instance<FMT, MN, 0>(a, grid, s); break;
    case 1: launch_instance<FMT, MN, 1>(a, grid, s); break;
    case 2: launch_instance<FMT, MN, 2>(a, grid, s); break;
    case 3: launch_instance<FMT, MN, 3>(a, grid, s); break;
    case 4: launch_instance<FMT, MN, 4>(a, grid, s); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

} // namespace

hipError_t launch_few_gemm(const KernelArgs &a, int format, bool mn, int instance, int grid, hipStream_t s) {
    static_assert(kFewInstanceCount == 5, "one case per instance");
    if (instance < 0 || instance >= kFewInstanceCount || grid <= 0 || a.tile_m != kFewInstances[instance].tile_m ||
        a.tile_n != kFewInstances[instance].tile_n)
        return hipErrorInvalidValue;
    switch (format) {
    case kFewBF16: return mn ? launch_format<kFewBF16, true>(a, instance, grid, s) : launch_format<kFewBF16, false>(a, instance, grid, s);
    case kFewF16: return mn ? launch_format<kFewF16, true>(a, instance, grid, s) : launch_format<kFewF16, false>(a, instance, grid, s);
    case kFewE4M3: return mn ? launch_format<kFewE4M3, true>(a, instance, grid, s) : launch_format<kFewE4M3, false>(a, instance, grid, s);
    case kFewE5M2: return mn ? launch_format<kFewE5M2, true>(a, instance, grid, s) : launch_format<kFewE5M2, false>(a, instance, grid, s);
    case kFewE5M2xE4M3: // an e5m2 gradient: dgrad only
        return mn ? launch_format<kFewE5M2xE4M3, true>(a, instance, grid, s) : hipErrorInvalidValue;
    default: return hipErrorInvalidValue;
    }
}

} // namespace gg

// Weight gradients of groups with few rows: grad_w[g] = grad_out[g]^T x[g], 16-bit and fp8.
//
// What bounds it: the writing of grad_w while a group has up to about a hundred rows, then the LDS
// reads of the operands. One workgroup of four waves computes 128 x 128 outputs (a wave 64 x 64), four
// workgroups per CU (128 registers per lane, 35 KB of LDS), so that some store while others load
// and multiply. A chunk of the group's rows (32, in a ring of two; fp8: 128, one) goes from global
// memory to LDS by DMA in row order (4 consecutive lanes on 64 contiguous bytes: 16 cycles per KB
// of the address unit) and is read transposed (ds_read_b64_tr_b16 / _b8) for both operands. Row r's
// 16-byte piece p sits at p ^ swz(r), which spreads the rows that one read pass covers over the banks
// (counters: the LDS is active 25-36 % of a launch, 30-43 % of that are bank conflicts, of the reads and the
// staged output together).
// x is the MFMA's first source, so a lane holds four consecutive columns of one output row; the tile
// is packed to 16 bits, staged through LDS and stored as whole 256-byte rows.
//
// A group without rows writes zeros. The resources end at the group's last row and columns past the
// operand's width get an offset past them, so both read zeros.
//
// Measured (MI355X, us per launch, persistent kernel -> this one): bf16 32 groups of 16 rows, 2880 x
// 2880 169 -> 97 (5.5 TB/s written), of 128 rows 172 -> 132; fp16 51 x 73, 5632 x 1280 198 -> 141; fp8
// 58 x 3, 2048 x 3072 200 -> 135; 11 x 316, 5376 x 3344 172 -> 143. Swept: chunks of 32 and 64 rows,
// rings of 1-4, 2-4 workgroups per CU (32 x 128 rows: 132 with 32 rows x 2, 4 per CU; 137 with 64 x 1,
// 4 per CU; 161 with 64 x 2, 2 per CU). Tiles go to the XCDs in runs of 128: one run per XCD over the
// whole launch left the XCDs of large groups behind (16 groups of 67-1286 rows 78 -> 64).
#include "gg_few.h"
#include "gg_kernel_impl.h"

namespace gg {
namespace {

typedef short    wtr16x4 __attribute__((ext_vector_type(4)));
typedef __bf16   wbf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 wf16x8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) wtr16x4 lds_wtr16;
typedef __attribute__((address_space(3))) i32x2   lds_wi32x2;

constexpr int kWT = kWgradFewTile; // 128 x 128 outputs per workgroup
constexpr int kWRow = 272;         // staged output row stride (256 bytes + 16)

template <int FMT>
__global__ void __launch_bounds__(kWgradFewThreads, 4) wgrad_few_kernel(const KernelArgs args) {
    constexpr bool kF8   = FMT >= kFewE4M3;
    constexpr bool kF16  = FMT == kFewF16;
    constexpr int  es    = kF8 ? 1 : 2;
    constexpr int  kc    = kF8 ? 128 : 32;   // rows per chunk
    constexpr int  S     = kF8 ? 1 : 2;      // chunks in the ring
    constexpr int  row_b = kWT * es;         // bytes of a staged row
    constexpr int  pieces = row_b / 16;      // per row: 16 or 8
    constexpr int  rows_dma = 64 / pieces;   // rows per DMA: 4 or 8
    constexpr int  kOp = kc * row_b, kD = kOp / 4096; // bytes of an operand's chunk, DMAs per wave
    __shared__ __attribute__((aligned(1024))) unsigned char lds[kWT * kWRow > 2 * S * kOp ? kWT * kWRow : 2 * S * kOp];
    const int tid = static_cast<int>(threadIdx.x), lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int N = args.n, MO = args.m_out;
    const int nt = (N + kWT - 1) / kWT, mt = (MO + kWT - 1) / kWT;

    LaneGroup lg{};
    if (args.d_lens != nullptr) {
        int total, first_bad, overflow;
        lg = lane_group_table(args.d_lens, args.d_offs, args.group_num, args.lens_rows, args.n_tiles, MO, lane, &total,
                              &first_bad, &overflow);
        if (blockIdx.x == 0 && tid == 0) {
            args.d_header->total_tiles = total;
            args.d_header->first_bad   = first_bad;
            args.d_header->overflow    = overflow;
            args.d_header->run_tiles   = 0;
        }
    }
    // in runs of one XCD's share of 1024 tiles: longer runs would leave the XCDs of large groups behind
    const int L = xcd_remap(static_cast<int>(blockIdx.x), args.total_tiles, min(static_cast<int>(gridDim.x), 1024), args.n_xcd);
    if (static_cast<int>(blockIdx.x) >= args.total_tiles)
        return;
    const int g = L / (mt * nt);
    int       tm, tn;
    band_coords(L - g * (mt * nt), mt, nt, 8, &tm, &tn);
    int64_t row0;
    int     m;
    if (args.d_lens != nullptr) {
        m    = __builtin_amdgcn_readlane(lg.m, g);
        row0 = static_cast<int64_t>(static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(lg.row0), g))) |
               (static_cast<int64_t>(__builtin_amdgcn_readlane(static_cast<int>(lg.row0 >> 32), g)) << 32);
    } else {
        const auto t = to_const_space(args.groups);
        m    = t[g].m;
        row0 = t[g].row0;
    }
    const int lda = args.lda * es, ldb = args.ldb * es;
    i32x4 ar = dma_rsrc(static_cast<const char *>(args.x) + row0 * lda, static_cast<uint32_t>(m) * static_cast<uint32_t>(lda));
    i32x4 br = dma_rsrc(static_cast<const char *>(args.w) + row0 * ldb, static_cast<uint32_t>(m) * static_cast<uint32_t>(ldb));
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        ar[i] = __builtin_amdgcn_readfirstlane(ar[i]);
        br[i] = __builtin_amdgcn_readfirstlane(br[i]);
    }
    // row r's 16-byte piece p sits at position p ^ swz(r)
    auto swz = [](int r) { return kF8 ? ((r >> 1) & 3) | (((r >> 5) & 1) << 2) : 2 * ((r & 3) | (((r >> 3) & 1) << 2)); };
    constexpr int kBad = static_cast<int>(0x80000000u);
    const int drow = lane / pieces, dpos = lane % pieces;
    const uint32_t base = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(&lds[0])) + wave * (kD * 1024);
    auto issue = [&](int c) {
        const uint32_t st = base + (c % S) * (2 * kOp);
#pragma unroll
        for (int d = 0; d < kD; ++d) {
            const int r = (wave * kD + d) * rows_dma + drow;
            const int col = (dpos ^ swz(r)) * (16 / es);
            const int ca = tm * kWT + col, cb = tn * kWT + col;
            dma16(st + d * 1024, ((c * kc + r) * lda + ca * es) | (ca >= MO ? kBad : 0), ar, 0);
            dma16(st + kOp + d * 1024, ((c * kc + r) * ldb + cb * es) | (cb >= N ? kBad : 0), br, 0);
        }
    };
    f32x4 acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
            acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int wm = wave >> 1, wn = wave & 1, fr = lane & 15, fq = lane >> 4;
    const int chunks = (m + kc - 1) / kc;
    if (S == 2 && chunks > 0)
        issue(0);
    for (int c = 0; c < chunks; ++c) {
        if constexpr (S == 1) {
            if (c > 0)
                asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); // the last chunk is read
            issue(c);
            wait_vm_lds_barrier<0>();
        } else {
            wait_vm_lds_barrier<0>(); // chunk c has landed and chunk c - 1 is read
            if (c + 1 < chunks)
                issue(c + 1);
        }
        const unsigned char *sc = lds + (c % S) * (2 * kOp);
        if constexpr (kF8) {
            auto frag = [&](int op, int blk) { // 16 columns from 16 blk, 128 rows
                i32x8 v;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int   row = 32 * fq + 8 * r + (fr >> 1);
                    const i32x2 t = __builtin_amdgcn_ds_read_tr8_b64_v2i32(
                        (lds_wi32x2 *)(sc + op * kOp + row * row_b + ((blk ^ swz(row)) << 4) + (fr & 1) * 8));
                    v[2 * r]     = t[0];
                    v[2 * r + 1] = t[1];
                }
                return v;
            };
            i32x8 fb[4];
#pragma unroll
            for (int j = 0; j < 4; ++j)
                fb[j] = frag(1, wn * 4 + j);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const i32x8 fa = frag(0, wm * 4 + i);
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(
                        fb[j], fa, acc[i][j], FMT == kFewE5M2 ? 1 : 0, FMT == kFewE4M3 ? 0 : 1, 0, 0, 0, 0);
            }
        } else {
            auto frag = [&](int op, int blk) { // 16 columns from 16 blk, 32 rows
                i32x4 v;
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int   row = 8 * fq + 4 * h + (fr >> 2);
                    const i32x2 t = __builtin_bit_cast(
                        i32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                   (lds_wtr16 *)(sc + op * kOp + row * row_b + (((2 * blk + ((fr & 3) >> 1)) ^ swz(row)) << 4) +
                                                 (fr & 1) * 8)));
                    v[2 * h]     = t[0];
                    v[2 * h + 1] = t[1];
                }
                return v;
            };
            i32x4 fb[4];
#pragma unroll
            for (int j = 0; j < 4; ++j)
                fb[j] = frag(1, wn * 4 + j);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const i32x4 fa = frag(0, wm * 4 + i);
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if constexpr (kF16)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(wf16x8, fb[j]),
                                                                           __builtin_bit_cast(wf16x8, fa), acc[i][j], 0, 0, 0);
                    else
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(wbf16x8, fb[j]),
                                                                            __builtin_bit_cast(wbf16x8, fa), acc[i][j], 0, 0, 0);
            }
        }
    }
    asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 3" ::: "memory");
    float scale = 1.f;
    if constexpr (kF8)
        scale = args.x_scale[0] * args.w_scale[g];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
            *reinterpret_cast<u32x2 *>(lds + (wm * 64 + 16 * i + fr) * kWRow + (wn * 64 + 16 * j + 4 * fq) * 2) =
                pack4<kF16>(kF8 ? acc[i][j] * scale : acc[i][j]);
    __syncthreads();
    const int col = tn * kWT + (tid & 15) * 8;
    uint16_t *o = static_cast<uint16_t *>(args.out) + (static_cast<int64_t>(g) * MO + static_cast<int64_t>(tm) * kWT) * N + col;
#pragma unroll
    for (int p = 0; p < 8; ++p) {
        const int   r = p * 16 + (tid >> 4);
        const u32x4 v = *reinterpret_cast<const u32x4 *>(lds + r * kWRow + (tid & 15) * 16);
        if (tm * kWT + r < MO && col < N)
            __builtin_nontemporal_store(v, reinterpret_cast<u32x4 *>(o + static_cast<int64_t>(r) * N));
    }
}

} // namespace

template <int FMT> void launch_format(const KernelArgs &a, int grid, hipStream_t s) {
    hipLaunchKernelGGL(wgrad_few_kernel<FMT>, dim3(static_cast<unsigned>(grid)), dim3(kWgradFewThreads), 0, s, a);
}

hipError_t launch_wgrad_few(const KernelArgs &a, int format, int grid, hipStream_t s) {
    switch (format) {
    case kFewBF16: launch_format<kFewBF16>(a, grid, s); break;
    case kFewF16: launch_format<kFewF16>(a, grid, s); break;
    case kFewE4M3: launch_format<kFewE4M3>(a, grid, s); break;
    case kFewE5M2: launch_format<kFewE5M2>(a, grid, s); break;
    case kFewE5M2xE4M3: launch_format<kFewE5M2xE4M3>(a, grid, s); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

} // namespace gg

// The weight gradient of a linear on CDNA4 bf16 MFMA (v_mfma_f32_16x16x32_bf16):
//
//   dw[n, k] = sum_m dy[m, n] * x[m, k]      dy bf16 [R, N], x bf16 [R, K]
//
// fp32 accumulation, one bf16 rounding (RNE) at the store: the reference's
// linear_dw, dy^T @ x in bf16 (python/xpu_kernels/int8/ops.py:207-238).
//
// Both operands are contracted along their *rows*, while an MFMA operand
// fragment wants 8 consecutive reduction values per lane.  The tiles therefore
// go into LDS exactly as they lie in memory (row-major, direct global->LDS
// loads), and the fragments come out with gfx950's transposing LDS read
// ds_read_b64_tr_b16.  Within each group of 16 lanes, lane j supplies the
// address of 4 consecutive bf16 and lane i = 4a + b receives element b of the
// vectors supplied by lanes a, a+4, a+8, a+12.  So when lane j points at row
// j/4, columns 4(j%4)..+3 of a 4 x 16 block, lane i receives column i of the
// 4 rows -- a transposed 4 x 16 read.  Two such reads (rows +0..3 and +4..7)
// give lane l the 8 reduction values m = 8(l/16)..+7 of operand row l%16,
// the fragment layout of the 16x16x32 MFMA.
//
// D = A * B with A from x (D rows = k) and B from dy (D columns = n), so lane
// l of a 16x16 block holds D[4(l/16)+i][l%16]: four consecutive k of one dw
// row, stored as one 8-byte write.
#include <algorithm>

#include "common.hpp"
#include "kernels.hpp"

namespace xpuint8 {
namespace {

typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef short v4s __attribute__((ext_vector_type(4)));
typedef short v8s __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v2f __attribute__((ext_vector_type(2)));
typedef __bf16 v2bf __attribute__((ext_vector_type(2)));

// 16 zero bytes: the DMA source for reduction rows past R.
__device__ __attribute__((aligned(16))) int8_t g_zero_line[16];

constexpr int kStepRows = 32;                // reduction rows per MFMA step

__device__ __forceinline__ void dma16(const int8_t* gsrc, int8_t* ldst) {
#if defined(__HIP_DEVICE_COMPILE__)
    __builtin_amdgcn_global_load_lds(gsrc, (__attribute__((address_space(3))) void*)ldst, 16, 0,
                                     0);
#endif
}

// The transposing read, issued as inline assembly.  Written with the builtin,
// the compiler must assume the read may see LDS that a pending direct-to-LDS
// load writes, and waits for *all* outstanding loads before it -- including
// the stage just issued, which removes the pipelining.  Here the ring's own
// vmcnt waits (before each barrier) order the loads; the reads' completion is
// awaited (lgkmcnt) before any fragment is used.
__device__ __forceinline__ uint32_t lds_addr(const int8_t* p) {
    return static_cast<uint32_t>(
        reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) const int8_t*)p));
}
template <int OFF>
__device__ __forceinline__ v4s tr_read_at(uint32_t addr) {
    static_assert(OFF >= 0 && OFF < 65536, "ds offset field");
    v4s r;
    asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(r) : "v"(addr), "n"(OFF));
    return r;
}

__device__ __forceinline__ uint32_t cvt_pk_bf16(float lo, float hi) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v2f{lo, hi}, v2bf));
}

// s_waitcnt immediate waiting for vmcnt <= n only.
__host__ __device__ constexpr int vmcnt_imm(int n) {
    return (n & 0xF) | ((n >> 4) << 14) | (0x7 << 4) | (0xF << 8);
}

// ---------------------------------------------------------------- split K
// Narrow outputs with a long contraction: the dense dx (C5: M = 4096 rows,
// K = 1280 outputs, R = 5120 contraction rows) and dW (N = 5120 rows, K = 1280,
// R = 4096), where 128 x 192 tiles of the persistent kernel below leave CUs idle
// (66.9 against 58.8 us for the dx, 61.9 against 54.9 for dW).  One block of 8
// waves owns a BB x 160 tile of out[b, k] (256 tiles at C5 for both), in two
// teams of 4 (2 x 2 waves of BB/2 x 80): team t owns half of the 32-row
// contraction steps through its own ring of S LDS stages, and the teams
// alternate between MFMAs and data movement every half step, so that on each
// SIMD one wave feeds the matrix core while the other reads fragments and
// issues loads:
//   A(s): team 0 runs its step s;  team 1 reads its step s's fragments and
//         issues its loads for step s + S - 1
//   B(s): team 1 runs its step s;  team 0 reads its step s + 1's fragments
//         and issues its loads for step s + S - 1
// with one s_barrier between phases.  D = A * B with A from the operand
// contracted along its rows, a[r, k] (dx: the weight; dW: x), and B from
// b (dx: dy[m, r], contracted along its contiguous dimension, BB = 128; dW,
// YT: dy[r, n], contracted along its rows, BB = 160).  A stage holds
//   for A, 10 blocks of 16 rows (contraction) x 32 columns (64 bytes), block
//     2cg + rb for rows 16rb.. and columns 32cg..: 16-byte chunk c of row r
//     at chunk 4r + (c ^ ((r >> 2) & 2)).  One direct-to-LDS load fills a
//     block from 16 row segments of 64 bytes (measured 8% faster at C5 than
//     32 rows x 32 bytes), and the two transposing reads of a fragment (rows
//     8g + 4h + q of the step, g, q = 0..3, 32 bytes each) cover the 64 banks
//     twice, the two-cycle minimum for their 512 bytes;
//   for B, the same (YT), or 8 blocks of 16 rows (m) x 64 bytes (one step of
//     32 bf16): chunk c of row r at position c ^ ((r >> 1) & 3), lane l's
//     fragment (row l%16, elements 8(l/16)..+7) one 16-byte read.
// The fp32 sums of the two halves meet in LDS (each team adds the other's
// partial for its share of the B blocks: IEEE addition is commutative, so the
// sum does not depend on which team forms it), and each team rounds and
// stores its share.  Lane l of block (a, b) holds D[4(l/16)+i][l%16]: four
// consecutive k of one output row, one 8-byte store.
__device__ __forceinline__ int swz_y(int r, int c) { return c ^ ((r >> 1) & 3); }
// chunk (16 bytes) of row r, chunk c within a 16-row x 64-byte block
__device__ __forceinline__ int chunk_at(int r, int c) { return 4 * r + (c ^ ((r >> 2) & 2)); }

template <int OFF>
__device__ __forceinline__ v8s plain_read_at(uint32_t addr) {
    static_assert(OFF >= 0 && OFF < 65536, "ds offset field");
    v8s r;
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(r) : "v"(addr), "n"(OFF));
    return r;
}

template <int S, bool YT>
__global__ __launch_bounds__(512, 1) void gemm_bf16_splitk_kernel(
    const uint16_t* __restrict__ A, int64_t lda, const uint16_t* __restrict__ Y, int64_t ldy,
    uint16_t* __restrict__ out, int64_t ldo, int R, int K, int NBR, int tiles_b, int tiles_k) {
    constexpr int BK = 160, TK = 5;                     // A side: k columns, blocks per wave
    constexpr int TB = YT ? 5 : 4, BB = 32 * TB;        // B side: blocks per wave, tile rows
    constexpr int AB = BK / 16, YB = BB / 16, NB = AB + YB;
    // block order in a stage: dy's blocks first (measured faster at C5 than
    // after the A operand's: 61.0 against 63.9 us for the dx, 59.8 against
    // 61.0 for dW)
    constexpr int A0 = YB, Y0 = 0;
    constexpr int PER = (NB + 3) / 4, REM = NB % 4;
    constexpr int STAGE = NB * 1024, RING = S * STAGE;
    constexpr int OWN0 = (TB + 1) / 2;                  // team 0 owns B blocks 0..OWN0-1
    static_assert(2 * RING >= 4 * TK * TB * 1024, "the exchanged partial sums fit");
    static_assert(2 * RING <= 160 * 1024, "LDS");
    __shared__ __attribute__((aligned(1024))) int8_t smem[2 * RING];

    // tile grid over the 8 XCDs (block b on XCD b % 8): each XCD a gx x
    // (8 / gx) block of tiles, gx chosen so that it reads the fewest operand
    // rows and columns
    int tbi = blockIdx.x % tiles_b, tki = blockIdx.x / tiles_b;
    {
        int best = 0, cost = 0;
        for (int gx = 1; gx <= 8; gx *= 2) {
            const int gy = 8 / gx;
            if (tiles_b % gx || tiles_k % gy) continue;
            const int c = (tiles_b / gx) * BB + (tiles_k / gy) * BK;
            if (!best || c < cost) best = gx, cost = c;
        }
        if (best) {
            const int x = blockIdx.x % 8, j = blockIdx.x / 8;
            const int lb = tiles_b / best, lk = tiles_k / (8 / best);
            tbi = (x % best) * lb + j % lb;
            tki = (x / best) * lk + j / lb;
        }
    }
    const int b0 = tbi * BB, k0 = tki * BK;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int team = wave >> 2, wt = wave & 3;
    const int wb = wt >> 1, wk = wt & 1;
    int8_t* const ring = smem + team * RING;

    const int RT = R / kStepRows, RH = (RT + 1) / 2;   // team 0 takes the first RH steps
    const int st0 = team * RH, nst = min(RT, st0 + RH) - st0;

    // DMA: wave wt brings blocks wt, wt + 4, ... of its team's stages.  Byte offsets from a wave-uniform base; a step adds 32
    // rows (row-contracted operands) or 64 bytes (dy of the dx).  Rows past
    // the output edge repeat the last row, columns past it a valid chunk
    // (neither is stored).
    const int8_t* const abase = reinterpret_cast<const int8_t*>(A + k0);
    const int8_t* const ybase =
        reinterpret_cast<const int8_t*>(YT ? Y + b0 : Y + int64_t(b0) * ldy);
    int off[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int j = min(wt + 4 * i, NB - 1);
        // row-contracted blocks: lane l fills chunk l of the block, i.e. row
        // r = l/4, chunk (l%4) ^ ((r >> 2) & 2) (an involution of l%4)
        const int r = lane >> 2, c = (lane & 3) ^ ((r >> 2) & 2);
        const bool isa = j >= A0 && j < A0 + AB;
        if (isa) {
            const int jj = j - A0, row = 16 * (jj & 1) + r;
            off[i] = row * int(lda) * 2 + (min(k0 + 32 * (jj >> 1) + 8 * c, K - 8) - k0) * 2;
        } else if constexpr (YT) {
            const int jj = j - Y0, row = 16 * (jj & 1) + r;
            off[i] = row * int(ldy) * 2 + (min(b0 + 32 * (jj >> 1) + 8 * c, NBR - 8) - b0) * 2;
        } else {
            const int rr = lane >> 2, c = swz_y(rr, lane & 3);
            off[i] = (min(b0 + 16 * (j - Y0) + rr, NBR - 1) - b0) * int(ldy) * 2 + 16 * c;
        }
    }
    const bool full_share = REM == 0 || wt < REM;
    auto issue = [&](int s) {
        const int step = st0 + s;
        int8_t* const st = ring + (s % S) * STAGE;
        const uint32_t arow = uint32_t(step * kStepRows) * uint32_t(lda) * 2u;
        const uint32_t yrow = YT ? uint32_t(step * kStepRows) * uint32_t(ldy) * 2u
                                 : uint32_t(step * 64);
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            if (i == PER - 1 && !full_share) break;
            const int j = wt + 4 * i;
            const int8_t* p = (j >= A0 && j < A0 + AB) ? abase + uint64_t(uint32_t(off[i]) + arow)
                                                       : ybase + uint64_t(uint32_t(off[i]) + yrow);
            dma16(p, st + j * 1024);
        }
    };
    auto wait_batches = [&](int later) {
        if (full_share) {
            if (later >= 2) __builtin_amdgcn_s_waitcnt(vmcnt_imm(2 * PER));
            else if (later == 1) __builtin_amdgcn_s_waitcnt(vmcnt_imm(PER));
            else __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
        } else {
            if (later >= 2) __builtin_amdgcn_s_waitcnt(vmcnt_imm(2 * (PER - 1)));
            else if (later == 1) __builtin_amdgcn_s_waitcnt(vmcnt_imm(PER - 1));
            else __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
        }
    };

    // fragment addresses within a stage.  Transposing reads of row-contracted
    // blocks: for the 16-column block at column kc of the tile, lane j of
    // group g reads step row 8g + 4h + j/4, 8 bytes at column kc + 4(j%4);
    // plain 16-byte reads for dy of the dx.
    const int g = lane >> 4, j = lane & 15;
    auto tr_off = [&](int first, int kc, int h) {
        const int cg = kc >> 5, half = (kc >> 4) & 1;
        const int R = 8 * g + 4 * h + (j >> 2), rb = R >> 4, r = R & 15;
        const int c = 2 * half + ((j & 3) >> 1);
        return uint32_t((first + 2 * cg + rb) * 1024 + 16 * chunk_at(r, c) + 8 * (j & 1));
    };
    uint32_t aoffs[TK][2], yoffs[YT ? TB : 1][2];
#pragma unroll
    for (int a = 0; a < TK; ++a)
#pragma unroll
        for (int h = 0; h < 2; ++h) aoffs[a][h] = tr_off(A0, wk * (BK / 2) + 16 * a, h);
    if constexpr (YT) {
#pragma unroll
        for (int b = 0; b < TB; ++b)
#pragma unroll
            for (int h = 0; h < 2; ++h) yoffs[b][h] = tr_off(Y0, wb * (BB / 2) + 16 * b, h);
    }
    const uint32_t yoff = (Y0 + wb * TB) * 1024 + j * 64 + swz_y(j, g) * 16;
    const uint32_t rbase = lds_addr(ring);

    v4f acc[TK][TB];
#pragma unroll
    for (int a = 0; a < TK; ++a)
#pragma unroll
        for (int b = 0; b < TB; ++b) acc[a][b] = v4f{0.f, 0.f, 0.f, 0.f};
    v4s al[TK], ah[TK];
    v4s yl[YT ? TB : 1], yh[YT ? TB : 1];
    v8s yf[YT ? 1 : TB];
    auto read_frags = [&](int s) {
        const uint32_t sb = rbase + (s % S) * STAGE;
        auto rda = [&](auto I) {
            constexpr int a = decltype(I)::value;
            if constexpr (a < TK) {
                al[a] = tr_read_at<0>(sb + aoffs[a][0]);
                ah[a] = tr_read_at<0>(sb + aoffs[a][1]);
            }
        };
        auto rdb = [&](auto I) {
            constexpr int b = decltype(I)::value;
            if constexpr (b < TB) {
                if constexpr (YT) {
                    yl[b] = tr_read_at<0>(sb + yoffs[b][0]);
                    yh[b] = tr_read_at<0>(sb + yoffs[b][1]);
                } else {
                    yf[b] = plain_read_at<b * 1024>(sb + yoff);
                }
            }
        };
        rda(std::integral_constant<int, 0>{});
        rda(std::integral_constant<int, 1>{});
        rda(std::integral_constant<int, 2>{});
        rda(std::integral_constant<int, 3>{});
        rda(std::integral_constant<int, 4>{});
        rdb(std::integral_constant<int, 0>{});
        rdb(std::integral_constant<int, 1>{});
        rdb(std::integral_constant<int, 2>{});
        rdb(std::integral_constant<int, 3>{});
        rdb(std::integral_constant<int, 4>{});
    };
    auto join = [](const v4s& lo, const v4s& hi) {
        const v8s v = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        return __builtin_bit_cast(v8bf, v);
    };
    auto compute = [&]() {
        // every read has landed before any fragment is used (the operands tie
        // the fragments to this wait)
        asm volatile("s_waitcnt lgkmcnt(0)"
                     : "+v"(al[0]), "+v"(al[1]), "+v"(al[2]), "+v"(al[3]), "+v"(al[4]),
                       "+v"(ah[0]), "+v"(ah[1]), "+v"(ah[2]), "+v"(ah[3]), "+v"(ah[4]));
        if constexpr (YT) {
            asm volatile("" : "+v"(yl[0]), "+v"(yl[1]), "+v"(yl[2]), "+v"(yl[3]), "+v"(yl[4]),
                              "+v"(yh[0]), "+v"(yh[1]), "+v"(yh[2]), "+v"(yh[3]), "+v"(yh[4]));
        } else {
            asm volatile("" : "+v"(yf[0]), "+v"(yf[1]), "+v"(yf[2]), "+v"(yf[3]));
        }
        v8bf bfr[TB];
#pragma unroll
        for (int b = 0; b < TB; ++b) {
            if constexpr (YT) bfr[b] = join(yl[b], yh[b]);
            else bfr[b] = __builtin_bit_cast(v8bf, yf[b]);
        }
#pragma unroll
        for (int a = 0; a < TK; ++a) {
            const v8bf af = join(al[a], ah[a]);
#pragma unroll
            for (int b = 0; b < TB; ++b)
                acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af, bfr[b], acc[a][b], 0, 0, 0);
        }
    };
    auto barrier = [&]() {
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
    };

    for (int s = 0; s < S - 1; ++s)
        if (s < nst) issue(s);
    if (nst > 0) wait_batches(min(S - 2, nst - 1));
    barrier();
    if (team == 0) {
        if (nst > 0) read_frags(0);
        barrier();
#pragma clang loop unroll(disable)
        for (int s = 0; s < RH; ++s) {
            if (s < nst) compute();                             // A(s)
            if (s + 1 < nst) wait_batches(min(S - 3, nst - 2 - s));
            barrier();
            if (s + 1 < nst) read_frags(s + 1);                 // B(s)
            if (s + S - 1 < nst) issue(s + S - 1);
            barrier();
        }
    } else {
        barrier();
#pragma clang loop unroll(disable)
        for (int s = 0; s < RH; ++s) {
            if (s < nst) read_frags(s);                         // A(s)
            if (s + S - 1 < nst) issue(s + S - 1);
            barrier();
            if (s < nst) compute();                             // B(s)
            if (s + 1 < nst) wait_batches(min(S - 2, nst - 2 - s));
            barrier();
        }
    }

    // exchange: each team gives the other its partial sums of the B blocks
    // the other owns (team 0 owns blocks 0 .. OWN0-1 of each wave, team 1 the
    // rest).  Team t's given blocks fill its own region of LDS, [wave][a][b]
    // x 64 lanes; constant block indices in each branch keep the
    // accumulators in registers.
    __syncthreads();
    v4f* const xchg = reinterpret_cast<v4f*>(smem);
    constexpr int CNT0 = TB - OWN0, CNT1 = OWN0;        // blocks given by team 0, 1
    auto slot = [&](auto T, int a, int b) {
        constexpr int t = decltype(T)::value;
        constexpr int first = t == 0 ? OWN0 : 0, cnt = t == 0 ? CNT0 : CNT1;
        constexpr int region = t == 0 ? 0 : 4 * TK * CNT0;
        return ((region + (wt * TK + a) * cnt + (b - first)) * 64) + lane;
    };
    auto finish = [&](auto T) {
        constexpr int t = decltype(T)::value;
        constexpr int lo = t == 0 ? 0 : OWN0, hi = t == 0 ? OWN0 : TB;   // owned blocks
        constexpr std::integral_constant<int, t> self{};
        constexpr std::integral_constant<int, 1 - t> other{};
#pragma unroll
        for (int a = 0; a < TK; ++a)
#pragma unroll
            for (int b = 0; b < TB; ++b)
                if (b < lo || b >= hi) xchg[slot(self, a, b)] = acc[a][b];
        __syncthreads();
#pragma unroll
        for (int a = 0; a < TK; ++a)
#pragma unroll
            for (int b = lo; b < hi; ++b) acc[a][b] += xchg[slot(other, a, b)];
        // lane l of block (a, b): output row b0 + (BB/2) wb + 16b + l%16,
        // columns k0 + 80 wk + 16a + 4(l/16) .. +3
#pragma unroll
        for (int b = lo; b < hi; ++b) {
            const int row = b0 + wb * (BB / 2) + 16 * b + (lane & 15);
            if (row >= NBR) continue;
#pragma unroll
            for (int a = 0; a < TK; ++a) {
                const int k = k0 + wk * 80 + 16 * a + 4 * (lane >> 4);
                if (k < K) {
                    const v4f v = acc[a][b];
                    *reinterpret_cast<uint2*>(out + int64_t(row) * ldo + k) =
                        make_uint2(cvt_pk_bf16(v[0], v[1]), cvt_pk_bf16(v[2], v[3]));
                }
            }
        }
    };
    if (team == 0) finish(std::integral_constant<int, 0>{});
    else finish(std::integral_constant<int, 1>{});
}

// fragments b = 0 .. COUNT-1 of a plainly read operand, 1 KB apart
template <int COUNT, int I = 0, int NF>
__device__ __forceinline__ void plain_read_frags(v8s (&f)[NF], uint32_t addr) {
    if constexpr (I < COUNT) {
        f[I] = plain_read_at<I * 1024>(addr);
        plain_read_frags<COUNT, I + 1>(f, addr);
    }
}

// ------------------------------------------------------------ large outputs
// Products with at least a round of large tiles: the persistent ping-pong
// scheme of the int8 GEMM in bf16, one block of 8 waves per CU over BB x BC
// tiles of out[b, c], in two groups of 4 waves (the tile's row halves) that
// alternate between MFMAs and data movement every half step, through a ring of
// four LDS slots of one 32-row contraction step that runs on from tile to tile.
//   phase A(s): group 0 runs step s's MFMAs; group 1 reads step s's fragments
//               and issues its loads for step s + 3
//   phase B(s): group 1 runs step s's MFMAs; group 0 reads step s + 1's
//               fragments and issues its loads for step s + 3
// A slot is refilled only after its last reader's phase, a step is complete
// (each wave waits for its own loads, then the barrier) before its first.
//
// The split-K kernel above gives a 128 x 160 tile 18 KB of operands per 32-row
// step for 320 clocks of MFMA per SIMD, more than the direct-to-LDS path
// moves (32-40 bytes per clock for row segments); a 256 x 320 tile needs 36 KB for
// 1280 clocks.  A wave's accumulators are the same 160 registers at
// 128 x 80 as there the whole block's.
//
// Operands in a slot (1 KB blocks, one direct-to-LDS load each):
//   contracted along its rows (a; y too with YT): 8 rows x 64 columns, so that
//     a load is 8 whole cache lines (16 x 64 bytes: 16 halves); block 4cg + rb
//     holds rows 8rb.. of columns 64cg..; the 32-byte chunk pair p of row r at
//     pair p ^ (2 ((r >> 1) & 1) + (rb & 1)), which puts the 8 row pieces that half a
//     wave's transposing read touches on distinct banks;
//   contracted along its columns (y of the dx): 16 rows x 64 bytes as in the
//     split-K kernel.
// Rows of the contraction past R are read as zeros from both operands.
//
// SL: contraction slice blockIdx.y of a split across blocks, `slice` (a multiple
// of 32) long but the last: a and y are offset to it, and its fp32 sums go to
// (float*)out + blockIdx.y * sl_stride instead of the bf16 output.
// Off: the lanes' byte offsets from a block's first row, at most 15 rows
// (uint32_t; uint64_t for leading dimensions past 2^27).
template <int BB, int BC, int WGM, bool YT, bool SL, class Off = uint32_t>
__global__ __launch_bounds__(512, 1) void gemm_bf16_pp_kernel(
    const uint16_t* __restrict__ A, int64_t lda, const uint16_t* __restrict__ Y, int64_t ldy,
    uint16_t* __restrict__ out, int64_t ldo, int R, int NC, int NBR, int tiles_b, int tiles_c,
    int slice, int64_t sl_stride) {
    if constexpr (SL) {
        const int64_t r0 = int64_t(blockIdx.y) * slice;
        A += r0 * lda;
        Y += YT ? r0 * ldy : r0;
        R = min(slice, R - int(r0));
    }
    constexpr int NW = 8, WGN = NW / WGM, S = 4;
    static_assert(WGM % 2 == 0 && WGM * WGN == NW, "two groups of four waves (row halves)");
    constexpr int WB = BB / WGM, WC = BC / WGN, TB = WB / 16, TC = WC / 16;
    static_assert(BC % 64 == 0 && (!YT || BB % 64 == 0), "whole 64-column blocks");
    constexpr int YB = BB / 16, CB = BC / 16, NB = YB + CB;    // 1 KB blocks per slot
    constexpr int PER = (NB + NW - 1) / NW, REM = NB % NW;
    static_assert(REM == 0 || REM == 4, "group 0 issues PER, group 1 PER or PER - 1");
    constexpr int STAGE = NB * 1024, RING = S * STAGE;
    // the epilogue's staging (16 rows x 256 bytes per wave): the slot of the
    // tile's last step, or an area of its own where a slot is smaller
    constexpr int STG = NW * 16 * 256, STG_OWN = STG > STAGE ? STG : 0;
    static_assert(RING + STG_OWN <= 160 * 1024, "LDS");
    static_assert(WC <= 128, "staged rows of at most 256 bytes");
    __shared__ __attribute__((aligned(1024))) int8_t smem[RING + STG_OWN];

    const int tiles = tiles_b * tiles_c;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wb = wave / WGN, wc = wave % WGN;
    const int grp = wb / (WGM / 2);
    const bool full_share = REM == 0 || grp == 0;

    // tile origin of sequence number i: XCD i % 8 takes a contiguous eighth of
    // the tiles (rounded up), in bands of 8 row tiles; false past its share
    const int share = (tiles + 7) / 8;
    auto tile_origin = [&](int i, int& b0, int& c0) {
        const int t = (i % 8) * share + i / 8;
        if (i / 8 >= share || t >= tiles) return false;
        constexpr int GROUP = 8;
        const int band = t / (GROUP * tiles_c);
        const int first = band * GROUP;
        const int gm = min(tiles_b - first, GROUP);
        const int in_band = t - band * GROUP * tiles_c;
        b0 = (first + in_band % gm) * BB;
        c0 = (in_band / gm) * BC;
        return true;
    };

    const int ST = (R - 1) / kStepRows + 1;
    const int8_t* base[PER];
    Off off[PER];
    auto setup = [&](int b0, int c0) {
        int ln;
        asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(ln));
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int j = min(wave + NW * i, NB - 1);
            if (!YT && j < YB) {
                const int r = ln >> 2, c = swz_y(r, ln & 3);
                // (blocks past the last row repeat it)
                const int r0 = min(b0 + 16 * j, NBR - 1);
                base[i] = reinterpret_cast<const int8_t*>(Y + int64_t(r0) * ldy);
                off[i] = Off(min(r, NBR - 1 - r0)) * Off(ldy) * 2u + 16 * c;
            } else {
                const bool isy = j < YB;
                const int jj = isy ? j : j - YB, cg = jj >> 2, rb = jj & 3;
                const int r = ln >> 3, p = ln & 7;
                const int c = 2 * ((p >> 1) ^ (2 * ((r >> 1) & 1) + (rb & 1))) + (p & 1);
                const int o0 = isy ? b0 : c0, lim = isy ? NBR : NC;
                const int64_t ld = isy ? ldy : lda;
                base[i] = reinterpret_cast<const int8_t*>((isy ? Y : A) + o0 + 8 * rb * ld);
                off[i] = Off(r) * Off(ld) * 2u + Off(min(o0 + 64 * cg + 8 * c, lim - 8) - o0) * 2u;
            }
        }
    };
    int ring0 = 0;                              // number of the tile's first step, mod S
    auto slot = [&](int s) { return ((ring0 + s + 1) & (S - 1)) * STAGE; };
    // this wave's loads of step `step` of the tile set up last, into ring position s
    auto issue_at = [&](int s, int step) {
        int8_t* const st = smem + slot(s);
        const int64_t arow = int64_t(step) * kStepRows * lda * 2;
        const int64_t yrow = YT ? int64_t(step) * kStepRows * ldy * 2 : int64_t(step) * 64;
        const int left = R - step * kStepRows;  // rows of the step
        if (left >= kStepRows) {
#pragma unroll
            for (int i = 0; i < PER; ++i) {
                if (i == PER - 1 && !full_share) continue;
                const int j = wave + NW * i;
                dma16(base[i] + (j < YB ? yrow : arow) + uint64_t(off[i]), st + j * 1024);
            }
        } else {
            // the last, partial step: the lane's contraction index within it (its
            // row, or the first of its eight columns) past R reads zeros
#pragma unroll
            for (int i = 0; i < PER; ++i) {
                if (i == PER - 1 && !full_share) continue;
                const int j = wave + NW * i;
                const int r = !YT && j < YB ? 8 * swz_y(lane >> 2, lane & 3)
                                            : 8 * ((j < YB ? j : j - YB) & 3) + (lane >> 3);
                const int8_t* p = base[i] + (j < YB ? yrow : arow) + uint64_t(off[i]);
                if (r >= left) p = g_zero_line;
                dma16(p, st + j * 1024);
            }
        }
    };
    auto wait_batches = [&](int later) {
        if (full_share) {
            if (later >= 2) __builtin_amdgcn_s_waitcnt(vmcnt_imm(2 * PER));
            else if (later == 1) __builtin_amdgcn_s_waitcnt(vmcnt_imm(PER));
            else __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
        } else {
            if (later >= 2) __builtin_amdgcn_s_waitcnt(vmcnt_imm(2 * (PER - 1)));
            else if (later == 1) __builtin_amdgcn_s_waitcnt(vmcnt_imm(PER - 1));
            else __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
        }
    };

    // fragment addresses within a slot: transposing reads of the 16-column
    // block blk of a row-contracted operand whose blocks start at `first`
    // (+512: the other four rows of each eight); plain 16-byte reads of dy
    const int g = lane >> 4, jl = lane & 15;
    auto tr_off = [&](int first, int blk) {
        const int cg = blk >> 2, sub = blk & 3;
        const int pair = sub ^ (2 * ((jl >> 3) & 1) + (g & 1));
        return uint32_t((first + 4 * cg + g) * 1024 + (jl >> 2) * 128 + 32 * pair +
                        16 * ((jl & 3) >> 1) + 8 * (jl & 1));
    };
    uint32_t aoff[TC], ytoff[YT ? TB : 1];
#pragma unroll
    for (int a = 0; a < TC; ++a) aoff[a] = tr_off(YB, wc * TC + a);
    if constexpr (YT) {
#pragma unroll
        for (int b = 0; b < TB; ++b) ytoff[b] = tr_off(0, wb * TB + b);
    }
    const uint32_t yoff = (wb * TB) * 1024 + jl * 64 + swz_y(jl, g) * 16;
    const uint32_t sbase = lds_addr(smem);

    v4f acc[TC][TB];
    v4s al[TC], ah[TC], yl[YT ? TB : 1], yh[YT ? TB : 1];
    v8s yf[YT ? 1 : TB];
    auto read_frags = [&](int s) {
        const uint32_t sb = sbase + slot(s);
#pragma unroll
        for (int a = 0; a < TC; ++a) {
            al[a] = tr_read_at<0>(sb + aoff[a]);
            ah[a] = tr_read_at<512>(sb + aoff[a]);
        }
        if constexpr (YT) {
#pragma unroll
            for (int b = 0; b < TB; ++b) {
                yl[b] = tr_read_at<0>(sb + ytoff[b]);
                yh[b] = tr_read_at<512>(sb + ytoff[b]);
            }
        } else {
            plain_read_frags<TB>(yf, sb + yoff);
        }
    };
    auto join = [](const v4s& lo, const v4s& hi) {
        const v8s v = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        return __builtin_bit_cast(v8bf, v);
    };
    auto compute = [&]() {
        // every read has landed before any fragment is used: the wait, then an
        // empty asm per fragment that its uses cannot be scheduled above
        asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(al[0]));
#pragma unroll
        for (int a = 0; a < TC; ++a) asm volatile("" : "+v"(al[a]), "+v"(ah[a]));
        if constexpr (YT) {
#pragma unroll
            for (int b = 0; b < TB; ++b) asm volatile("" : "+v"(yl[b]), "+v"(yh[b]));
        } else {
#pragma unroll
            for (int b = 0; b < TB; ++b) asm volatile("" : "+v"(yf[b]));
        }
        v8bf af[TC];
#pragma unroll
        for (int a = 0; a < TC; ++a) af[a] = join(al[a], ah[a]);
#pragma unroll
        for (int b = 0; b < TB; ++b) {
            v8bf bf;
            if constexpr (YT) bf = join(yl[b], yh[b]);
            else bf = __builtin_bit_cast(v8bf, yf[b]);
#pragma unroll
            for (int a = 0; a < TC; ++a)
                acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[a], bf, acc[a][b], 0, 0, 0);
        }
    };
    auto barrier = [&]() {
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
    };
    // lane l of block (a, b): output row b0 + WB wb + 16b + l%16, columns c0 +
    // WC wc + 16a + 4(l/16) .. +3; 16 rows per pass through the wave's staging
    // area, 16-byte chunk c of row r at c ^ r, leaving as contiguous 16-byte stores
    auto epilogue = [&](int b0, int c0) {
        if constexpr (SL) {
            float* const part = reinterpret_cast<float*>(out) + int64_t(blockIdx.y) * sl_stride;
#pragma unroll
            for (int b = 0; b < TB; ++b) {
                const int row = b0 + wb * WB + 16 * b + (lane & 15);
#pragma unroll
                for (int a = 0; a < TC; ++a) {
                    const int col = c0 + wc * WC + 16 * a + 4 * (lane >> 4);
                    if (row < NBR && col < NC)
                        *reinterpret_cast<v4f*>(part + int64_t(row) * ldo + col) = acc[a][b];
                }
            }
            return;
        }
        int8_t* const stg = smem + (STG_OWN ? RING : slot(ST - 1)) + wave * (16 * 256);
        constexpr int CH = WC / 8, ITEMS = 16 * CH;
#pragma unroll
        for (int b = 0; b < TB; ++b) {
            const int r = lane & 15;
#pragma unroll
            for (int a = 0; a < TC; ++a) {
                const int c = 16 * a + 4 * (lane >> 4);
                const v4f v = acc[a][b];
                *reinterpret_cast<uint2*>(stg + r * 256 + (((c >> 3) ^ r) << 4) + (c & 7) * 2) =
                    make_uint2(cvt_pk_bf16(v[0], v[1]), cvt_pk_bf16(v[2], v[3]));
            }
            __builtin_amdgcn_s_waitcnt(0xC07F);                   // lgkmcnt(0)
#pragma unroll
            for (int i = 0; i < (ITEMS + 63) / 64; ++i) {
                const int flat = i * 64 + lane, rr = flat / CH, c = flat % CH;
                if (ITEMS % 64 == 0 || flat < ITEMS) {
                    const uint4 v = *reinterpret_cast<const uint4*>(stg + rr * 256 + ((c ^ rr) << 4));
                    const int row = b0 + wb * WB + 16 * b + rr, col = c0 + wc * WC + 8 * c;
                    if (row < NBR && col < NC)
                        *reinterpret_cast<uint4*>(out + int64_t(row) * ldo + col) = v;
                }
            }
            __builtin_amdgcn_s_waitcnt(0xC07F);                   // reads done before reuse
        }
    };

    int ti = blockIdx.x, b0, c0;
    if (!tile_origin(ti, b0, c0)) return;
    setup(b0, c0);
    for (int s = 0; s < S - 1; ++s)
        if (s < ST) issue_at(s, s);
    wait_batches(min(S - 2, ST - 1));
    barrier();
    for (;;) {
#pragma unroll
        for (int a = 0; a < TC; ++a)
#pragma unroll
            for (int b = 0; b < TB; ++b) acc[a][b] = v4f{0.f, 0.f, 0.f, 0.f};
        const int tnext = ti + int(gridDim.x);
        int b0n = 0, c0n = 0;
        const bool more = tile_origin(tnext, b0n, c0n);
        // with a next tile the loads of its steps 0-2 go out in this tile's last
        // three steps, so the ring never drains
        const bool cont = more && ST >= S - 1;
        const int smain = cont ? ST - (S - 1) : ST;
        if (grp == 0) {
            read_frags(0);
            barrier();
#pragma clang loop unroll(disable)
            for (int s = 0; s < smain; ++s) {
                compute();                                      // A(s)
                if (s + 1 < ST) wait_batches(min(S - 3, ST - 2 - s));
                barrier();
                if (s + 1 < ST) read_frags(s + 1);              // B(s)
                if (s + S - 1 < ST) issue_at(s + S - 1, s + S - 1);
                barrier();
            }
            if (cont) {
                setup(b0n, c0n);
#pragma clang loop unroll(disable)
                for (int s = smain; s < ST; ++s) {
                    compute();                                  // A(s)
                    if (s + 1 < ST) wait_batches(S - 3);
                    barrier();
                    if (s + 1 < ST) read_frags(s + 1);          // B(s)
                    issue_at(s + S - 1, s + S - 1 - ST);
                    barrier();
                }
            }
        } else {
            barrier();
#pragma clang loop unroll(disable)
            for (int s = 0; s < smain; ++s) {
                read_frags(s);                                  // A(s)
                if (s + S - 1 < ST) issue_at(s + S - 1, s + S - 1);
                if (s + 1 < ST) wait_batches(min(S - 2, ST - 2 - s));
                barrier();
                compute();                                      // B(s)
                barrier();
            }
            if (cont) {
                setup(b0n, c0n);
#pragma clang loop unroll(disable)
                for (int s = smain; s < ST; ++s) {
                    read_frags(s);                              // A(s)
                    issue_at(s + S - 1, s + S - 1 - ST);
                    if (s + 1 < ST) wait_batches(S - 2);
                    barrier();
                    compute();                                  // B(s)
                    barrier();
                }
            }
        }
        // every fragment read has completed; with too few steps for the loop to
        // have issued the next tile's first loads, they go out here
        if (more && !cont) {
            setup(b0n, c0n);
            for (int s = 0; s < S - 1; ++s)
                if (s < ST) issue_at(ST + s, s);
        }
        epilogue(b0, c0);
        if (!more) break;
        __builtin_amdgcn_s_waitcnt(0);                          // stores, loads, LDS all done
        barrier();
        ring0 = (ring0 + ST) & (S - 1);
        ti = tnext;
        b0 = b0n;
        c0 = c0n;
    }
}

// out[m, k] = bf16(sum over s of part[s][m, k]), the slices added in order in
// fp32; four columns per thread (K % 4 == 0), grid-stride.
__global__ __launch_bounds__(256) void sum_slices_bf16_kernel(const float* __restrict__ part,
                                                              int nsl, int64_t sl_stride,
                                                              uint16_t* __restrict__ out,
                                                              int64_t ldo, int64_t M, int64_t K) {
    const int64_t q = K / 4, total = M * q;
    for (int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; t < total;
         t += int64_t(gridDim.x) * blockDim.x) {
        const int64_t m = t / q, k = (t - m * q) * 4;
        const float* p = part + m * K + k;
        float4 v = *reinterpret_cast<const float4*>(p);
        for (int s = 1; s < nsl; ++s) {
            const float4 w = *reinterpret_cast<const float4*>(p + s * sl_stride);
            v.x = v.x + w.x; v.y = v.y + w.y; v.z = v.z + w.z; v.w = v.w + w.w;
        }
        *reinterpret_cast<uint2*>(out + m * ldo + k) =
            make_uint2(cvt_pk_bf16(v.x, v.y), cvt_pk_bf16(v.z, v.w));
    }
}

}  // namespace

// Whether a product takes the split-K kernel: a contraction of whole 32-row
// steps long enough for two teams, and enough bb x 160 tiles to fill the chip
// in one round.  (The byte offsets of the row-contracted operands, up to R rows,
// stay below 2^32.)
static bool bf16_splitk_applies(int nb, int bb, int R, int K, int64_t lda, int64_t ldy, bool yt) {
    if (nb <= 64 || R % kStepRows || R < 2048 || K % 8 || (yt && nb % 8)) return false;
    if (int64_t(R) * lda * 2 >= (int64_t(1) << 32)) return false;
    if (yt && int64_t(R) * ldy * 2 >= (int64_t(1) << 32)) return false;
    if (!yt && int64_t(bb) * ldy * 2 >= (int64_t(1) << 32)) return false;
    const int64_t tiles = int64_t((nb + bb - 1) / bb) * ((K + 159) / 160);
    return tiles >= 128 && tiles <= 256;
}

// The persistent kernel's tiles of out[b, c], by index; 256 x 320 is taken for
// the dx only and 256 x 256 for dW only (whose transposing reads of both
// operands need the registers), 256 x 320 and 192 x 256 for whole contractions
// only.
struct Bf16Tile {
    int bb, bc;
};
constexpr Bf16Tile kBf16Tiles[] = {{256, 320}, {256, 256}, {192, 256},
                                   {128, 256}, {128, 192}, {128, 128}};
constexpr int kBf16FirstSliced = 3, kBf16MaxSlices = 8;

struct Bf16Plan {
    int tile, slices, slice;    // slice: rows of the contraction per slice
};

// The tile and the contraction slices with the least predicted time.  rounds of
// tiles, each the slice's 32-row steps (0.066 us per 10^4 outputs for the dx,
// 0.073 for dW, whose operands both come through transposing reads, plus 0.24 /
// 0.27 us of barriers, waits and load issue) and an epilogue; slices add their
// fp32 stores and a pass that reads them back.  Fitted to eight tiles and up to
// eight slices on 110 products (M 128-4096, N 512-10240, K 512-5120; scatter 6%
// for the dx, 4% for dW); choosing by it is 0.6% and 0.5% off the fastest of them on
// average.  Against the 128 x 128 kernels and the power-of-two slices
// it replaces, us:
//   dx 4096 x 1280 x 5120 (M, N, K)  83.7 -> 53.0 (256 x 320, one round)
//   dx 3682 x 3248 x 4864            176.4 -> 104.2
//   dx 322 x 5648 x 2048             87.9 -> 26.4 (128 x 128, four slices)
//   dx 205 x 2672 x 768              51.1 -> 14.9 (2672 % 32 kept it unsplit)
//   dW 2893 x 544 x 768 (M, N, K)    46.0 -> 17.2 (eight slices)
//   dW 1970 x 672 x 512              32.1 -> 16.3
// and over all 110 1.69 times as fast (dx) and 1.23 (dW).
// work: the bytes of fp32 partial sums that may be used.
static Bf16Plan bf16_plan(int64_t nbr, int64_t nc, int R, bool yt, int64_t work) {
    const double c0 = yt ? 3.98 : 4.57, mm = yt ? 0.0732 : 0.0658, st = yt ? 0.273 : 0.238,
                 fs = yt ? 0.97 : 0.947, ep = yt ? 0.92 : 1.26, fe = yt ? 0.18 : 0.0,
                 s0 = yt ? 4.5 : 2.5, sp = yt ? 0.8e-6 : 0.85e-6, se = yt ? 0.51 : 0.91;
    const int64_t cus = device_cus();
    Bf16Plan best{5, 1, R};
    double time = 0;
    for (int i = 0; i < int(sizeof(kBf16Tiles) / sizeof(kBf16Tiles[0])); ++i) {
        if (i == (yt ? 0 : 1)) continue;
        const int64_t bb = kBf16Tiles[i].bb, bc = kBf16Tiles[i].bc;
        const int64_t tiles = ((nbr + bb - 1) / bb) * ((nc + bc - 1) / bc);
        const double area = 1e-4 * double(bb * bc);
        for (int n = 1; n <= (i < kBf16FirstSliced ? 1 : kBf16MaxSlices); ++n) {
            const int len = n == 1 ? R : int((int64_t(R) + n - 1) / n + 31) / 32 * 32;
            if (n > 1 && (len < 128 || (R - 1) / len + 1 != n || n * nbr * nc * 4 > work)) continue;
            const int64_t rounds = ((tiles + 7) / 8 * n + cus / 8 - 1) / (cus / 8);
            const double fill = double(tiles * n) / double(cus * rounds);
            double t = c0 + double(rounds) * (((len - 1) / 32 + 1) * (mm * area + st) *
                                                  (fs + (1 - fs) * fill) +
                                              ep * area * (fe + (1 - fe) * fill));
            if (n > 1) t += s0 + sp * double(nbr) * double(nc) * n + double(rounds) * se * area;
            if (time == 0 || t < time) best = Bf16Plan{i, n, len}, time = t;
        }
    }
    return best;
}

int64_t bf16_dx_work_bytes(int M, int N, int K) {
    if (bf16_splitk_applies(M, 128, N, K, K, N, false)) return 0;
    const int n = bf16_plan(M, K, N, false, int64_t(1) << 62).slices;
    return n > 1 ? int64_t(n) * M * K * 4 : 0;
}
int64_t bf16_dw_work_bytes(int R, int N, int K) {
    if (bf16_splitk_applies(N, 160, R, K, K, N, true)) return 0;
    const int n = bf16_plan(N, K, R, true, int64_t(1) << 62).slices;
    return n > 1 ? int64_t(n) * N * K * 4 : 0;
}

GemmChoice bf16_choice(int nbr, int nc, int R, bool yt) {
    if (bf16_splitk_applies(nbr, yt ? 160 : 128, R, nc, nc, yt ? nbr : R, yt))
        return GemmChoice{kSplitKKernel, yt ? 160 : 128, 160, 1};
    const Bf16Plan p = bf16_plan(nbr, nc, R, yt, int64_t(1) << 62);
    return GemmChoice{kPersistentKernel, kBf16Tiles[p.tile].bb, kBf16Tiles[p.tile].bc, p.slices};
}

// out[b, c] = sum over r of a[r, c] * y (y[b, r], or y[r, b] with YT) on the
// persistent kernel by the plan
template <bool YT>
static hipError_t launch_bf16_pp(hipStream_t st, const uint16_t* a, int64_t lda, const uint16_t* y,
                                 int64_t ldy, uint16_t* out, int64_t ldo, int R, int nc, int nbr,
                                 float* part, int64_t part_bytes) {
    const bool wide = std::max(lda, ldy) >= (int64_t(1) << 27);
    const Bf16Plan p =
        wide ? Bf16Plan{5, 1, R} : bf16_plan(nbr, nc, R, YT, part ? part_bytes : 0);
    const int bb = kBf16Tiles[p.tile].bb, bc = kBf16Tiles[p.tile].bc;
    const int tb = (nbr + bb - 1) / bb, tc = (nc + bc - 1) / bc;
    const int64_t tiles = int64_t(tb) * tc;
    const dim3 grid(unsigned(std::min<int64_t>((tiles + 7) / 8 * 8, device_cus() / 8 * 8)),
                    unsigned(p.slices));
    const int64_t stride = int64_t(nbr) * nc;
#define XPU_BF16_PP(BB, BC, WGM, SL, ...)                                                         \
    hipLaunchKernelGGL((gemm_bf16_pp_kernel<BB, BC, WGM, YT, SL, ##__VA_ARGS__>), grid,          \
                       dim3(512), 0, st, a, lda, y, ldy,                                           \
                       SL ? reinterpret_cast<uint16_t*>(part) : out, SL ? int64_t(nc) : ldo, R,   \
                       nc, nbr, tb, tc, p.slice, stride)
    if (wide) {
        XPU_BF16_PP(128, 128, 2, false, uint64_t);
    } else if (p.slices > 1) {
        switch (p.tile) {
            case 3: XPU_BF16_PP(128, 256, 2, true); break;
            case 4: XPU_BF16_PP(128, 192, 2, true); break;
            default: XPU_BF16_PP(128, 128, 2, true); break;
        }
        if (const hipError_t e = hipGetLastError(); e != hipSuccess) return e;
        int64_t blocks = (int64_t(nbr) * (nc / 4) + 255) / 256;
        if (blocks > (int64_t(1) << 20)) blocks = int64_t(1) << 20;
        hipLaunchKernelGGL(sum_slices_bf16_kernel, dim3(unsigned(blocks)), dim3(256), 0, st, part,
                           p.slices, stride, out, ldo, int64_t(nbr), int64_t(nc));
    } else {
        switch (p.tile) {
            case 0:
                if constexpr (!YT) XPU_BF16_PP(256, 320, 2, false);
                break;
            case 1:
                if constexpr (YT) XPU_BF16_PP(256, 256, 2, false);
                break;
            case 2: XPU_BF16_PP(192, 256, 2, false); break;
            case 3: XPU_BF16_PP(128, 256, 2, false); break;
            case 4: XPU_BF16_PP(128, 192, 2, false); break;
            default: XPU_BF16_PP(128, 128, 2, false); break;
        }
    }
#undef XPU_BF16_PP
    return hipGetLastError();
}

// The workspace that xpuint8_linear_dx_workspace_size names: fp32 partial sums
// of the fewest power-of-two slices giving 192 blocks of 128 x 160 tiles where
// those number below 128 (each slice a whole number of 32-row steps and at least
// 1024 rows); 0 slices when none applies.  The product splits its contraction as
// bf16_plan finds best within the workspace it is given.
int bf16_nn_slices(int M, int N, int K) {
    if (M <= 64 || K % 8 || N % kStepRows) return 0;
    const int64_t tiles = int64_t((M + 127) / 128) * ((K + 159) / 160);
    if (tiles >= 128) return 0;
    int s = 1;
    while (tiles * s < 192 && (N / kStepRows) % (2 * s) == 0 && N / (2 * s) >= 1024) s *= 2;
    if (s == 1) return 0;
    if (int64_t(N / s) * K * 2 >= (int64_t(1) << 32) || 128 * int64_t(N) * 2 >= (int64_t(1) << 31))
        return 0;
    return s;
}

hipError_t gemm_bf16_nn(hipStream_t st, const void* dy, int64_t ldy, const void* w, int64_t ldw,
                        void* out, int64_t ldo, int M, int N, int K, float* part,
                        int64_t part_bytes) {
    const uint16_t* a = static_cast<const uint16_t*>(w);
    const uint16_t* y = static_cast<const uint16_t*>(dy);
    if (bf16_splitk_applies(M, 128, N, K, ldw, ldy, false)) {
        const int tm = (M + 127) / 128, tk = (K + 159) / 160;
        hipLaunchKernelGGL((gemm_bf16_splitk_kernel<4, false>), dim3(unsigned(tm * tk)), dim3(512),
                           0, st, a, ldw, y, ldy, static_cast<uint16_t*>(out), ldo, N, K, M, tm, tk);
        return hipGetLastError();
    }
    return launch_bf16_pp<false>(st, a, ldw, y, ldy, static_cast<uint16_t*>(out), ldo, N, K, M,
                                 part, part_bytes);
}

hipError_t gemm_bf16_tn(hipStream_t st, const void* dy, int64_t ldy, const void* x, int64_t ldx,
                        void* dw, int64_t ldo, int R, int N, int K, float* part,
                        int64_t part_bytes) {
    constexpr int STAGES_TN = 4;                // 2 x 4 x 20 KB of LDS
    const uint16_t* a = static_cast<const uint16_t*>(x);
    const uint16_t* y = static_cast<const uint16_t*>(dy);
    if (bf16_splitk_applies(N, 160, R, K, ldx, ldy, true)) {
        const int tn = (N + 159) / 160, tk = (K + 159) / 160;
        hipLaunchKernelGGL((gemm_bf16_splitk_kernel<STAGES_TN, true>), dim3(unsigned(tn * tk)),
                           dim3(512), 0, st, a, ldx, y, ldy, static_cast<uint16_t*>(dw), ldo, R, K,
                           N, tn, tk);
        return hipGetLastError();
    }
    return launch_bf16_pp<true>(st, a, ldx, y, ldy, static_cast<uint16_t*>(dw), ldo, R, K, N, part,
                                part_bytes);
}

}  // namespace xpuint8

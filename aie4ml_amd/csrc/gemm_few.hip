// Dense, and MatMul in the floating-point formats, with few output tiles: small batches (inference on one to some hundred rows) and narrow
// layers.
//
// The tiled kernels give one workgroup a 128 x 128 (or larger) output tile and all of K: 16 rows of a 4096 x 4096 layer are 32
// such tiles, each a chain of 32 K tiles, and nine tenths of the chip idle. Here a workgroup takes a tile of 16 to 64 rows and columns,
// and its waves share K between them: wave w reduces the 128-byte K tiles w, w + NW, .. into accumulators of its own, straight from
// global memory (operands are read once per workgroup, so there is nothing for LDS to share), several tiles ahead; the
// partial sums meet in LDS, where every thread finishes four neighbouring outputs. Integer sums wrap, so the split changes no bit;
// floating-point sums get another order, as with any tiling.
// Bound by the latency of the loads (16 x 4096 -> 4096: waves wait on counters 44 % of their time, the matrix unit is busy 1 %).
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "float_formats.hpp"
#include "gemm_few.hpp"
#include "round64.hpp"

namespace a4g {

template <int KIND>
struct FewOps {
    static constexpr bool FLOAT = KIND == FEW_BF16 || KIND == FEW_F32 || KIND == FEW_FP8;
    static constexpr bool WIDE_A = KIND == FEW_I16X8 || KIND == FEW_I16X16;  // two bytes an element of A, one a plane of B
    static constexpr bool PLANES_B = KIND == FEW_I16X16;
    static constexpr int SUMS = KIND == FEW_I16X16 ? 3 : 1;  // accumulators that reach the epilogue
    using acc_t = std::conditional_t<FLOAT, v4f, v4i>;
};

// eight int16 pairs -> signed high bytes and low bytes less 128, in order
__device__ __forceinline__ void split_planes(const v4i& x, const v4i& y, v4i& hi, v4i& lo) {
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const unsigned w0 = static_cast<unsigned>(t < 2 ? x[2 * t] : y[2 * t - 4]), w1 = static_cast<unsigned>(t < 2 ? x[2 * t + 1] : y[2 * t - 3]);
        hi[t] = static_cast<int>(__builtin_amdgcn_perm(w1, w0, 0x07050301u));
        lo[t] = static_cast<int>(__builtin_amdgcn_perm(w1, w0, 0x06040200u) ^ 0x80808080u);
    }
}

// NW waves share K; the tile is TM x TN blocks of 16 x 16. DEPTH K tiles of a wave are on their way or in use.
// WF: the weights also lie in fragment order (a4g_rowpack_weights_i8: 1 KiB per 32 columns and 32 bytes of k, whole 128-byte tiles,
// zeros behind the end): a fragment is four contiguous runs of 256 bytes and needs no turn through LDS.
template <int KIND, int NW, int TM, int TN, int DEPTH, bool WF>
__global__ __launch_bounds__(NW * 64) void gemm_few_kernel(GemmArgs g, int tiles_m) {
    static_assert(!WF || KIND == FEW_I8, "fragment order is the int8 weights'");
    using O = FewOps<KIND>;
    using acc_t = typename O::acc_t;  // of a 16 x 16 block: four neighbouring columns of the lane's row
    constexpr int NA = O::WIDE_A ? 4 : 2;                     // 16-byte chunks of A per lane, block and K tile
    constexpr int ACCS = KIND == FEW_I16X8 ? 2 : O::SUMS;     // accumulators a wave keeps per block
    constexpr int GROUPS = TM * TN * 64;                      // groups of four neighbouring outputs of the tile
    constexpr int PER_THREAD = (GROUPS + NW * 64 - 1) / (NW * 64);
    extern __shared__ __attribute__((aligned(16))) int8_t few_smem[];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int frow = lane & 15, quarter = lane >> 4;
    // an XCD takes consecutive tiles, rows fastest: the tiles that share weights find them in one L2
    const int cols = WF ? (g.N + 31) / 32 * 32 : g.N;  // fragment order mixes the columns of a group of 32
    const int tiles_n = (cols + TN * 16 - 1) / (TN * 16), tiles = tiles_m * tiles_n;
    const int tile = tiles < 8 ? static_cast<int>(blockIdx.x) : static_cast<int>((blockIdx.x & 7) * ((tiles + 7) / 8) + blockIdx.x / 8);  // grid_for_tiles
    if (tile >= tiles) return;
    const int m0 = tile % tiles_m * (TM * 16), n0 = tile / tiles_m * (TN * 16);

    const int ka = O::WIDE_A ? 2 * g.K : g.K, kb = g.K;  // bytes of a row of A, of a row of (a plane of) B
    const int lda = static_cast<int>(g.lda), ldb = static_cast<int>(g.ldb);
    // rows past the end of a matrix lie outside its descriptor and read as zero
    const auto rsrc_a = __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(g.A + blockIdx.y * g.stride_a + static_cast<int64_t>(m0) * g.lda), 0,
                                                          (min(TM * 16, g.M - m0) - 1) * lda + ka, 0x00020000);
    const int b_range = (min(TN * 16, g.N - n0) - 1) * ldb + (kb + 15) / 16 * 16;
    const int64_t b_at = blockIdx.y * g.stride_b + static_cast<int64_t>(n0) * g.ldb;
    const int ktiles = (kb + 127) / 128;
    const auto rsrc_b = __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(WF ? g.Wf : g.Bt + b_at), 0, WF ? (g.N + 31) / 32 * ktiles * 4096 : b_range, 0x00020000);
    const auto rsrc_b2 = __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>((O::PLANES_B ? g.Bt_lo : g.Bt) + b_at), 0, b_range, 0x00020000);

    // ---- operands of a K tile (128 bytes of a row of B): a load takes whole 128-byte lines (eight lanes a line, 256 bytes and
    // sixteen lanes for two-byte elements), goes to the wave's own patch of LDS and is read back as fragments: lane
    // (row, quarter) the 16 bytes of k at 64 c + 16 quarter, c = 0, 1. Fragments straight from memory touch 16 lines for 64 bytes
    // each and ran at half the rate (64 x 4096 -> 4096 int8: 10.3 us, 6.8 this way). The chunk of A that crosses the end of a row
    // is fetched as the row's last 16 bytes, see gemm_rs_kernel; chunks past the end read as zero, and so do the tiles past
    // the wave's last one that the ring asks for.
    constexpr unsigned NOWHERE = 0x80000000u;
    constexpr int CPA = O::WIDE_A ? 16 : 8;  // 16-byte chunks of a row of A in a K tile
    constexpr int RPA = 64 / CPA, LA = TM * 16 / RPA, LB = TN * 2, PLANES = O::PLANES_B ? 2 : 1;
    constexpr int PATCH_A = TM * 16 * CPA * 16, PATCH_B = WF ? 0 : TN * 16 * 128, PATCH = PATCH_A + PLANES * PATCH_B;
    const int arow = lane / CPA, achunk = lane % CPA, brow = lane >> 3, bchunk = lane & 7;
    int8_t* const patch = few_smem + wave * PATCH;
    // The patch as it is read. A lane reads what other lanes wrote, and the compiler, which follows one lane's addresses, moved reads
    // ahead of writes that it could tell apart from them; behind an offset that it cannot see (0) every read may meet every write, so
    // they stay in order, and LDS instructions of a wave complete in order. (A wavefront fence also holds back the loads from
    // memory: 732 x 5120 -> 1800 fp8 22.0 us, 24.0 with one.)
    int opaque = 0;
    asm volatile("" : "+v"(opaque));
    const int8_t* const patch_in = patch + opaque;
    // chunk c of row r lies at chunk c ^ ((r >> 1) & 7) (two-byte rows: c ^ (r & 15)): sixteen rows' fragments touch all banks
    auto swz_a = [](int r) { return O::WIDE_A ? r & 15 : (r >> 1) & 7; };
    v4i ra[DEPTH][LA], rb[DEPTH][PLANES][LB];
    // column of the first of the four outputs that lane quarter q of the tile's block j of 16 holds: in order, or, in fragment
    // order, the columns that operand rows 16 h + 4 q .. of the group of 32 stand for (direct_col_of_operand_row)
    auto column = [&](int j, int q) {
        const int blk = (n0 >> 4) + j;
        return WF ? (blk >> 1) * 32 + direct_col_of_operand_row((blk & 1) * 16 + 4 * q) : n0 + 16 * j + 4 * q;
    };
    auto load_tile = [&](int slot, int kt) __attribute__((always_inline)) {
        const int kbyte = kt * 128 + bchunk * 16;
        const unsigned off_b = kbyte < kb ? static_cast<unsigned>(brow * ldb + kbyte) : NOWHERE;
#pragma unroll
        for (int j = 0; j < LB; ++j) {
            if constexpr (WF) {  // chunk c = j & 1 of block j >> 1
                const int blk = (n0 >> 4) + (j >> 1);
                const int at = (((blk >> 1) * ktiles + kt) * 4 + 2 * (j & 1) + (quarter >> 1)) * 1024 + ((quarter & 1) * 32 + (blk & 1) * 16 + frow) * 16;
                rb[slot][0][j] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rsrc_b, kt < ktiles ? static_cast<unsigned>(at) : NOWHERE, 0, 0));
                continue;
            }
            rb[slot][0][j] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rsrc_b, off_b + j * 8 * ldb, 0, 0));
            if constexpr (O::PLANES_B)
                rb[slot][1][j] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rsrc_b2, off_b + j * 8 * ldb, 0, 0));
        }
        const int at = kt * CPA * 16 + achunk * 16;
        const unsigned off_a = at < ka ? static_cast<unsigned>(arow * lda + min(at, ka - 16)) : NOWHERE;
#pragma unroll
        for (int i = 0; i < LA; ++i)
            ra[slot][i] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rsrc_a, off_a + i * RPA * lda, 0, 0));
    };
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) load_tile(d, wave + d * NW);

    // what the thread's outputs need besides the sums
    int par_add[PER_THREAD][4], par_shift[PER_THREAD][4], par_cols[PER_THREAD][4];
    v4f par_bias[PER_THREAD];
    const int32_t* colsum = (g.a_unsigned || O::WIDE_A) ? g.colsum + blockIdx.y * g.stride_colsum : nullptr;
#pragma unroll
    for (int p = 0; p < PER_THREAD; ++p) {
        const int idx = tid + p * NW * 64;
        const int n = column((idx >> 6) % TN, quarter);
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const int nn = min(n + t, g.N - 1);
            if constexpr (O::FLOAT) {
                par_bias[p][t] = g.bias ? reinterpret_cast<const float*>(g.bias)[nn] : 0.f;
            } else {
                par_add[p][t] = g.bias ? g.bias[nn] : 0;
                par_cols[p][t] = colsum ? colsum[nn] : 0;
                par_shift[p][t] = g.shifts ? g.shifts[static_cast<int64_t>(nn) * g.shift_stride] : g.shift;
            }
        }
    }

    acc_t acc[TM][TN][ACCS];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int s = 0; s < ACCS; ++s) acc[i][j][s] = acc_t{0, 0, 0, 0};
    int row_sum[TM] = {};  // FEW_I16X16: sum of the lane's activations

    const int flip = g.a_unsigned ? static_cast<int>(0x80808080u) : 0;
    // the K tile that crosses the end of the rows: what lies behind them goes, what belongs to them moves into place
    auto finish_rows = [&](int slot, int kt) __attribute__((always_inline)) {
        if (kt == ktiles - 1) {  // wave-uniform, and no load inside
            const int at = kt * CPA * 16 + achunk * 16;
#pragma unroll
            for (int i = 0; i < LA; ++i)
                if (at < ka) ra[slot][i] = chunk_in_place(ra[slot][i], ka - at, ka);
            if constexpr (O::FLOAT) {  // what lies between K and the next chunk of a MatMul's operand is not its own: 0 * NaN
                const int rem = kb - (kt * 128 + bchunk * 16);
#pragma unroll
                for (int j = 0; j < LB; ++j)
#pragma unroll
                    for (int t = 0; t < 4; ++t) {
                        const int v = rem - 4 * t;  // bytes of this dword that belong to K
                        if (v <= 0) rb[slot][0][j][t] = 0;
                        else if (v < 4) rb[slot][0][j][t] &= static_cast<int>((1u << (8 * v)) - 1u);
                    }
            }
        }
    };
    v4i fa[TM][NA], fb[PLANES][TN][2];  // fragments of the tile in hand
    // Registers of a tile -> the wave's patch -> fragments, in blocks of sixteen rows. The 64 x 64 tiles have one K tile on its way: a
    // block is read back as soon as its rows have arrived (447 x 4736 -> 2295 fp8 15.6 us, 17.6 with all writes ahead of all reads). So do
    // bfloat16 and float32 (200 sizes each 1.5 and 0.8 % faster); int8 on 32 x 32 tiles would lose its fourth wave per SIMD to it (20 %).
    constexpr bool BLOCKS = TM == 4 || KIND == FEW_BF16 || KIND == FEW_F32;
    auto put_a = [&](int slot, int i) __attribute__((always_inline)) {
#pragma unroll
        for (int t = i * (LA / TM); t < (i + 1) * (LA / TM); ++t) {
            const int r = arow + t * RPA;
            *reinterpret_cast<v4i*>(patch + r * CPA * 16 + ((achunk ^ swz_a(r)) * 16)) = ra[slot][t];
        }
    };
    auto get_a = [&](int i, int c) __attribute__((always_inline)) {
        const int chunk = O::WIDE_A ? (c >> 1) * 8 + quarter * 2 + (c & 1) : c * 4 + quarter;
        fa[i][c] = *reinterpret_cast<const v4i*>(patch_in + (i * 16 + frow) * CPA * 16 + ((chunk ^ swz_a(frow)) * 16));
    };
    auto put_b = [&](int slot, int j) __attribute__((always_inline)) {
#pragma unroll
        for (int p = 0; p < (WF ? 0 : PLANES); ++p)
#pragma unroll
            for (int t = 2 * j; t < 2 * j + 2; ++t) {
                const int r = brow + t * 8;
                *reinterpret_cast<v4i*>(patch + PATCH_A + p * PATCH_B + r * 128 + ((bchunk ^ ((r >> 1) & 7)) * 16)) = rb[slot][p][t];
            }
    };
    auto get_b = [&](int slot, int p, int j, int c) __attribute__((always_inline)) {
        fb[p][j][c] = WF ? rb[slot][0][2 * j + c] : *reinterpret_cast<const v4i*>(patch_in + PATCH_A + p * PATCH_B + (j * 16 + frow) * 128 + (((c * 4 + quarter) ^ ((frow >> 1) & 7)) * 16));
    };
    auto multiply = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int c = 0; c < 2; ++c) {
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                v4i a[2];
                if constexpr (O::WIDE_A) {
                    const v4i x = fa[i][2 * c], y = fa[i][2 * c + 1];
                    split_planes(x, y, a[0], a[1]);
                    if constexpr (KIND == FEW_I16X16) {
                        typedef short v2s __attribute__((ext_vector_type(2)));
                        constexpr v2s ones = {1, 1};
#pragma unroll
                        for (int t = 0; t < 4; ++t) {
                            const int wx = x[t], wy = y[t];
                            row_sum[i] = __builtin_amdgcn_sdot2(__builtin_bit_cast(v2s, wx), ones, row_sum[i], false);
                            row_sum[i] = __builtin_amdgcn_sdot2(__builtin_bit_cast(v2s, wy), ones, row_sum[i], false);
                        }
                    }
                } else {
                    a[0] = fa[i][c];
                    if constexpr (KIND == FEW_I8) a[0] ^= flip;  // uint8 -> int8; 128 * colsum is added at the end
                }
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    const v4i& b = fb[0][j][c];
                    acc_t(&s)[ACCS] = acc[i][j];
                    if constexpr (KIND == FEW_I8) {
                        s[0] = __builtin_amdgcn_mfma_i32_16x16x64_i8(b, a[0], s[0], 0, 0, 0);
                    } else if constexpr (KIND == FEW_I16X8) {
                        s[0] = __builtin_amdgcn_mfma_i32_16x16x64_i8(b, a[0], s[0], 0, 0, 0);
                        s[1] = __builtin_amdgcn_mfma_i32_16x16x64_i8(b, a[1], s[1], 0, 0, 0);
                    } else if constexpr (KIND == FEW_I16X16) {
                        const v4i& bl = fb[1][j][c];
                        s[0] = __builtin_amdgcn_mfma_i32_16x16x64_i8(b, a[0], s[0], 0, 0, 0);
                        s[1] = __builtin_amdgcn_mfma_i32_16x16x64_i8(bl, a[0], s[1], 0, 0, 0);  // hl and lh share a sum: 2 * 2^29
                        s[2] = __builtin_amdgcn_mfma_i32_16x16x64_i8(bl, a[1], s[2], 0, 0, 0);
                        s[1] = __builtin_amdgcn_mfma_i32_16x16x64_i8(b, a[1], s[1], 0, 0, 0);
                    } else if constexpr (KIND == FEW_BF16) {
                        s[0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, b), __builtin_bit_cast(v8bf, a[0]), s[0], 0, 0, 0);
                    } else if constexpr (KIND == FEW_F32) {
                        const v4f bf = __builtin_bit_cast(v4f, b), af = __builtin_bit_cast(v4f, a[0]);
#pragma unroll
                        for (int t = 0; t < 4; ++t) s[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(bf[t], af[t], s[0], 0, 0, 0);
                    } else if (c == 0) {  // fp8: the tile's 128 bytes of k at once, both chunks of a lane per operand
                        typedef int v8i __attribute__((ext_vector_type(8)));
                        const v4i &b1 = fb[0][j][1], &a1 = fa[i][1];
                        const v8i bw = {b[0], b[1], b[2], b[3], b1[0], b1[1], b1[2], b1[3]};
                        const v8i aw = {a[0][0], a[0][1], a[0][2], a[0][3], a1[0], a1[1], a1[2], a1[3]};
                        s[0] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(bw, aw, s[0], 0, 0, 0, 0, 0, 0);
                    }
                }
            }
        }
    };
    for (int base = wave; base < ktiles; base += DEPTH * NW) {
#pragma unroll
        for (int d = 0; d < DEPTH; ++d) {
            finish_rows(d, base + d * NW);
            if constexpr (BLOCKS) {
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    put_b(d, j);
#pragma unroll
                    for (int c = 0; c < 2; ++c)
#pragma unroll
                        for (int p = 0; p < PLANES; ++p) get_b(d, p, j, c);
                }
#pragma unroll
                for (int i = 0; i < TM; ++i) {
                    put_a(d, i);
#pragma unroll
                    for (int c = 0; c < NA; ++c) get_a(i, c);
                }
            } else {
#pragma unroll
                for (int i = 0; i < TM; ++i) put_a(d, i);
#pragma unroll
                for (int j = 0; j < TN; ++j) put_b(d, j);
            }
            if constexpr (!WF) load_tile(d, base + (d + DEPTH) * NW);  // past the wave's last tile: zeros
            if constexpr (!BLOCKS) {
#pragma unroll
                for (int c = 0; c < NA; ++c)
#pragma unroll
                    for (int i = 0; i < TM; ++i) get_a(i, c);
#pragma unroll
                for (int c = 0; c < 2; ++c)
#pragma unroll
                    for (int p = 0; p < PLANES; ++p)
#pragma unroll
                        for (int j = 0; j < TN; ++j) get_b(d, p, j, c);
            }
            multiply();
            if constexpr (WF) load_tile(d, base + (d + DEPTH) * NW);  // the weights' registers were operands
        }
    }

    // ---- the waves' sums meet in LDS, where the patches were: group (block, lane) of sum s of wave w
    __syncthreads();
    acc_t* part = reinterpret_cast<acc_t*>(few_smem);
    int* part_rows = reinterpret_cast<int*>(few_smem + NW * O::SUMS * GROUPS * 16);
#pragma unroll
    for (int i = 0; i < TM; ++i) {
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            if constexpr (KIND == FEW_I16X8) {  // a.w = 256 sum(hi.w) + sum((lo - 128).w) + 128 sum(w), wrapping
#pragma unroll
                for (int t = 0; t < 4; ++t)
                    acc[i][j][0][t] = static_cast<int>((static_cast<unsigned>(acc[i][j][0][t]) << 8) + static_cast<unsigned>(acc[i][j][1][t]));
            }
#pragma unroll
            for (int s = 0; s < O::SUMS; ++s) part[(wave * O::SUMS + s) * GROUPS + (i * TN + j) * 64 + lane] = acc[i][j][s];
        }
        if constexpr (KIND == FEW_I16X16) part_rows[(wave * TM + i) * 64 + lane] = row_sum[i];
    }
    __syncthreads();

    const int lo = g.relu ? max(kind_lo(g.out_kind), 0) : kind_lo(g.out_kind), hi = kind_hi(g.out_kind);
#pragma unroll
    for (int p = 0; p < PER_THREAD; ++p) {
        const int idx = tid + p * NW * 64;
        if (GROUPS % (NW * 64) != 0 && idx >= GROUPS) return;
        const int blk = idx >> 6, i = blk / TN, j = blk % TN;
        const int m = m0 + i * 16 + frow, n = column(j, quarter);
        acc_t sum[O::SUMS];
#pragma unroll
        for (int s = 0; s < O::SUMS; ++s) {
            sum[s] = part[s * GROUPS + idx];
#pragma unroll
            for (int w = 1; w < NW; ++w) {
                const acc_t v = part[(w * O::SUMS + s) * GROUPS + idx];
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    if constexpr (O::FLOAT) sum[s][t] += v[t];
                    else sum[s][t] = static_cast<int>(static_cast<unsigned>(sum[s][t]) + static_cast<unsigned>(v[t]));
                }
            }
        }
        v4i bits;  // the four results, one dword, two or four of them in use
        int bytes = 1;
        if constexpr (O::FLOAT) {
            float y[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                y[t] = sum[0][t] + par_bias[p][t];
                if (g.relu) y[t] = fmaxf(y[t], 0.f);
            }
            if constexpr (KIND == FEW_F32) {
                bits = __builtin_bit_cast(v4i, v4f{y[0], y[1], y[2], y[3]});
                bytes = 4;
            } else if constexpr (KIND == FEW_BF16) {
                bits = v4i{static_cast<int>(f32_to_bf16_bits(y[0]) | (f32_to_bf16_bits(y[1]) << 16)),
                           static_cast<int>(f32_to_bf16_bits(y[2]) | (f32_to_bf16_bits(y[3]) << 16)), 0, 0};
                bytes = 2;
            } else {
                bits = v4i{static_cast<int>(f32_to_fp8_bits(y[0]) | (f32_to_fp8_bits(y[1]) << 8) | (f32_to_fp8_bits(y[2]) << 16) | (f32_to_fp8_bits(y[3]) << 24)), 0, 0, 0};
            }
        } else {
            int y[4];
            if constexpr (KIND == FEW_I16X16) {
                long long rows = 0;
#pragma unroll
                for (int w = 0; w < NW; ++w)
#pragma unroll
                    for (int h = 0; h < 4; ++h) rows += part_rows[(w * TM + i) * 64 + 16 * h + frow];
                with_round_mode(g.mode, [&](auto mode) {
#pragma unroll
                    for (int t = 0; t < 4; ++t) {
                        const Round64 rr = make_round64(par_shift[p][t], g.mode);
                        const long long v = static_cast<long long>(sum[0][t]) * 65536 + static_cast<long long>(sum[1][t]) * 256 + sum[2][t] +
                                            128ll * (rows + par_cols[p][t]) + par_add[p][t];
                        y[t] = requant64_m<decltype(mode)::value>(v, rr.c0, rr.s, rr.en, lo, hi);
                    }
                });
            } else {
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    const RoundCfg rc = make_round(g.mode, min(max(par_shift[p][t], 0), 31));
                    y[t] = clamp_i(apply_round(static_cast<int>(static_cast<unsigned>(sum[0][t]) + static_cast<unsigned>(par_add[p][t]) + 128u * static_cast<unsigned>(par_cols[p][t])), rc), lo, hi);
                }
            }
            if (g.out_kind == A4G_I16 || g.out_kind == A4G_U16) {
                bits = v4i{static_cast<int>(pack2_halves(y[0], y[1])), static_cast<int>(pack2_halves(y[2], y[3])), 0, 0};
                bytes = 2;
            } else {
                bits = v4i{static_cast<int>(pack4_bytes(y[0], y[1], y[2], y[3])), 0, 0, 0};
            }
        }
        if (m < g.M && n < g.N) {
            int8_t* dst = static_cast<int8_t*>(g.C) + (blockIdx.y * g.stride_c + static_cast<int64_t>(m) * g.ldc + n) * bytes;
            store_chunk_ragged(dst, bits, min(4, g.N - n) * bytes);
        }
    }
}

template <int KIND, int NW, int TM, int TN, int DEPTH, bool WF = false>
static hipError_t launch_few_tile(const GemmArgs& g, int batch, hipStream_t stream) {
    using O = FewOps<KIND>;
    constexpr int PATCHES = NW * 2048 * (TM * (O::WIDE_A ? 2 : 1) + (WF ? 0 : TN * (O::PLANES_B ? 2 : 1)));
    constexpr int SUMS = NW * O::SUMS * TM * TN * 1024 + (KIND == FEW_I16X16 ? NW * TM * 256 : 0);
    constexpr int LDS = PATCHES > SUMS ? PATCHES : SUMS;
    static_assert(LDS <= 160 * 1024, "LDS budget");
    auto kern = gemm_few_kernel<KIND, NW, TM, TN, DEPTH, WF>;
    static bool attr_set = false;  // benign race: the attribute is idempotent
    if (!attr_set) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
        if (e != hipSuccess) return e;
        attr_set = true;
    }
    const int tiles_m = (g.M + TM * 16 - 1) / (TM * 16), tiles_n = ((WF ? (g.N + 31) / 32 * 32 : g.N) + TN * 16 - 1) / (TN * 16);
    kern<<<dim3(grid_for_tiles(static_cast<int64_t>(tiles_m) * tiles_n), batch), NW * 64, LDS, stream>>>(g, tiles_m);
    return hipGetLastError();
}

// Rows and columns of a tile, in blocks of 16. Wider tiles read less per output, narrower ones make more workgroups and
// have less to wait for at the start and at the end.
struct FewForm {
    int tm, tn;
};
static constexpr FewForm FEW_FORMS[4] = {{1, 1}, {2, 1}, {2, 2}, {4, 4}};

template <int KIND>
static hipError_t launch_few_kind(const GemmArgs& g, int batch, int form, hipStream_t stream) {
    if constexpr (KIND == FEW_I8) {
        if (g.Wf && batch == 1 && aligned16(g.Wf) && wreg_applicable(g) && rowpacked_bytes(g.N, g.K) < (int64_t{1} << 31)) {
            // (no size picks 32 x 16)
            return form == 0 ? launch_few_tile<KIND, 4, 1, 1, 4, true>(g, batch, stream) : launch_few_tile<KIND, 4, 2, 2, 2, true>(g, batch, stream);
        }
    }
    switch (form) {
    case 0: return launch_few_tile<KIND, 4, 1, 1, 4>(g, batch, stream);
    case 1: return launch_few_tile<KIND, 4, 2, 1, 3>(g, batch, stream);
    case 2: return launch_few_tile<KIND, 4, 2, 2, 2>(g, batch, stream);
    default:
        if constexpr (KIND != FEW_I16X16) return launch_few_tile<KIND, 4, 4, 4, 1>(g, batch, stream);
        else return hipErrorInvalidValue;
    }
}

// What a launch takes, in us: `start`, plus `tile` for every K tile of 128 bytes and every workgroup that a CU gets (at least one), plus
// `more` for every workgroup of a CU after its first. The tiled kernels by the same law with their 128 x 128 tiles. Fitted to 1400 random
// sizes in every format (4200 in int8) at which every form and the tiled kernel were timed: 1 to 16384 rows, 32 to 8192 inputs, 8 to
// 8192 outputs, from a workgroup in all to hundreds for a CU; where the law is coarse the constants are the ones that pick best.
// What is picked is within 0.1 % of the fastest on average at 600 other sizes a format (int8 0.3 %, bfloat16 and int16 0.5 %, float32 0.8 %). Measured, this kernel / the tiled ones, us:
// 16 x 4096 -> 4096 int8 5.4 / 22.3, int16 7.5 / 51, bfloat16 6.7 / 38, float32 14 / 235, fp8 4.6 / 24; 128 x 768 -> 768 int8
// 4.6 / 7.7; 1024 x 768 -> 768 int8 6.9 / 7.8. Not taken: 2048 x 768 -> 768 int8 10.1 / 9.6, 8192 x 60 -> 2048 int8 62 / 21,
// 3639 x 512 -> 150 int16 x int16 19.5 / 13.6.
struct FewCost {
    float start, tile, more;
};
struct FewCosts {
    FewCost form[4];
    FewCost whole, stored, ragged;  // the tiled kernels: operands on whole chunks, with results that do not leave from registers, neither
};
static constexpr FewCosts FEW_COSTS[] = {
    /* FEW_I8     */ {{{4.05f, 0.0472f, 0.65f}, {4.53f, 0.0558f, 1.14f}, {4.26f, 0.0892f, 0.81f}, {7.92f, 0.2474f, 1.31f}},
                      {5.43f, 0.5193f, 3.54f}, {6.68f, 0.5456f, 3.98f}, {8.82f, 0.6466f, 4.35f}},
    /* FEW_I16X8  */ {{{4.97f, 0.076f, 1.28f}, {5.92f, 0.1001f, 4.11f}, {4.97f, 0.1958f, 2.19f}, {10.26f, 0.3652f, 11.32f}},
                      {5.63f, 0.7455f, 3.83f}, {5.63f, 0.7455f, 3.83f}, {6.16f, 0.8082f, 5.64f}},
    /* FEW_I16X16 */ {{{5.68f, 0.0917f, 2.23f}, {6.52f, 0.1483f, 5.98f}, {5.8f, 0.2706f, 5.62f}, {}},
                      {6.55f, 1.297f, 12.71f}, {6.55f, 1.297f, 12.71f}, {6.28f, 1.344f, 10.37f}},
    /* FEW_BF16   */ {{{3.52f, 0.0509f, 0.7f}, {3.53f, 0.0705f, 0.74f}, {3.78f, 0.0864f, 0.88f}, {5.99f, 0.1925f, 2.94f}},
                      {8.0f, 0.5162f, 4.42f}, {8.0f, 0.5162f, 4.42f}, {10.36f, 0.5061f, 3.54f}},
    /* FEW_F32    */ {{{3.62f, 0.0654f, 0.9f}, {3.9f, 0.1175f, 0.84f}, {4.33f, 0.1585f, 1.05f}, {5.8f, 0.6075f, 2.47f}},
                      {7.17f, 1.886f, 6.34f}, {7.17f, 1.886f, 6.34f}, {7.5f, 1.901f, 8.99f}},
    /* FEW_FP8    */ {{{3.68f, 0.039f, 0.8f}, {3.8f, 0.0697f, 0.97f}, {3.9f, 0.0913f, 1.11f}, {6.68f, 0.2032f, 2.64f}},
                      {10.56f, 0.4347f, 5.38f}, {10.56f, 0.4347f, 5.38f}, {10.99f, 0.6238f, 5.57f}},
};

static float launch_us(const FewCost& c, int ktiles, float workgroups) {
    float per_cu = std::max(1.f, workgroups / 256.f);
    per_cu = 0.5f * (per_cu + std::ceil(per_cu));  // a last round that is not full overlaps the one before it in part
    return c.start + c.tile * static_cast<float>(ktiles) * per_cu + c.more * (per_cu - 1.f);
}

// Reductions of up to 768 on aligned rows have a kernel of their own with little fixed cost (launch_wreg); what is faster here has the
// weights in fragment order, if they are, and tiles of 16 x 16 or 32 x 32 (those of 64 x 64 are behind launch_wreg at every such size).
static bool weights_in_registers(const GemmArgs& g, FewKind kind, int batch) { return kind == FEW_I8 && batch == 1 && wreg_applicable(g); }

static int few_form(const GemmArgs& g, FewKind kind, int batch, float* us) {
    const int ktiles = (g.K + 127) / 128;
    int best = 0;
    *us = 1e30f;
    for (int f = 0; f < (kind == FEW_I16X16 || weights_in_registers(g, kind, batch) ? 3 : 4); ++f) {
        const float rows = static_cast<float>((g.M + FEW_FORMS[f].tm * 16 - 1) / (FEW_FORMS[f].tm * 16));
        const float cols = static_cast<float>((g.N + FEW_FORMS[f].tn * 16 - 1) / (FEW_FORMS[f].tn * 16));
        const float t = launch_us(FEW_COSTS[kind].form[f], ktiles, rows * cols * static_cast<float>(batch));
        if (t < *us) {
            *us = t;
            best = f;
        }
    }
    return best;
}

bool few_preferred(const GemmArgs& g, FewKind kind, int batch) {
    const bool wide = kind == FEW_I16X8 || kind == FEW_I16X16;
    if (g.K * (wide ? 2 : 1) < 16 || g.M <= 0 || 64 * g.lda >= (int64_t{1} << 31) || 64 * g.ldb >= (int64_t{1} << 31)) return false;
    if (!whole_chunk_rows(g.Bt, g.ldb, g.stride_b, g.K) || (kind == FEW_I16X16 && !whole_chunk_rows(g.Bt_lo, g.ldb, g.stride_b, g.K))) return false;
    float us, other;
    few_form(g, kind, batch, &us);
    if (weights_in_registers(g, kind, batch)) {
        other = 6.6f + static_cast<float>(g.M) * static_cast<float>(g.N) * static_cast<float>(g.K) * 1.4e-9f;
    } else {
        const bool whole = g.K * (wide ? 2 : 1) % 16 == 0 && g.lda % 16 == 0 && g.stride_a % 16 == 0 && aligned16(g.A);
        const float tiles = static_cast<float>((g.M + 127) / 128) * static_cast<float>((g.N + 127) / 128) * static_cast<float>(batch);
        // (direct_epilogue_ok in gemm.hip)
        const bool direct = (g.out_kind == A4G_I8 || g.out_kind == A4G_U8) && g.N % 16 == 0 && g.ldc % 16 == 0 && aligned16(g.C);
        const FewCosts& c = FEW_COSTS[kind];
        other = launch_us(!whole ? c.ragged : direct ? c.whole : c.stored, (g.K + 127) / 128, tiles);
    }
    return us < other;
}

hipError_t launch_few(const GemmArgs& g, FewKind kind, int batch, hipStream_t stream) {
    float us;
    const int form = few_form(g, kind, batch, &us);
    switch (kind) {
    case FEW_I8: return launch_few_kind<FEW_I8>(g, batch, form, stream);
    case FEW_I16X8: return launch_few_kind<FEW_I16X8>(g, batch, form, stream);
    case FEW_I16X16: return launch_few_kind<FEW_I16X16>(g, batch, form, stream);
    case FEW_BF16: return launch_few_kind<FEW_BF16>(g, batch, form, stream);
    case FEW_F32: return launch_few_kind<FEW_F32>(g, batch, form, stream);
    default: return launch_few_kind<FEW_FP8>(g, batch, form, stream);
    }
}

}  // namespace a4g

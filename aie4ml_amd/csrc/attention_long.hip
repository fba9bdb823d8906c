// Fused attention core for any number of keys: O = srs( softmax_int( srs(Q K^T) ) V ) in one launch, the same integer
// operations in the same order as MatMul (matmul.cpp:80-115) -> Softmax (softmax.cpp:19-127 / 252-384) -> MatMul.
//
// attention_kernel keeps a row's logits in registers, which ends at 512 keys. Here a wave walks the keys of its 32 query
// rows three times and keeps nothing per key: (1) the row maximum, taken on the raw accumulators (rounding and saturation
// are monotone, so one rounding per row is enough: half a vector instruction per logit), (2) the sum of the scores,
// (3) the probabilities, which go straight into the second matrix product. The logits of (2) and (3) are formed again:
// two products of 32 x 32 logits more (two matrix instructions each at dimension 64) and about two vector instructions per logit
// cost less than what storing them would: 1024 keys of 128 rows are 128 KiB, which leaves one wave per SIMD, and a lone wave issues
// vector instructions at half the rate of two.
// Bound by vector issue and by the latencies between its steps (12 vector instructions per logit in all, by the counter). Two workgroups of four waves
// share a CU; the score table is stored once per LDS bank (a single copy would serialise the gathers: two per logit).
// Measured (head dimension 64, as many queries as keys): 48 heads of 1024 keys 42.6 us, 192 heads 114 us (0.57 ns per 1000
// logits with the chip full, 0.36 in attention_kernel at 512 keys); MatMul, Softmax and MatMul head by head through memory
// took more than 1000 us for the 48 heads. By walks, of the 192 heads' time: 13 / 26 / 54 us, the rest is each workgroup's
// start and end. Scores gathered a tile ahead of their use: no gain (112 us), and four waves per SIMD do not fit the
// registers (128 a lane: 190 us with the spills).
#include <climits>
#include <type_traits>

#include "attention_common.hpp"

namespace a4g {

// DT: head dimension / 32. BIT, FASTP: as in attention_kernel (rounding kind of the logits, 3 the float form;
// probabilities that need no clamp). NW: waves per workgroup.
template <int DT, int BIT, bool FASTP, int NW>
__global__ __launch_bounds__(NW * 64, NW == 8 ? 1 : 2) void attention_long_kernel(AttnArgs a) {
    constexpr int D = DT * 32, THREADS = NW * 64, ROWS = NW * 32;
    constexpr int CHUNK = 64, PITCH = CHUNK + 16;  // keys of V^T in LDS at a time (two buffers): 80-byte rows spread over all banks
    constexpr int KD = DT == 4 ? 2 : 4;            // tiles of K fragments on their way or in use
    __shared__ int table[256 * 64];                // entry of gap d for lane l at dword d * 64 + l
    extern __shared__ __attribute__((aligned(16))) int8_t attn_smem[];
    int8_t* vt = attn_smem;                                           // 2 x [D][PITCH], keys in the order of the probability registers
    int* colsum = reinterpret_cast<int*>(attn_smem + 2 * D * PITCH);  // sum over all keys of V[k][n]

    const int nblk = (a.sq + ROWS - 1) / ROWS;
    // consecutive items on one XCD: they read the same head's keys and values
    const int item = (gridDim.x & 7) == 0 ? static_cast<int>((blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3)) : static_cast<int>(blockIdx.x);
    const int bh = item / nblk;
    const int b = bh / a.heads, h = bh - b * a.heads;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int m = lane & 31, half = lane >> 5;
    const int hoff = half * 16;
    const int ntile = (a.sk + 31) >> 5, full = a.sk >> 5;  // tiles of 32 keys; those that are whole

    // rows past the last key read as zero; tile numbers are clamped to the last one, so that the scalar part of the
    // address stays inside the descriptor
    const int k_ss = static_cast<int>(a.k_ss);
    const __amdgpu_buffer_rsrc_t rsrc_k =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(a.K + b * a.k_sb + h * a.k_sh), 0, (a.sk - 1) * k_ss + a.d, 0x00020000);
    const int kvoff = m * k_ss + hoff;
    v4i qf[DT], kf[KD][DT];
    auto load_k = [&](int slot, int t) __attribute__((always_inline)) {
        const int at = min(t, ntile - 1) * 32 * k_ss;
#pragma unroll
        for (int ks = 0; ks < DT; ++ks)
            kf[slot][ks] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rsrc_k, kvoff + ks * 32, at, 0));
    };
    const int row = (item - bh * nblk) * ROWS + wave * 32 + m;
    {
        const int8_t* Qp = a.Q + b * a.q_sb + h * a.q_sh + static_cast<int64_t>(row < a.sq ? row : a.sq - 1) * a.q_ss;
#pragma unroll
        for (int ks = 0; ks < DT; ++ks) {
            const bool missing = a.d < D && ks * 32 + hoff >= a.d;  // a piece of the row that does not exist counts nothing
            qf[ks] = *reinterpret_cast<const v4i*>(Qp + (missing ? 0 : ks * 32 + hoff));
            if (missing) qf[ks] = v4i{0, 0, 0, 0};
        }
    }
#pragma unroll
    for (int j = 0; j < KD; ++j) load_k(j, j);

    // the score table: each entry computed once, then copied to its 64 slots
    {
        int* once = reinterpret_cast<int*>(vt);
        if (tid < 256) once[tid] = table_entry(a.sm, tid);
        if (tid < D) colsum[tid] = 0;
        __syncthreads();
        for (int i = tid * 4; i < 256 * 64; i += THREADS * 4) {
            const int e = once[i >> 6];
            *reinterpret_cast<v4i*>(table + i) = v4i{e, e, e, e};
        }
    }

    // float form (BIT == 3): sums start from the bit pattern of 1.5 * 2^23 and leave the matrix unit as floats, see
    // attention_kernel
    constexpr int START = BIT == 3 ? 0x4B400000 : 0;
    v16i start16 = {START, START, START, START, START, START, START, START, START, START, START, START, START, START, START, START};
    if (BIT == 3) asm volatile("" : "+v"(start16));  // kept in registers: formed again for every tile it costs 24 moves
    const float lbias = 128.f - 12582912.f * a.lscale;
    auto product = [&](int slot) __attribute__((always_inline)) {
        v16i sums = start16;
#pragma unroll
        for (int ks = 0; ks < DT; ++ks) sums = __builtin_amdgcn_mfma_i32_32x32x32_i8(kf[slot][ks], qf[ks], sums, 0, 0, 0);
        return sums;
    };
    // Walks all tiles: before(tile) ahead of every one, then f(tile, accumulators, whether keys of the tile are missing).
    // The matrix unit works a tile ahead of f, the loads KD tiles ahead of the matrix unit; towards the end of a walk both
    // turn to the first tiles of the next one. The loads stand outside the branches, so that the waits for them count exactly.
    const int padded = (ntile + KD - 1) / KD * KD;
    v16i acc_next = product(0);
    auto walk = [&](auto&& before, auto&& f) __attribute__((always_inline)) {
        for (int t0 = 0; t0 < padded; t0 += KD) {
#pragma unroll
            for (int j = 0; j < KD; ++j) {
                const int t = t0 + j;
                before(t);
                const v16i acc = acc_next;
                load_k(j, t + KD < padded ? t + KD : j);
                acc_next = product((j + 1) % KD);
                if (t < full) f(t, acc, std::false_type{});
                else if (t < ntile) f(t, acc, std::true_type{});
            }
        }
    };
    auto nothing = [](int) {};

    // ---- first walk: row maximum of the raw sums
    int mx = INT_MIN;
    float mxf = 0.f;
    walk(nothing, [&](int t, const v16i& acc, auto masked) __attribute__((always_inline)) {
        constexpr bool MASKED = decltype(masked)::value;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const int left = MASKED ? a.sk - (t * 32 + 8 * g + 4 * half) : 4;  // keys that exist among the group's four
            if (BIT == 3) {
                float f[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int bits = acc[4 * g + i];
                    f[i] = i < left ? __builtin_bit_cast(float, bits) : 0.f;
                }
                mxf = __builtin_fmaxf(__builtin_fmaxf(mxf, f[0]), f[1]);
                mxf = __builtin_fmaxf(__builtin_fmaxf(mxf, f[2]), f[3]);
            } else {
                int y[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) y[i] = i < left ? acc[4 * g + i] : INT_MIN;
                mx = max(max(mx, y[0]), y[1]);
                mx = max(max(mx, y[2]), y[3]);
            }
        }
    });
    unsigned mxb;  // the maximum of the rounded, saturated logits, biased by 128
    if (BIT == 3) {
        mxf = __builtin_fmaxf(mxf, __builtin_bit_cast(float, lane_xor<32>(__builtin_bit_cast(int, mxf))));
        mxb = __builtin_amdgcn_cvt_pk_u8_f32(fmaf(mxf, a.lscale, lbias), 0, 0u);
    } else {
        mx = max(mx, lane_xor<32>(mx));  // lanes m and m + 32 share a row
        mxb = static_cast<unsigned>((clamp_i(fast_round_k<BIT>(mx, a.lr), -128, 127) ^ 0x80) & 0xFF);
    }
    __syncthreads();  // the score table is complete

    const unsigned mrep = mxb * 0x01010101u;
    const char* tbytes = reinterpret_cast<const char*>(table);
    const unsigned lane4 = static_cast<unsigned>(lane) << 2;
    // the scores of a group of four keys: requantise, pack (biased by 128), gap to the maximum per byte, table
    auto scores = [&](int t, int g, const v16i& acc, auto masked, int (&e)[4]) __attribute__((always_inline)) {
        constexpr bool MASKED = decltype(masked)::value;
        const int left = MASKED ? a.sk - (t * 32 + 8 * g + 4 * half) : 4;
        unsigned w;
        if (BIT == 3) {
            float f[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int bits = acc[4 * g + i];
                f[i] = fmaf(__builtin_bit_cast(float, bits), a.lscale, lbias);
                f[i] = i < left ? f[i] : 0.f;
            }
            w = __builtin_amdgcn_cvt_pk_u8_f32(f[0], 0, 0u);
            w = __builtin_amdgcn_cvt_pk_u8_f32(f[1], 1, w);
            w = __builtin_amdgcn_cvt_pk_u8_f32(f[2], 2, w);
            w = __builtin_amdgcn_cvt_pk_u8_f32(f[3], 3, w);
        } else {
            int y[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                y[i] = clamp_i(fast_round_k<BIT>(acc[4 * g + i], a.lr), -128, 127);
                y[i] = i < left ? y[i] : -128;
            }
            w = pack4_bytes(y[0], y[1], y[2], y[3]) ^ 0x80808080u;
        }
        const unsigned d4 = mrep - w;  // per byte, never borrows
        e[0] = *reinterpret_cast<const int*>(tbytes + __builtin_amdgcn_perm(d4, lane4, 0x0c0c0400u));
        e[1] = *reinterpret_cast<const int*>(tbytes + __builtin_amdgcn_perm(d4, lane4, 0x0c0c0500u));
        e[2] = *reinterpret_cast<const int*>(tbytes + __builtin_amdgcn_perm(d4, lane4, 0x0c0c0600u));
        e[3] = *reinterpret_cast<const int*>(tbytes + __builtin_amdgcn_perm(d4, lane4, 0x0c0c0700u));
        if (MASKED) {
#pragma unroll
            for (int i = 0; i < 4; ++i) e[i] = i < left ? e[i] : 0;
        }
    };

    // ---- second walk: row sum of the scores
    int sum = 0;
    walk(nothing, [&](int t, const v16i& acc, auto masked) __attribute__((always_inline)) {
        int e[4][4];
#pragma unroll
        for (int g = 0; g < 4; ++g) scores(t, g, acc, masked, e[g]);
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            sum = sum + e[g][0] + e[g][1];
            sum = sum + e[g][2] + e[g][3];
        }
    });
    sum += lane_xor<32>(sum);
    const int inv = row_inverse(a.sm, sum);

    // ---- third walk: probabilities (uint8, read as int8 after ^ 0x80) feed the second product from registers. V arrives
    // 64 keys at a time, a 4 x 4 block of bytes per thread, transposed on its way into LDS: within each group of 32 keys,
    // position 16 * half + 4 * g + i holds key 8 * g + 4 * half + i, the order of a lane's probabilities. Rows past the
    // last key read as zero.
    constexpr int NB = (CHUNK / 4) * (D / 4);
    static_assert(NB <= THREADS, "one block of V per thread");
    const int n0 = (tid % (D / 4)) * 4, k0 = (tid / (D / 4)) * 4;  // the thread's four columns and four keys of a chunk
    const bool loader = tid < NB;
    const int pos = (k0 & ~31) + ((k0 >> 2) & 1) * 16 + ((k0 & 31) >> 3) * 4;
    const int v_ss = static_cast<int>(a.v_ss);
    const __amdgpu_buffer_rsrc_t rsrc_v =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(a.V + b * a.v_sb + h * a.v_sh), 0, (a.sk - 1) * v_ss + a.d, 0x00020000);
    const int vvoff = (loader ? k0 : 0) * v_ss + (n0 < a.d ? n0 : 0);  // columns past the head dimension are never stored
    unsigned av[4];
    auto load_v = [&](int chunk) __attribute__((always_inline)) {
        const int at = min(chunk * CHUNK, a.sk - 1) * v_ss;
#pragma unroll
        for (int i = 0; i < 4; ++i) av[i] = __builtin_amdgcn_raw_buffer_load_b32(rsrc_v, vvoff + i * v_ss, at, 0);
    };
    int part[4] = {0, 0, 0, 0};
    v16i oacc[DT];
#pragma unroll
    for (int u = 0; u < DT; ++u) oacc[u] = v16i{0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    const unsigned inv16 = static_cast<unsigned>(inv) << (16 - a.sm.out_shift);  // FASTP only: 0 <= inv, shift <= 16
    load_v(0);
    walk(
        [&](int t) __attribute__((always_inline)) {
            if (t & 1) return;
            if (t < ntile) {
                // Two buffers, one barrier per chunk: whoever writes this one has passed the barrier of the chunk before,
                // and everybody who passed that one is done with the chunk before it, which lay here.
                if (loader) {
                    unsigned cv[4];
                    transpose4x4(av, cv);
                    const int ones = t + (k0 >> 5) < ntile ? 0x01010101 : 0;  // a second tile past the last one is not multiplied
                    int8_t* to = vt + ((t >> 1) & 1) * D * PITCH + n0 * PITCH + pos;
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        *reinterpret_cast<unsigned*>(to + j * PITCH) = cv[j];
                        part[j] = __builtin_amdgcn_sdot4(static_cast<int>(cv[j]), ones, part[j], false);
                    }
                }
                __syncthreads();
            }
            load_v((t >> 1) + 1);
        },
        [&](int t, const v16i& acc, auto masked) __attribute__((always_inline)) {
            int e[4][4];
#pragma unroll
            for (int g = 0; g < 4; ++g) scores(t, g, acc, masked, e[g]);
            v4i pf;
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                if (FASTP) {
                    // a score (15 bits) times inv16 (below 2^16 whenever no clamp is needed): p in bits 16..23, nothing above
                    unsigned q[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i) q[i] = __umul24(static_cast<unsigned>(e[g][i]), inv16);
                    const unsigned lo = __builtin_amdgcn_perm(q[1], q[0], 0x0c0c0602u);
                    const unsigned hi = __builtin_amdgcn_perm(q[3], q[2], 0x06020c0cu);
                    pf[g] = static_cast<int>((lo | hi) ^ 0x80808080u);
                } else {
                    int p[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i) p[i] = clamp_i(__mul24(e[g][i], inv) >> a.sm.out_shift, 0, 255);
                    pf[g] = static_cast<int>(pack4_bytes(p[0], p[1], p[2], p[3]) ^ 0x80808080u);
                }
            }
            const int8_t* from = vt + ((t >> 1) & 1) * D * PITCH + m * PITCH + (t & 1) * 32 + hoff;
#pragma unroll
            for (int u = 0; u < DT; ++u) {
                const v4i vf = *reinterpret_cast<const v4i*>(from + 32 * u * PITCH);
                oacc[u] = __builtin_amdgcn_mfma_i32_32x32x32_i8(vf, pf, oacc[u], 0, 0, 0);
            }
        });
    if (loader) {
#pragma unroll
        for (int j = 0; j < 4; ++j) atomicAdd(&colsum[n0 + j], part[j]);
    }
    __syncthreads();

    // ---- + 128 * colsum (undoes the ^ 0x80), requantise, 16 contiguous bytes per lane
    int8_t* Op = a.O + b * a.o_sb + h * a.o_sh + static_cast<int64_t>(row) * a.o_ss;
    const bool row_ok = row < a.sq;
#pragma unroll
    for (int u = 0; u < DT; ++u) {
        unsigned ow[4];
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const v4i cs = *reinterpret_cast<const v4i*>(colsum + 32 * u + 8 * g + 4 * half);
            int y[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) y[i] = clamp_i(fast_round(oacc[u][4 * g + i] + 128 * cs[i], a.orr), -128, 127);
            ow[g] = pack4_bytes(y[0], y[1], y[2], y[3]);
        }
        const auto s02 = __builtin_amdgcn_permlane32_swap(ow[0], ow[2], false, false);
        const auto s13 = __builtin_amdgcn_permlane32_swap(ow[1], ow[3], false, false);
        const v4i o = {static_cast<int>(s02[0]), static_cast<int>(s02[1]), static_cast<int>(s13[0]), static_cast<int>(s13[1])};
        if (row_ok && 32 * u + 16 * half < a.d) *reinterpret_cast<v4i*>(Op + 32 * u + 16 * half) = o;
    }
}

template <int DT, int BIT, bool FASTP>
static void launch_long(const AttnArgs& a, int64_t heads_in_all, hipStream_t stream) {
    constexpr int NW = DT == 4 ? 8 : 4;
    constexpr int LDS = 2 * DT * 32 * (64 + 16) + DT * 32 * 4;
    auto kern = attention_long_kernel<DT, BIT, FASTP, NW>;
    static bool attr_set = false;  // benign race: the attribute is idempotent
    if (!attr_set) {
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
        attr_set = true;
    }
    kern<<<static_cast<int>(heads_in_all * ((a.sq + NW * 32 - 1) / (NW * 32))), NW * 64, LDS, stream>>>(a);
}

template <int DT>
static void launch_long_dim(const AttnArgs& a, int64_t heads_in_all, hipStream_t stream) {
    const bool fastp = a.noclamp && a.sm.out_shift <= 16;
#define A4G_ATTN_LONG(B)                                                \
    if (fastp) launch_long<DT, B, true>(a, heads_in_all, stream);       \
    else launch_long<DT, B, false>(a, heads_in_all, stream);
    switch (a.lscale > 0.f ? 3 : fast_round_kind(a.lr)) {
    case 0: A4G_ATTN_LONG(0) break;
    case 1: A4G_ATTN_LONG(1) break;
    case 2: A4G_ATTN_LONG(2) break;
    default: A4G_ATTN_LONG(3) break;
    }
#undef A4G_ATTN_LONG
}

}  // namespace a4g

using namespace a4g;

extern "C" int a4g_attention_long_i8(const int8_t* Q, const int8_t* K, const int8_t* V, int8_t* O, int64_t batch, int64_t heads,
                                     int64_t sq, int64_t sk, int64_t d, const int64_t* strides, int logit_shift,
                                     int logit_round_mode, int softmax_kind, int exp_kq, int hccs_B, int hccs_S, int hccs_Dmax,
                                     int inv_shift, int use_clb, int out_shift, int out_round_mode, a4g_stream_t stream_) {
    const char* who = "a4g_attention_long_i8";
    AttnArgs a{};
    if (int rc = attention_params(who, batch, heads, sq, sk, d, logit_shift, logit_round_mode, softmax_kind, exp_kq, hccs_B, hccs_S,
                                  hccs_Dmax, inv_shift, use_clb, out_shift, out_round_mode, &a))
        return rc;
    // 32768 keys: the output's sums (255 * 128 per key) stay within 31 bits, as its rounding assumes
    A4G_REQUIRE(d % 16 == 0 && d <= 128 && sk <= 32768, A4G_ERR_UNSUPPORTED,
                "%s: covers head dimensions that are multiples of 16 up to 128 and up to 32768 keys, got d=%lld sk=%lld", who,
                (long long)d, (long long)sk);
    A4G_REQUIRE(batch * heads * ((sq + 127) / 128) <= INT32_MAX && sq <= (1 << 24), A4G_ERR_UNSUPPORTED, "%s: too many rows", who);
    if (batch == 0) return A4G_OK;
    if (int rc = attention_operands(who, Q, K, V, O, strides, &a)) return rc;
    A4G_REQUIRE((sk + 32) * strides[8] < (int64_t{1} << 31), A4G_ERR_UNSUPPORTED,
                "%s: the values of one head must span less than 2 GiB (row stride %lld bytes)", who, (long long)strides[8]);
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    if (d <= 32) launch_long_dim<1>(a, batch * heads, stream);
    else if (d <= 64) launch_long_dim<2>(a, batch * heads, stream);
    else launch_long_dim<4>(a, batch * heads, stream);
    return check_hip(hipGetLastError(), who);
}

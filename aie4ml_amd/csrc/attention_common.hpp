// What the two fused attention kernels share: the launch arguments, the 4 x 4 byte transposition of V, and the checks of
// the C entry points.
#pragma once

#include "common.hpp"
#include "softmax_common.hpp"

namespace a4g {

struct AttnArgs {
    const int8_t* Q;
    const int8_t* K;
    const int8_t* V;
    int8_t* O;
    int64_t q_sb, q_sh, q_ss;  // byte strides: batch, head, row (the feature axis is contiguous)
    int64_t k_sb, k_sh, k_ss;
    int64_t v_sb, v_sh, v_ss;
    int64_t o_sb, o_sh, o_ss;
    int heads, sq;
    int d;      // head dimension that exists, a multiple of 16 up to the kernel's width: the 16-byte pieces of a row past it do not
    int sk;     // key / value rows that exist (the ragged form; the kernel's tiles cover the next tile count that has an instance)
    int items;  // (batch, head, block of query rows) triples in all
    FastRound lr, orr;  // logits and output requantisation
    SoftmaxParams sm;
    int noclamp;
    float lscale;  // 2^-logit_shift, for the float form of the logit requantisation
};

// 4x4 byte transpose: in a[i] byte j  ->  out c[j] byte i.
__device__ __forceinline__ void transpose4x4(const unsigned a[4], unsigned c[4]) {
    const unsigned lo01 = __builtin_amdgcn_perm(a[1], a[0], 0x05010400u);
    const unsigned hi01 = __builtin_amdgcn_perm(a[1], a[0], 0x07030602u);
    const unsigned lo23 = __builtin_amdgcn_perm(a[3], a[2], 0x05010400u);
    const unsigned hi23 = __builtin_amdgcn_perm(a[3], a[2], 0x07030602u);
    c[0] = __builtin_amdgcn_perm(lo23, lo01, 0x05040100u);
    c[1] = __builtin_amdgcn_perm(lo23, lo01, 0x07060302u);
    c[2] = __builtin_amdgcn_perm(hi23, hi01, 0x05040100u);
    c[3] = __builtin_amdgcn_perm(hi23, hi01, 0x07060302u);
}


// Everything about a call that does not depend on the kernel chosen for it: argument checks and the launch arguments.
static inline int attention_params(const char* who, int64_t batch, int64_t heads, int64_t sq, int64_t sk, int64_t d, int logit_shift,
                                   int logit_round_mode, int softmax_kind, int exp_kq, int hccs_B, int hccs_S, int hccs_Dmax,
                                   int inv_shift, int use_clb, int out_shift, int out_round_mode, AttnArgs* a) {
    A4G_REQUIRE(batch >= 0 && heads >= 1 && sq >= 1 && sk >= 1 && d >= 1, A4G_ERR_INVALID_ARGUMENT,
                "%s: bad shape batch=%lld heads=%lld sq=%lld sk=%lld d=%lld", who, (long long)batch, (long long)heads,
                (long long)sq, (long long)sk, (long long)d);
    A4G_REQUIRE(valid_round(logit_round_mode) && valid_round(out_round_mode), A4G_ERR_INVALID_ARGUMENT,
                "%s: unknown rounding mode", who);
    A4G_REQUIRE(logit_shift >= 0 && logit_shift <= 24 && out_shift >= 0 && out_shift <= 24, A4G_ERR_INVALID_ARGUMENT,
                "%s: accumulator output shift must be in [0,24], got %d and %d", who, logit_shift, out_shift);
    A4G_REQUIRE(softmax_kind == 0 || softmax_kind == 1, A4G_ERR_INVALID_ARGUMENT, "%s: softmax_kind must be 0 (exp) or 1 (hccs)",
                who);
    bool noclamp = false;
    if (softmax_kind == 0) {
        if (int rc = make_exp_params(who, exp_kq, inv_shift, A4G_U8, &a->sm, &noclamp)) return rc;
    } else {
        if (int rc = make_hccs_params(who, sk, hccs_B, hccs_S, hccs_Dmax, inv_shift, use_clb, A4G_U8, &a->sm, &noclamp))
            return rc;
    }
    a->heads = static_cast<int>(heads);
    a->sq = static_cast<int>(sq);
    a->sk = static_cast<int>(sk);
    a->d = static_cast<int>(d);
    a->lr = make_fast_round(logit_round_mode, logit_shift);
    a->orr = make_fast_round(out_round_mode, out_shift);
    a->noclamp = noclamp;
    // nearest-even logits take the float form: d * 2^14 + 2^(7 + shift) < 2^24 for the head dimensions covered
    a->lscale = (logit_round_mode == A4G_RND_CONV_EVEN && logit_shift >= 1 && logit_shift <= 15 && d <= 512)
                    ? ldexpf(1.f, -logit_shift) : 0.f;
    return A4G_OK;
}

// Operands: pointers, alignment, strides (byte strides {batch, head, row} of Q, K, V, O in that order).
static inline int attention_operands(const char* who, const int8_t* Q, const int8_t* K, const int8_t* V, int8_t* O,
                                     const int64_t* strides, AttnArgs* a) {
    const int64_t sk = a->sk, d = a->d;
    A4G_REQUIRE(Q && K && V && O && strides, A4G_ERR_INVALID_ARGUMENT, "%s: null pointer", who);
    bool ok = aligned16(Q) && aligned16(K) && aligned16(V) && aligned16(O);
    for (int i = 0; i < 12; ++i) ok = ok && strides[i] % 16 == 0 && strides[i] >= 0;
    A4G_REQUIRE(ok, A4G_ERR_UNSUPPORTED, "%s: pointers and strides must be multiples of 16 bytes", who);
    A4G_REQUIRE(strides[2] >= d && strides[5] >= d && strides[8] >= d && strides[11] >= d, A4G_ERR_INVALID_ARGUMENT,
                "%s: row stride smaller than the head dimension", who);
    A4G_REQUIRE((sk + 32) * strides[5] < (int64_t{1} << 31), A4G_ERR_UNSUPPORTED,
                "%s: the keys of one head must span less than 2 GiB (row stride %lld bytes)", who, (long long)strides[5]);
    a->Q = Q; a->K = K; a->V = V; a->O = O;
    a->q_sb = strides[0]; a->q_sh = strides[1]; a->q_ss = strides[2];
    a->k_sb = strides[3]; a->k_sh = strides[4]; a->k_ss = strides[5];
    a->v_sb = strides[6]; a->v_sh = strides[7]; a->v_ss = strides[8];
    a->o_sb = strides[9]; a->o_sh = strides[10]; a->o_ss = strides[11];
    return A4G_OK;
}

}  // namespace a4g

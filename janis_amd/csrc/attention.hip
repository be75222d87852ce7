// SDPA with several query rows per head (prompts; cpu/cpu_attn.go:64-119) on
// the matrix cores of gfx950: head_dim 128, bf16 or f16 keys and values, bf16
// or fp32 queries, any Hq / Hk, the offset causal mask.
//
// A block of 4 waves takes 128 rows of one kv head -- row r is query r / G of
// head r % G, so the heads that share the keys read them from LDS once -- and
// walks the keys in tiles of 64 with an online softmax; a wave owns 32 rows.
// Both products run transposed, S^T = K Q^T and O^T = V^T P^T, so that a lane
// holds one row (lane % 32) in both accumulators: the row's maximum, sum and
// rescale are per-lane scalars, and the scores become the second product's B
// operand where they are, with no exchange between lanes (its K order is the
// order the first product left the keys in, applied to V as it is staged).
//
// Keys and values enter as they are stored. Queries and probabilities are fp32
// and enter as sums of 16-bit terms, one matrix instruction per term into the
// same fp32 accumulator:
//   f16 keys:  a row of q times a power of two that brings its largest element
//              to [2^13, 2^14) (its inverse joins the softmax scale), as one f16
//              term for bf16 q (exact for elements down to 2^-30 of the largest)
//              and two for fp32 q (within 2^-24 of the element, or 2^-38 of the
//              largest where that is more);
//              p * 2^13, at most 2^15, as two f16 terms: within 2^-24 of p or, f16
//              having nothing below 2^-24, 2^-38 of the row's maximum, 1;
//   bf16 keys: one bf16 term for bf16 q, three for fp32 q (24 bits); p as three
//              bf16 terms.
// The floor under f16 probabilities shows only where the keys that hold the weight
// have next to no values (an attention sink), so that the result comes from the
// small ones. Each row's result is held against it, by the sum of the squares of the
// block's values (3 % of a call's time), and a row that it could have cost more than
// about 2^-22 is computed again as rows that are not finite are.
// Relative error against float64 with scores of standard deviation 2.3, 512 and
// 4000 keys: 3.9e-7 and 7.9e-7 (fp32 q, f16 keys), where the per-row kernel
// (sdpa_rows_kernel) has 7.3e-7 and 1.5e-6; with bf16 q and keys 2.8e-7 and
// 6.9e-7 against 3.8e-7 and 1.1e-6.
//
// The products also meet keys past a row's limit with p = 0, where an infinity
// or NaN in V would give NaN; the per-row kernel never reads those. So a row
// whose result is not finite is computed again with that kernel's arithmetic over
// the block's keys, and that result stands.
//
// Per 32 rows x 64 keys a wave issues 16 MFMAs for each q term and 16 for each p term
// (512 cycles each 16) and ~1100 cycles of VALU. K/V tiles come through registers into
// two LDS buffers (64 KiB: two blocks per CU), the next tile's loads in flight
// during the current one. What bounds it, by counters (32 heads over 8, 1500 queries
// of 4000 bf16 keys): the MFMA pipes are busy 33 % of the time and VALU 31, one after
// the other at one or two waves per SIMD (376 blocks on 256 CUs); the waves issue in
// 41 % of their cycles, are ready behind another instruction in 36 and wait for
// memory, LDS or barriers in 23. LDS is active 31 % of the time, half of that in bank
// conflicts. 512 queries of 512 keys are 128 blocks: half of the CUs idle, the MFMA
// pipes 5 % busy.
// Measured on MI355X (replayed graphs; the per-row kernel before): 512 queries of
// 512 keys 3230 -> 30 us (fp32 q, f16 keys), 1500 of 4000 143 ms -> 220 us (bf16), 16 of
// 4112 2.8 ms -> 26 us (fp32 q, f16 keys).
#include "jh_common.hpp"

namespace jh {
namespace {

constexpr int kDh = 128;
constexpr int kRows = 128;  // rows per block
constexpr int kKeys = 64;   // keys per tile
constexpr int kTileBytes = kKeys * kDh * 2;
constexpr int kAgain = 8;    // rows computed again together
constexpr float kLog2e = 1.44269504088896340736f;
// p is held as p * 2^kPShift, and a row's maximum is moved when it grew by more than
// kLazy (log2): f16 terms have nothing below 2^-24 and nothing past 2^16, so p is kept
// high there; bf16 terms have fp32's range, and each move costs 64 products.
template <bool F16>
constexpr float kPShift = F16 ? 13.0f : 7.0f;
template <bool F16>
constexpr float kLazy = F16 ? 2.0f : 8.0f;

typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ float load_act(const void* p, int64_t i, int dt) {
    return dt == JH_BF16 ? bf16_to_f32(static_cast<const uint16_t*>(p)[i]) : static_cast<const float*>(p)[i];
}

template <bool F16>
__device__ __forceinline__ floatx16 mfma(uint4 a, uint4 b, floatx16 c) {
    if constexpr (F16)
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c,
                                                      0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b),
                                                       c, 0, 0, 0);
}

// (a, b) as N packed 16-bit terms, each the nearest to what the earlier ones
// left (the remainders are exact in fp32).
template <bool F16, int N>
__device__ __forceinline__ void split_pair(float a, float b, uint32_t (&t)[N]) {
#pragma unroll
    for (int n = 0; n < N; n++) {
        const f32x2_t f = {a, b};
        if constexpr (F16) {
            const f16x2_t v = __builtin_convertvector(f, f16x2_t);
            t[n] = __builtin_bit_cast(uint32_t, v);
            a -= (float)v.x;
            b -= (float)v.y;
        } else {
            t[n] = __builtin_bit_cast(uint32_t, __builtin_convertvector(f, bf16x2_t));
            a -= __uint_as_float(t[n] << 16);
            b -= __uint_as_float(t[n] & 0xFFFF0000u);
        }
    }
}

__device__ __forceinline__ bool finite(float v) { return (__float_as_uint(v) & 0x7F800000u) != 0x7F800000u; }

struct SdpaArgs {
    const void* q;
    int q_dt;
    const uint16_t *k, *v;
    void* out;
    int out_dt;
    int Hk, G, Lq, Lk, n_tiles, BHk;
    int64_t kcap;
    float scale;
    int causal;
    int kps;      // keys per split (a multiple of kKeys)
    int nsplit;
    float* part_o;   // [B*Hk * G*Lq, nsplit, 128] (split)
    float* part_ml;  // [B*Hk * G*Lq, nsplit, 2]
};

// F16: f16 keys and values (else bf16). QN: 16-bit terms of q.
template <bool F16, int QN, bool SPLIT>
__global__ __launch_bounds__(256, QN == 3 ? 1 : 2) void sdpa_mfma_kernel(SdpaArgs a) {
    constexpr int PN = F16 ? 2 : 3;
    // two slots of a key tile [64][128] (16-byte chunk c of key k at c ^ (k % 16))
    // and a value tile transposed, [128][64] (4-key chunk s of feature d at
    // s ^ (d / 2 % 16)): the lanes of a fragment read spread over 256 bytes
    __shared__ __attribute__((aligned(16))) uint8_t lds[4 * kTileBytes];
    const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5, c32 = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // heads fastest: with 8 kv heads a head's tiles share one XCD's L2; tiles
    // from the last (the longest under the causal mask)
    const int bhk = blockIdx.x % a.BHk, tile = a.n_tiles - 1 - blockIdx.x / a.BHk;
    const int b = bhk / a.Hk, hk = bhk - b * a.Hk;
    const int n_rows = a.G * a.Lq;
    auto limit_of = [&](int r) { return a.causal ? max(0, a.Lk - a.Lq + r / a.G + 1) : a.Lk; };
    const int kb = SPLIT ? (int)blockIdx.y * a.kps : 0;
    const int ke_all = SPLIT ? min(a.Lk, kb + a.kps) : a.Lk;
    const int w0 = tile * kRows + 32 * wave;  // the wave's first row
    // key limits: this lane's row, the wave's smallest and largest, the block's largest
    const int row = min(w0 + c32, n_rows - 1);
    const int lim = min(ke_all, limit_of(row));
    const int lim_lo = min(ke_all, limit_of(min(w0, n_rows - 1)));
    const int lim_hi = w0 < n_rows ? min(ke_all, limit_of(min(w0 + 31, n_rows - 1))) : 0;
    const int ke = min(ke_all, limit_of(min(tile * kRows + kRows, n_rows) - 1));
    const int64_t q_off = ((int64_t)(b * a.Hk * a.G + hk * a.G + row % a.G) * a.Lq + row / a.G) * kDh;

    // q as B fragments: MFMA step kk takes features 16 kk + 8 h .. +8 of the row
    uint4 qf[QN][8];
    float c = fabsf(a.scale) * kLog2e;  // the scale's sign goes into q
    {
        const float sgn = a.scale < 0.0f ? -1.0f : 1.0f;
        float qscale = sgn, amax = 0.0f, v[8][8];
#pragma unroll
        for (int kk = 0; kk < 8; kk++) {
            const int64_t at = q_off + 16 * kk + 8 * h;
            if (a.q_dt == JH_F32) {
                const float4* const p = reinterpret_cast<const float4*>(static_cast<const float*>(a.q) + at);
                const float4 x = p[0], y = p[1];
                v[kk][0] = x.x, v[kk][1] = x.y, v[kk][2] = x.z, v[kk][3] = x.w;
                v[kk][4] = y.x, v[kk][5] = y.y, v[kk][6] = y.z, v[kk][7] = y.w;
            } else {
                const uint4 x = *reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(a.q) + at);
                const uint32_t w[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
                for (int p = 0; p < 4; p++)
                    v[kk][2 * p] = __uint_as_float(w[p] << 16), v[kk][2 * p + 1] = __uint_as_float(w[p] & 0xFFFF0000u);
            }
        }
        if constexpr (F16) {
#pragma unroll
            for (int kk = 0; kk < 8; kk++)
#pragma unroll
                for (int e = 0; e < 8; e++) amax = fmaxf(amax, fabsf(v[kk][e]));
            amax = pair32<true>(amax);
            const int ex = (int)(__float_as_uint(amax) >> 23);
            const int f = min(max(267 - ex, 1), 253);  // exponent field of 2^(13 - exponent of amax)
            qscale = sgn * __uint_as_float((uint32_t)f << 23);
            c *= __uint_as_float((uint32_t)(254 - f) << 23);
        }
#pragma unroll
        for (int kk = 0; kk < 8; kk++) {
            uint32_t t[4][QN];
#pragma unroll
            for (int p = 0; p < 4; p++)
                split_pair<F16, QN>(v[kk][2 * p] * qscale, v[kk][2 * p + 1] * qscale, t[p]);
#pragma unroll
            for (int n = 0; n < QN; n++) qf[n][kk] = make_uint4(t[0][n], t[1][n], t[2][n], t[3][n]);
        }
        if (c < 1e-37f) c = 1e-37f;  // f16, a row of q near zero: equal weights, and masked scores stay -inf
    }

    floatx16 o[4];
#pragma unroll
    for (int t = 0; t < 4; t++)
#pragma unroll
        for (int r = 0; r < 16; r++) o[t][r] = 0.0f;
    const float ninf = -__builtin_inff();
    float m = ninf, l = 0.0f;  // the row's reference maximum (log2 units) and this lane's part of its sum

    const int64_t head = (int64_t)bhk * a.kcap * kDh;
    const auto rk = make_rsrc(a.k + head, (uint32_t)a.Lk * kDh * 2);  // keys past Lk read 0
    const auto rv = make_rsrc(a.v + head, (uint32_t)a.Lk * kDh * 2);
    const int sr = tid >> 4, sc = tid & 15;  // staging: row and 16-byte chunk
    u32x4_t kr[4], vr[4];
    float v2 = 0.0f;  // F16: sum of the squares of the values this thread stages
    auto load = [&](int k0) {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            kr[j] = __builtin_amdgcn_raw_buffer_load_b128(rk, (uint32_t)((k0 + sr + 16 * j) * kDh + 8 * sc) * 2, 0, 0);
            vr[j] = __builtin_amdgcn_raw_buffer_load_b128(rv, (uint32_t)((k0 + 4 * sr + j) * kDh + 8 * sc) * 2, 0, 0);
        }
    };
    auto stage = [&](uint8_t* buf) {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int k = sr + 16 * j;
            *reinterpret_cast<u32x4_t*>(buf + k * 256 + 16 * (sc ^ (k & 15))) = kr[j];
        }
        if constexpr (F16)
#pragma unroll
            for (int j = 0; j < 4; j++)
#pragma unroll
                for (int d = 0; d < 4; d++) {
                    const f16x2_t v = __builtin_bit_cast(f16x2_t, (uint32_t)vr[j][d]);
                    v2 = __builtin_amdgcn_fdot2(v, v, v2, false);
                }
        uint8_t* const vt = buf + kTileBytes;
#pragma unroll
        for (int d = 0; d < 4; d++) {
            // features 8 sc + 2 d and + 1 of keys 4 sr .. + 3
            const uint32_t r0 = vr[0][d], r1 = vr[1][d], r2 = vr[2][d], r3 = vr[3][d];
            const int f = 8 * sc + 2 * d;
            const int at = 8 * (sr ^ ((f >> 1) & 15));
            *reinterpret_cast<uint2*>(vt + f * 128 + at) =
                make_uint2(__builtin_amdgcn_perm(r1, r0, 0x05040100u), __builtin_amdgcn_perm(r3, r2, 0x05040100u));
            *reinterpret_cast<uint2*>(vt + (f + 1) * 128 + at) =
                make_uint2(__builtin_amdgcn_perm(r1, r0, 0x07060302u), __builtin_amdgcn_perm(r3, r2, 0x07060302u));
        }
    };
    auto compute = [&](const uint8_t* buf, int k0) {
        floatx16 s[2];
#pragma unroll
        for (int g = 0; g < 2; g++) {
#pragma unroll
            for (int r = 0; r < 16; r++) s[g][r] = 0.0f;
            const uint8_t* const kt = buf + (32 * g + c32) * 256;
#pragma unroll
            for (int kk = 0; kk < 8; kk++) {
                const uint4 kf = *reinterpret_cast<const uint4*>(kt + 16 * ((2 * kk + h) ^ (c32 & 15)));
#pragma unroll
                for (int n = QN - 1; n >= 0; n--) s[g] = mfma<F16>(kf, qf[n][kk], s[g]);
            }
        }
        // register r of s[g] is key k0 + 32 g + 8 (r / 4) + 4 h + r % 4
        if (k0 + kKeys > lim_lo) {
#pragma unroll
            for (int g = 0; g < 2; g++)
#pragma unroll
                for (int r = 0; r < 16; r++)
                    if (k0 + 32 * g + 8 * (r >> 2) + 4 * h + (r & 3) >= lim) s[g][r] = ninf;
        }
        float mt = ninf;
#pragma unroll
        for (int r = 0; r < 16; r++) mt = fmaxf(mt, fmaxf(s[0][r], s[1][r]));
        mt = pair32<true>(mt) * c;
        if (__any(mt > m + kLazy<F16>)) {
            const float mn = fmaxf(m, mt);
            const float f = mn == ninf ? 1.0f : __builtin_amdgcn_exp2f(m - mn);
            l *= f;
#pragma unroll
            for (int t = 0; t < 4; t++)
#pragma unroll
                for (int r = 0; r < 16; r++) o[t][r] *= f;
            m = mn;
        }
        const float neg = m == ninf ? 0.0f : kPShift<F16> - m;
        float ls = 0.0f;
#pragma unroll
        for (int g = 0; g < 2; g++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                s[g][r] = __builtin_amdgcn_exp2f(fmaf(s[g][r], c, neg));
                ls += s[g][r];
            }
        l += ls;
        // B of step kk: keys 16 kk + 4 h + 0..3, then 16 kk + 8 + 4 h + 0..3
        const uint8_t* const vt = buf + kTileBytes;
        auto value_frag = [&](int kk, int d) {
            const int f = 32 * d + c32, x = (f >> 1) & 15;
            const uint2 lo = *reinterpret_cast<const uint2*>(vt + f * 128 + 8 * ((4 * kk + h) ^ x));
            const uint2 hi = *reinterpret_cast<const uint2*>(vt + f * 128 + 8 * ((4 * kk + 2 + h) ^ x));
            return make_uint4(lo.x, lo.y, hi.x, hi.y);
        };
#pragma unroll
        for (int kk = 0; kk < 4; kk++) {
            uint32_t t[4][PN];
#pragma unroll
            for (int p = 0; p < 4; p++)
                split_pair<F16, PN>(s[kk >> 1][8 * (kk & 1) + 2 * p], s[kk >> 1][8 * (kk & 1) + 2 * p + 1], t[p]);
#pragma unroll
            for (int d = 0; d < 4; d++) {
                const uint4 vf = value_frag(kk, d);
#pragma unroll
                for (int n = PN - 1; n >= 0; n--)
                    o[d] = mfma<F16>(vf, make_uint4(t[0][n], t[1][n], t[2][n], t[3][n]), o[d]);
            }
        }
    };

    if (kb < ke) {
        load(kb);
        stage(lds);
        if (kb + kKeys < ke) load(kb + kKeys);
        __syncthreads();
        int slot = 0;
        for (int k0 = kb; k0 < ke; k0 += kKeys, slot ^= 1) {
            // LDS slot `slot` holds this tile, the registers the next one
            if (k0 + kKeys < ke) stage(lds + (slot ^ 1) * 2 * kTileBytes);
            if (k0 + 2 * kKeys < ke) load(k0 + 2 * kKeys);
            if (k0 < lim_hi) compute(lds + slot * 2 * kTileBytes, k0);
            __syncthreads();
        }
    }

    l = pair32<false>(l);
    // lane (h, row) holds features 32 t + 8 (r / 4) + 4 h + r % 4
    bool bad = !finite(l);
#pragma unroll
    for (int t = 0; t < 4; t++)
#pragma unroll
        for (int r = 0; r < 16; r++) bad |= !finite(o[t][r]);
    if constexpr (F16) {
        // p * 2^13 is off by up to 2^-25 where it is small, so the result by about
        // 2^-25 / sqrt(3) of the root of the sum of V^2: under 2^-22 of the result
        // unless that is as small as here. (An infinity in V counts as the largest
        // sum of finite values.)
        __shared__ float v2s[4];
        v2 = wave_sum(v2);
        if (lane == 0) v2s[wave] = v2;
        __syncthreads();
        const float all = fminf((v2s[0] + v2s[1]) + (v2s[2] + v2s[3]), 0x1p39f * (float)(ke_all - kb));
        float o2 = 0.0f;
#pragma unroll
        for (int t = 0; t < 4; t++)
#pragma unroll
            for (int r = 0; r < 16; r++) o2 = fmaf(o[t][r], o[t][r], o2);
        o2 = pair32<false>(o2);  // by every lane
        bad |= l > 0.0f && o2 < 0x1p-7f * all;
    }
    const uint64_t votes = __ballot(bad && w0 + c32 < n_rows);
    uint32_t again = (uint32_t)votes | (uint32_t)(votes >> 32);  // rows of the wave to compute again
    const int64_t grow = (int64_t)bhk * n_rows;
    if (w0 + c32 < n_rows && !((again >> c32) & 1u)) {
        if constexpr (SPLIT) {
            float* const po = a.part_o + ((grow + row) * a.nsplit + blockIdx.y) * kDh;
#pragma unroll
            for (int t = 0; t < 4; t++)
#pragma unroll
                for (int g = 0; g < 4; g++)
                    *reinterpret_cast<float4*>(po + 32 * t + 8 * g + 4 * h) =
                        make_float4(o[t][4 * g], o[t][4 * g + 1], o[t][4 * g + 2], o[t][4 * g + 3]);
            if (h == 0)
                *reinterpret_cast<float2*>(a.part_ml + ((grow + row) * a.nsplit + blockIdx.y) * 2) = make_float2(m, l);
        } else {
#pragma unroll
            for (int t = 0; t < 4; t++)
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    const int64_t at = q_off + 32 * t + 8 * g + 4 * h;
                    const float x = o[t][4 * g] / l, y = o[t][4 * g + 1] / l, z = o[t][4 * g + 2] / l,
                                w = o[t][4 * g + 3] / l;
                    if (a.out_dt == JH_F32)
                        *reinterpret_cast<float4*>(static_cast<float*>(a.out) + at) = make_float4(x, y, z, w);
                    else
                        *reinterpret_cast<uint2*>(static_cast<uint16_t*>(a.out) + at) =
                            make_uint2(pack_bf16x2(x, y), pack_bf16x2(z, w));
                }
        }
    }
    // Rows to compute again: sdpa_rows_kernel's arithmetic over the block's keys, kAgain
    // rows of the wave together, so that they share each key's and value's loads (a
    // lane scores a key, and holds two features of the results). q is read from LDS,
    // which the tiles no longer need (the loop's last barrier is behind every wave). A
    // row whose scores are numbers takes m (at most kLazy below its maximum); others
    // take a pass over the keys for it. Bound: VALU, about 1800 cycles per row and 64
    // keys. All rows of 32 heads over 8 not finite, 512 of 512 keys: 631 us, 3.2 ms in
    // the per-row kernel; 300 of 300 of one head: 105 us and 141.
    float* const qs = reinterpret_cast<float*>(lds + wave * (kAgain * kDh * 4));
    while (again) {
        auto widen2 = [](uint32_t u) {
            if constexpr (F16) {
                const f16x2_t x = __builtin_bit_cast(f16x2_t, u);
                return make_float2((float)x.x, (float)x.y);
            } else {
                return make_float2(__uint_as_float(u << 16), __uint_as_float(u & 0xFFFF0000u));
            }
        };
        auto row_at = [&](int r) { return ((int64_t)(b * a.Hk * a.G + hk * a.G + r % a.G) * a.Lq + r / a.G) * kDh; };
        int rr[kAgain], lj[kAgain], count = 0, j = 0;
        float sub[kAgain];  // the row's maximum, in nats
        bool pass = false;
#pragma unroll
        for (int t = 0; t < kAgain; t++) {
            if (again) j = __ffs(again) - 1, again &= again - 1, count = t + 1;  // past the last: a repeat
            rr[t] = w0 + j;
            lj[t] = min(ke_all, limit_of(rr[t]));
            sub[t] = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(m), j)) * (1.0f / kLog2e);
            pass |= !finite(__uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(l), j)));
            const int64_t at = row_at(rr[t]);
            qs[t * kDh + lane] = load_act(a.q, at + lane, a.q_dt);
            qs[t * kDh + lane + 64] = load_act(a.q, at + lane + 64, a.q_dt);
        }
        __builtin_amdgcn_wave_barrier();
        const int end = lj[kAgain - 1];  // the last row's limit is the largest
        auto scores = [&](int key, float (&s)[kAgain]) {
            const uint4* const kp = reinterpret_cast<const uint4*>(a.k + head) + (int64_t)min(key, end - 1) * 16;
            uint4 w[16];
#pragma unroll
            for (int i = 0; i < 16; i++) w[i] = kp[i];
#pragma unroll
            for (int t = 0; t < kAgain; t++) s[t] = 0.0f;
#pragma unroll
            for (int i = 0; i < 16; i++) {
                // one chunk after the other: or all of q is read ahead, and spilled
                int from = 8 * i;
                static_assert(kAgain == 8, "the asm's operands");
                asm volatile("" : "+v"(from), "+v"(s[0]), "+v"(s[1]), "+v"(s[2]), "+v"(s[3]), "+v"(s[4]), "+v"(s[5]),
                             "+v"(s[6]), "+v"(s[7]));
                const float2 x0 = widen2(w[i].x), x1 = widen2(w[i].y), x2 = widen2(w[i].z), x3 = widen2(w[i].w);
#pragma unroll
                for (int t = 0; t < kAgain; t++) {
                    const float4 q0 = *reinterpret_cast<const float4*>(qs + t * kDh + from);
                    const float4 q1 = *reinterpret_cast<const float4*>(qs + t * kDh + from + 4);
                    s[t] = fmaf(q0.x, x0.x, s[t]), s[t] = fmaf(q0.y, x0.y, s[t]);
                    s[t] = fmaf(q0.z, x1.x, s[t]), s[t] = fmaf(q0.w, x1.y, s[t]);
                    s[t] = fmaf(q1.x, x2.x, s[t]), s[t] = fmaf(q1.y, x2.y, s[t]);
                    s[t] = fmaf(q1.z, x3.x, s[t]), s[t] = fmaf(q1.w, x3.y, s[t]);
                }
            }
#pragma unroll
            for (int t = 0; t < kAgain; t++) s[t] *= a.scale;
        };
        float sc[kAgain];
        if (pass) {
#pragma unroll
            for (int t = 0; t < kAgain; t++) sub[t] = ninf;
            for (int k0 = kb; k0 < end; k0 += 64) {
                scores(k0 + lane, sc);
#pragma unroll
                for (int t = 0; t < kAgain; t++)
                    if (k0 + lane < lj[t]) sub[t] = fmaxf(sub[t], sc[t]);
            }
#pragma unroll
            for (int t = 0; t < kAgain; t++) sub[t] = wave_max(sub[t]);
        }
        float ls[kAgain], r0[kAgain], r1[kAgain], e[kAgain];
#pragma unroll
        for (int t = 0; t < kAgain; t++) ls[t] = r0[t] = r1[t] = 0.0f;
        for (int k0 = kb; k0 < end; k0 += 64) {
            scores(k0 + lane, sc);
#pragma unroll
            for (int t = 0; t < kAgain; t++) {
                // a split whose scores are all -inf adds nothing (and without splits
                // the sum of 0 makes the row NaN)
                const float d = sc[t] - (sub[t] == ninf ? 0.0f : sub[t]);
                e[t] = k0 + lane < lj[t] ? (float)exp((double)d) : 0.0f;
                ls[t] += e[t];
            }
            const uint32_t* const vp = reinterpret_cast<const uint32_t*>(a.v + head) + lane;
            for (int j0 = 0; j0 < min(64, end - k0); j0 += 16) {
                uint32_t vw[16];
#pragma unroll
                for (int i = 0; i < 16; i++) vw[i] = vp[(int64_t)min(k0 + j0 + i, end - 1) * 64];
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    const float2 x = widen2(vw[i]);
#pragma unroll
                    for (int t = 0; t < kAgain; t++) {
                        if (k0 + j0 + i >= lj[t]) continue;  // not even 0 times the value
                        const float p =
                            __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(e[t]), j0 + i));
                        r0[t] = fmaf(p, x.x, r0[t]);
                        r1[t] = fmaf(p, x.y, r1[t]);
                    }
                }
            }
        }
#pragma unroll
        for (int t = 0; t < kAgain; t++) {
            ls[t] = wave_sum(ls[t]);
            if (t >= count) break;
            if constexpr (SPLIT) {
                const int64_t part = (grow + rr[t]) * a.nsplit + blockIdx.y;
                // (m, l) in the units of the other rows, whose sums hold 2^kPShift: into m
                // over bf16 values, whose sums it could overflow, into the sums over f16
                // ones (a larger m leaves the merge fewer bits). What rounding m to fp32
                // takes from it goes into the sums.
                constexpr float up = F16 ? 0.0f : kPShift<F16>, by = F16 ? 8192.0f : 1.0f;
                static_assert(!F16 || kPShift<F16> == 13.0f, "2^kPShift");
                const float ms = sub[t] * kLog2e + up;
                const float f = by * (sub[t] == ninf ? 1.0f : (float)exp((double)sub[t] - ((double)ms - up) * 0.69314718055994531));
                *reinterpret_cast<float2*>(a.part_o + part * kDh + 2 * lane) = make_float2(r0[t] * f, r1[t] * f);
                if (lane == 0) *reinterpret_cast<float2*>(a.part_ml + part * 2) = make_float2(ms, ls[t] * f);
            } else {
                const int64_t at = row_at(rr[t]) + 2 * lane;
                store_y(a.out, at, r0[t] / ls[t], a.out_dt);
                store_y(a.out, at + 1, r1[t] / ls[t], a.out_dt);
            }
        }
        __builtin_amdgcn_wave_barrier();
    }
}

// The splits of one row added in split order: one wave per row, lane s holding
// split s's maximum and sum (at most 64 splits), the values requested 8 splits at
// a time, so that a row costs three memory round trips up to 16 splits.
constexpr int kMaxSplits = 64;
__global__ __launch_bounds__(256) void sdpa_mfma_merge_kernel(const float* __restrict__ part_o,
                                                              const float* __restrict__ part_ml, int64_t rows,
                                                              int n_rows, int G, int Lq, int nsplit,
                                                              void* __restrict__ out, int out_dt) {
    const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (row >= rows) return;
    const int64_t bhk = row / n_rows;
    const int r = (int)(row - bhk * n_rows);
    const float2 ml = reinterpret_cast<const float2*>(part_ml)[row * nsplit + min(lane, nsplit - 1)];
    const float mx = wave_max(ml.x);
    // (a split without keys of the row: a sum of 0 and values of 0)
    const float w = lane >= nsplit ? 0.0f : ml.x == mx ? 1.0f : __builtin_amdgcn_exp2f(ml.x - mx);
    const float l = wave_sum(lane >= nsplit ? 0.0f : ml.y * w);
    float x0 = 0.0f, x1 = 0.0f;
    for (int s0 = 0; s0 < nsplit; s0 += 8) {
        float2 o[8];
#pragma unroll
        for (int j = 0; j < 8; j++)
            o[j] = *reinterpret_cast<const float2*>(part_o + (row * nsplit + min(s0 + j, nsplit - 1)) * kDh + 2 * lane);
#pragma unroll
        for (int j = 0; j < 8; j++) {
            if (s0 + j >= nsplit) break;
            const float ws = __shfl(w, s0 + j, 64);
            x0 = fmaf(o[j].x, ws, x0);
            x1 = fmaf(o[j].y, ws, x1);
        }
    }
    const int64_t at = ((bhk * G + r % G) * Lq + r / G) * kDh + 2 * lane;
    store_y(out, at, x0 / l, out_dt);
    store_y(out, at + 1, x1 / l, out_dt);
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

}  // namespace

// Calls the matrix-core kernel takes; others run sdpa_rows_kernel. Its loads
// and stores are 16 bytes wide (buffers so aligned) with 32-bit offsets inside
// a head. fp32 keys and values (no model's caches hold them) stay there, and so
// does a scale of (next to) zero: times it, the largest scores of bf16 are to
// vanish, and the factor above is kept from zero.
bool sdpa_mfma_ok(const void* q, int q_dt, const void* k, const void* v, int kv_dt, const void* out, int64_t B,
                  int64_t Hq, int64_t Hk, int64_t Lq, int64_t Lk, int64_t Dh, float scale) {
    return fabsf(scale) >= 1e-30f && Dh == kDh && Lq > 1 && Lk > 0 && (kv_dt == JH_BF16 || kv_dt == JH_F16) &&
           (q_dt == JH_BF16 || q_dt == JH_F32) && Lk < ((int64_t)1 << 22) && Hq / Hk * Lq < ((int64_t)1 << 30) &&
           B * Hk * ((Hq / Hk * Lq + kRows - 1) / kRows) < ((int64_t)1 << 30) && aligned16(q) && aligned16(k) &&
           aligned16(v) && aligned16(out);
}

size_t sdpa_mfma_workspace_bytes(int64_t B, int64_t Hq, int64_t Lq, int64_t nsplit) {
    return nsplit > 1 ? sizeof(float) * (size_t)(B * Hq * Lq * nsplit) * (kDh + 2) : 0;
}

// Splits of the keys: the count with the least modelled time among those whose
// partials fit max_bytes. On MI355X a 64-key
// tile of 128 rows took 2.4 us in a block alone on its CU and 3.1 us in each of two
// that share one, the merge 4 us and its partials (written and read at about 4
// TB/s). Forced counts beside the model's: 512 queries of 512 keys whole 30 us (fp32 q,
// f16 keys; the model's), in halves 34; 1500 of 4000 whole 227 (bf16; the model's), in
// halves 216, in 16 349; 16 of 4112 whole 159, in halves 86, in 16 28, in 22 (the
// model's) 26.
int64_t sdpa_mfma_splits(int64_t B, int64_t Hq, int64_t Hk, int64_t Lq, int64_t Lk, int num_cus, size_t max_bytes) {
    const int64_t blocks = B * Hk * ((Hq / Hk * Lq + kRows - 1) / kRows), tiles = (Lk + kKeys - 1) / kKeys;
    int64_t best = 1;
    double least = 0;
    for (int64_t n = 1; n <= tiles && n <= kMaxSplits && sdpa_mfma_workspace_bytes(B, Hq, Lq, n) <= max_bytes; n++) {
        const int64_t per_cu = (blocks * n + num_cus - 1) / num_cus;
        const double work = (3.1 * (double)(per_cu / 2) + 2.4 * (double)(per_cu % 2)) * (double)((tiles + n - 1) / n);
        const double t = work + (n > 1 ? 4.0 + (double)(B * Hq * Lq * n) * (2 * (kDh + 2) * 4) / 4e6 : 0.0);
        if (n == 1 || t < least) best = n, least = t;
    }
    return best;
}

Status launch_sdpa_mfma(const void* q, int q_dt, const void* k, const void* v, int kv_dt, void* out, int out_dt,
                        int64_t B, int64_t Hq, int64_t Hk, int64_t Lq, int64_t Lk, int64_t kcap, float scale,
                        bool causal, int64_t nsplit, void* workspace, hipStream_t st) {
    const int64_t G = Hq / Hk, tiles = (G * Lq + kRows - 1) / kRows, rows = B * Hq * Lq;
    SdpaArgs a{};
    a.q = q, a.q_dt = q_dt;
    a.k = static_cast<const uint16_t*>(k), a.v = static_cast<const uint16_t*>(v);
    a.out = out, a.out_dt = out_dt;
    a.Hk = (int)Hk, a.G = (int)G, a.Lq = (int)Lq, a.Lk = (int)Lk, a.n_tiles = (int)tiles, a.BHk = (int)(B * Hk);
    a.kcap = kcap;
    a.scale = scale;
    a.causal = causal ? 1 : 0;
    a.kps = (int)(((Lk + nsplit - 1) / nsplit + kKeys - 1) / kKeys * kKeys);
    a.nsplit = (int)nsplit;
    a.part_o = static_cast<float*>(workspace);
    a.part_ml = a.part_o + (nsplit > 1 ? rows * nsplit * kDh : 0);
    const dim3 grid((unsigned)(tiles * B * Hk), (unsigned)nsplit);
    auto go = [&](auto one, auto many) {
        if (nsplit > 1) hipLaunchKernelGGL(many, grid, dim3(256), 0, st, a);
        else hipLaunchKernelGGL(one, grid, dim3(256), 0, st, a);
    };
    const bool qf = q_dt == JH_F32;
    if (kv_dt == JH_F16)
        qf ? go(sdpa_mfma_kernel<true, 2, false>, sdpa_mfma_kernel<true, 2, true>)
           : go(sdpa_mfma_kernel<true, 1, false>, sdpa_mfma_kernel<true, 1, true>);
    else
        qf ? go(sdpa_mfma_kernel<false, 3, false>, sdpa_mfma_kernel<false, 3, true>)
           : go(sdpa_mfma_kernel<false, 1, false>, sdpa_mfma_kernel<false, 1, true>);
    if (nsplit > 1)
        hipLaunchKernelGGL(sdpa_mfma_merge_kernel, dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, st, a.part_o,
                           a.part_ml, rows, (int)(G * Lq), (int)G, (int)Lq, (int)nsplit, out, out_dt);
    return Status::ok();
}

}  // namespace jh

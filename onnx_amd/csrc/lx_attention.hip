// lx_attention.hip -- long attention heads in one launch (launch_attention_long): scores, scaled masked Softmax and
// context without the [S, SK] scores and probabilities in memory.
//
// Four waves per block: two times 32 query rows of one head, two waves each, one walking the even and one the odd key
// tiles of 32; their sums join at the end.  (A tile is a chain of products, maximum, exponentials and products that one
// wave per SIMD does not cover: [8,12,512,512] heads of 32 52 us with one wave per 32 rows, 46 with two in blocks of
// 128 rows, 38 in blocks of 64, which spread evenly over the CUs.)  Products run
// on the bf16 matrix unit with every operand in three bf16 parts, as k_matmul_f32_b3's (lx_matmul.hip): p1 = bf16(x),
// p2 = bf16(x - p1), p3 = bf16(x - p1 - p2), six part products per product, accumulated in float32: for the scores the
// small ones of all D first, for the context in an accumulator of their own (in one, every MFMA rounded at the size of
// the whole sum).  Against 64 bits, the three float32 nodes in brackets, [2,4,512,512] heads of 64: normal values
// 1.5e-7 (3.5e-7), ReLU'd V 8.1e-8 (8.7e-8), a tenth of Q, K and V 7.1e-8 (9.8e-8), 3% of the keys 1.0e-7 (1.8e-7);
// [2,4,197,197] 1.4e-7 (3.5e-7), 7.0e-8 (1.5e-7), 6.9e-8 (9.7e-8), 8.2e-8 (1.4e-7).  Both products run transposed, so that nothing crosses lanes in between:
//   scores^T  = K Q^T  : lane l holds query l % 32 and keys 8 (r / 4) + 4 (l / 32) + r % 4 of the tile (r = 0..15);
//   context^T = V^T P^T: r = 8 c + j is then the lane's k slot j of the 16 keys c, the order V's tile is stored in.
// The Softmax is the running one: a reference m per row (the row's largest score so far; it follows a new largest
// only when that is over m + 8, so the sums hardly ever rescale), probabilities 2^40 exp(s - m) (the scale keeps the
// parts of the smallest ones exact), their sum and the context divided at the end.  As the reference's ReduceMax
// starts at 0, a row whose scores all lie so far below 0 that exp(s) is 0 gives NaN.
//
// The scale is applied and the mask added in one or two fused steps (the quotient as x zh + x zl with the divisor's
// reciprocal in two floats, after Brisebarre, Muller and Raina 2004; a product for a power of two).  exp(x) is
// v_exp_f32 of the rounded x log2(e) with the rounding error put back to first order.
//
// Values the parts cannot hold (not finite or 2^60 and more in Q, K or V, nonzero below 2^-109 in V) end the walk, and the
// block runs again on the fp32 MFMA; so do a divisor outside [2^-20, 2^60] and a factor of 2^21 and more, which would
// bring the parts lost of tiny Q and K back into the scores.
//
// Bound: the VALU (16 scores per lane and tile, about 17 instructions each with the splitting, beside 24 or 48 MFMAs
// of 32 cycles), and at few heads the chain itself.  The three launches it replaces move the scores through memory
// four times: [8,12,512,512] heads of 32 took 34 + 32 + 25 us against 42 here, [4,12,197,197] heads of 64
// 24 + 8.5 + 18 against 26.6 (94 and 54 us a captured graph, 45 and 27).
#include <hip/hip_runtime.h>

#include "lx_device.h"
#include "lx_kernels.h"

namespace lx {

typedef float v16f __attribute__((ext_vector_type(16)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
typedef float v2f __attribute__((ext_vector_type(2)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uint32_t attn_bf16_pair(float x0, float x1) {
    const v2f x = {x0, x1};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(x, v2bf));
}

// the three parts of eight floats
__device__ __forceinline__ void attn_split8(const float (&x)[8], v4u (&p)[3]) {
    float r[8];
#pragma unroll
    for (int i = 0; i < 8; i++) r[i] = x[i];
#pragma unroll
    for (int z = 0; z < 3; z++) {
#pragma unroll
        for (int i = 0; i < 4; i++) p[z][i] = attn_bf16_pair(r[2 * i], r[2 * i + 1]);
        if (z == 2) break;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            r[2 * i] -= __builtin_bit_cast(float, p[z][i] << 16);
            r[2 * i + 1] -= __builtin_bit_cast(float, p[z][i] & 0xffff0000u);
        }
    }
}

__device__ __forceinline__ v16f attn_mfma(v4u a, v4u b, v16f acc) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, a), __builtin_bit_cast(v8bf, b), acc, 0, 0, 0);
}
// lo + the small part products of A B over 16 k
__device__ __forceinline__ v16f attn_mfma5(const v4u (&a)[3], const v4u (&b)[3], v16f lo) {
    lo = attn_mfma(a[2], b[0], lo);
    lo = attn_mfma(a[0], b[2], lo);
    lo = attn_mfma(a[1], b[1], lo);
    lo = attn_mfma(a[1], b[0], lo);
    return attn_mfma(a[0], b[1], lo);
}

// 2^40 exp(x) for x <= 8 (0 from about x = -87): 2^t with t = x log2(e) rounded, times exp(x - t ln 2) to first order
// (the difference is a rounding error of t; -inf gives NaN there and 0 in 2^t, hence the maximum)
__device__ __forceinline__ float attn_exp40(float x) {
    constexpr float kL = 0x1.715476p+0f, kLn2 = 0x1.62e430p-1f, kLn2lo = -0x1.05c610p-29f;  // log2(e), ln 2 in two floats
    const float t = x * kL;
    const float r = __builtin_fmaxf(__builtin_fmaf(t, -kLn2lo, __builtin_fmaf(t, -kLn2, x)), -1.f);
    const float e = __builtin_amdgcn_exp2f(t) * 0x1p40f;
    return __builtin_fmaf(e, r, e);
}

// DC: 16-wide chunks of D (2 or 4); VT: 32-wide tiles of DV (1 or 2)
template <int DC, int VT>
struct AttnLong {
    static constexpr int kHalf = 128;                         // threads of a key half
    static constexpr int kDch = 2 * DC;                       // eight-wide chunks of a key
    static constexpr int kKStep = 32 * 16 + 16;               // bytes of one chunk of the tile's keys, padded
    static constexpr int kKPart = kDch * kKStep, kVPart = VT * 4 * 512;
    static constexpr int kStage = 3 * (kKPart + kVPart);
    static constexpr int kItemsK = 32 * kDch, kItemsV = VT * 128, kItems = (kItemsK + kItemsV + kHalf - 1) / kHalf;
    static constexpr int kLdK = DC * 16 + 4, kLdV = VT * 32;  // fp32 tiles
    static_assert(4 * 32 * (kLdK + kLdV) <= 4 * kStage && (4 * VT + 1) * 2048 <= 4 * kStage, "the fp32 tiles and the merge fit");
};

// key of slot r (0..15) of half h of a tile
__device__ __forceinline__ constexpr int attn_key(int r, int h) { return 8 * (r / 4) + 4 * h + r % 4; }

template <int DC, int VT, int NOUT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(DC + VT <= 3 ? 3 : DC + VT == 6 ? 1 : 2))) void k_attention_long(AttentionArgs a,
                                                                                                 int vecm, int vecy, int fast,
                                                                                                 int vecq) {
    using T = AttnLong<DC, VT>;
    __shared__ __attribute__((aligned(1024))) char sm[2][2][T::kStage];  // [step][key half]
    __shared__ int bad[2];  // set where a tile (alternating) holds a value the parts cannot hold
    const int t = threadIdx.x & (T::kHalf - 1), l = t & 63, h = l >> 5;  // t: index in the half's staging
    const int w4 = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), w = w4 & 1, kh = w4 >> 1;  // key tiles 2 step + kh
    const int S = a.s, SK = a.sk, D = a.d, DV = a.dv;
    const int qt = (S + 63) / 64;
    const uint32_t z = blockIdx.x / (uint32_t)qt;
    const int i = (int)(blockIdx.x - z * qt) * 64 + 32 * w + (l & 31);  // this lane's query
    int64_t qo = 0, ko = 0, vo = 0, yo = 0;
    {
        uint32_t b = z;  // (the host bounds the batches to 2^31)
        for (int d = a.nbatch - 1; d >= 0; d--) {
            const uint32_t n = (uint32_t)a.bdims[d], x = b % n;
            b /= n;
            qo += x * a.q_bstr[d];
            ko += x * a.k_bstr[d];
            vo += x * a.v_bstr[d];
            yo += x * a.y_bstr[d];
        }
    }
    const int nt = (SK + 31) / 32;
    const int64_t row = (int64_t)z * S + min(i, S - 1);
    const float *mrow = nullptr;
    if constexpr (NOUT != 0) mrow = a.mask + mask_row_offset<NOUT>((uint32_t)row, a.mask_rows);
    const float m1 = NOUT != 0 && !a.mask_inner ? mrow[0] : 0.f;
    // the scale: 0 a product with sf, 1 the two-float quotient, 2 a division
    const float sv = a.scale ? a.scale[0] : 1.f;
    float sf = sv, sl = 0.f;
    int smode = 0;
    const uint32_t sb = __builtin_bit_cast(uint32_t, sv), se = (sb >> 23) & 0xffu;
    if (a.scale && a.scale_div) {
        sf = 1.f / sv;
        sl = __builtin_fmaf(-sf, sv, 1.f) / sv;
        smode = se < 127 - 20 || se > 127 + 60 ? 2 : (sb & 0x7fffffu) ? 1 : 0;
    }
    if (threadIdx.x < 2) bad[threadIdx.x] = 0;

    float mx = -3.0e38f, top = -__builtin_inff(), sum = 0.f;  // reference, largest score, sum of this lane's half
    v16f o[VT], olo[VT];  // the context: the sums of the large and of the small part products
    auto clear = [&]() {
        mx = -3.0e38f;
        top = -__builtin_inff();
        sum = 0.f;
#pragma unroll
        for (int v = 0; v < VT; v++)
#pragma unroll
            for (int r = 0; r < 16; r++) o[v][r] = olo[v][r] = 0.f;
    };
    // the mask elements of this lane's keys of tile kt
    auto load_mask = [&](int kt, float (&mv)[16]) {
        if (NOUT == 0 || !a.mask_inner) {
#pragma unroll
            for (int r = 0; r < 16; r++) mv[r] = m1;
        } else {
#pragma unroll
            for (int g = 0; g < 4; g++) {
                const int key = 32 * kt + 8 * g + 4 * h;
                if (vecm) {
                    const float4 v = *reinterpret_cast<const float4 *>(mrow + min(key, SK - 4));
                    mv[4 * g] = v.x; mv[4 * g + 1] = v.y; mv[4 * g + 2] = v.z; mv[4 * g + 3] = v.w;
                } else {
#pragma unroll
                    for (int e = 0; e < 4; e++) mv[4 * g + e] = mrow[min(key + e, SK - 1)];
                }
            }
        }
    };
    // the products to scores: scale, mask, -inf past the keys
    auto scores = [&](int kt, v16f &s, const float (&mv)[16]) {
        if (smode == 0) {
#pragma unroll
            for (int r = 0; r < 16; r++) s[r] = __builtin_fmaf(s[r], sf, mv[r]);
        } else if (smode == 1) {
#pragma unroll
            for (int r = 0; r < 16; r++) s[r] = __builtin_fmaf(s[r], sf, __builtin_fmaf(s[r], sl, mv[r]));
        } else {
#pragma unroll
            for (int r = 0; r < 16; r++) s[r] = s[r] / sv + mv[r];
        }
        if (32 * kt + 32 > SK) {
#pragma unroll
            for (int r = 0; r < 16; r++)
                if (32 * kt + attn_key(r, h) >= SK) s[r] = -__builtin_inff();
        }
    };
    // scores to probabilities: the running maximum (rescaling the sums where it moved), exp, sum
    auto softmax = [&](bool first, v16f &s) {
        float tm = s[0];
#pragma unroll
        for (int r = 1; r < 16; r++) tm = fmaxf(tm, s[r]);
        tm = fmaxf(tm, __shfl_xor(tm, 32));
        top = fmaxf(top, tm);
        const bool move = tm > mx + 8.f || first;
        if (__any(move)) {
            const float nm = move ? fmaxf(mx, tm) : mx;
            const float al = attn_exp40(mx - nm) * 0x1p-40f;
            mx = nm;
            sum = sum * al;
#pragma unroll
            for (int v = 0; v < VT; v++)
#pragma unroll
                for (int r = 0; r < 16; r++) o[v][r] *= al, olo[v][r] *= al;
        }
        float part[4];
#pragma unroll
        for (int g = 0; g < 4; g++) {
#pragma unroll
            for (int e = 0; e < 4; e++) s[4 * g + e] = attn_exp40(s[4 * g + e] - mx);
            part[g] = (s[4 * g] + s[4 * g + 1]) + (s[4 * g + 2] + s[4 * g + 3]);
        }
        sum += (part[0] + part[1]) + (part[2] + part[3]);
    };

    // Whole tiles of heads of exactly DC * 16 and VT * 32 (fast: K rows contiguous and 16-byte aligned): buffer loads,
    // a tile's base in scalar registers and one constant 32-bit offset per lane (addresses, clamps and selects of the
    // general form took half of the tile's instructions).
    int foff[T::kItems];
#pragma unroll
    for (int n = 0; n < T::kItems; n++) {
        const int it = t + T::kHalf * n, j = it - T::kItemsK, g = j / (32 * VT);
        foff[n] = it < T::kItemsK ? (int)((it / T::kDch * a.k_cs + it % T::kDch * 8) * 4)
                                  : (int)(((16 * (g / 2) + 4 * (g % 2)) * a.v_rs + j % (32 * VT) * a.v_cs) * 4);
    }
    auto load_fast = [&](int n, int kt, float (&x)[8]) {
        const int it = 64 * w + T::kHalf * n;  // (items of a wave are of one kind)
        if (it < T::kItemsK) {
            const auto rs = __builtin_amdgcn_make_buffer_rsrc((void *)(a.k + ko + (int64_t)kt * 32 * a.k_cs), 0, 0x7fffffff, 0x00027000);
#pragma unroll
            for (int e = 0; e < 8; e += 4) {
                const float4 v = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(rs, foff[n], 4 * e, 0));
                x[e] = v.x; x[e + 1] = v.y; x[e + 2] = v.z; x[e + 3] = v.w;
            }
        } else if (it < T::kItemsK + T::kItemsV) {
            const auto rs = __builtin_amdgcn_make_buffer_rsrc((void *)(a.v + vo + (int64_t)kt * 32 * a.v_rs), 0, 0x7fffffff, 0x00027000);
            const int r4 = (int)a.v_rs * 4;
#pragma unroll
            for (int e = 0; e < 8; e++)
                x[e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, foff[n], (e % 4 + 8 * (e / 4)) * r4, 0));
        }
    };
    // staging: item n of the tile is eight consecutive elements of a key (K), or one column of eight keys (V)
    auto load_item = [&](int n, int kt, float (&x)[8]) {
        const int it = t + T::kHalf * n;
        if (it < T::kItemsK) {
            const int key = 32 * kt + it / T::kDch, d0 = it % T::kDch * 8;
            const float *p = a.k + ko + (int64_t)min(key, SK - 1) * a.k_cs;
#pragma unroll
            for (int e = 0; e < 8; e++) x[e] = p[(int64_t)min(d0 + e, D - 1) * a.k_rs];
#pragma unroll
            for (int e = 0; e < 8; e++) x[e] = key < SK && d0 + e < D ? x[e] : 0.f;
        } else if (it < T::kItemsK + T::kItemsV) {
            const int j = it - T::kItemsK, dv = j % (32 * VT), g = j / (32 * VT);  // g: 16 keys g / 2, half g % 2
            const float *p = a.v + vo + (int64_t)min(dv, DV - 1) * a.v_cs;
            const int k0 = 32 * kt + 16 * (g / 2) + 4 * (g % 2);
#pragma unroll
            for (int e = 0; e < 8; e++) x[e] = p[(int64_t)min(k0 + e % 4 + 8 * (e / 4), SK - 1) * a.v_rs];
#pragma unroll
            for (int e = 0; e < 8; e++) x[e] = k0 + e % 4 + 8 * (e / 4) < SK && dv < DV ? x[e] : 0.f;
        }
    };
    auto load_tile = [&](int kt, float (&x)[T::kItems][8]) {
        if (fast && 32 * (kt + 1) <= SK) {
#pragma unroll
            for (int n = 0; n < T::kItems; n++) load_fast(n, kt, x[n]);
        } else {
#pragma unroll
            for (int n = 0; n < T::kItems; n++) load_item(n, kt, x[n]);
        }
    };
    auto store_item = [&](int n, const float (&x)[8], char *st, int *flag) {
        const int it = t + T::kHalf * n;
        if (it >= T::kItemsK + T::kItemsV) return;
        const bool isk = it < T::kItemsK;
        // magnitudes as integers (a NaN is the largest), zero the largest less one
        uint32_t big = 0, tiny = 0xffffffffu;
#pragma unroll
        for (int e = 0; e < 8; e += 2) {
            const uint32_t u0 = __builtin_bit_cast(uint32_t, x[e]) << 1, u1 = __builtin_bit_cast(uint32_t, x[e + 1]) << 1;
            big = max(max(u0, u1), big);
            if (!isk) tiny = min(min(u0 - 1u, u1 - 1u), tiny);
        }
        if (big >= (127u + 60u) << 24 || tiny < (18u << 24) - 1u) *flag = 1;
        v4u p[3];
        attn_split8(x, p);
        const int j = it - T::kItemsK;
        char *d = isk ? st + it % T::kDch * T::kKStep + it / T::kDch * 16
                      : st + 3 * T::kKPart + ((j % (32 * VT) / 32 * 4 + j / (32 * VT)) * 32 + j % 32) * 16;
        const int ps = isk ? T::kKPart : T::kVPart;
#pragma unroll
        for (int q = 0; q < 3; q++) *reinterpret_cast<v4u *>(d + q * ps) = p[q];
    };

    clear();
    bool again = smode == 2 || (smode == 0 && se > 127 + 20 && !a.scale_div);
    if (!again) {
        // Q in parts: lane l holds query l % 32, elements 16 c + 8 (l / 32) ..
        v4u qp[DC][3];
        float x0[T::kItems][8];
        load_tile(kh, x0);
        __syncthreads();
#pragma unroll
        for (int c = 0; c < DC; c++) {
            float x[8];
            const float *p = a.q + qo + (int64_t)min(i, S - 1) * a.q_rs;
            if (vecq) {
#pragma unroll
                for (int e = 0; e < 8; e += 4) {
                    const float4 v = *reinterpret_cast<const float4 *>(p + 16 * c + 8 * h + e);
                    x[e] = v.x; x[e + 1] = v.y; x[e + 2] = v.z; x[e + 3] = v.w;
                }
            } else {
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    const int d = 16 * c + 8 * h + e;
                    x[e] = p[(int64_t)min(d, D - 1) * a.q_cs];
                    x[e] = d < D ? x[e] : 0.f;
                }
            }
            bool fin = true;
#pragma unroll
            for (int e = 0; e < 8; e++) fin = fin && fabsf(x[e]) < 0x1p60f;
            if (!fin) bad[0] = 1;
            attn_split8(x, qp[c]);
        }
#pragma unroll
        for (int n = 0; n < T::kItems; n++) store_item(n, x0[n], sm[0][kh], &bad[0]);
        __syncthreads();
        for (int st = 0; 2 * st < nt; st++) {
            // every wave reads the same verdict: the next step's goes to the other word, this word's next write
            // comes after the barrier below
            if ((again = bad[st & 1] != 0)) break;
            const int kt = 2 * st + kh, kn = kt + 2;  // (tiles past the keys hold zeros)
            float mv[16];
            load_mask(kt, mv);
            load_tile(kn, x0);
            const char *ks = sm[st & 1][kh] + (l & 31) * 16 + h * T::kKStep;
            v16f s;
            v4u k1[DC];  // the small part products of every chunk, then the large ones
#pragma unroll
            for (int r = 0; r < 16; r++) s[r] = 0.f;
#pragma unroll
            for (int c = 0; c < DC; c++) {
                v4u kp[3];
#pragma unroll
                for (int q = 0; q < 3; q++)
                    kp[q] = *reinterpret_cast<const v4u *>(ks + q * T::kKPart + 2 * c * T::kKStep);
                k1[c] = kp[0];
                s = attn_mfma5(kp, qp[c], s);
            }
#pragma unroll
            for (int c = 0; c < DC; c++) s = attn_mfma(k1[c], qp[c][0], s);
            scores(kt, s, mv);
            softmax(st == 0, s);
            v4u pp[2][3];
#pragma unroll
            for (int c = 0; c < 2; c++) {
                float x[8];
#pragma unroll
                for (int e = 0; e < 8; e++) x[e] = s[8 * c + e];
                attn_split8(x, pp[c]);
            }
            const char *vs = sm[st & 1][kh] + 3 * T::kKPart + (h * 32 + (l & 31)) * 16;
#pragma unroll
            for (int c = 0; c < 2; c++) {  // (the two accumulations of VT tiles side by side: neighbouring MFMAs are independent)
                v4u vp[VT][3];
#pragma unroll
                for (int v = 0; v < VT; v++)
#pragma unroll
                    for (int q = 0; q < 3; q++)
                        vp[v][q] = *reinterpret_cast<const v4u *>(vs + q * T::kVPart + (v * 4 + c * 2) * 512);
#pragma unroll
                for (int z = 0; z < 6; z++)
#pragma unroll
                    for (int v = 0; v < VT; v++) {
                        constexpr int pa[6] = {2, 0, 1, 1, 0, 0}, pb[6] = {0, 2, 1, 0, 1, 0};
                        v16f &t = z == 5 ? o[v] : olo[v];
                        t = attn_mfma(vp[v][pa[z]], pp[c][pb[z]], t);
                    }
            }
#pragma unroll
            for (int n = 0; n < T::kItems; n++) store_item(n, x0[n], sm[(st + 1) & 1][kh], &bad[(st + 1) & 1]);
            __syncthreads();
        }
    }
    float total = 1.f;  // what the context is divided by
    if (again) {
        // on the fp32 MFMA, the tiles in float32: a walk for the maxima and sums, then one with the divided
        // probabilities (at most 1: no sum overflows that the nodes' does not)
        clear();
        float *kf = reinterpret_cast<float *>(sm[0][0]), *vf = kf + 32 * T::kLdK;
        const float *qr = a.q + qo + (int64_t)min(i, S - 1) * a.q_rs;
        for (int n = 0; n < 2 * nt; n++) {
            const bool second = n >= nt;
            const int kt = second ? n - nt : n;
            if (n == nt) total = sum + __shfl_xor(sum, 32);
            float mv[16];
            load_mask(kt, mv);
            __syncthreads();
            for (int e = threadIdx.x; e < 32 * DC * 16; e += 256) {
                const int key = e / (DC * 16), d = e % (DC * 16);
                kf[key * T::kLdK + d] = 32 * kt + key < SK && d < D ? a.k[ko + (int64_t)(32 * kt + key) * a.k_cs + (int64_t)d * a.k_rs] : 0.f;
            }
            for (int e = threadIdx.x; e < 32 * VT * 32; e += 256) {
                const int key = e / (VT * 32), d = e % (VT * 32);
                vf[key * T::kLdV + d] = 32 * kt + key < SK && d < DV ? a.v[vo + (int64_t)(32 * kt + key) * a.v_rs + (int64_t)d * a.v_cs] : 0.f;
            }
            __syncthreads();
            v16f s;
#pragma unroll
            for (int r = 0; r < 16; r++) s[r] = 0.f;
            for (int c = 0; c < DC; c++)
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    const int d = 16 * c + 8 * h + j;
                    const float qv = d < D ? qr[(int64_t)d * a.q_cs] : 0.f;
                    s = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[(l & 31) * T::kLdK + d], qv, s, 0, 0, 0);
                }
            scores(kt, s, mv);
            if (!second) {
                softmax(n == 0, s);
                continue;
            }
#pragma unroll
            for (int r = 0; r < 16; r++) s[r] = attn_exp40(s[r] - mx) / total;
#pragma unroll
            for (int v = 0; v < VT; v++)
#pragma unroll
                for (int r = 0; r < 16; r++)
                    o[v] = __builtin_amdgcn_mfma_f32_32x32x2f32(vf[attn_key(r, h) * T::kLdV + 32 * v + (l & 31)], s[r], o[v], 0, 0, 0);
        }
        total = 1.f;
    } else {
#pragma unroll
        for (int v = 0; v < VT; v++)
#pragma unroll
            for (int r = 0; r < 16; r++) o[v][r] = o[v][r] + olo[v][r];

        // the second half's context, sum and maxima join the first's (both stages are read: the barrier above)
        float *x = reinterpret_cast<float *>(sm) + (w * 64 + l) * 4;
        constexpr int kRow = 2 * 64 * 4;  // floats of four values of every lane
        if (kh) {
#pragma unroll
            for (int v = 0; v < VT; v++)
#pragma unroll
                for (int g = 0; g < 4; g++)
                    *reinterpret_cast<float4 *>(x + (4 * v + g) * kRow) =
                        make_float4(o[v][4 * g], o[v][4 * g + 1], o[v][4 * g + 2], o[v][4 * g + 3]);
            *reinterpret_cast<float4 *>(x + 4 * VT * kRow) = make_float4(mx, sum, top, 0.f);
        }
        __syncthreads();
        if (!kh) {
            const float4 q = *reinterpret_cast<const float4 *>(x + 4 * VT * kRow);
            const float m = fmaxf(mx, q.x), fa = attn_exp40(mx - m) * 0x1p-40f, fb = attn_exp40(q.x - m) * 0x1p-40f;
            sum = sum * fa + q.y * fb;
            top = fmaxf(top, q.z);
#pragma unroll
            for (int v = 0; v < VT; v++)
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    const float4 y = *reinterpret_cast<const float4 *>(x + (4 * v + g) * kRow);
                    o[v][4 * g] = o[v][4 * g] * fa + y.x * fb;
                    o[v][4 * g + 1] = o[v][4 * g + 1] * fa + y.y * fb;
                    o[v][4 * g + 2] = o[v][4 * g + 2] * fa + y.z * fb;
                    o[v][4 * g + 3] = o[v][4 * g + 3] * fa + y.w * fb;
                }
        }
        total = sum + __shfl_xor(sum, 32);
    }
    if (i >= S || kh) return;
    // a row whose exp(s) are all 0 is 0 / 0 in the reference (its maximum starts at 0)
    if (top < -103.97208f) total = __builtin_nanf("");
    // divided with the reciprocal in two floats (the fp32 walk's total is 1 and its context may be infinite)
    const float inv = 1.f / total, invlo = __builtin_fmaf(-inv, total, 1.f) * inv;
#pragma unroll
    for (int v = 0; v < VT; v++)
#pragma unroll
        for (int r = 0; r < 16; r++) {
            if (again) o[v][r] *= inv;
            else o[v][r] = __builtin_fmaf(o[v][r], inv, o[v][r] * invlo);
        }
    float *Y = a.y + yo + (int64_t)i * a.y_rs;
#pragma unroll
    for (int v = 0; v < VT; v++)
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const int dv = 32 * v + 8 * g + 4 * h;
            if (vecy) {
                if (dv < DV)
                    *reinterpret_cast<float4 *>(Y + dv) =
                        make_float4(o[v][4 * g], o[v][4 * g + 1], o[v][4 * g + 2], o[v][4 * g + 3]);
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++)
                    if (dv + e < DV) Y[(int64_t)(dv + e) * a.y_cs] = o[v][4 * g + e];
            }
        }
}

template <int DC, int VT>
static void attention_long_launch(const AttentionArgs &a, int vecm, int vecy, hipStream_t s) {
    // K rows contiguous and 16-byte aligned, offsets within a tile below 2^31 bytes
    int fast = a.d == DC * 16 && a.dv == VT * 32 && a.k_rs == 1 && a.k_cs % 4 == 0 && (uintptr_t)a.k % 16 == 0 &&
               a.k_cs < (1 << 23) && a.v_rs < (1 << 22) && a.v_cs < (1 << 21);
    int vecq = a.d == DC * 16 && a.q_cs == 1 && a.q_rs % 4 == 0 && (uintptr_t)a.q % 16 == 0;
    for (int d = 0; d < a.nbatch; d++) {
        fast = fast && a.k_bstr[d] % 4 == 0;
        vecq = vecq && a.q_bstr[d] % 4 == 0;
    }
    const dim3 g((unsigned)(a.batch * ((a.s + 63) / 64))), blk(256);
    switch (a.mask ? a.mask_rows.nouter : 0) {
    case 1: hipLaunchKernelGGL((k_attention_long<DC, VT, 1>), g, blk, 0, s, a, vecm, vecy, fast, vecq); break;
    case 2: hipLaunchKernelGGL((k_attention_long<DC, VT, 2>), g, blk, 0, s, a, vecm, vecy, fast, vecq); break;
    default:
        if (a.mask) hipLaunchKernelGGL((k_attention_long<DC, VT, -1>), g, blk, 0, s, a, vecm, vecy, fast, vecq);
        else hipLaunchKernelGGL((k_attention_long<DC, VT, 0>), g, blk, 0, s, a, vecm, vecy, fast, vecq);
    }
}

// Whether heads run here: kernel sizes, and the estimated time (us) below that of the three launches.  Here: rounds of
// blocks of 64 rows, `per` of them on a CU; a block takes `block` and, per step of 64 keys, `step` (`inexact` times that
// where D or DV is not the tile's and the loads are the general ones), `more` for every other block on its CU.  Each step
// is a chain of products, maximum, exponentials and products, so few heads over many keys wait for it where the three
// launches spread over the chip (128 rows and 1024 keys of one head of 64: 56.5 against 21.7 us).  The three launches:
// `nodes`, then by the scores' elements, their rows 16-byte aligned or not (four passes over them), and, where the context's K does not split, by the keys.  Fitted to 577 shapes (heads of 16
// to 64, 1 to 384 of them, 65 to 2048 rows and 73 to 2048 keys): what it picks is within 10% of the faster one in 574.
bool attention_long_fits(const AttentionArgs &a) {
    if (a.s <= 64 || a.sk <= kAttentionLongKeys || a.d < 1 || a.d > 64 || a.dv < 1 || a.dv > 64 || a.batch < 1) return false;
    const int64_t blocks = a.batch * ((a.s + 63) / 64);
    if (blocks > 0x7fffffff) return false;
    struct Cost {
        double launch, block, step, more, inexact, tail;
        int per;
    };
    static const Cost kCost[3] = {{8.7, 4.1, 1.6, 1.2, 1.5, 0.4, 3}, {5.8, 8.7, 1.6, 1.6, 1.5, 0.6, 2}, {5.2, 9.6, 2.6, 0, 1.7, 1.2, 1}};
    const bool wide = a.d > 32, tall = a.dv > 32;
    const Cost &c = kCost[wide + tall];
    const double steps = (double)((a.sk + 63) / 64), fixed = c.block + (a.sk % 32 ? c.tail : 0);
    const double step = c.step * (a.d == (wide ? 64 : 32) && a.dv == (tall ? 64 : 32) ? 1 : c.inexact);
    const int64_t per_cu = (blocks + 255) / 256, rest = per_cu % c.per;
    double here = c.launch + (double)(per_cu / c.per) * (fixed + steps * (step + c.more * (c.per - 1)));
    if (rest) here += fixed + steps * (step + c.more * (double)(rest - 1));
    const double scores = 1e-6 * (double)a.batch * a.s * a.sk;
    const double nodes = wide || tall ? 19 + scores * (a.sk % 4 ? 13.9 : 4.5) + (a.sk % 64 ? 0.023 * a.sk : 0) + (a.sk % 4 ? 4.4 : 0)
                                      : 18.5 + scores * (a.sk % 4 ? 11.5 : 3.8) + (a.sk % 64 ? 0.032 * a.sk : 0);
    return here < nodes;
}

hipError_t launch_attention_long(const AttentionArgs &a, hipStream_t s) {
    if (!attention_long_fits(a)) return hipErrorInvalidValue;
    // 16-byte mask reads: rows of a multiple of 4 keys at aligned offsets; 16-byte stores of y likewise
    int vecm = a.mask && a.mask_inner && a.sk % 4 == 0 && (uintptr_t)a.mask % 16 == 0;
    for (int d = 0; d < a.mask_rows.nouter; d++) vecm = vecm && a.mask_rows.a_str[d] % 4 == 0;
    int vecy = a.y_cs == 1 && a.dv % 4 == 0 && a.y_rs % 4 == 0 && (uintptr_t)a.y % 16 == 0;
    for (int d = 0; d < a.nbatch; d++) vecy = vecy && a.y_bstr[d] % 4 == 0;
    if (a.d <= 32) {
        if (a.dv <= 32) attention_long_launch<2, 1>(a, vecm, vecy, s);
        else attention_long_launch<2, 2>(a, vecm, vecy, s);
    } else {
        if (a.dv <= 32) attention_long_launch<4, 1>(a, vecm, vecy, s);
        else attention_long_launch<4, 2>(a, vecm, vecy, s);
    }
    return hipGetLastError();
}

}  // namespace lx

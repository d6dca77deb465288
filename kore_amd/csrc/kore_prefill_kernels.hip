// kore_prefill_kernels.hip - gfx950 kernels of kore's batched causal attention
// (forward_batch(), kore.cpp:1542-1563), any even head_dim up to 256 and any
// number of q-heads per kv-head.
//
//   prefill_kernel          causal attention of a chunk of query rows over the
//                           cache, both products on fp16 MFMA with every
//                           operand split into two or three fp16 parts
//   prefill_fp32            the same on fp32 MFMA, where the parts would lose bits
//   prefill_combine_kernel  merge of the key ranges that a query row's work
//                           was split into
//
// Why split fp16.  The fp32 matrix rate (157 TFLOP/s) bounds the two products;
// fp16 runs 16 times as fast, and x = hi + lo with hi = fp16(x), lo = fp16(x -
// hi) carries 23 of 24 bits, so three products (hi hi + hi lo + lo hi, each exact,
// summed in fp32) cost 3 / 16 of the fp32 ones.  The sums take 16 products per
// fp32 rounding instead of two, and the score's small cross terms are summed
// first, so the result is nearer to the exact one than the fp32 kernel's was
// (28/4/128, 2048 rows, mean of six draws: 5.0e-7 of the 2-norm against 9.1e-7;
// 12/2/128, 333 rows at 7001: 6.6e-7 against 1.28e-6).  A head_dim that is neither
// 64 nor 128 ran on VALU with fp64 scores; to lose nothing there a third part
// holds the last bit (six products) and the scores' 16-dim pieces are summed in
// fp64 (33/3/96, 700 rows at 100: 2.4e-7 against 3.9e-7).  A call of a few keys may
// differ by one rounding of the MFMA's sum either way (one row alone: 1.4e-8, and V
// itself before).
//
// Measured, one layer, against the kernels before (fp32 MFMA; VALU for 33/3/96):
// 28/4/128 2048 rows 261 -> 146 us (115 -> 206 TFLOP/s), 12/2/128 333 rows at
// 7001 151 -> 75 us, 33/3/96 700 rows at 100 730 -> 93 us.  Before the checks that
// send a tile to prefill_fp32, and the units that follow the weights, these took
// 141, 72 and 82 us, with wrong results for the data that needs them.
// What bounds it: MFMAs 27 % of a SIMD's cycles, other vector instructions 29 to 33 %,
// and a wave does one after the other (39 % of the waves' time waits for an issue).
//
// Range.  fp16 holds 2^-24 .. 65504, so every operand is scaled by a power of
// two (exact) that brings its largest magnitude to 2^13 .. 2^14: a query row
// by its own, K and V by groups of eight keys, a query's softmax weights by one
// that follows them.  A value's parts go down to 2^-25, so what a small one loses
// is 2^-38 of its group's largest.  Where that could be seen in an output (V
// whose keys, dims, groups or tiles lie far apart in size, or K and q that make a
// score coarse) or a value is not finite, the workgroup starts again on
// prefill_fp32, as the fp32 products were: such values reach exactly the rows that
// attend them.  With one key's V 1e6 times the others' 28/4/128, 2048 rows take
// 410 us, 33/3/96, 700 rows 118.

#include "kore_attn_kernels.h"
#include "kore_attn_device.h"

#include <algorithm>
#include <vector>

namespace kore_attn_gpu {
namespace {

typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float float2v __attribute__((ext_vector_type(2)));
typedef float float8v __attribute__((ext_vector_type(8)));
// vectors of floats at any float's address (q, out and odd geometries' rows)
typedef float f2u __attribute__((ext_vector_type(2), aligned(4)));
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));

// v_mfma_f32_32x32x16_f16: lane l supplies A[l % 32][8 (l / 32) + e] and B[8
// (l / 32) + e][l % 32], e = 0..7; D register r of lane l is D[8 (r / 4) + 4
// (l / 32) + r % 4][l % 32].
__device__ __forceinline__ floatx16 mfma32h(half8 a, half8 b, floatx16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

// v_mfma_f32_32x32x2_f32: A[l % 32][l / 32], B[l / 32][l % 32], D as above
__device__ __forceinline__ floatx16 mfma32f(float a, float b, floatx16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

// the fp16 parts of eight values times sc (a power of two), PARTS of them: hi,
// lo and what those two leave (one bit of 24)
template <int PARTS>
__device__ __forceinline__ void split8(const float8v &x, float sc, half8 *p) {
#pragma unroll
    for (int e = 0; e < 8; e += 2) {
        const half2v h = __builtin_convertvector((float2v{x[e] * sc, x[e + 1] * sc}), half2v);
        const float r0 = fmaf(x[e], sc, -(float)h[0]), r1 = fmaf(x[e + 1], sc, -(float)h[1]);
        const half2v l = __builtin_convertvector((float2v{r0, r1}), half2v);
        p[0][e] = h[0];
        p[0][e + 1] = h[1];
        p[1][e] = l[0];
        p[1][e + 1] = l[1];
        if constexpr (PARTS == 3) {
            const half2v r = __builtin_convertvector((float2v{r0 - (float)l[0], r1 - (float)l[1]}), half2v);
            p[2][e] = r[0];
            p[2][e + 1] = r[1];
        }
    }
}

// the larger magnitude, NaN if either is
__device__ __forceinline__ float nmax(float a, float b) { return __builtin_elementwise_maximum(a, b); }
__device__ __forceinline__ float wave_nmax(float x) {
    x = nmax(x, dpp<0x128>(x));
    x = nmax(x, dpp<0x124>(x));
    x = nmax(x, dpp<0x122>(x));
    x = nmax(x, dpp<0x121>(x));
    float a, b;
    pair16(x, a, b);
    x = nmax(a, b);
    pair32(x, a, b);
    return nmax(a, b);
}
__device__ __forceinline__ float pow2(int e) { return __builtin_bit_cast(float, (uint32_t)(e + 127) << 23); }
// exponent s with max |x| 2^s in [2^13, 2^14), at most 126 (zeros, tiny values)
__device__ __forceinline__ int scale_exp(float mx) { return mx > 0.f ? min(14 - __builtin_amdgcn_frexp_expf(mx), 126) : 126; }
constexpr int kZeroExp = 127;   // the scale of a V group of zeros

// workgroups of prefill_kernel that fit a CU (registers, LDS)
constexpr int per_cu(int hdp, bool exact) { return hdp <= (exact ? 128 : 96) ? 2 : 1; }

constexpr int kMfma = 0x8, kDsRead = 0x100;   // __builtin_amdgcn_sched_group_barrier classes
constexpr int kBK = 32;           // keys per tile
// Limits of the two- and three-part products.  Weights are scaled so that a
// tile's largest lies in 2^kTMin .. 2^kTMax (fp16 ends below 2^16), and is put to
// 2^kTNew where it does not; below 2^kTMin it matters only to an output that is
// small in the same units: kEnough is 2^22 against the 2^-11 that a lost part is
// worth (2^-25 times V's 2^14).  At 2^kTMin the parts still have 24 bits beside V
// groups of 2^-kSpread, a spread that tokens whose V differ 50-fold do not reach
// (28/4/128, 2048 rows: 151 us; with a limit of 2^-3 459, in the fp32 loop).
constexpr float kTMax = 15.f, kTMin = 8.f;
constexpr int kTNew = 11;
constexpr float kEnough = 0x1p22f;
constexpr int kSpread = 6;        // log2 of the spread of V's group scales in a tile
constexpr int kRange = 40;        // ... and over a workgroup's tiles (exponents stay in fp32's range)
constexpr int kNone = 1 << 20;    // a unit before any key (pow2 drops it)

// What both loops of prefill_kernel share: a workgroup's place in the work, a
// lane's query row, its share of a tile in registers, and the output.
template <int HDP, bool EXACT>
struct PrefillLane {
    static constexpr int KS = HDP / 16;             // k-steps of the scores
    static constexpr int NT = HDP / 32;             // output blocks
    static constexpr int C8 = HDP / 8;              // 8-dim chunks of a K row
    static constexpr int NUK = (HDP + 63) / 64;     // (key, chunk) units of K per lane
    static constexpr int VD = HDP % 128 == 0 ? 2 : 1;           // dims per V unit
    static constexpr int NUV = (HDP / VD + 63) / 64;
    static constexpr int kKB = C8 * 33 * 16, kVB = 4 * HDP * 16;        // bytes of one part of a tile
    static constexpr int PARTS = EXACT ? 2 : 3;     // fp16 parts of an operand
    static constexpr int kVOff = PARTS * kKB, kMeta = PARTS * (kKB + kVB), kBuf = kMeta + 48;
    static constexpr int kVOff32 = 2 * kKB;         // V of the fp32 loop's tiles
    static constexpr int NBUF = 2 * kBuf <= 160 * 1024 ? 2 : 1;

    const float *q, *kg, *vg;
    const float2 *cs;
    float *out, *part_o, *part_ml;
    int hd_, n_kseg, n_split, n_items, g, item, part, seg, F, ws, n_keys, t_begin, t_end, my_kmin, my_kmax;
    int lane, wave, qi, qg, qpos, vkey0;
    bool qvalid;
    size_t qoff;
    // ---- this wave's share of a tile: keys 8 wave .. + 7 of K as (key, chunk)
    // units, keys {0..3, 8..11} + 16 (wave / 2) + 4 (wave % 2) of V as dims
    float8v rk[NUK], rv[NUV][VD];

    __device__ __forceinline__ int hd() const { return EXACT ? HDP : hd_; }
    // not EXACT, offsets and masks that derive from the lane are many: computed
    // anew for every tile, as keeping them costs the loop spills
    __device__ __forceinline__ int fresh_lane() const {
        int l = lane;
        if constexpr (!EXACT) asm volatile("" : "+v"(l));
        return l;
    }

    // wi: the workgroup's place in the work list
    template <class Args>
    __device__ __forceinline__ PrefillLane(const Args &a, int wi) {
        q = a.q; cs = a.cs; out = a.out; part_o = a.part_o; part_ml = a.part_ml;
        hd_ = a.hd; n_kseg = a.n_kseg; n_split = a.n_split; n_items = a.n_items;
        const int tid = threadIdx.x, nkv = a.n_head_kv, n_rep = a.n_rep;
        lane = tid & 63;
        wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        g = wi % nkv;
        // split plan: item << 2 | part (0 whole, 1 / 2 first / second half)
        const int code = n_split > 0 ? (int)a.unit[wi / nkv] : 0;
        part = code & 3;
        seg = n_split > 0 ? 0 : (wi / nkv) % n_kseg;
        item = n_split > 0 ? code >> 2 : wi / nkv / n_kseg;
        F = a.n_tok * n_rep;
        const int n_head = nkv * n_rep, f0 = kPrefillRows * (n_items - 1 - item);    // the item's first row
        n_keys = a.pos0 + a.n_tok;
        const int n_tiles = (a.pos0 + min(f0 + kPrefillRows - 1, F - 1) / n_rep) / kBK + 1;
        ws = f0 + 32 * wave;                                     // this wave's first row
        my_kmin = a.pos0 + min(ws, F - 1) / n_rep;               // key limits of its first and last row
        my_kmax = ws < F ? a.pos0 + min(ws + 31, F - 1) / n_rep : -1;
        // key tiles of this workgroup: a key segment, a half of a split item
        // (the plan splits only items of at least two tiles), or all of them
        const int t_half = n_tiles / 2;
        t_begin = part == 2 ? t_half : seg * a.seg_tiles;
        t_end = part == 1 ? t_half : (n_kseg == 1 ? n_tiles : min(n_tiles, t_begin + a.seg_tiles));

        qi = lane & 31;
        qg = lane >> 5;
        const int fq = ws + qi, fqc = min(fq, F - 1), qz = fqc / n_rep;
        qvalid = fq < F;
        qpos = a.pos0 + qz;
        qoff = ((size_t)qz * n_head + (size_t)g * n_rep + (fqc - qz * n_rep)) * hd();
        kg = a.kc + (size_t)g * a.slots * hd();
        vg = a.vc + (size_t)g * a.slots * hd();
        vkey0 = 16 * (wave >> 1) + 4 * (wave & 1);
    }

    // rows past the last key repeat it (they are masked): uniform bases, 32-bit lane offsets
    __device__ __forceinline__ void load_tile(int t) {
        const int lane = fresh_lane();
        const int k0 = t * kBK, last = n_keys - 1 - k0;
        const float *kt = kg + (size_t)k0 * hd();
#pragma unroll
        for (int i = 0; i < NUK; ++i) {
            const int u = min(lane + 64 * i, HDP - 1);
            const unsigned row = __umul24(min(8 * wave + u / C8, last), hd());
            const int d = 8 * (u % C8);
            if constexpr (EXACT) {
                const float4 x = ld4(kt + (row + d)), y = ld4(kt + (row + d + 4));
                rk[i][0] = x.x; rk[i][1] = x.y; rk[i][2] = x.z; rk[i][3] = x.w;
                rk[i][4] = y.x; rk[i][5] = y.y; rk[i][6] = y.z; rk[i][7] = y.w;
            } else {
#pragma unroll
                for (int e = 0; e < 8; e += 2) {   // head_dim is even: pairs are whole
                    const float2 x = *(const float2 *)(kt + (row + min(d + e, hd() - 2)));
                    rk[i][e] = x.x;
                    rk[i][e + 1] = x.y;
                }
            }
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float *vt = vg + (size_t)(k0 + min(vkey0 + (j & 3) + 8 * (j >> 2), last)) * hd();
#pragma unroll
            for (int i = 0; i < NUV; ++i) {
                const unsigned d = VD * min(lane + 64 * i, HDP / VD - 1);
                if constexpr (VD == 2) {
                    const float2 x = *(const float2 *)(vt + (EXACT ? d : min(d, (unsigned)hd() - 2)));
                    rv[i][0][j] = x.x;
                    rv[i][1][j] = x.y;
                } else {
                    rv[i][0][j] = vt[EXACT ? d : min(d, (unsigned)hd() - 1)];
                }
            }
        }
    }
    // dims past head_dim (read from its last ones) count as zeros
    __device__ __forceinline__ void clear_pad() {
        const int lane = fresh_lane();
        if constexpr (!EXACT) {
#pragma unroll
            for (int i = 0; i < NUK; ++i)
#pragma unroll
                for (int e = 0; e < 8; ++e) rk[i][e] = 8 * (min(lane + 64 * i, HDP - 1) % C8) + e < hd() ? rk[i][e] : 0.f;
#pragma unroll
            for (int i = 0; i < NUV; ++i)
#pragma unroll
                for (int d = 0; d < VD; ++d)
#pragma unroll
                    for (int j = 0; j < 8; ++j) rv[i][d][j] = VD * (lane + 64 * i) < hd() ? rv[i][d][j] : 0.f;
        }
    }
    // roped q of the lane's row, dims 16 s + 8 qg + e
    __device__ __forceinline__ void load_q(float8v *y) const {
        const float *qp = q + qoff;
        const int half = hd() / 2;
        const float *cp = (const float *)(cs + (size_t)qpos * half);
        if constexpr (EXACT) {                     // dim d + hd() / 2 is the same lane's, HDP / 32 steps on
#pragma unroll
            for (int s = 0; s < KS / 2; ++s) {
                const int d = 16 * s + 8 * qg;
                f4u lo[2], hi[2], c[4];
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    lo[k] = *(const f4u *)(qp + d + 4 * k);
                    hi[k] = *(const f4u *)(qp + half + d + 4 * k);
                }
#pragma unroll
                for (int k = 0; k < 4; ++k) c[k] = *(const f4u *)(cp + 2 * d + 4 * k);
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    float y0, y1;
                    rope_pair(lo[e / 4][e % 4], hi[e / 4][e % 4], make_float2(c[e / 2][2 * (e % 2)], c[e / 2][2 * (e % 2) + 1]),
                              y0, y1);
                    y[s][e] = y0;
                    y[s + KS / 2][e] = y1;
                }
            }
        } else {
#pragma unroll
            for (int s = 0; s < KS; ++s) {
                const int d = 16 * s + 8 * qg;
                const bool low = d + 8 <= half, high = d >= half && d + 8 <= hd();
                if (low || high) {                 // eight dims on one side of the rotation
                    const int d0 = low ? d : d - half;
                    f4u lo[2], hi[2], c[4];
#pragma unroll
                    for (int k = 0; k < 2; ++k) {
                        lo[k] = *(const f4u *)(qp + d0 + 4 * k);
                        hi[k] = *(const f4u *)(qp + half + d0 + 4 * k);
                    }
#pragma unroll
                    for (int k = 0; k < 4; ++k) c[k] = *(const f4u *)(cp + 2 * d0 + 4 * k);
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        float y0, y1;
                        rope_pair(lo[e / 4][e % 4], hi[e / 4][e % 4],
                                  make_float2(c[e / 2][2 * (e % 2)], c[e / 2][2 * (e % 2) + 1]), y0, y1);
                        y[s][e] = low ? y0 : y1;
                    }
                } else {
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        float y0 = 0.f, y1 = 0.f;
                        if (d + e < hd()) {
                            const int d0 = d + e < half ? d + e : d + e - half;
                            rope_pair(qp[d0], qp[d0 + half], make_float2(cp[2 * d0], cp[2 * d0 + 1]), y0, y1);
                        }
                        y[s][e] = d + e < half ? y0 : y1;
                    }
                }
            }
        }
    }
    // output: lane (qi, qg) register r of block tt is dim 32 tt + 8 (r / 4) + 4 qg + r % 4
    __device__ __forceinline__ void finish(const floatx16 *acc, float m_run, float l_run, int unit) const {
        {
            float lo, hi;
            pair32(l_run, lo, hi);
            l_run = lo + hi;
        }
        const int sh = -unit;
        if (n_kseg > 1 || part != 0) {
            if (ws >= F) return;
            const size_t pe = part != 0 ? (((size_t)g * n_split + item) * 4 + wave) * 2 + (part - 1)
                                        : (((size_t)g * n_items + item) * 4 + wave) * n_kseg + seg;
            float *dst = part_o + (pe * 32 + qi) * HDP;
#pragma unroll
            for (int tt = 0; tt < NT; ++tt)
#pragma unroll
                for (int r = 0; r < 16; r += 4)
                    st4(dst + 32 * tt + 2 * r + 4 * qg, make_float4(ldexpf(acc[tt][r], sh), ldexpf(acc[tt][r + 1], sh),
                                                                    ldexpf(acc[tt][r + 2], sh), ldexpf(acc[tt][r + 3], sh)));
            if (qg == 0) {
                part_ml[(pe * 32 + qi) * 2 + 0] = m_run;
                part_ml[(pe * 32 + qi) * 2 + 1] = l_run;
            }
            return;
        }
        if (!qvalid) return;
        const float inv = 1.f / l_run;
        float *dst = out + qoff;
#pragma unroll
        for (int tt = 0; tt < NT; ++tt)
#pragma unroll
            for (int r = 0; r < 16; r += 4) {
                const int d = 32 * tt + 2 * r + 4 * qg;
                float x[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) x[e] = ldexpf(EXACT ? acc[tt][r + e] * inv : acc[tt][r + e] / l_run, sh);
                if (EXACT || d + 4 <= hd()) *(f4u *)(dst + d) = f4u{x[0], x[1], x[2], x[3]};
                else if (d + 2 <= hd()) *(f2u *)(dst + d) = f2u{x[0], x[1]};
            }
    }

    // The tiles in turn, one ahead: the first turn only writes the first tile.
    // check(bo, t): whether tile t can be computed here; false ends the loop (what
    // was loaded after the tile is dropped).  The same in every wave.
    template <class Write, class Check, class Compute>
    __device__ __forceinline__ bool run(Write write, Check check, Compute compute) {
        for (int t = t_begin - 1; t < t_end; ++t) {
            const int bo = NBUF == 1 ? 0 : ((t - t_begin) & 1) * kBuf;
            if (t >= t_begin) {
                if (!check(bo, t)) return false;
                compute(bo, t);
            }
            if (t + 1 < t_end) {
                if constexpr (NBUF == 1) __syncthreads();
                write(NBUF == 1 ? 0 : kBuf - bo);
                if (t + 2 < t_end) load_tile(t + 2);
            }
            __syncthreads();
        }
        return true;
    }
};

// The same work in fp32 (its MFMAs run at a sixteenth of the rate), for operands
// whose splits would lose bits and for infinities and NaN.  A function of its
// own: inlined, its registers cost the fast loop spills, each reload waiting for
// the tile in flight (28/4/128, 2048 rows: 448 us).
template <int HDP, bool EXACT>
__device__ __attribute__((noinline)) void prefill_fp32(uint64_t args, int work, uint32_t lds_at) {
    typedef const __attribute__((address_space(4))) PrefillArgs Args;
    typedef __attribute__((address_space(3))) unsigned char Lds;
    using Lane = PrefillLane<HDP, EXACT>;
    constexpr int KS = Lane::KS, NT = Lane::NT, C8 = Lane::C8, NUK = Lane::NUK, VD = Lane::VD, NUV = Lane::NUV;
    constexpr int kMeta = Lane::kMeta, kVOff32 = Lane::kVOff32;
    // arguments come in vector registers: back to scalar ones
    const uint64_t at = (uint64_t)__builtin_amdgcn_readfirstlane((uint32_t)(args >> 32)) << 32 |
                        (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)args);
    Args &a = *(Args *)at;
    unsigned char *lds = (unsigned char *)(Lds *)(uintptr_t)__builtin_amdgcn_readfirstlane(lds_at);
    Lane L(a, __builtin_amdgcn_readfirstlane(work));
    const int lane = L.lane, wave = L.wave, qi = L.qi, qg = L.qg, qpos = L.qpos;
    const float scale_log2 = a.scale_log2;
    L.load_tile(L.t_begin);
    float8v y[KS];
    L.load_q(y);
    floatx16 acc[NT];
#pragma unroll
    for (int tt = 0; tt < NT; ++tt) acc[tt] = floatx16{};
    float m_run = -INFINITY, l_run = 0.f;
    // Tiles: K as chunks of 4 dims [hd / 4][33 keys], V as groups
    // of 4 keys [8][hd], 16 bytes a unit, and which of +inf, -inf and NaN V has.
    auto write_tile32 = [&](int bo) {
        L.clear_pad();
        bool top = false, low = false, nan = false;
#pragma unroll
        for (int i = 0; i < NUK; ++i) {
            const int u = lane + 64 * i;
            unsigned char *dst = lds + bo + (2 * (u % C8) * 33 + 8 * wave + u / C8) * 16;
            if (HDP % 64 == 0 || u < HDP) {
                st4((float *)dst, make_float4(L.rk[i][0], L.rk[i][1], L.rk[i][2], L.rk[i][3]));
                st4((float *)(dst + 33 * 16), make_float4(L.rk[i][4], L.rk[i][5], L.rk[i][6], L.rk[i][7]));
            }
        }
#pragma unroll
        for (int i = 0; i < NUV; ++i) {
            const int u = lane + 64 * i;
#pragma unroll
            for (int d = 0; d < VD; ++d) {
                const float8v x = L.rv[i][d];
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    top |= x[e] == __builtin_inff();
                    low |= x[e] == -__builtin_inff();
                    nan |= x[e] != x[e];
                }
                unsigned char *dst = lds + bo + kVOff32 + ((4 * (wave >> 1) + (wave & 1)) * HDP + VD * u + d) * 16;
                if ((HDP / VD) % 64 == 0 || u < HDP / VD) {
                    st4((float *)dst, make_float4(x[0], x[1], x[2], x[3]));
                    st4((float *)(dst + 2 * HDP * 16), make_float4(x[4], x[5], x[6], x[7]));
                }
            }
        }
        const int odd = (__builtin_amdgcn_ballot_w64(top) != 0) | (__builtin_amdgcn_ballot_w64(low) != 0) << 1 |
                        (__builtin_amdgcn_ballot_w64(nan) != 0) << 2;
        if (lane == 0) ((int *)(lds + bo + kMeta))[8 + wave] = odd;
    };

    auto compute_tile32 = [&](int bo, int t) {
        const int k0 = t * kBK;
        if (k0 > L.my_kmax) return;
        const unsigned char *kp = lds + bo + (66 * qg + qi) * 16, *vp = lds + bo + kVOff32 + (qg * HDP + qi) * 16;
        const int4 ov = *(const int4 *)(lds + bo + kMeta + 32);
        const int odd = __builtin_amdgcn_readfirstlane(ov.x | ov.y | ov.z | ov.w);
        floatx16 s{};
        double sd[EXACT ? 1 : 16];
#pragma unroll
        for (int st = 0; st < KS; ++st) {           // 16 dims, then one rounding at the score's size (none in fp64)
            floatx16 x{};
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const float4 k4 = ld4((const float *)(kp + (4 * st + c) * 33 * 16));
#pragma unroll
                for (int e = 0; e < 4; ++e) x = mfma32f(comp(k4, e), y[st][4 * c + e], x);
            }
            if constexpr (EXACT) {
                s += x;
            } else {
#pragma unroll
                for (int r = 0; r < 16; ++r) sd[r] = st == 0 ? (double)x[r] : sd[r] + (double)x[r];
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        float mt = -INFINITY;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            if constexpr (!EXACT) s[r] = (float)sd[r];
            if (k0 + 8 * (r / 4) + 4 * qg + (r % 4) > qpos) {
                s[r] = -INFINITY;
                if constexpr (!EXACT) sd[r] = -INFINITY;
            }
            mt = fmaxf(mt, s[r] * scale_log2);
        }
        {
            float lo, hi;
            pair32(mt, lo, hi);
            mt = fmaxf(lo, hi);
        }
        const float m_new = fmaxf(m_run, mt), m_use = m_new == -INFINITY ? 0.f : m_new;
        const float alpha = fast_exp2(m_run - m_use);
        m_run = m_new;
        float p[16], ps = 0.f;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            if constexpr (EXACT) p[r] = fast_exp2(fmaf(s[r], scale_log2, -m_use));
            else p[r] = fast_exp2((float)fma(sd[r], (double)scale_log2, (double)-m_use));
            ps += p[r];
        }
        l_run = fmaf(l_run, alpha, ps);
#pragma unroll
        for (int tt = 0; tt < NT; ++tt) {
            floatx16 d{};
            auto v_at = [&](int j) { return ld4((const float *)(vp + (2 * j * HDP + 32 * tt) * 16)); };
#pragma unroll
            for (int j = 0; j < 4; ++j) {            // keys 8 j + 4 qg + e
                const float4 v4 = v_at(j);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float v = comp(v4, e);
                    d = mfma32f(__builtin_fabsf(v) < __builtin_inff() ? v : 0.f, p[4 * j + e], d);
                }
            }
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[tt][r] = fmaf(acc[tt][r], alpha, d[r]);
            if (odd) {
                // how many +inf, -inf and NaN every (query, dim) gets from keys it
                // attends (a weight of 0 for a masked key must not make NaN of them)
                auto count = [&](auto is, float add) {
                    floatx16 n{};
#pragma unroll
                    for (int ks = 0; ks < 2; ++ks) {
                        half8 c, on;                 // keys 16 ks + 8 (e / 4) + 4 qg + e % 4
#pragma unroll
                        for (int e = 0; e < 8; ++e) {
                            const int j = 2 * ks + e / 4;
                            c[e] = is(comp(v_at(j), e % 4)) ? (_Float16)1.f : (_Float16)0.f;
                            on[e] = k0 + 8 * j + 4 * qg + e % 4 <= qpos ? (_Float16)1.f : (_Float16)0.f;
                        }
                        n = mfma32h(c, on, n);
                    }
#pragma unroll
                    for (int r = 0; r < 16; ++r) acc[tt][r] += n[r] > 0.f ? add : 0.f;
                };
                if (odd & 1) count([](float x) { return x == __builtin_inff(); }, __builtin_inff());
                if (odd & 2) count([](float x) { return x == -__builtin_inff(); }, -__builtin_inff());
                if (odd & 4) count([](float x) { return x != x; }, __builtin_nanf(""));
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    L.run(write_tile32, [](int, int) { return true; }, compute_tile32);
    L.finish(acc, m_run, l_run, 0);
}

// Workgroup = 4 waves of one kv-head g.  The query rows of a kv-head, n_tok
// positions times n_rep heads, are one list f = z n_rep + i (position major),
// cut into strips of 32 (a wave) and items of 4 strips (a workgroup): whatever
// n_rep is, a strip's rows lie within 32 / n_rep + 1 positions, so the waves of
// a workgroup want the same keys and little is computed for the causal mask to
// drop.  Per tile of 32 keys a wave computes S^T = K Q^T (keys x queries, 3 hd
// / 16 MFMAs), so every lane owns the scores of one query; the softmax weights
// of its 16 keys, split in registers, are the B operand of O^T += V^T P^T (6 hd
// / 32 MFMAs) without leaving the lane: the k order of the second product is
// the order in which the first leaves its keys, and V^T is laid out in LDS to
// match.
//
// Tiles: each wave loads a quarter of the next tile (8 keys of K, 8 of V) into
// registers while the current tile is computed, then scales, splits and writes
// it to the other LDS buffer, one barrier per tile.  K is kept as chunks of 8
// dims [hd / 8][33 keys] and V as groups of 8 keys [4][hd], both 16 bytes a
// unit: an MFMA operand is one 16-byte read, 32 lanes wide and consecutive
// (no bank conflicts), and the 33rd key spreads the writes of a row's chunks
// over the banks.  The splits are made once per workgroup, i.e. per 128 query
// rows; making them in every wave would cost more VALU time than the MFMAs.
//
// The softmax runs in base 2.  EXACT keeps an integer reference maximum per
// query (any reference gives the same normalised result) that moves only when
// the true maximum exceeds it by more than 4, so the rescale of the accumulators
// is rare and exact; otherwise the reference is the maximum itself, whose weight
// is then 1 and whose argument, near 0 for the keys that count, rounds least.
// The exponent's argument fma(score, scale, -reference) has one rounding.
//
// HDP: head_dim rounded up to a multiple of 32.  EXACT (head_dim == HDP, 64 or
// 128): two fp16 parts per operand, 23 of 24 bits; otherwise three, the whole
// fp32 value, scores summed in fp64 and each tile's output summed apart.
template <int HDP, bool EXACT>
__global__ __launch_bounds__(kThreads, per_cu(HDP, EXACT)) void prefill_kernel(PrefillArgs a) {
    using Lane = PrefillLane<HDP, EXACT>;
    constexpr int KS = Lane::KS, NT = Lane::NT, C8 = Lane::C8, NUK = Lane::NUK, VD = Lane::VD, NUV = Lane::NUV;
    constexpr int PARTS = Lane::PARTS, kKB = Lane::kKB, kVB = Lane::kVB, kVOff = Lane::kVOff, kMeta = Lane::kMeta;
    __shared__ __align__(16) unsigned char lds[Lane::NBUF * Lane::kBuf];
    __shared__ int leave;                           // the last tile was one for the fp32 loop
    // work index: items run from the longest (last rows) down; the second part
    // of the grid takes them from the short end, so that the two workgroups of
    // a CU (b and b + fold) add up to about the same work
    const int bx = blockIdx.x;
    const int wi = bx < a.fold ? bx : (int)gridDim.x - 1 - (bx - a.fold);
    Lane L(a, wi);
    const int lane = L.lane, wave = L.wave, qi = L.qi, qg = L.qg, qpos = L.qpos;
    if (threadIdx.x == 0) leave = 0;
    bool off = false;                               // this wave's last tile was one for the fp32 loop

    // scales, splits and writes the loaded share to a buffer, with 2^-scale of
    // the K group, the scale exponent of the V group and whether this share
    // (or the last tile's result) is one for the fp32 loop
    auto write_tile = [&](int bo) {
        const int lane = L.fresh_lane();
        L.clear_pad();
        float mk = 0.f, mv = 0.f, md[NUV][VD];
#pragma unroll
        for (int i = 0; i < NUK; ++i)
#pragma unroll
            for (int e = 0; e < 8; ++e) mk = nmax(mk, __builtin_fabsf(L.rk[i][e]));
#pragma unroll
        for (int i = 0; i < NUV; ++i)
#pragma unroll
            for (int d = 0; d < VD; ++d) {
                md[i][d] = 0.f;
#pragma unroll
                for (int e = 0; e < 8; ++e) md[i][d] = nmax(md[i][d], __builtin_fabsf(L.rv[i][d][e]));
                mv = nmax(mv, md[i][d]);
            }
        mk = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, wave_nmax(mk))));
        mv = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, wave_nmax(mv))));
        constexpr float kInf = __builtin_inff();
        const int ek = scale_exp(mk), ev = mv > 0.f ? scale_exp(mv) : kZeroExp;
        const float sk = pow2(ek), sv = pow2(ev);
        // V's group: every key's largest value has to be within 2^-10 of the group's
        // (a row may attend that key alone, or give it nearly all the weight), every
        // dim's within 2^-12 (or zero, which is exact).  That one dim is large in every
        // key shows the first for ordinary data.
        const float thr_d = mv * 0x1p-12f, thr_k = mv * 0x1p-10f;
        float every = __builtin_inff(), dims = __builtin_inff();   // one dim's least over the keys; the dims' least
#pragma unroll
        for (int j = 0; j < 8; ++j) every = fminf(every, __builtin_fabsf(L.rv[0][0][j]));
#pragma unroll
        for (int i = 0; i < NUV; ++i)
#pragma unroll
            for (int d = 0; d < VD; ++d) dims = fminf(dims, EXACT || md[i][d] > 0.f ? md[i][d] : mv);
        bool far = (__builtin_amdgcn_ballot_w64(dims < thr_d) != 0) | (__builtin_amdgcn_ballot_w64(every >= thr_k) == 0);
#pragma unroll
        for (int i = 0; i < NUK; ++i) {
            const int u = lane + 64 * i;
            half8 h[PARTS];
            split8<PARTS>(L.rk[i], sk, h);
            if (HDP % 64 == 0 || u < HDP)
#pragma unroll
                for (int q = 0; q < PARTS; ++q)
                    *(half8 *)(lds + bo + q * kKB + ((u % C8) * 33 + 8 * wave + u / C8) * 16) = h[q];
        }
#pragma unroll
        for (int i = 0; i < NUV; ++i) {
            const int u = lane + 64 * i;
#pragma unroll
            for (int d = 0; d < VD; ++d) {
                half8 h[PARTS];
                split8<PARTS>(L.rv[i][d], sv, h);
                if ((HDP / VD) % 64 == 0 || u < HDP / VD)
#pragma unroll
                    for (int q = 0; q < PARTS; ++q)
                        *(half8 *)(lds + bo + kVOff + q * kVB + (wave * HDP + VD * u + d) * 16) = h[q];
            }
        }
        if (far) {                                       // every dim, zeros apart, and every key
            bool low = false;
#pragma unroll
            for (int i = 0; i < NUV; ++i)
#pragma unroll
                for (int d = 0; d < VD; ++d) low |= md[i][d] < thr_d && md[i][d] > 0.f;
            far = __builtin_amdgcn_ballot_w64(low) != 0;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                float x = 0.f;
#pragma unroll
                for (int i = 0; i < NUV; ++i)
#pragma unroll
                    for (int d = 0; d < VD; ++d) x = fmaxf(x, __builtin_fabsf(L.rv[i][d][j]));
                far |= __builtin_amdgcn_ballot_w64(x >= thr_k) == 0;
            }
        }
        const int bad = off | far | !(mk < kInf) | !(mv < kInf) | (ev == 126);   // 126: too small for its scale
        if (lane == 0) {
            float *s = (float *)(lds + bo + kMeta);
            s[wave] = pow2(-ek);
            ((int *)s)[4 + wave] = ev;
            ((int *)s)[8 + wave] = bad;
        }
    };
    if (L.t_begin < L.t_end) L.load_tile(L.t_begin);

    // Q^T operand of the fast loop, scaled to the row's own power of two; cq brings
    // a score to the log2 domain
    half8 qp8[KS][PARTS];
    float cq;
    {
        float8v y[KS];
        L.load_q(y);
        float mq = 0.f;
#pragma unroll
        for (int s = 0; s < KS; ++s)
#pragma unroll
            for (int e = 0; e < 8; ++e) mq = fmaxf(mq, __builtin_fabsf(y[s][e]));
        float ma, mb;
        pair32(mq, ma, mb);
        const int eq = scale_exp(fmaxf(ma, mb));   // a non-finite row's scores are NaN whatever the scale
        const float sq = pow2(eq);
#pragma unroll
        for (int s = 0; s < KS; ++s) split8<PARTS>(y[s], sq, qp8[s]);
        cq = ldexpf(a.scale_log2, -eq);
    }

    floatx16 acc[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[t] = floatx16{};
    float m_run = EXACT ? 0.f : -INFINITY, l_run = 0.f;   // softmax reference; this lane's half of the sum
    int unit = kNone;                              // acc holds the output times 2^unit (kNone: no key yet)
    float base = -INFINITY, t_min = kTMin;         // EXACT: m_run - unit; kTMin while acc is below kEnough, else -inf
    bool settled = false;                          // not EXACT: every query's acc is above kEnough
    int a_min = kZeroExp, a_max = -kZeroExp;       // V's scales so far
    bool begun = false;                            // acc is no longer zero

    auto compute_tile = [&](int bo, int t) {
        const int k0 = t * kBK;
        if (k0 > L.my_kmax) return;
        int ko = bo + (33 * qg + qi) * 16;
        const unsigned char *vp = lds + bo + kVOff + (qg * HDP + qi) * 16;
        const float *sp = (const float *)(lds + bo + kMeta);
        const float4 ck = ld4(sp);
        const int4 av = *(const int4 *)(sp + 4);
        auto k_at = [&](int st, int part) { return *(const half8 *)(lds + ko + 2 * st * 33 * 16 + part * kKB); };
        floatx16 s{};
        double sd[EXACT ? 1 : 16];
        if constexpr (EXACT) {
            // the cross terms first: they are small, and the sum then takes one
            // rounding at its own size per 16 dims
#pragma unroll
            for (int st = 0; st < KS; ++st) {
                s = mfma32h(k_at(st, 0), qp8[st][1], s);
                s = mfma32h(k_at(st, 1), qp8[st][0], s);
            }
            asm volatile("" : "+v"(ko));   // K's hi parts are read again: kept, they would take 2 KS registers too many
#pragma unroll
            for (int st = 0; st < KS; ++st) s = mfma32h(k_at(st, 0), qp8[st][0], s);
            // operands are read a few MFMAs ahead, no further (registers)
            __builtin_amdgcn_sched_group_barrier(kDsRead, 6, 0);
#pragma unroll
            for (int i = 0; i < 3 * KS - 6; ++i) {
                __builtin_amdgcn_sched_group_barrier(kMfma, 1, 0);
                __builtin_amdgcn_sched_group_barrier(kDsRead, 1, 0);
            }
            __builtin_amdgcn_sched_group_barrier(kMfma, 6, 0);
        } else {
            // 16 dims at a time on the MFMA, to 2^-24 of the operands, their sums in fp64
#pragma unroll
            for (int st = 0; st < KS; ++st) {
                const half8 kh = k_at(st, 0), kl = k_at(st, 1), kr = k_at(st, 2);
                floatx16 x{};
                x = mfma32h(kr, qp8[st][0], x);
                x = mfma32h(kh, qp8[st][2], x);
                x = mfma32h(kl, qp8[st][1], x);
                x = mfma32h(kl, qp8[st][0], x);
                x = mfma32h(kh, qp8[st][1], x);
                x = mfma32h(kh, qp8[st][0], x);
#pragma unroll
                for (int r = 0; r < 16; ++r) sd[r] = st == 0 ? (double)x[r] : sd[r] + (double)x[r];
            }
#pragma unroll
            for (int r = 0; r < 16; ++r) s[r] = (float)sd[r];
        }
        // the factors to the log2 domain (never 0, which an operand of zeros or of tiny values would make it: a
        // masked score of -inf times 0 is NaN)
        constexpr float kTiny = 0x1p-126f;
        const float cj[4] = {fmaxf(cq * ck.x, kTiny), fmaxf(cq * ck.y, kTiny), fmaxf(cq * ck.z, kTiny),
                             fmaxf(cq * ck.w, kTiny)};
        // s[r]: query qi, key k0 + 8 (r / 4) + 4 qg + r % 4; the causal mask only
        // matters on tiles that reach past the strip's first row
        const bool diag = k0 + kBK - 1 > L.my_kmin;
        float mt = -INFINITY;
        if (diag) {
#pragma unroll
            for (int r = 0; r < 16; ++r)
                if (k0 + 8 * (r / 4) + 4 * qg + (r % 4) > qpos) {
                    s[r] = -INFINITY;
                    if constexpr (!EXACT) sd[r] = -INFINITY;
                }
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
            mt = fmaxf(mt, fmaxf(fmaxf(s[4 * j], s[4 * j + 1]), fmaxf(s[4 * j + 2], s[4 * j + 3])) * cj[j]);
        {
            float lo, hi;
            pair32(mt, lo, hi);
            mt = fmaxf(lo, hi);
        }
        // A key's weight takes V's scale off: it is brought to 2^(unit - scale).  z is
        // log2 of the tile's largest so scaled; where that leaves its range (or, not
        // EXACT, the maximum rises) the query's reference or unit moves, and acc with
        // it.  unit's moves are powers of two, so acc loses nothing by them.
        const int av0 = __builtin_amdgcn_readfirstlane(av.x), av1 = __builtin_amdgcn_readfirstlane(av.y);
        const int av2 = __builtin_amdgcn_readfirstlane(av.z), av3 = __builtin_amdgcn_readfirstlane(av.w);
        const int a_t = min(min(av0, av1), min(av2, av3)), a_hi = max(max(av0, av1), max(av2, av3));
        if (a_t != kZeroExp) {
            a_min = min(a_min, a_t);
            a_max = max(a_max, a_t);
        }
        off = a_hi - a_t > kSpread || a_max - a_min > kRange;
        float8v p0, p1;
        auto weights = [&](float m) {                // the keys' weights; returns their sum
            float ps = 0.f;
#pragma unroll
            for (int r = 0; r < 8; ++r) {
                if constexpr (EXACT) {
                    p0[r] = fast_exp2(fmaf(s[r], cj[r / 4], -m));
                    p1[r] = fast_exp2(fmaf(s[8 + r], cj[2 + r / 4], -m));
                } else {
                    p0[r] = fast_exp2((float)fma(sd[r], (double)cj[r / 4], (double)-m));
                    p1[r] = fast_exp2((float)fma(sd[8 + r], (double)cj[2 + r / 4], (double)-m));
                }
                ps += p0[r] + p1[r];
            }
            return ps;
        };
        float alpha = 1.f;
        if constexpr (!EXACT) {                      // the maximum is the reference
            const float m_new = fmaxf(m_run, mt), m_use = m_new == -INFINITY ? 0.f : m_new;
            alpha = fast_exp2(m_run - m_use);
            m_run = m_new;
            const float ps = weights(m_use);
            l_run = fmaf(l_run, alpha, ps);
        }
        const float z = EXACT ? mt - base - (float)a_t : mt - m_run + (float)(unit - a_t);
        bool move = z > kTMax;
        if constexpr (EXACT) move |= z < t_min;
        else move |= (alpha != 1.f) | (!settled && z < kTMin);
        // Small elements of q and K are off by 2^-25, scaled, beside partners of up to
        // 2^14: a score by some 2^-7 times its factor.  That has to be below 2^-21 (3e-7
        // of a weight), or below what fp32 leaves of a score as large as the tile's
        // largest (a channel that is large in q and in K).
        const float cm = fmaxf(fmaxf(cj[0], cj[1]), fmaxf(cj[2], cj[3]));
        if (__builtin_amdgcn_ballot_w64(move | (cm > 0x1p-14f))) {
            off |= __builtin_amdgcn_ballot_w64(cm > 0x1p-15f * __builtin_fabsf(mt) && cm > 0x1p-14f) != 0;
            move &= mt != -INFINITY;
            if (__builtin_amdgcn_ballot_w64(move)) {
                float am = 0.f;
                if (begun) {
                    float lo, hi;
#pragma unroll
                    for (int tt = 0; tt < NT; ++tt)
#pragma unroll
                        for (int r = 0; r < 16; ++r) am = fmaxf(am, __builtin_fabsf(acc[tt][r]));
                    pair32(am, lo, hi);
                    am = fmaxf(lo, hi);
                }
                const bool first = EXACT ? base == -INFINITY : unit == kNone;
                if constexpr (EXACT) {
                    const float m_new = move && (first || mt > m_run) ? ceilf(mt) : m_run;
                    alpha = first ? 0.f : fast_exp2(m_run - m_new);        // a power of two
                    m_run = m_new;
                    l_run *= alpha;
                }
                am *= alpha;
                const float at = mt - m_run + (float)(unit - a_t);
                const bool turn = move && a_t != kZeroExp && (first || at > kTMax || (at < kTMin && am < kEnough));
                const int step = turn ? kTNew - (int)ceilf(fmaxf(mt - m_run, -60.f)) + a_t - unit : 0;
                unit += step;
                am = ldexpf(am, step);
                alpha = ldexpf(alpha, step);
                if constexpr (EXACT) {
                    t_min = am < kEnough ? kTMin : -INFINITY;
                    if (move) base = m_run - (float)unit;
                } else {
                    settled = __builtin_amdgcn_ballot_w64(am < kEnough) == 0;
                }
                if (begun)
#pragma unroll
                    for (int tt = 0; tt < NT; ++tt)
#pragma unroll
                        for (int r = 0; r < 16; ++r) acc[tt][r] *= alpha;
            }
        }
        begun = true;
        if constexpr (EXACT) {
            const float ps = weights(m_run);
            l_run += ps;
        }
        half8 pp[2][PARTS];
        split8<PARTS>(p0, pow2(unit - (qg ? av1 : av0)), pp[0]);
        split8<PARTS>(p1, pow2(unit - (qg ? av3 : av2)), pp[1]);
        // k-step ks of block tt, the small terms and the hi hi one
        auto v_at = [&](int tt, int ks, int part) {
            return *(const half8 *)(vp + (2 * ks * HDP + 32 * tt) * 16 + part * kVB);
        };
        auto pv_lo = [&](floatx16 d, int tt, int ks) {
            const half8 vh = v_at(tt, ks, 0), vl = v_at(tt, ks, 1);
            if constexpr (PARTS == 3) {
                d = mfma32h(v_at(tt, ks, 2), pp[ks][0], d);
                d = mfma32h(vh, pp[ks][2], d);
                d = mfma32h(vl, pp[ks][1], d);
            }
            d = mfma32h(vl, pp[ks][0], d);
            return mfma32h(vh, pp[ks][1], d);
        };
        auto pv_hi = [&](floatx16 d, int tt, int ks) { return mfma32h(v_at(tt, ks, 0), pp[ks][0], d); };
#pragma unroll
        for (int tt = 0; tt < NT; ++tt) {
            if constexpr (EXACT) {
                acc[tt] = pv_hi(pv_lo(acc[tt], tt, 0), tt, 0);
                acc[tt] = pv_hi(pv_lo(acc[tt], tt, 1), tt, 1);
            } else {   // the tile's sum, then one rounding at the size of acc
                acc[tt] += pv_hi(pv_hi(pv_lo(pv_lo(floatx16{}, tt, 0), tt, 1), tt, 0), tt, 1);
            }
            if constexpr (!EXACT) __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (EXACT) {
            __builtin_amdgcn_sched_group_barrier(kDsRead, 4, 1);
#pragma unroll
            for (int i = 0; i < 2 * NT - 2; ++i) {
                __builtin_amdgcn_sched_group_barrier(kMfma, 3, 1);
                __builtin_amdgcn_sched_group_barrier(kDsRead, 2, 1);
            }
            __builtin_amdgcn_sched_group_barrier(kMfma, 6, 1);
        }
        if (off && t + 1 == L.t_end && lane == 0) leave = 1;
    };

    auto check = [&](int bo, int t) {               // flags written before the last barrier
        const int4 bv = *(const int4 *)(lds + bo + kMeta + 32);
        return !__builtin_amdgcn_readfirstlane(bv.x | bv.y | bv.z | bv.w);
    };
    if (L.t_begin < L.t_end && (!L.run(write_tile, check, compute_tile) ||
                                __builtin_amdgcn_readfirstlane(leave))) {
        __syncthreads();                            // every wave has left the fast loop's buffers
        prefill_fp32<HDP, EXACT>((uint64_t)__builtin_amdgcn_kernarg_segment_ptr(), wi,
                                 (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)lds);
        return;
    }
    // no key at all: the segment or half is left out of the merge
    L.finish(acc, EXACT && base == -INFINITY && l_run == 0.f ? -INFINITY : m_run, l_run, unit);
}

// Block = 32 query rows of one strip of a kv-head: the log-sum-exp merge of the
// key segments (or of the two halves of a split item); thread (row tid / 8, c =
// tid % 8) owns the float4s c, c + 8, ... of its row.  Segments in batches of
// four, every load of a batch issued before its arithmetic (one memory round
// trip per batch).
template <int HDP, bool EXACT>
__global__ __launch_bounds__(256) void prefill_combine_kernel(PrefillArgs a) {
    constexpr int N4 = HDP / 32;                        // float4 per thread
    const int hd = EXACT ? HDP : a.hd, F = a.n_tok * a.n_rep;
    int g, item;
    const int id = blockIdx.x, gi = id >> 2, wave = id & 3;
    const int S = a.n_split > 0 ? 2 : a.n_kseg;
    const int per = a.n_split > 0 ? a.n_split : a.n_items;
    g = gi / per;
    item = gi - g * per;
    const size_t base = (size_t)id * S;
    const int r = threadIdx.x >> 3, c = threadIdx.x & 7;
    const int f = kPrefillRows * (a.n_items - 1 - item) + 32 * wave + r;
    if (f >= F) return;
    constexpr int kSeg = 4;
    const float2 *ml = reinterpret_cast<const float2 *>(a.part_ml);
    float m = -INFINITY;
    for (int s0 = 0; s0 < S; s0 += 2 * kSeg) {
        float mv[2 * kSeg];
#pragma unroll
        for (int u = 0; u < 2 * kSeg; ++u) mv[u] = s0 + u < S ? ml[(base + s0 + u) * 32 + r].x : -INFINITY;
#pragma unroll
        for (int u = 0; u < 2 * kSeg; ++u) m = fmaxf(m, mv[u]);
    }
    float den = 0.f;
    float4 acc[N4];
#pragma unroll
    for (int j = 0; j < N4; ++j) acc[j] = zero4();
    for (int s0 = 0; s0 < S; s0 += kSeg) {
        float2 st[kSeg];
        float4 x[kSeg][N4];
#pragma unroll
        for (int u = 0; u < kSeg; ++u)
            if (s0 + u < S) {
                st[u] = ml[(base + s0 + u) * 32 + r];
                const float *po = a.part_o + ((base + s0 + u) * 32 + r) * HDP + 4 * c;
#pragma unroll
                for (int j = 0; j < N4; ++j) x[u][j] = ld4(po + 32 * j);
            }
#pragma unroll
        for (int u = 0; u < kSeg; ++u)
            if (s0 + u < S && st[u].x != -INFINITY) {       // a segment may hold masked keys only
                const float w = exp2f(st[u].x - m);
                den = fmaf(w, st[u].y, den);
#pragma unroll
                for (int j = 0; j < N4; ++j) {
                    acc[j].x = fmaf(w, x[u][j].x, acc[j].x);
                    acc[j].y = fmaf(w, x[u][j].y, acc[j].y);
                    acc[j].z = fmaf(w, x[u][j].z, acc[j].z);
                    acc[j].w = fmaf(w, x[u][j].w, acc[j].w);
                }
            }
    }
    const float inv = 1.f / den;
    const int z = f / a.n_rep;
    float *op = a.out + ((size_t)z * a.n_head_kv * a.n_rep + (size_t)g * a.n_rep + (f - z * a.n_rep)) * hd;
#pragma unroll
    for (int j = 0; j < N4; ++j) {
        const int d = 32 * j + 4 * c;
        const float x[4] = {acc[j].x, acc[j].y, acc[j].z, acc[j].w};
        float y[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) y[e] = EXACT ? x[e] * inv : x[e] / den;
        if (EXACT || d + 4 <= hd) *(f4u *)(op + d) = f4u{y[0], y[1], y[2], y[3]};
        else if (d + 2 <= hd) *(f2u *)(op + d) = f2u{y[0], y[1]};
    }
}

// ---------------------------------------------------------------- dispatch

// head_dim 64 and 128 take the two-part kernel; with a single key tile, where
// the last bit of V is most of the error, the three-part one (4 keys: 0.9e-7
// fp32 before, 1.0e-7 two parts)
bool exact(const PrefillArgs &a) { return (a.hd == 64 || a.hd == 128) && a.pos0 + a.n_tok > kBK; }

template <int HDP, bool EXACT>
hipError_t launch_t(const PrefillArgs &a, hipStream_t s) {
    const dim3 grid(a.n_split > 0 ? a.n_units * a.n_head_kv : a.n_items * a.n_head_kv * a.n_kseg);
    hipLaunchKernelGGL((prefill_kernel<HDP, EXACT>), grid, dim3(kThreads), 0, s, a);
    if (a.n_split > 0 || a.n_kseg > 1) {
        const dim3 cgrid(a.n_head_kv * (a.n_split > 0 ? a.n_split : a.n_items) * 4);
        hipLaunchKernelGGL((prefill_combine_kernel<HDP, EXACT>), cgrid, dim3(256), 0, s, a);
    }
    return hipGetLastError();
}

}  // namespace

int prefill_padded_dim(int head_dim) { return (head_dim + 31) / 32 * 32; }

size_t prefill_part_floats(int head_dim, int num_cu) {
    return (size_t)2 * num_cu * kPrefillRows * (prefill_padded_dim(head_dim) + 2);
}

void prefill_plan(PrefillArgs &a, int num_cu) {
    a.n_items = (a.n_tok * a.n_rep + kPrefillRows - 1) / kPrefillRows;
    a.n_split = 0;
    a.n_units = 0;
    a.n_kseg = 1;
    a.fold = num_cu;
    const int cu = per_cu(prefill_padded_dim(a.hd), exact(a)), n_wg = a.n_items * a.n_head_kv, F = a.n_tok * a.n_rep;
    auto tiles = [&](int i) {   // key tiles of item i (its last row)
        const int f0 = kPrefillRows * (a.n_items - 1 - i);
        return (a.pos0 + std::min(f0 + kPrefillRows - 1, F - 1) / a.n_rep) / kBK + 1;
    };
    // Split the key range when the workgroups of a chunk do not fill every
    // CU: as many segments as keep all of them in one wave, each of at least
    // 2 key tiles.  A 64-row chunk has 16 workgroups (7B): unsplit, each walks
    // all its key tiles alone.
    if (n_wg < num_cu) a.n_kseg = std::max(1, std::min(cu * num_cu / n_wg, tiles(0) / 2));
    a.seg_tiles = (tiles(0) + a.n_kseg - 1) / a.n_kseg;
    // Two workgroups fit per CU and the grid is folded so that each CU's pair
    // adds up to about the mean work; with between one and two workgroups per
    // CU some CUs hold one item only, while the pairs' sums run up to about
    // the longest item plus the shortest.  Splitting the longest items into
    // two halves of their key tiles fills the grid to two per CU and lets the
    // pairs (r-th longest unit with the r-th shortest) even out.
    if (a.n_kseg != 1 || n_wg < num_cu || n_wg >= cu * num_cu) return;
    int split = std::min(a.n_items, (cu * num_cu - n_wg) / a.n_head_kv);
    while (split > 0 && tiles(split - 1) < 4) --split;   // halves of at least two tiles
    if (split == 0 || a.n_items + split > kMaxPrefillUnits) return;
    struct Unit { int tiles, code; };
    std::vector<Unit> u;
    u.reserve(a.n_items + split);
    for (int i = 0; i < a.n_items; ++i) {
        const int t = tiles(i);
        if (i < split) {
            u.push_back({t / 2, i << 2 | 1});
            u.push_back({t - t / 2, i << 2 | 2});
        } else {
            u.push_back({t, i << 2});
        }
    }
    std::stable_sort(u.begin(), u.end(), [](const Unit &x, const Unit &y) { return x.tiles > y.tiles; });
    for (size_t r = 0; r < u.size(); ++r) a.unit[r] = (uint16_t)u[r].code;
    a.n_split = split;
    a.n_units = (int)u.size();
}

hipError_t launch_prefill(const PrefillArgs &a, hipStream_t s) {
    switch (prefill_padded_dim(a.hd)) {
        case 32: return launch_t<32, false>(a, s);
        case 64: return exact(a) ? launch_t<64, true>(a, s) : launch_t<64, false>(a, s);
        case 96: return launch_t<96, false>(a, s);
        case 128: return exact(a) ? launch_t<128, true>(a, s) : launch_t<128, false>(a, s);
        case 160: return launch_t<160, false>(a, s);
        case 192: return launch_t<192, false>(a, s);
        case 224: return launch_t<224, false>(a, s);
        case 256: return launch_t<256, false>(a, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace kore_attn_gpu

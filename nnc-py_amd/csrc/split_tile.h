// fp32 products on the 16-bit matrix units of gfx950, shared by implicit-GEMM
// convolution and GEMM/MatMul.
//
// v_mfma_f32_32x32x2_f32 runs at 157 TFLOP/s, the bf16 instructions at 16
// times that, with fp32 accumulators. An fp32 operand is therefore cut into
// three bf16 pieces of 8 bits each, which hold all 24 of its bits (a known
// way to have fp32 products from 16-bit units; SplitB16):
//
//   x 2^24 = h + m + l   h = bf16(x 2^24), m = bf16(rest), l = the rest
//
// with |m| <= 2^-8 |h| and |l| <= 2^-17 |h| up to a rounding. Six products
// (h h, h m, m h, m m, l h, h l), each exact in fp32, add up to the product
// of the operands but for m l + l m + l l, at most 2^-24 of it: what the fp32
// instruction rounds off a product. The factor 2^24 on either operand, taken
// out of the sum at the end, keeps the smallest fp32 values' pieces among
// normal numbers, so the pieces are the operand at any size: whatever scales
// meet inside a row, each term has fp32's precision by itself, and products
// with one nonzero term (selections, whole numbers of 16 bits or less) are
// exact.
//
// What the factor takes away is at the other end: |x| from 2^104, sums from
// 2^80, infinities and NaN. Each of them makes a sum of the tile infinite or
// NaN, so a workgroup looks at its segment's finished sums (no test of the
// operands in the loop) and, if one is not finite, computes that segment
// again with the fp32 instruction out of the same LDS image (WholeF32), and
// its later segments straight away. Such tiles take about the time that the
// fp32 instruction needs, plus the segment thrown away; outputs beside the
// large value in a tile then have the fp32 instruction's rounding.
//
// The h h products go to one accumulator and the smaller ones to a second,
// added once at the end: the large sum takes one rounding per 16 k (the
// instruction adds a step's products before it rounds) instead of one per 2,
// and the small ones cost it none. Tiles with registers to spare (at most two
// blocks per wave) also move it to a second level every four slices.
//
// The operands are cut once per workgroup, between global memory and LDS:
// fp32 to registers two 16-k steps ahead, pieces to LDS one step ahead of
// the MFMAs, the cutting's VALU work interleaved with the MFMAs
// (split_order). Cutting them after the LDS read instead repeats it for each
// wave that shares a row: 249 against 341 TFLOP/s in an issue-rate probe (two
// waves per SIMD).
#pragma once

#include <type_traits>

#include "mfma_tile.h"

namespace nnc {

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32v2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32v4 __attribute__((ext_vector_type(4)));

struct SplitB16 {
    static constexpr int PLANES = 3, PRODUCTS = 6;
    static constexpr int OPS = 13;  // VALU operations per pair
    static constexpr bool CHECKED = true;
    typedef bf16x8 Frag;
    static __device__ __forceinline__ uint32_t pack(float a, float b) {
        return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, bf16x2));
    }
    static __device__ __forceinline__ void cut(float x0, float x1, uint32_t (&p)[PLANES]) {
        const float s0 = x0 * 0x1p24f, s1 = x1 * 0x1p24f;
        p[0] = pack(s0, s1);
        const float r0 = s0 - __uint_as_float(p[0] << 16), r1 = s1 - __uint_as_float(p[0] & 0xffff0000u);
        p[1] = pack(r0, r1);
        p[2] = pack(r0 - __uint_as_float(p[1] << 16), r1 - __uint_as_float(p[1] & 0xffff0000u));
    }
    static __device__ __forceinline__ floatx16 mma(Frag a, Frag b, floatx16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
    }
    // the sum, and whether the pieces hold it
    static __device__ __forceinline__ float sum(float hi, float lo, bool& ok) {
        const float s = hi + lo;
        ok &= __builtin_fabsf(s) < __builtin_inff();
        return s * 0x1p-48f;
    }
};

// The operands whole, for the fp32 instruction: plane p of a 16-k step's half
// holds k 4p .. 4p + 3 of its eight.
struct WholeF32 {
    static constexpr int PLANES = 2, PRODUCTS = 8;
    static constexpr bool CHECKED = false;
    typedef f32x4 Frag;
    static __device__ __forceinline__ float sum(float hi, float, bool&) { return hi; }
};

// LDS image of one operand's 16-k step: plane p, k-half q (8 k each), row x
// at p * PLANE + q * HALF + 16 x bytes: an MFMA lane's 8 k are one 16-byte
// read, 32 lanes read 512 contiguous bytes. Halves are 64 bytes off a
// multiple of 128 so that a store's eight lanes on four rows and both halves
// hit all 32 banks.
template <class Md, int X>
struct SplitOperand {
    static constexpr int HALF = X * 16 + 64, PLANE = 2 * HALF, BYTES = Md::PLANES * PLANE;
};

template <class Md, class T>
struct SplitStage {
    typedef SplitOperand<Md, T::BM> A;
    typedef SplitOperand<Md, T::BN> B;
    static constexpr int STAGE = A::BYTES + B::BYTES;  // bytes; two stages
};

template <class T>
constexpr int split_lds_bytes() {
    return 2 * SplitStage<SplitB16, T>::STAGE;
}

// One operand's staging registers: per thread and 16-k step, RUN consecutive
// k of each of NG rows (x, x + X / NG, ...); two steps (sets Q) in flight.
// The thread stages the same rows throughout a tile.
template <class T, int X, int RUN_>
struct SplitStaged {
    static constexpr int PER = X * 16 / T::THREADS, RUN = RUN_, NG = PER / RUN;
    static_assert(NG >= 1 && NG * RUN == PER && (RUN == 4 || RUN == 8 || RUN == 16), "k per thread");
    int x, koff;
    float v[2][PER];

    // cuts set Q and stores it to the operand's image at S
    template <class Md, int Q>
    __device__ __forceinline__ void store(char* S) {
        typedef SplitOperand<Md, X> O;
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            const float* u = v[Q] + g * RUN;
            if constexpr (std::is_same<Md, WholeF32>::value) {
#pragma unroll
                for (int i = 0; i < RUN; i += 4) {
                    const int k = koff + i;
                    *reinterpret_cast<f32x4*>(S + ((k >> 2) & 1) * O::PLANE + (k >> 3) * O::HALF + (x + g * (X / NG)) * 16) =
                        f32x4{u[i], u[i + 1], u[i + 2], u[i + 3]};
                }
            } else {
                uint32_t w[RUN / 2][Md::PLANES];
#pragma unroll
                for (int i = 0; i < RUN / 2; ++i) Md::cut(u[2 * i], u[2 * i + 1], w[i]);
#pragma unroll
                for (int p = 0; p < Md::PLANES; ++p) {
                    char* d = S + p * O::PLANE + (koff >> 3) * O::HALF + (x + g * (X / NG)) * 16 + (koff & 4) * 2;
                    if constexpr (RUN == 4) {
                        *reinterpret_cast<u32v2*>(d) = u32v2{w[0][p], w[1][p]};
                    } else {
#pragma unroll
                        for (int q = 0; q < RUN / 8; ++q)
                            *reinterpret_cast<u32v4*>(d + q * O::HALF) =
                                u32v4{w[4 * q][p], w[4 * q + 1][p], w[4 * q + 2][p], w[4 * q + 3][p]};
                    }
                }
            }
        }
    }
};

// How the last 16-k steps of an operand end: K a multiple of 32, of 4, any.
enum KEnd { kEndSlice, kEndQuad, kEndAny };

// An operand with rows contiguous in k: element (x, k) at base[x*ld + k], rows
// of any alignment (buffer loads need 4-byte alignment only). Four lanes
// load a row's 64 bytes of a step, so an instruction touches 16 whole
// 64-byte pieces; with two lanes per row and 8 k per lane it touched 32
// half-used ones, twice the L1 accesses (522 per 128x128 step against a step
// of 384 MFMA cycles). kEndQuad: a lane's four k are all inside or all past
// K, a select on its offset; kEndAny: the last steps load their k < K 4 bytes
// at a time (16 bytes over a row's end would read the next row, and past the
// matrix in its last) behind a branch in each step.
template <class T, int X, KEnd END>
struct KcSplit : SplitStaged<T, X, 4> {
    typedef SplitStaged<T, X, 4> S;
    using S::koff;
    using S::NG;
    using S::v;
    using S::x;
    static constexpr bool BRANCH = END == kEndAny;
    static __device__ __forceinline__ int64_t origin(int x0, int64_t ld) { return (int64_t)x0 * ld; }
    __amdgpu_buffer_rsrc_t r;
    uint32_t vo[NG];  // byte offsets of this thread's rows at its first k, or kOutOfRange
    __device__ __forceinline__ void init() {
        x = threadIdx.x / 4;
        koff = (threadIdx.x % 4) * 4;
    }
    __device__ __forceinline__ void tile(const float* base, int64_t ld, int xlim) {
        r = make_rsrc(base);
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            const int row = x + g * (X / NG);
            vo[g] = keep_or_oob((uint32_t)(row * (int)ld + koff) * 4u, row < xlim);
        }
    }
    template <int Q>
    __device__ __forceinline__ void load(int k0, int K, bool on) {
        const bool in = END == kEndQuad ? on & (k0 + koff < K) : on;
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            const uint32_t o = in ? vo[g] : kOutOfRange;
            if (END != kEndAny || k0 + 16 <= K) {
                const f32x4 q = __builtin_bit_cast(
                    f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)o, (int)((uint32_t)k0 * 4u), 0));
                v[Q][4 * g] = q[0], v[Q][4 * g + 1] = q[1], v[Q][4 * g + 2] = q[2], v[Q][4 * g + 3] = q[3];
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    v[Q][4 * g + i] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
                        r, (int)(k0 + koff + i < K ? o + 4u * i : kOutOfRange), (int)((uint32_t)k0 * 4u), 0));
            }
        }
    }
};

// A wave's MFMA operands of one step, read from a stage.
template <class Md, class T>
struct SplitFrags {
    typedef SplitStage<Md, T> D;
    typename Md::Frag a[Md::PLANES][T::TM], b[Md::PLANES][T::TN];
    __device__ __forceinline__ void read(const char* S, int wave, int lane) {
        const int wi = (wave / T::WN) * T::WAVE_M, wj = (wave % T::WN) * T::WAVE_N;
        const int ra = (lane >> 5) * D::A::HALF + (wi + (lane & 31)) * 16;
        const int rb = D::A::BYTES + (lane >> 5) * D::B::HALF + (wj + (lane & 31)) * 16;
#pragma unroll
        for (int p = 0; p < Md::PLANES; ++p) {
#pragma unroll
            for (int tm = 0; tm < T::TM; ++tm)
                a[p][tm] = *reinterpret_cast<const typename Md::Frag*>(S + ra + p * D::A::PLANE + tm * 512);
#pragma unroll
            for (int tn = 0; tn < T::TN; ++tn)
                b[p][tn] = *reinterpret_cast<const typename Md::Frag*>(S + rb + p * D::B::PLANE + tn * 512);
        }
    }
    template <int P, int Q>
    __device__ __forceinline__ void product(floatx16 (&c)[T::TM][T::TN]) const {
#pragma unroll
        for (int tm = 0; tm < T::TM; ++tm)
#pragma unroll
            for (int tn = 0; tn < T::TN; ++tn) c[tm][tn] = Md::mma(a[P][tm], b[Q][tn], c[tm][tn]);
    }
    __device__ __forceinline__ void mma(floatx16 (&hi)[T::TM][T::TN], floatx16 (&lo)[T::TM][T::TN]) const {
        if constexpr (std::is_same<Md, WholeF32>::value) {
#pragma unroll
            for (int p = 0; p < 2; ++p)
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int tm = 0; tm < T::TM; ++tm)
#pragma unroll
                        for (int tn = 0; tn < T::TN; ++tn) {
                            const float x = a[p][tm][e], y = b[p][tn][e];
                            hi[tm][tn] = __builtin_amdgcn_mfma_f32_32x32x2f32(x, y, hi[tm][tn], 0, 0, 0);
                        }
        } else {
            product<0, 0>(hi);
            product<1, 0>(lo);
            product<0, 1>(lo);
            product<1, 1>(lo);
            product<2, 0>(lo);
            product<0, 2>(lo);
        }
    }
};

// Instruction order of one step's block: its LDS reads, then every MFMA
// followed by its share of the cutting (the compiler otherwise cuts first
// and multiplies after: 177 against 190 TFLOP/s, Gemm_nt 4096^3 with bf16
// pieces).
template <class Md, class T, int PER>
__device__ __forceinline__ void split_order() {
    if constexpr (Md::CHECKED) {
        constexpr int M = Md::PRODUCTS * T::TM * T::TN;
        constexpr int V = PER * Md::OPS / 2;  // PER: k per thread of both operands
        __builtin_amdgcn_sched_group_barrier(0x100, Md::PLANES * (T::TM + T::TN), 0);
#pragma unroll
        for (int q = 0; q < M; ++q) {
            __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x2, (V + M - 1) / M, 0);
        }
    }
}

// This wave's LDS stores done, then the workgroup barrier; loads to
// registers stay in flight across it.
__device__ __forceinline__ void split_barrier() {
    __builtin_amdgcn_sched_barrier(0);
    dma_barrier<63>();
    __builtin_amdgcn_sched_barrier(0);
}

// base += hi; hi = 0
template <class T>
__device__ __forceinline__ void split_flush(floatx16 (&hi)[T::TM][T::TN], floatx16 (&base)[T::TM][T::TN]) {
#pragma unroll
    for (int tm = 0; tm < T::TM; ++tm)
#pragma unroll
        for (int tn = 0; tn < T::TN; ++tn)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const float x = hi[tm][tn][r], y = base[tm][tn][r];
                base[tm][tn][r] = y + x;
                hi[tm][tn][r] = 0.f;
            }
}

// One pass of workgroup `wg` over its segments from `seg` on (`walk` just
// past it). The operands run ahead across segment boundaries: a load cursor
// walks the slices (32 k, two steps) one to one and a half ahead of the
// MFMAs, so a new tile starts with its first step in LDS and its next two in
// registers. False: a sum of `seg` is not finite; nothing of it was written.
//
// P: the product. `a`, `b`: its staged operands (SplitStaged); tile(t): the
// loads' tile; load_a<Q>, load_b<Q>(slice, half, on): 16 k into set Q (zeros
// when off); advance(new_tile): the loads' slice moves on by one; begin(it):
// ... to `it` of the tile just set; out(seg, sum): a finished segment.
template <class Md, class T, class P>
__device__ __forceinline__ bool split_pass(P& p, const StreamK& sk, SegmentWalker& walk, Segment& seg, char* lds) {
    typedef SplitStage<Md, T> D;
    constexpr int PER = decltype(p.a)::PER + decltype(p.b)::PER;
    constexpr bool TWO_LEVEL = T::TM * T::TN <= 2;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    SegmentWalker lw = walk;  // load cursor: segment ls, slice lit
    Segment ls = seg;
    int lit = seg.kb;
    bool on = true;
    auto next_slice = [&]() {
        if (!on) return;
        if (++lit < ls.ke) {
            p.step();
        } else {
            on = lw.next(sk, ls);
            lit = ls.kb;
            if (on) {
                p.tile(ls.tile);
                p.begin(lit);
            }
        }
    };
    p.tile(ls.tile);
    p.begin(lit);
    p.template load_a<0>(lit, 0, true);
    p.template load_b<0>(lit, 0, true);
    p.template load_a<1>(lit, 1, true);
    p.template load_b<1>(lit, 1, true);
    p.a.template store<Md, 0>(lds);
    p.b.template store<Md, 0>(lds + D::A::BYTES);
    next_slice();
    p.template load_a<0>(lit, 0, on);
    p.template load_b<0>(lit, 0, on);
    split_barrier();
    while (true) {
        floatx16 hi[T::TM][T::TN], lo[T::TM][T::TN], base[T::TM][T::TN];
#pragma unroll
        for (int tm = 0; tm < T::TM; ++tm)
#pragma unroll
            for (int tn = 0; tn < T::TN; ++tn)
#pragma unroll
                for (int r = 0; r < 16; ++r) hi[tm][tn][r] = lo[tm][tn][r] = base[tm][tn][r] = 0.f;
        for (int it = seg.kb; it < seg.ke; ++it) {
            if (TWO_LEVEL && ((it - seg.kb) & 3) == 3) split_flush<T>(hi, base);
            SplitFrags<Md, T> f;
            // first half out of stage 0; the second half's pieces to stage 1
            f.read(lds, wave, lane);
            p.a.template store<Md, 1>(lds + D::STAGE);
            if (!P::LOADS_BRANCH) p.template load_a<1>(lit, 1, on);
            p.b.template store<Md, 1>(lds + D::STAGE + D::A::BYTES);
            if (!P::LOADS_BRANCH) p.template load_b<1>(lit, 1, on);
            f.mma(hi, lo);
            split_order<Md, T, PER>();
            if (P::LOADS_BRANCH) {
                p.template load_a<1>(lit, 1, on);
                p.template load_b<1>(lit, 1, on);
            }
            split_barrier();
            // second half out of stage 1; the next slice's first to stage 0
            next_slice();
            f.read(lds + D::STAGE, wave, lane);
            p.a.template store<Md, 0>(lds);
            if (!P::LOADS_BRANCH) p.template load_a<0>(lit, 0, on);
            p.b.template store<Md, 0>(lds + D::A::BYTES);
            if (!P::LOADS_BRANCH) p.template load_b<0>(lit, 0, on);
            f.mma(hi, lo);
            split_order<Md, T, PER>();
            if (P::LOADS_BRANCH) {
                p.template load_a<0>(lit, 0, on);
                p.template load_b<0>(lit, 0, on);
            }
            split_barrier();
        }
        if (TWO_LEVEL) split_flush<T>(hi, base);
        bool ok = true;
#pragma unroll
        for (int tm = 0; tm < T::TM; ++tm)
#pragma unroll
            for (int tn = 0; tn < T::TN; ++tn)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const float x = TWO_LEVEL ? base[tm][tn][r] : hi[tm][tn][r], y = lo[tm][tn][r];
                    hi[tm][tn][r] = Md::sum(x, y, ok);
                }
        if (Md::CHECKED && __builtin_amdgcn_readfirstlane(__syncthreads_or(!ok))) return false;
        p.out(seg, hi);
        if (!walk.next(sk, seg)) return true;
    }
}

template <class T, class P>
__device__ __forceinline__ void split_run(P& p, const StreamK& sk, int wg, char* lds) {
    SegmentWalker walk(sk, wg);
    Segment seg;
    if (!walk.next(sk, seg)) return;
    if (!split_pass<SplitB16, T>(p, sk, walk, seg, lds)) split_pass<WholeF32, T>(p, sk, walk, seg, lds);
}

// 16 consecutive k from k0 of a k-contiguous row at byte offset `row`, zeros
// past K, for a wave that holds its operands in registers: four 16-byte loads
// (buffer loads need 4-byte alignment only). TAIL: K may end inside one of
// them, whose k < K then come one by one (16 bytes over the last row's end
// would read past the matrix).
template <bool TAIL>
__device__ __forceinline__ void ws_row(__amdgpu_buffer_rsrc_t r, uint32_t row, int k0, int K, bool on, float (&v)[16]) {
    const int kt = TAIL ? K & ~3 : K;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const uint32_t o = row + (uint32_t)(k0 + 4 * u) * 4u;
        const f32x4 x = load_f32x4(r, (on & (k0 + 4 * u < kt)) ? o : kOutOfRange);
        v[4 * u] = x[0], v[4 * u + 1] = x[1], v[4 * u + 2] = x[2], v[4 * u + 3] = x[3];
    }
    if constexpr (TAIL) {
        const bool here = on & (kt >= k0) & (kt < k0 + 16);
        float t[3];
#pragma unroll
        for (int e = 0; e < 3; ++e) {
            const uint32_t o = row + (uint32_t)(kt + e) * 4u;
            t[e] = load_f32(r, (here & (kt + e < K)) ? o : kOutOfRange);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int e = 0; e < 3; ++e) v[4 * u + e] = kt == k0 + 4 * u ? t[e] : v[4 * u + e];
    }
}

// A wave's 32 x 32 product of operands that it holds whole in registers (the
// short convolutions and GEMMs): lane (row l % 32, half l / 32) has NS slices
// of 16 consecutive k of its row of either operand, one fp32 instruction per
// k of each half.
template <int NS>
__device__ __forceinline__ floatx16 wave_product(const float (&a)[NS][16], const float (&b)[NS][16]) {
    floatx16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.f;
#pragma unroll
    for (int q = 0; q < NS; ++q)
#pragma unroll
        for (int c = 0; c < 16; ++c) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[q][c], b[q][c], acc, 0, 0, 0);
    return acc;
}

// The same in bf16 pieces, twelve 8-pass instructions a slice in place of
// sixteen 16-pass ones and 208 VALU operations beside them. A wave with a sum
// that is not finite goes over its registers again with the fp32 instruction.
template <int NS>
__device__ __forceinline__ floatx16 wave_product_pieces(const float (&a)[NS][16], const float (&b)[NS][16]) {
    floatx16 hi, lo;
#pragma unroll
    for (int r = 0; r < 16; ++r) hi[r] = lo[r] = 0.f;
#pragma unroll
    for (int q = 0; q < NS; ++q)
#pragma unroll
        for (int s = 0; s < 16; s += 8) {
            uint32_t pa[4][3], pb[4][3];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                SplitB16::cut(a[q][s + 2 * i], a[q][s + 2 * i + 1], pa[i]);
                SplitB16::cut(b[q][s + 2 * i], b[q][s + 2 * i + 1], pb[i]);
            }
            bf16x8 fa[3], fb[3];
#pragma unroll
            for (int p = 0; p < 3; ++p) {
                fa[p] = __builtin_bit_cast(bf16x8, u32v4{pa[0][p], pa[1][p], pa[2][p], pa[3][p]});
                fb[p] = __builtin_bit_cast(bf16x8, u32v4{pb[0][p], pb[1][p], pb[2][p], pb[3][p]});
            }
            hi = SplitB16::mma(fa[0], fb[0], hi);
            lo = SplitB16::mma(fa[1], fb[0], lo);
            lo = SplitB16::mma(fa[0], fb[1], lo);
            lo = SplitB16::mma(fa[1], fb[1], lo);
            lo = SplitB16::mma(fa[2], fb[0], lo);
            lo = SplitB16::mma(fa[0], fb[2], lo);
        }
    bool ok = true;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const float x = hi[r], y = lo[r];
        hi[r] = SplitB16::sum(x, y, ok);
    }
    return __all(ok) ? hi : wave_product<NS>(a, b);
}

template <int NS, bool PIECES>
__device__ __forceinline__ floatx16 wave_product_as(const float (&a)[NS][16], const float (&b)[NS][16]) {
    if constexpr (PIECES) return wave_product_pieces<NS>(a, b);
    else return wave_product<NS>(a, b);
}

}  // namespace nnc

// er_gemv_tok.hip -- token-batched GEMV Y[t, M] = W[M, K] . X[t, K] for two
// and more tokens, on the int8 matrix cores.
//
// The batched entry points (Dequant_Q8_0.metal:143-197, 214-500;
// GEMVKernel.swift:682-702) read fp32 activations, so the products stay the
// ones of the one-token kernels (er_gemv.hip): three exact int8 limbs per
// activation (er_xlimbs.h) against the raw integer quants, in int32.  With one
// token that is a v_dot4 per four weights and limb; with several the same
// integers come out of v_mfma_i32_16x16x32_i8, which multiplies 16 weight rows
// with 4 tokens x 3 limbs at a time, and the row's bytes, its nibble split and
// its scales are read and formed once for all the tokens.
//
// Every row value has the bits of the one-token call of the same matrix: the
// integer sums are exact, each 64-weight slot's contribution is formed by the
// same fp32 operations, and the slots are added in the order of the one-token
// kernel that the matrix's M and K select (TokOrder).  Whether a token's rows
// are evaluated in fp32 instead (the conditioning rule of er_xlimbs.h) is
// decided as that kernel decides it, from the same pieces of x and, where the
// order of the sums could matter, in its order.  So batching tokens never
// changes a result.
//
// Work split.  A workgroup of 8 waves owns 16 RT RG rows and 4 TG tokens; RG
// row groups x KW slices of K (KW RG = 8).  It converts the tokens' x once,
// into LDS in the operand order of the matrix instruction, in phases of as
// many 256-weight units as the LDS holds, and each wave walks its slice unit
// by unit, RT row tiles of 16 at once, their raw bytes loaded one unit ahead.
// A lane holds one weight row (lane % 16) and one token of each group (lane /
// 16), so the four limb sums of a (row, token) are one lane's registers and
// the rescaling needs no cross-lane step.
//
// Bound: vector instructions, and the waits of one or two waves per SIMD for
// LDS reads and each other.  Per 64-weight slot a (16 rows x 4 tokens) tile
// costs about 17 of them (Q4_K; Q8_0 15, Q6_K 30) plus 14 (8, 38) per row tile
// for the quants and scales, against 2 (2, 4) matrix instructions (taking those
// out changes no time); the conversion of x costs as much as 1.5 row tiles (of
// 16 tokens) per workgroup, which is why the rows of a workgroup go up with
// the launch (plan_tok).  Counters of 77 tokens: the vector units busy 63% of
// the time the CUs are (Q4_K 14336 x 4096; Q8_0 49%, with the LDS active 52%;
// Q6_K 4096 x 14336 63%), the matrix cores 13 to 22%, and 1120 workgroups on
// 256 CUs leave the last of five rounds three eighths full (Q4_K, Q8_0).
// Measured, us a call in a graph, the one-token kernels over the tokens ->
// these (the planner's choice; weights of several matrices in turn, 600 MB):
//   tokens            5             16             32             77
//   Q4_K 14336x4096   25.4 -> 18.2   51.0 -> 31.6   97.8 -> 44.8  232 -> 133
//   Q8_0 14336x4096   40.3 -> 26.5  120 -> 36.4    237 -> 51.0    565 -> 147
//   Q6_K 4096x14336   40.4 -> 36.6  103 -> 57.7    201 -> 89.7    482 -> 228
#include "er_gemv_cfg.h"

// One wave-uniform unit of work: super-block sb (256 weights) of the slice.
// Packed: sb [0, 8), pmask [8, 12): slots of the unit that belong to the
// slice, base [12, 20): 4 + position of slot 0 in the slice's addition tree,
// ins [20]: the slots' chains are complete after this unit, flush [21]: the
// slice's last unit, count [22, 30): leaves of the slice's tree.
#define ER_TOK_NONE 0u

struct TokUnit {
    uint32_t v;
    __device__ __forceinline__ uint32_t sb() const { return v & 255u; }
    __device__ __forceinline__ uint32_t pmask() const { return (v >> 8) & 15u; }
    __device__ __forceinline__ int base() const { return (int)((v >> 12) & 255u) - 4; }
    __device__ __forceinline__ bool ins() const { return (v >> 20) & 1u; }
    __device__ __forceinline__ bool flush() const { return (v >> 21) & 1u; }
    __device__ __forceinline__ uint32_t count() const { return (v >> 22) & 255u; }
};

// Unit i of K slice ks under order o (0: past the slice's end).
//  whole rows (o.ns >= 1): leaf l of the tree adds slots l + lpr j, j < ns, in
//   order; slice ks holds leaves [ks lpr / KW, (ks + 1) lpr / KW); units run
//   over j for each four leaves.
//  K-sliced (o.ns == 0): the row value is the sum, in order, of 8 trees over
//   spw consecutive slots; slice ks holds trees [8 ks / KW, 8 (ks + 1) / KW).
ER_DEV uint32_t tok_unit(const TokOrder &o, uint32_t S, uint32_t ks, uint32_t i) {
    if (o.ns) {
        const uint32_t leaves = o.lpr >> __builtin_ctz(o.kw), n = (i * o.mg) >> 16, j = i - n * o.ns;
        const uint32_t l0 = ks * leaves + 4u * n;  // first leaf of the unit
        if (4u * n >= leaves || l0 >= S) return ER_TOK_NONE;
        const uint32_t slot = l0 + o.lpr * j;
        const uint32_t ins = j + 1u == o.ns ? 1u : 0u;
        const uint32_t live = min(leaves, S - ks * leaves);  // leaves with a slot (S % 4 == 0)
        const uint32_t flush = ins && 4u * n + 4u >= live ? 1u : 0u;
        const uint32_t pm = slot < S ? 15u : 0u;
        return (min(slot, S - 4u) >> 2) | pm << 8 | (4u * n + 4u) << 12 | ins << 20 | flush << 21 | live << 22;
    }
    const uint32_t n = (i * o.mg) >> 16, k = i - n * o.upt, per = 8u >> __builtin_ctz(o.kw);
    if (n >= per) return ER_TOK_NONE;
    const uint32_t s0 = (ks * per + n) * o.spw, s1 = min(s0 + o.spw, S);
    if (s0 >= S) return ER_TOK_NONE;
    const uint32_t sb = (s0 >> 2) + k;
    if (4u * sb >= s1) return ER_TOK_NONE;
    uint32_t pm = 0;
    for (uint32_t p = 0; p < 4u; ++p) pm |= (4u * sb + p >= s0 && 4u * sb + p < s1 ? 1u : 0u) << p;
    const uint32_t flush = 4u * sb + 4u >= s1 ? 1u : 0u;
    return sb | pm << 8 | (4u * sb + 4u - s0) << 12 | 1u << 20 | flush << 21 | (s1 - s0) << 22;
}

typedef int i32x4 __attribute__((ext_vector_type(4)));

// 16 rows x (4 tokens x 3 limbs): c[l] = sum over 32 positions of limb l of
// this lane's token with this lane's weight row.
ER_DEV i32x4 tok_mfma(u32x2 x, u32x2 w) {
    return __builtin_amdgcn_mfma_i32_16x16x32_i8(__builtin_bit_cast(long, x), __builtin_bit_cast(long, w),
                                                 i32x4{0, 0, 0, 0}, 0, 0, 0);
}

// dwords 0 <-> 2 and 1 <-> 3 across the wave halves: the upper half's dwords
// 0, 1 change places with the lower half's dwords 2, 3
ER_DEV u32x4 tok_swap_halves(const u32x4 &q) {
    const auto a = __builtin_amdgcn_permlane32_swap(q.x, q.z, false, false);
    const auto b = __builtin_amdgcn_permlane32_swap(q.y, q.w, false, false);
    return u32x4{a[0], b[0], a[1], b[1]};
}
// the same between odd and even rows of 16 lanes: odd rows' dwords 0, 1 change
// places with the preceding even rows' dwords 2, 3
ER_DEV u32x4 tok_swap_rows(const u32x4 &q) {
    const auto a = __builtin_amdgcn_permlane16_swap(q.x, q.z, false, false);
    const auto b = __builtin_amdgcn_permlane16_swap(q.y, q.w, false, false);
    return u32x4{a[0], b[0], a[1], b[1]};
}

// Orders a wave's LDS accesses before and after it for the compiler (the LDS
// itself serves a wave in order).
ER_DEV void tok_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Ends the branch of register level n.  Without it the compiler merges the
// like stores of several levels' branches into one through a chosen address,
// which puts the array in scratch memory.
#define tok_branch(n) asm volatile("; level %0" ::"i"(n))

// (a << 8) + b, as one v_lshl_add (of a chain of them the compiler would make
// two shifts and an add3).  The instruction itself must come from the
// compiler: it keeps the wait states between a matrix instruction and the
// first read of its result, which it does not for an instruction in asm.
ER_DEV int tok_lshl8_add(int a, int b) {
    int r = (int)(((uint32_t)a << 8) + (uint32_t)b);
    asm volatile("" : "+v"(r));
    return r;
}

template <int P>
struct TokInt {
    static constexpr int value = P;
};

// group_sum over aligned groups of L lanes, L uniform.
ER_DEV float tok_group_sum(float v, uint32_t L) {
    switch (L) {
        case 64: return group_sum<64>(v);
        case 32: return group_sum<32>(v);
        case 16: return group_sum<16>(v);
        case 8: return group_sum<8>(v);
        default: return group_sum<4>(v);
    }
}

// Formats.  A unit is one 256-weight super-block of a row (for Q8_0 eight
// blocks); its slot p (64 weights) meets slot p of the x unit.
//   load(): a row tile's unit.  Lane 4 i + c takes granules (16 bytes) c, c + 4,
//    ... of row i, so that four neighbouring lanes ask for 64 bytes of one
//    row.  (Loading in operand order, 16 rows per 16 neighbouring lanes, made
//    every lane a request of its own: Q8_0 14336 x 4096 took 40 us for 4
//    tokens, and 237 us for 77 against 109 without the loads.)
//   stash(): those granules into the wave's stage in LDS, rows STRIDE apart.
//   prep(): the unit's scales of this lane's row, from the stage.
//   op<p>(): slot p's matrix operands and scales (quarter r = lane / 16 of the
//    positions); p runs from 0 to 3.
//   dot(): the slot's contribution, added to acc as the one-token kernels do.
//
// x operand layout in LDS: per (unit, slot, token) and quarter r = 0..3 (what
// one lane supplies) three limb granules of 16 bytes, each {8 values of the
// first product, 8 of the second}.  FAC: bytes per (unit, token) of scales and chunk sums.
struct TokQ4K {
    static constexpr int FMT = ER_FMT_Q4_K;
    static constexpr uint32_t FAC = 64, STRIDE = 144;
    using One = CuQ4K;
    struct Ld {
        u32x4 v[3];  // v[2]: granule 8, read by c = 0 (a copy in the others)
    };
    struct Sc {
        uint32_t s[2], m[2];
        float d, dmin;
        u32x4 q;  // the current pair of slots
    };
    struct Xf {
        float4 f;  // group scale, chunk sums XL and XH, -
    };
    struct Op {
        u32x2 lo, hi;
        float s0, s1, m0, m1;
    };
    ER_DEV void load(Ld &l, const uint8_t *row, uint32_t sb, uint32_t c) {
        const uint8_t *bp = row + sb * 144u;
        l.v[0] = ld16_a16(bp + 16u * c);
        l.v[1] = ld16_a16(bp + 64u + 16u * c);
        l.v[2] = ld16_a16(bp + 128u);
    }
    ER_DEV void stash(const Ld &l, uint8_t *st, uint32_t c) {
        *(u32x4 *)(st + 16u * c) = l.v[0];
        *(u32x4 *)(st + 64u + 16u * c) = l.v[1];
        if (c == 0) *(u32x4 *)(st + 128u) = l.v[2];
    }
    ER_DEV uint32_t shift(uint32_t, uint32_t) { return 0u; }
    ER_DEV Sc prep(const uint8_t *st) {
        const u32x4 h = *(const u32x4 *)__builtin_assume_aligned(st, 16);
        Sc c;
        c.s[0] = h.y & 0x3f3f3f3fu;
        c.m[0] = h.z & 0x3f3f3f3fu;
        c.s[1] = (h.w & 0x0f0f0f0fu) | ((h.y >> 2) & 0x30303030u);
        c.m[1] = ((h.w >> 4) & 0x0f0f0f0fu) | ((h.z >> 2) & 0x30303030u);
        c.d = f16_to_f32(h.x & 0xffffu);
        c.dmin = f16_to_f32(h.x >> 16);
        return c;
    }
    // quarter r holds bytes [16 r, 16 r + 16) of a pair of 32-byte slots; after
    // the swaps dwords 0, 1 are slot 2k's positions {0, 16, 8, 24}[r] + [0, 8)
    // and dwords 2, 3 those of slot 2k + 1
    template <int P>
    ER_DEV Op op(const uint8_t *st, Sc &c, uint32_t r) {
        if constexpr (P % 2 == 0)
            c.q = tok_swap_halves(*(const u32x4 *)__builtin_assume_aligned(st + 16u + 32u * P + 16u * r, 16));
        const u32x2 b = P & 1 ? u32x2{c.q.z, c.q.w} : u32x2{c.q.x, c.q.y};
        Op o;
        o.lo = b & 0x0f0f0f0fu;
        o.hi = (b >> 4) & 0x0f0f0f0fu;
        const uint32_t s = c.s[P >> 1], m = c.m[P >> 1];
        o.s0 = P & 1 ? ub2(s) : ub0(s);
        o.s1 = P & 1 ? ub3(s) : ub1(s);
        o.m0 = P & 1 ? ub2(m) : ub0(m);
        o.m1 = P & 1 ? ub3(m) : ub1(m);
        return o;
    }
    ER_DEV Xf xfac(const uint8_t *fac, uint32_t slot) {
        return Xf{*(const float4 *)__builtin_assume_aligned(fac + 16u * slot, 16)};
    }
    // a limb sum of 32 nibbles fits: |c0 2^16 + c1 2^8 + c2| <= 480 * 4227200
    // < 2^31, so it is put together in int32 and rounded to fp32 once (the
    // one-token form rounds once too: c1 2^8 + c2 < 2^24 is exact)
    ER_DEV float whole(const i32x4 &c) { return (float)tok_lshl8_add(tok_lshl8_add(c[0], c[1]), c[2]); }
    ER_DEV float dot(const Op &o, const Sc &c, const u32x4 &x, const Xf &xf, float acc) {
        const float T0 = whole(tok_mfma(u32x2{x.x, x.y}, o.lo)), T1 = whole(tok_mfma(u32x2{x.z, x.w}, o.hi));
        const float sT = __builtin_fmaf(o.s0, T0, o.s1 * T1);
        const float mX = __builtin_fmaf(o.m0, xf.f.y, o.m1 * xf.f.z);
        return acc + __builtin_fmaf(c.d * xf.f.x, sT, -c.dmin * mX);
    }
};

struct TokQ8 {
    static constexpr int FMT = ER_FMT_Q8_0;
    static constexpr uint32_t FAC = 64, STRIDE = 272;
    using One = CuQ8;
    struct Ld {
        u32x4 v[5];  // v[4]: granule 16, read by c = 0
    };
    struct Sc {};
    struct Xf {
        float sg;
    };
    struct Op {
        u32x2 a, b;
        float dA, dB;
    };
    ER_DEV void load(Ld &l, const uint8_t *row, uint32_t sb, uint32_t c) {
        const uint8_t *bp = row + sb * 272u;  // 4-byte aligned (the fused entries' rule)
#pragma unroll
        for (int n = 0; n < 4; ++n) l.v[n] = ld16_a4(bp + 64 * n + 16u * c);
        l.v[4] = ld16_a4(bp + 256);
    }
    ER_DEV void stash(const Ld &l, uint8_t *st, uint32_t c) {
#pragma unroll
        for (int n = 0; n < 4; ++n) *(u32x4 *)(st + 64 * n + 16u * c) = l.v[n];
        if (c == 0) *(u32x4 *)(st + 256) = l.v[4];
    }
    ER_DEV uint32_t shift(uint32_t, uint32_t) { return 0u; }
    ER_DEV Sc prep(const uint8_t *) { return Sc{}; }
    // block A: positions {0, 16, 8, 24}[r] + [0, 8) in dwords 0, 1; block B in 2, 3
    template <int P>
    ER_DEV Op op(const uint8_t *st, Sc &, uint32_t r) {
        const uint8_t *bp = st + 68 * P;
        const u32x4 q = tok_swap_halves(ld16_u2(bp + 2 + 34u * (r >> 1) + 16u * (r & 1u)));
        return Op{u32x2{q.x, q.y}, u32x2{q.z, q.w}, f16_to_f32(ld2(bp)), f16_to_f32(ld2(bp + 34))};
    }
    ER_DEV Xf xfac(const uint8_t *fac, uint32_t slot) { return Xf{*(const float *)(fac + 16u * slot)}; }
    ER_DEV float dot(const Op &o, const Sc &, const u32x4 &x, const Xf &xf, float acc) {
        const i32x4 ca = tok_mfma(u32x2{x.x, x.y}, o.a), cb = tok_mfma(u32x2{x.z, x.w}, o.b);
        const float TA = xl_combine(ca[0], ca[1], ca[2]), TB = xl_combine(cb[0], cb[1], cb[2]);
        const float a = __builtin_fmaf(xf.sg * o.dA, TA, acc);
        return __builtin_fmaf(xf.sg * o.dB, TB, a);
    }
};

// Q6_K blocks are 2-byte aligned: the stage holds the 16-byte-aligned window
// of 14 granules around each row's block (the last of them reaches past the
// block by less than 16 bytes and never past the 16-byte line its last byte
// is in).  Slot p = 2h + c: four granules m of 16 weights with their own scale.
// One operand register pair holds granule m in quarters 0, 1 and granule m + 1
// in quarters 2, 3; each granule's product comes from a copy with the other's
// quarters cleared.
struct TokQ6K {
    static constexpr int FMT = ER_FMT_Q6_K;
    static constexpr uint32_t FAC = 96, STRIDE = 224;
    using One = CuQ6K;
    struct Ld {
        u32x4 v[4];  // v[3]: granules 12, 13, read by c < 2
    };
    struct Sc {
        u32x4 s, ql, qh;  // scales; the current half's quants
        float d;
    };
    struct Xf {
        float4 x32;
        float sgA, sgB;
    };
    struct Op {
        u32x2 q[4];
        float s[4];
    };
    ER_DEV void load(Ld &l, const uint8_t *row, uint32_t sb, uint32_t c) {
        const uint8_t *bp = (const uint8_t *)((uintptr_t)(row + sb * 210u) & ~(uintptr_t)15);
#pragma unroll
        for (int n = 0; n < 3; ++n) l.v[n] = ld16_a16(bp + 64 * n + 16u * c);
        l.v[3] = ld16_a16(bp + 192 + 16u * (c & 1u));
    }
    ER_DEV void stash(const Ld &l, uint8_t *st, uint32_t c) {
#pragma unroll
        for (int n = 0; n < 3; ++n) *(u32x4 *)(st + 64 * n + 16u * c) = l.v[n];
        if (c < 2u) *(u32x4 *)(st + 192 + 16u * c) = l.v[3];
    }
    // offset of the block in its window; rowLow: the row's address, low bits
    ER_DEV uint32_t shift(uint32_t rowLow, uint32_t sb) { return (rowLow + sb * 210u) & 15u; }
    ER_DEV Sc prep(const uint8_t *st) {
        Sc c;
        c.s = ld16_u2(st + 192);
        c.d = f16_to_f32(ld2(st + 208));
        return c;
    }
    // quarters 0, 1 hold the two slots' granules 0 / 2 (16 bytes each), 2, 3
    // their granules 1 / 3; after the swaps dwords 0, 1 are slot c = 0's and
    // 2, 3 slot c = 1's, eight weights per quarter
    template <int P>
    ER_DEV Op op(const uint8_t *st, Sc &k, uint32_t r) {
        constexpr int h = P >> 1, c = P & 1;
        if constexpr (c == 0) {
            k.ql = tok_swap_rows(ld16_u2(st + 64 * h + 16u * r));
            k.qh = tok_swap_rows(ld16_u2(st + 128 + 32 * h + 16u * (r & 1u)));
        }
        const u32x2 l = c ? u32x2{k.ql.z, k.ql.w} : u32x2{k.ql.x, k.ql.y};
        const u32x2 g = (c ? u32x2{k.qh.z, k.qh.w} : u32x2{k.qh.x, k.qh.y}) >> (r & 2u);
        const uint32_t lowHalf = r < 2u ? ~0u : 0u;
        const u32x2 a = (l & 0x0f0f0f0fu) | ((g << 4) & 0x30303030u);  // granules 0 | 1
        const u32x2 b = ((l >> 4) & 0x0f0f0f0fu) | (g & 0x30303030u);  // granules 2 | 3
        Op o;
        o.q[0] = a & lowHalf;
        o.q[1] = a & ~lowHalf;
        o.q[2] = b & lowHalf;
        o.q[3] = b & ~lowHalf;
        // scales sc[8h + 2m + c]: bytes c, 2 + c of dwords 2h, 2h + 1
        const uint32_t sx = h ? k.s.z : k.s.x, sy = h ? k.s.w : k.s.y;
        o.s[0] = sb(sx, c);
        o.s[1] = sb(sx, 2 + c);
        o.s[2] = sb(sy, c);
        o.s[3] = sb(sy, 2 + c);
        return o;
    }
    ER_DEV Xf xfac(const uint8_t *fac, uint32_t slot) {
        const float4 g = *(const float4 *)__builtin_assume_aligned(fac + 64u + 16u * (slot >> 1), 16);
        return Xf{*(const float4 *)__builtin_assume_aligned(fac + 16u * slot, 16), g.x, g.z};
    }
    ER_DEV float dot(const Op &o, const Sc &c, const u32x4 &x, const Xf &xf, float acc) {
        const u32x2 xa = u32x2{x.x, x.y}, xb = u32x2{x.z, x.w};
        const i32x4 c0 = tok_mfma(xa, o.q[0]), c1 = tok_mfma(xa, o.q[1]);
        const i32x4 c2 = tok_mfma(xb, o.q[2]), c3 = tok_mfma(xb, o.q[3]);
        float v = o.s[0] * __builtin_fmaf(xf.sgA, xl_combine(c0[0], c0[1], c0[2]), -xf.x32.x);
        v = __builtin_fmaf(o.s[1], __builtin_fmaf(xf.sgA, xl_combine(c1[0], c1[1], c1[2]), -xf.x32.y), v);
        v = __builtin_fmaf(o.s[2], __builtin_fmaf(xf.sgB, xl_combine(c2[0], c2[1], c2[2]), -xf.x32.z), v);
        v = __builtin_fmaf(o.s[3], __builtin_fmaf(xf.sgB, xl_combine(c3[0], c3[1], c3[2]), -xf.x32.w), v);
        return __builtin_fmaf(c.d, v, acc);
    }
};

// Row sources: bytes of row r, and where token t's value of it goes.  NORM,
// PAIRS, act: as the K-sliced kernels' (gemv_cuk_rows).
struct TokOne {
    static constexpr bool NORM = false, PAIRS = false;
    const uint8_t *W;
    float *y;
    size_t rowBytes;
    uint32_t M;
    __device__ __forceinline__ const TokOne &again() const { return *this; }
    __device__ __forceinline__ const uint8_t *row(uint32_t r) const { return W + (size_t)r * rowBytes; }
    __device__ __forceinline__ void store(uint32_t r, uint32_t t, float v) const { y[(size_t)t * M + r] = v; }
};
// again(): the source for the end of the kernel.  TokQ8Multi (first kernel
// argument: the Q8Multi block) and TokQ8Pairs (first arguments: TokSiluArgs)
// read their fields from the argument segment a second time: held over the
// whole kernel they spilled scalar registers.
struct TokQ8Multi : CukQ8Multi {
    __device__ __forceinline__ TokQ8Multi(const Q8Multi &mm, size_t rb) : CukQ8Multi(mm, rb) {}
    __device__ __forceinline__ TokQ8Multi again() const {
        auto *ka = (const __attribute__((address_space(4))) Q8Multi *)__builtin_amdgcn_kernarg_segment_ptr();
        asm volatile("" : "+s"(ka));
        Q8Multi m;
        for (int i = 0; i < 3; ++i) {
            m.W[i] = ka->W[i];
            m.y[i] = ka->y[i];
            m.res[i] = ka->res[i];
            m.M[i] = ka->M[i];
        }
        m.halfMask = ka->halfMask;
        m.normW = normW;
        m.eps = eps;
        return TokQ8Multi(m, rowBytes);
    }
    __device__ __forceinline__ void store(uint32_t r, uint32_t t, float v) const { store_at(r, t, v); }
};
struct TokSiluArgs {
    const uint8_t *Wg, *Wu;
    const float *x;
    float *y;
    const float *normW;
    float eps;
    uint32_t M;
};
struct TokQ8Pairs : CukQ8Pairs {
    __device__ __forceinline__ TokQ8Pairs again() const {
        auto *ka = (const __attribute__((address_space(4))) TokSiluArgs *)__builtin_amdgcn_kernarg_segment_ptr();
        asm volatile("" : "+s"(ka));
        return TokQ8Pairs(CukQ8Pairs{ka->Wg, ka->Wu, ka->y, rowBytes, normW, eps, ka->M});
    }
    __device__ __forceinline__ TokQ8Pairs(const CukQ8Pairs &p) : CukQ8Pairs(p) {}
    __device__ __forceinline__ void store(uint32_t r, uint32_t t, float v) const { y[(size_t)t * M + (r >> 1)] = v; }
};

// The sum of x^2 over a token's row, added as the one-token kernel does:
// lane-group kernels (4 waves, 16-value chunks, butterfly over the wave) or
// K-sliced ones (8 waves over their slices, group_sum).  One wave; the result
// is wave-uniform.  Four of those waves' pieces are loaded together (one after
// the other, each waiting for its own, cost a workgroup of 16 tokens ~15 us).
ER_DEV float tok_sum_sq(const TokOrder &o, const float *__restrict__ x, uint32_t K) {
    const uint32_t lane = lane_id(), S = K >> 6;
    float tot = 0.0f;
    if (o.ns) {
        static_assert(ER_GEMV_WAVES == 4, "the lane-group kernels' four waves together");
        const uint32_t C16 = K >> 4;
        float ss[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        for (uint32_t c = 0; c < C16; c += 256u) {
            float4 f[4][4];
#pragma unroll
            for (uint32_t w = 0; w < 4u; ++w)
#pragma unroll
                for (int q = 0; q < 4; ++q) f[w][q] = ((const float4 *)(x + 16u * min(c + 64u * w + lane, C16 - 1u)))[q];
#pragma unroll
            for (uint32_t w = 0; w < 4u; ++w)
                if (c + 64u * w + lane < C16)
#pragma unroll
                    for (int q = 0; q < 4; ++q) ss[w] = xl_add_sq(ss[w], f[w][q]);
        }
#pragma unroll
        for (uint32_t w = 0; w < 4u; ++w) {
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) ss[w] += __shfl_xor(ss[w], off, 64);
            tot += ss[w];
        }
        return tot;
    }
    const uint32_t vpl = S <= 64u ? 8u : 16u, ppg = 64u / vpl;  // values of a piece, pieces per 64-group
    for (uint32_t w0 = 0; w0 < ER_CU_WAVES; w0 += 4u) {
        float ss[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        for (uint32_t p = 0; p < ppg * o.spw; p += 64u) {
            float4 f[4][4];
#pragma unroll
            for (uint32_t w = 0; w < 4u; ++w) {
                const uint32_t h = min(ppg * (w0 + w) * o.spw + p + lane, ppg * S - 1u);
#pragma unroll
                for (uint32_t q = 0; q < 4u; ++q) f[w][q] = *(const float4 *)(x + vpl * h + 4u * min(q, vpl / 4u - 1u));
            }
#pragma unroll
            for (uint32_t w = 0; w < 4u; ++w) {
                const uint32_t s0 = (w0 + w) * o.spw, s1 = min(s0 + o.spw, S);
                if (ppg * s0 + p + lane < ppg * s1)
#pragma unroll
                    for (uint32_t q = 0; q < 4u; ++q) ss[w] += q < vpl / 4u ? xl_sq(f[w][q]) : 0.0f;
            }
        }
#pragma unroll
        for (uint32_t w = 0; w < 4u; ++w) tot += group_sum<64>(ss[w]);
    }
    return tot;
}

// The conditioning rule as the one-token kernel decides it, its sums added in
// that kernel's lanes and waves: value16(k, v) gives the 16 values of x from k
// on as converted, grp holds S float2 of this wave's LDS.  One wave; the result
// is wave-uniform.  For tokens whose sums lie so near the rule's threshold that
// the order of the additions could decide (xl_ill_near).
template <class V>
ER_DEV bool tok_ill_in_order(const TokOrder &o, uint32_t S, float f, float2 *grp, V value16) {
    const uint32_t lane = lane_id();
    const bool half = o.conv & 1u;
    tok_fence();
#pragma unroll 1
    for (uint32_t c0 = 0; c0 < 4u * S; c0 += 64u) {
        const uint32_t c = c0 + lane;
        float v[16], ma = 0.0f, mb = 0.0f;
        value16(16u * min(c, 4u * S - 1u), v);
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            ma = fmaxf(ma, fabsf(v[q]));
            mb = fmaxf(mb, fabsf(v[8 + q]));
        }
        float mx = dpp_max_nonneg<ER_DPP_QUAD_XOR1>(fmaxf(ma, mb)), sg, inv;
        mx = dpp_max_nonneg<ER_DPP_QUAD_XOR2>(mx);
        xl_scale(mx, &sg, &inv);
        const float rest = xl_rest_energy16(v, ma, mb, mx, half);
        if ((c & 3u) == 0u && c < 4u * S) grp[c >> 2] = float2{sg, rest};
    }
    tok_fence();
    const uint32_t ppg = half ? 8u : 4u;  // pieces (lanes) of a 64-group
    const uint32_t nw = o.ns ? o.conv >> 1 : ER_CU_WAVES, stride = o.ns ? 64u * nw : 64u;
    float e = 0.0f, r = 0.0f;
#pragma unroll 1
    for (uint32_t w = 0; w < nw; ++w) {
        const uint32_t p0 = o.ns ? 64u * w : ppg * w * o.spw, p1 = ppg * (o.ns ? S : min((w + 1u) * o.spw, S));
        float ew = 0.0f, rw = 0.0f;
#pragma unroll 1
        for (uint32_t p = p0; p < p1; p += stride) {
            const uint32_t i = p + lane;
            if (i < p1 && (i & (ppg - 1u)) == 0u) {
                const float2 g = grp[half ? i >> 3 : i >> 2];
                ew = __builtin_fmaf(g.y > 0.0f ? g.x : 0.0f, g.x, ew);
                rw += g.y;
            }
        }
        e += group_sum<64>(ew);
        r += group_sum<64>(rw);
    }
    return xl_ill_rule(e, r, f);
}

// Rows of the workgroup: RG groups of RT tiles of 16; tokens: 4 TG.  MODE:
// ER_TOK_PLAIN (a leaf is one slot and slices start at a unit), ER_TOK_CHAIN
// (several slots per leaf, o.ns > 1), ER_TOK_SPLIT (K-sliced rows whose
// slices start inside a unit).
#define ER_TOK_PLAIN 0
#define ER_TOK_CHAIN 1
#define ER_TOK_SPLIT 2
template <class F, int RT, int TG, int MODE, class Rows>
ER_DEV void gemv_tok(const Rows &rows, const float *__restrict__ x, uint32_t M, uint32_t K, uint32_t T,
                     const TokOrder o) {
    extern __shared__ __attribute__((aligned(16))) uint32_t lds[];
    constexpr uint32_t TT = 4u * TG, NT = 64u * ER_CU_WAVES;
    __shared__ uint32_t units[ER_TOK_MAX_UNITS];  // slice ks, index i at ks * ups + i
    __shared__ float rmsv[TT];
    __shared__ float2 chk[NT / 32u];
    __shared__ uint32_t nfw[ER_CU_WAVES];  // [wave] tokens it saw a non-finite chunk sum of
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t S = K >> 6, kw = o.kw, rg = ER_CU_WAVES / kw, rowsWg = 16u * RT * rg;
    const uint32_t ks = wave % kw, grp = wave / kw;
    // token tiles of one row block run on one XCD (workgroup b on XCD b % 8),
    // next to each other, so the block's weights are fetched into its L2 once
    const uint32_t nTok = (T + TT - 1u) / TT, xcd = blockIdx.x & 7u, seq = blockIdx.x >> 3;
    const uint32_t blk = seq / nTok * 8u + xcd, t0 = (seq % nTok) * TT;
    if (blk * rowsWg >= M) return;
    const uint32_t nT = min(TT, T - t0);  // live tokens
    const uint32_t r = lane >> 4;         // quarter of the positions, and token of each group

    // x of a phase: a wave pass is one token's x of four units (one 16-value
    // chunk per lane); this wave makes passes wave, wave + 8, ...
    const uint32_t U = 1u << o.lupp;  // units per slice and phase
    const uint32_t lq = __builtin_ctz(kw) + o.lupp - 2u, passes = nT << lq;
    const uint32_t c16 = lane & 15u;
    // weights 256 sb of unit v (slice v / U) of phase ph; any unit of the row
    // where the slice has none
    auto x_block = [&](uint32_t ph, uint32_t v) {
        const uint32_t sl = v >> o.lupp, i = (ph << o.lupp) + (v & (U - 1u)), n = __umul24(i, o.mg) >> 16;
        const uint32_t b = o.ns ? (__umul24(sl, o.lpr >> __builtin_ctz(kw)) >> 2) + n +
                                      __umul24(o.lpr >> 2, i - __umul24(n, o.ns))
                                : (__umul24((sl << (3u - __builtin_ctz(kw))) + n, o.spw) >> 2) + i - __umul24(n, o.upt);
        return min(b, (S >> 2) - 1u) * 256u;
    };
    constexpr int NW = Rows::NORM ? 4 : 1;
    auto load_x = [&](uint32_t ph, uint32_t ps, float4 (&xr)[4], float4 (&wr)[NW]) {
        const uint32_t pc = min(ps, passes - 1u), t = pc >> lq;
        const uint32_t k0 = x_block(ph, 4u * (pc - (t << lq)) + r) + 16u * c16;
        const float *xp = x + (size_t)(t0 + t) * K + k0;
#pragma unroll
        for (int q = 0; q < 4; ++q) xr[q] = ((const float4 *)xp)[q];
        if constexpr (Rows::NORM) {
            if (rows.normW) {
#pragma unroll
                for (int q = 0; q < 4; ++q) wr[q] = ((const float4 *)(rows.normW + k0))[q];
            }
        }
    };
    float4 xr[2][4], wr[2][NW];
    load_x(0, wave, xr[0], wr[0]);
    __builtin_amdgcn_sched_barrier(0);

    if constexpr (Rows::NORM) {
        for (uint32_t t = wave; t < nT; t += ER_CU_WAVES) {
            const float ss = rows.normW ? tok_sum_sq(o, x + (size_t)(t0 + t) * K, K) : 0.0f;
            if (lane == 0) rmsv[t] = rows.normW ? 1.0f / __builtin_sqrtf(ss / (float)K + rows.eps) : 1.0f;
        }
        __syncthreads();
    }
    // this lane's granule of a slot's limbs: quarter r of limb lane % 4 (3: a
    // copy, its sums are not read) of token lane % 16 / 4.  A quarter's three
    // limbs lie side by side: 8 lanes of a read meet no bank twice
    const uint32_t xl = r * 48u + min(lane & 3u, 2u) * 16u + ((lane & 15u) >> 2) * 192u;

    // LDS of a phase: limbs, then the factors; after the last phase the
    // partial row sums
    uint8_t *limbs = (uint8_t *)lds;
    uint8_t *facs = limbs + (size_t)(kw << o.lupp) * TT * 768u;
    // finished trees go to part[(tree TT + t) rowsWg + row] in LDS, past the
    // factors: tree ks * per + nfin (whole rows: one per slice), or, with one
    // slice of K, added up in order as they finish
    const uint32_t per = o.ns || kw == 1u ? 1u : 8u / kw, nPart = per * kw, stp = TT * rowsWg;
    float *part = (float *)(facs + (kw << o.lupp) * (TT * F::FAC));
    uint32_t nfm = 0;  // tokens with a non-finite chunk sum
    // x under RMSNorm as converted: whole rows with token t's factor, K-sliced
    // ones without it (their row values take it)
    auto normed = [&](const float4 &f, const float4 &w, uint32_t t) {
        if (!o.ns) return float4{f.x * w.x, f.y * w.y, f.z * w.z, f.w * w.w};
        const float s = rmsv[t];
        return float4{f.x * s * w.x, f.y * s * w.y, f.z * s * w.z, f.w * s * w.w};
    };
    auto convert = [&](uint32_t ps, const float4 (&xr)[4], const float4 (&wr)[NW]) {
        const uint32_t t = ps >> lq, v = 4u * (ps - (t << lq)) + r;
        float xv[16];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            float4 f = xr[q];
            if constexpr (Rows::NORM) {
                if (rows.normW) f = normed(f, wr[q], t);
            }
            xv[4 * q] = f.x;
            xv[4 * q + 1] = f.y;
            xv[4 * q + 2] = f.z;
            xv[4 * q + 3] = f.w;
        }
        XlChunk ck;
        xl_chunk(xv, ck, o.conv & 1u);
        if (__builtin_amdgcn_ballot_w64(!__builtin_isfinite(ck.sum)) != 0) nfm |= 1u << t;
        // the chunk's slot, and the granules of its two 8-value pieces
        constexpr bool Q6 = F::FMT == ER_FMT_Q6_K;
        const uint32_t m = (c16 >> 1) & 3u;  // Q6_K granule
        const uint32_t slot = Q6 ? 2u * (c16 >> 3) + (c16 & 1u) : c16 >> 2;
        const uint32_t g0 = Q6 ? 2u * (m & 1u) : c16 & 1u, half = Q6 ? m >> 1 : (c16 >> 1) & 1u;
        uint8_t *lp = limbs + ((v * 4u + slot) * TT + t) * 192u + 48u * g0 + 8u * half;
#pragma unroll
        for (int l = 0; l < ER_XL_PLANES; ++l) {
            *(u32x2 *)__builtin_assume_aligned(lp + 16 * l, 8) = u32x2{ck.lb[l][0], ck.lb[l][1]};
            *(u32x2 *)__builtin_assume_aligned(lp + 16 * l + (Q6 ? 48 : 96), 8) = u32x2{ck.lb[l][2], ck.lb[l][3]};
        }
        uint8_t *fp = facs + (v * TT + t) * F::FAC;
        if constexpr (Q6) {
            ((float *)fp)[4u * slot + m] = 32.0f * ck.sum;
            if ((lane & 3u) == 0) *(float2 *)(fp + 64u + 8u * (c16 >> 2)) = float2{ck.sg, ck.rest};
        } else {
            const float pr = dpp_add<ER_DPP_QUAD_XOR1>(ck.sum);
            const float po = __int_as_float(
                __builtin_amdgcn_update_dpp(0, __float_as_int(pr), ER_DPP_QUAD_XOR2, 0xf, 0xf, false));
            if ((lane & 3u) == 0) *(float4 *)(fp + 16u * slot) = float4{ck.sg, pr, po, ck.rest};
        }
    };

    // weights: RT row tiles, a pair of them in the stage at a time; the first
    // unit's bytes leave right after the first x.  Lane l loads row l / 4 of a
    // tile and computes row l % 16.
    constexpr int PT = RT < 2 ? RT : 2;
    const uint32_t row0 = blk * rowsWg + grp * (16u * RT), lc = lane & 3u;
    uint8_t *stage = (uint8_t *)part + o.part + wave * (PT * 16u * F::STRIDE);
    uint8_t *stW = stage + (lane >> 2) * F::STRIDE;
    const uint8_t *stR = stage + (lane & 15u) * F::STRIDE;
    const uint8_t *rp[RT];
    uint32_t low[RT];  // the computed row's address, low bits (Q6_K)
#pragma unroll
    for (int q = 0; q < RT; ++q) {
        rp[q] = rows.row(min(row0 + 16u * q + (lane >> 2), M - 1u));
        low[q] = F::FMT == ER_FMT_Q6_K ? (uint32_t)(uintptr_t)rows.row(min(row0 + 16u * q + (lane & 15u), M - 1u)) : 0u;
    }
    typename F::Ld ld[RT];
    TokUnit cu{(uint32_t)__builtin_amdgcn_readfirstlane((int)tok_unit(o, S, ks, 0))};
    // the first pair's bytes leave before x is converted, the others after it
    // (an absent unit: super-block 0).  With all four tiles' loads ahead of it
    // the conversion began when they had left, 6 us into the launch.
#pragma unroll
    for (int q = 0; q < PT; ++q) F::load(ld[q], rp[q], cu.sb(), lc);
    __builtin_amdgcn_sched_barrier(0);

    // the units, for the walk: written behind the first loads and read after
    // the conversion's barrier, so the table costs no barrier of its own (with
    // one, and the rows summed through LDS at the end, a call took 0.3 to 0.8
    // us more: Q4_K 4096 x 4096 x 5 10.3 -> 9.7 us, 14336 x 4096 x 5 19.4 ->
    // 18.9, Q8_0 1024 x 1024 x 4 6.2 -> 5.3); formed on scalars at every unit
    // instead, long slices lose it again (4096 x 14336 x 5 27.7 -> 28.6)
    if (grp == 0)
        for (uint32_t i = lane; i < o.ups; i += 64u) units[ks * o.ups + i] = tok_unit(o, S, ks, i);
    auto unit = [&](uint32_t i) {
        return TokUnit{i < o.ups ? (uint32_t)__builtin_amdgcn_readfirstlane((int)units[ks * o.ups + i]) : ER_TOK_NONE};
    };

    // st: the addition tree as a binary counter, level l the sum of 2^l of its
    // steps (a unit's four leaves, or one leaf where slices start inside a
    // unit) while bit l of their count is set; ch: the leaves' chains
    constexpr int LV = MODE == ER_TOK_SPLIT ? 5 : 3, NC = MODE == ER_TOK_CHAIN ? 4 : 1;
    float st[LV][RT][TG], ch[NC][RT][TG];
    auto each = [&](auto f) {
#pragma unroll
        for (int q = 0; q < RT; ++q)
#pragma unroll
            for (int g = 0; g < TG; ++g) f(q, g);
    };
    each([&](int q, int g) {
#pragma unroll
        for (int l = 0; l < LV; ++l) st[l][q][g] = 0.0f;
#pragma unroll
        for (int l = 0; l < NC; ++l) ch[l][q][g] = 0.0f;
    });
    auto insert = [&](auto self, auto L, float (&v)[RT][TG], uint32_t n) -> void {
        constexpr int l = decltype(L)::value;
        if constexpr (l == LV) {  // all 2^LV steps
            each([&](int q, int g) { st[0][q][g] = v[q][g]; });
            tok_branch(2 * LV);
        } else {
            if ((n >> l) & 1u) {
                each([&](int q, int g) { v[q][g] = st[l][q][g] + v[q][g]; });
                self(self, TokInt<l + 1>{}, v, n);
            } else {
                each([&](int q, int g) { st[l][q][g] = v[q][g]; });
                tok_branch(l);
            }
        }
    };
    float *mine = part + (ks * per * TT + r) * rowsWg + grp * (16u * RT) + (lane & 15u);
    for (uint32_t l = 0; l < per; ++l)  // slices past the row's end add nothing
        each([&](int q, int g) { mine[(l * TT + 4 * g) * rowsWg + 16 * q] = 0.0f; });
    uint32_t nfin = 0;
    const uint32_t ct = tid / (NT / TT);
    float ce = 0.0f, cr = 0.0f;  // conditioning sums of token ct

    for (uint32_t ph = 0; (ph << o.lupp) < o.ups; ++ph) {
        if (ph) {
            __syncthreads();  // the last phase's limbs are read
            load_x(ph, wave, xr[0], wr[0]);
        }
        for (uint32_t ps = wave; ps < passes; ps += 2u * ER_CU_WAVES) {
            load_x(ph, ps + ER_CU_WAVES, xr[1], wr[1]);
            convert(ps, xr[0], wr[0]);
            if (ps + ER_CU_WAVES >= passes) break;
            load_x(ph, ps + 2u * ER_CU_WAVES, xr[0], wr[0]);
            convert(ps + ER_CU_WAVES, xr[1], wr[1]);
        }
        if (ph == 0) {
#pragma unroll
            for (int q = PT; q < RT; ++q) F::load(ld[q], rp[q], cu.sb(), lc);
        }
        __syncthreads();
        // the conditioning sums of this phase's x groups, a slice's own once
        // (Q6_K slot p shares its x groups with the slot beside it, and a unit
        // is never split there: group p counts with the unit); NT / TT
        // neighbouring threads share a token
        if (ct < nT) {
            for (uint32_t g = tid & (NT / TT - 1u); g < (kw << o.lupp) * 4u; g += NT / TT) {
                const uint32_t v = g >> 2, p = g & 3u, i = (ph << o.lupp) + (v & (U - 1u));
                const uint32_t pk = i < o.ups ? units[(v >> o.lupp) * o.ups + i] : ER_TOK_NONE;
                if (!((pk >> (8u + p)) & 1u)) continue;
                const uint8_t *fp = facs + (v * TT + ct) * F::FAC;
                float sg, rest;
                if constexpr (F::FMT == ER_FMT_Q6_K) {
                    const float2 f = *(const float2 *)(fp + 64u + 8u * p);
                    sg = f.x;
                    rest = f.y;
                } else {
                    const float4 f = *(const float4 *)(fp + 16u * p);
                    sg = f.x;
                    rest = f.w;
                }
                ce = __builtin_fmaf(rest > 0.0f ? sg : 0.0f, sg, ce);
                cr += rest;
            }
        }
        for (uint32_t i = 0; i < U; ++i) {
            const TokUnit nu = unit((ph << o.lupp) + i + 1u);
            const uint32_t v = ks * U + i;
            const uint8_t *lp = limbs + v * (4u * TT * 192u) + xl;
            const uint8_t *fp = facs + (v * TT + r) * F::FAC;
            float a2[MODE == ER_TOK_PLAIN ? 2 : 1][RT][TG];  // the unit's pair sums
            float vs[MODE == ER_TOK_SPLIT ? 4 : 1][RT][TG];  // the unit's slots
#pragma unroll
            for (int h = 0; h < RT; h += PT) {
                // this pair into the stage (the wave's own: its LDS accesses run
                // in order), its next unit's loads behind it
                tok_fence();
#pragma unroll
                for (int q = 0; q < PT; ++q) F::stash(ld[h + q], stW + q * (16u * F::STRIDE), lc);
                tok_fence();
                if (nu.v != ER_TOK_NONE) {
#pragma unroll
                    for (int q = 0; q < PT; ++q) F::load(ld[h + q], rp[h + q], nu.sb(), lc);
                }
                __builtin_amdgcn_sched_barrier(0);
                const uint8_t *src[PT];
                typename F::Sc sc[PT];
#pragma unroll
                for (int q = 0; q < PT; ++q) {
                    src[q] = stR + q * (16u * F::STRIDE) + F::shift(low[h + q], cu.sb());
                    sc[q] = F::prep(src[q]);
                }
                auto slot = [&](auto P) {
                    constexpr int p = decltype(P)::value;
                    // (never skipped in plain mode, but the branch keeps the slots
                    // apart: as one basic block they were ordered with the operands
                    // of all four live at once, and spilled)
                    typename F::Op op[PT];
                    if ((cu.pmask() >> p) & 1u) {
                        u32x4 xo[TG];
                        typename F::Xf xf[TG];
#pragma unroll
                        for (int q = 0; q < PT; ++q) op[q] = F::template op<p>(src[q], sc[q], r);
#pragma unroll
                        for (int g = 0; g < TG; ++g) {
                            xo[g] = *(const u32x4 *)__builtin_assume_aligned(lp + (p * TT + 4u * g) * 192u, 16);
                            xf[g] = F::xfac(fp + 4u * g * F::FAC, p);
                        }
#pragma unroll
                        for (int q = 0; q < PT; ++q)
#pragma unroll
                            for (int g = 0; g < TG; ++g) {
                                if constexpr (MODE == ER_TOK_CHAIN) {
                                    float &c = ch[p][h + q][g];
                                    c = F::dot(op[q], sc[q], xo[g], xf[g], c);
                                } else {
                                    const float d = F::dot(op[q], sc[q], xo[g], xf[g], 0.0f);
                                    if constexpr (MODE == ER_TOK_PLAIN)
                                        a2[p >> 1][h + q][g] = p & 1 ? a2[p >> 1][h + q][g] + d : d;
                                    else
                                        vs[p][h + q][g] = d;
                                }
                            }
                    } else if constexpr (MODE == ER_TOK_SPLIT && p % 2 == 0) {
#pragma unroll
                        for (int q = 0; q < PT; ++q) (void)F::template op<p>(src[q], sc[q], r);  // slot p + 1's bytes
                    }
                    __builtin_amdgcn_sched_barrier(0);
                };
                slot(TokInt<0>{});
                slot(TokInt<1>{});
                slot(TokInt<2>{});
                slot(TokInt<3>{});
            }
            if constexpr (MODE == ER_TOK_SPLIT) {
#pragma unroll
                for (int p = 0; p < 4; ++p)
                    if ((cu.pmask() >> p) & 1u) insert(insert, TokInt<0>{}, vs[p], (uint32_t)(cu.base() + p));
            }
            if constexpr (MODE != ER_TOK_SPLIT) {
                if (MODE == ER_TOK_PLAIN ? cu.v != ER_TOK_NONE : cu.ins()) {
                    float u[RT][TG];
                    each([&](int q, int g) {
                        if constexpr (MODE == ER_TOK_CHAIN) {
                            u[q][g] = (ch[0][q][g] + ch[1][q][g]) + (ch[2][q][g] + ch[3][q][g]);
#pragma unroll
                            for (int l = 0; l < 4; ++l) ch[l][q][g] = 0.0f;
                        } else {
                            u[q][g] = a2[0][q][g] + a2[1][q][g];
                        }
                    });
                    insert(insert, TokInt<0>{}, u, (uint32_t)cu.base() >> 2);
                }
            }
            if (cu.flush()) {
                // the slice's tree, its missing leaves adding nothing: the
                // levels present, low to high (all 2^LV steps: in st[0])
                const uint32_t n = MODE == ER_TOK_SPLIT ? cu.count() : cu.count() >> 2;
                float s[RT][TG];
                const bool full = n >> LV;
                each([&](int q, int g) {
                    // levels present come one after the other from the lowest:
                    // x + 0 is x, so an absent level adds zero
                    float a = full || (n & 1u) ? st[0][q][g] : 0.0f;
#pragma unroll
                    for (int l = 1; l < LV; ++l) a = ((n >> l) & 1u ? st[l][q][g] : 0.0f) + a;
                    s[q][g] = a;
                });
                each([&](int q, int g) {
                    float *p = mine + (nfin * TT + 4 * g) * rowsWg + 16 * q;
                    *p = kw == 1u ? *p + s[q][g] : s[q][g];
                });
                nfin += kw == 1u ? 0u : 1u;
            }
            cu = nu;
        }
    }
    // the launch's checks per token
    constexpr uint32_t CW = NT / TT < 64u ? NT / TT : 64u, CN = NT / TT / CW;  // partial sums per token: CN
    ce = group_sum<CW>(ce);
    cr = group_sum<CW>(cr);
    if (tid % CW == 0) chk[tid / CW] = float2{ce, cr};
    if (lane == 0) nfw[wave] = nfm;
    __syncthreads();
    // every wave decides for itself, so that rows with no such token are stored
    // straight from their sums: bit t of ill (fp32 over every term), of
    // nf (over the non-finite ones)
    uint32_t nf = 0;
#pragma unroll
    for (uint32_t w = 0; w < ER_CU_WAVES; ++w) nf |= nfw[w];
    float ee = 0.0f, rr = 0.0f;
#pragma unroll
    for (uint32_t w = 0; w < CN; ++w) {
        const float2 c = chk[min(lane, TT - 1u) * CN + w];
        ee += c.x;
        rr += c.y;
    }
    constexpr float illF = F::FMT == ER_FMT_Q8_0 ? 1.0f : 4.0f;
    uint32_t ill = (uint32_t)__builtin_amdgcn_ballot_w64(lane < nT && xl_ill_rule(ee, rr, illF));
    uint32_t near = (uint32_t)__builtin_amdgcn_ballot_w64(lane < nT && xl_ill_near(ee, rr, illF));
#pragma unroll 1
    for (; near; near &= near - 1u) {  // alike in every wave
        const uint32_t t = __builtin_ctz(near);
        const float *xt = x + (size_t)(t0 + t) * K;
        const bool b = tok_ill_in_order(o, S, illF, (float2 *)stage, [&](uint32_t k, float (&v)[16]) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                float4 f = ((const float4 *)(xt + k))[q];
                if constexpr (Rows::NORM) {
                    if (rows.normW) f = normed(f, ((const float4 *)(rows.normW + k))[q], t);
                }
                v[4 * q] = f.x;
                v[4 * q + 1] = f.y;
                v[4 * q + 2] = f.z;
                v[4 * q + 3] = f.w;
            }
        });
        ill = b ? ill | 1u << t : ill & ~(1u << t);
    }
    const uint32_t bad = (uint32_t)__builtin_amdgcn_readfirstlane((int)(ill | nf));
    const Rows end = rows.again();
    // row value (t, row) at part[t rowsWg + row]: slices as the tree's top
    // levels (whole rows) or in order
    const uint32_t lr = __builtin_ctz(rowsWg);
    auto value = [&](uint32_t at) {
        float v;
        if (o.ns) {
            if (nPart == 1u) {
                v = part[at];
            } else if (nPart == 2u) {
                v = part[at] + part[at + stp];
            } else if (nPart == 4u) {
                v = (part[at] + part[at + stp]) + (part[at + 2u * stp] + part[at + 3u * stp]);
            } else {
                v = ((part[at] + part[at + stp]) + (part[at + 2u * stp] + part[at + 3u * stp])) +
                    ((part[at + 4u * stp] + part[at + 5u * stp]) + (part[at + 6u * stp] + part[at + 7u * stp]));
            }
        } else {
            v = 0.0f;
            for (uint32_t q = 0; q < nPart; ++q) v += part[at + q * stp];
            if constexpr (Rows::NORM) v *= rmsv[at >> lr];
        }
        return v;
    };
    auto store_rows = [&](auto val) {
        if constexpr (Rows::PAIRS) {
            for (uint32_t i = tid; i < (nT << (lr - 1u)); i += NT) {
                const uint32_t t = i >> (lr - 1u), at = 2u * i, row = blk * rowsWg + (at & (rowsWg - 1u));
                if (row < M) end.store(row, t0 + t, Rows::act(val(at)) * val(at + 1u));
            }
        } else {
            for (uint32_t i = tid; i < (nT << lr); i += NT) {
                const uint32_t row = blk * rowsWg + (i & (rowsWg - 1u));
                if (row < M) end.store(row, t0 + (i >> lr), val(i));
            }
        }
    };
    if (bad == 0u) {
        store_rows(value);
        return;
    }
    // Tokens whose x the limbs do not carry (er_nonfinite.h, the conditioning
    // rule of er_xlimbs.h): their rows again in fp32 from the raw weights, one
    // row per lane group as the one-token kernels do.
    for (uint32_t i = tid; i < (nT << lr); i += NT) part[i] = value(i);  // only this thread reads slice 0 of (row, t)
    __syncthreads();
    const uint32_t L = o.nfl, G = NT / L, li = lane % L;
    for (uint32_t i = tid / L; i < (rowsWg + G - 1u) / G * G; i += G) {
        const uint32_t rw = min(blk * rowsWg + i, M - 1u);
        for (uint32_t t = 0; t < nT; ++t) {
            if (!((bad >> t) & 1u)) continue;
            const bool all = (ill >> t) & 1u;
            const float *xt = x + (size_t)(t0 + t) * K;
            float sp[1] = {0.0f}, h = 0.0f;
            nf_terms<1>([&](int, uint32_t k) { return weight_at<F::FMT>(end.row(rw), k); },
                        [&](uint32_t k) {
                            if constexpr (Rows::NORM)
                                return rows.normW ? xt[k] * rmsv[t] * rows.normW[k] : xt[k];
                            else
                                return xt[k];
                        },
                        nullptr, K >> 4, li, L, sp, h, all);
            const float v = tok_group_sum(sp[0], L), hs = tok_group_sum(h, L);
            if (li == 0 && i < rowsWg && (all || hs > 0.0f)) part[(t << lr) + i] = v;
        }
    }
    __syncthreads();
    store_rows([&](uint32_t at) { return part[at]; });
}

// er_gemv_<fmt>_tok[c|s]_r<RT>_t<4 TG> (W, x, y, M, K, T, order; c, s: MODE), and the fused
// Q8_0 rows and gate/up + SiLU (2M rows); 1-D grid of 8 ceil(blocks / 8)
// ceil(T / (4 TG)) workgroups, dynamic LDS as plan_tok sizes it.
#define ER_TOK_ENTRY(fmt, F, RT, TG, TT, C, tag)                                                            \
    extern "C" __global__ void __launch_bounds__(64 * ER_CU_WAVES)                                           \
        er_gemv_##fmt##_tok##tag##_r##RT##_t##TT(const uint8_t *__restrict__ W, const float *__restrict__ x,   \
                                                 float *__restrict__ y, uint32_t M, uint32_t K, uint32_t T,  \
                                                 TokOrder o) {                                               \
        const TokOne rows{W, y, F::One::row_bytes(K), M};                                                     \
        gemv_tok<F, RT, TG, C>(rows, x, M, K, T, o);                                                          \
    }
#define ER_TOK_Q8F_ENTRY(RT, TG, TT, C, tag)                                                                 \
    extern "C" __global__ void __launch_bounds__(64 * ER_CU_WAVES)                                           \
        er_gemv_q8_0_multi_tok##tag##_r##RT##_t##TT(Q8Multi mm, const float *__restrict__ x, uint32_t K,       \
                                                    uint32_t T, TokOrder o) {                                \
        const TokQ8Multi rows(mm, CuQ8::row_bytes(K));                                                        \
        gemv_tok<TokQ8, RT, TG, C>(rows, x, mm.M[0] + mm.M[1] + mm.M[2], K, T, o);                            \
    }                                                                                                        \
    extern "C" __global__ void __launch_bounds__(64 * ER_CU_WAVES)                                           \
        er_gemv_q8_0_silu_tok##tag##_r##RT##_t##TT(const uint8_t *__restrict__ Wg,                            \
                                                   const uint8_t *__restrict__ Wu,                           \
                                                   const float *__restrict__ x, float *__restrict__ y,       \
                                                   const float *__restrict__ normW, float eps, uint32_t M,   \
                                                   uint32_t K, uint32_t T, TokOrder o) {                     \
        const TokQ8Pairs rows(CukQ8Pairs{Wg, Wu, y, CuQ8::row_bytes(K), normW, eps, M});                      \
        gemv_tok<TokQ8, RT, TG, C>(rows, x, 2u * M, K, T, o);                                                 \
    }
#define ER_TOK_ENTRIES(RT, TG, TT)                         \
    ER_TOK_ENTRY(q4k, TokQ4K, RT, TG, TT, ER_TOK_PLAIN, )  \
    ER_TOK_ENTRY(q4k, TokQ4K, RT, TG, TT, ER_TOK_CHAIN, c) \
    ER_TOK_ENTRY(q4k, TokQ4K, RT, TG, TT, ER_TOK_SPLIT, s) \
    ER_TOK_ENTRY(q6k, TokQ6K, RT, TG, TT, ER_TOK_PLAIN, )  \
    ER_TOK_ENTRY(q8_0, TokQ8, RT, TG, TT, ER_TOK_PLAIN, )  \
    ER_TOK_ENTRY(q8_0, TokQ8, RT, TG, TT, ER_TOK_CHAIN, c) \
    ER_TOK_Q8F_ENTRY(RT, TG, TT, ER_TOK_PLAIN, )
ER_TOK_CONFIGS(ER_TOK_ENTRIES)
// the kinds and modes with more values live, where (4, 2) spills
#define ER_TOK_ENTRIES_SMALL(RT, TG, TT)                   \
    ER_TOK_ENTRY(q6k, TokQ6K, RT, TG, TT, ER_TOK_CHAIN, c) \
    ER_TOK_ENTRY(q8_0, TokQ8, RT, TG, TT, ER_TOK_SPLIT, s) \
    ER_TOK_Q8F_ENTRY(RT, TG, TT, ER_TOK_CHAIN, c)          \
    ER_TOK_Q8F_ENTRY(RT, TG, TT, ER_TOK_SPLIT, s)
ER_TOK_CONFIGS_SMALL(ER_TOK_ENTRIES_SMALL)

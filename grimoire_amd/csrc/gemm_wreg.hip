// gemm_wreg.hip -- grouped expert products for batches of a few to a few
// hundred rows per expert, bf16 MFMA with exactly decoded weights.
//
// What bounds it: up to ~64 rows per expert the weight stream (every touched
// expert's rows once), above that the matrix core.  A tile is up to 128
// activation rows (down: 64, INT4: 16) x 256 weight rows (INT4: 128) per
// work-group of four waves, two (INT4: four) work-groups per CU; the number
// of 16-row activation blocks NT is chosen per tile from its live rows, so an
// expert with few rows neither multiplies nor loads padding.
//
//   - Weights never touch LDS.  v_mfma_f32_16x16x32_bf16 takes its second
//     operand as 16 columns x 4 groups of 8 K: lane (column c = l % 16,
//     group g = l / 16).  K is permuted so that a lane's group owns 16
//     consecutive bytes of the row: the four lanes of a column read one
//     64-byte piece (a "segment": 128 K of 4-bit codes, 32 K of bf16) and
//     each 16-byte register holds the operands of J MFMA steps (4 for
//     4-bit, 1 for bf16).  A stage is SP segments of the wave's rows, double
//     buffered in registers (MXFP4 down, 128 experts x 8 rows, K 2048, N 4096:
//     SP 2 116 us, SP 4 132: more lines in flight than the L2 holds; SP 1 a
//     third slower).
//   - Activations (bf16 rows, one or two planes) come through LDS by
//     buffer_load ... lds, double buffered, gathered by row through the
//     route -> token map; 16-byte slots XOR-swizzled by row so that the
//     operand reads are free of bank conflicts.  Each wave's fragment reads
//     are inline asm with their own lgkmcnt waits (a compiler-visible LDS
//     read would wait for every load in flight).
//   - One barrier per stage.
//
// Weights decode to bf16 exactly: e2m1 x e8m0 through the fp4 converter;
// INT4 codes as 16 + q (a bf16 of exponent 4 keeps q in its mantissa), the
// offset 16 + zero point taken out per 128-K segment with the segment's sum
// of x (one more MFMA against ones), then the group scale in fp32.  (128 + q,
// one operation fewer, would lose three more bits to the offset.)
//
// Measured (one MI355X, kernel alone): MXFP4, 128 experts x 8 rows, K = N =
// 2880: gate_up 259 us = 4.4 TB/s of weights, down 143 us (rows of 1440 bytes
// put odd rows' pieces across memory lines); K 4096, N 2048: gate_up 228 us =
// 5.0 TB/s.  bf16, 64 experts x 9 rows, K 2048: gate_up 112 us = 4.8 TB/s,
// down 46 us = 5.8 TB/s.  INT4, 128 experts x 1 row, K 4096, N 1024: gate_up
// 97 us = 5.7 TB/s.  32 experts x 512 rows, K = N = 2880 MXFP4: gate_up 680
// us = 0.80 PFLOP/s, down (two planes) 625 us = 0.87.  1000 tokens of the
// layer (128 experts, top-4, K = N = 2880, Zipf(1.1) popularity): gate_up 676
// -> 341 us, down 596 -> 232 us against the 128-row tile kernel (gemm.hip).
#include "gemm_wreg.hpp"

#include "dispatch_one.hpp"
#include "topk.hpp"

#include <algorithm>
#include <utility>

namespace grim {

typedef __bf16 bf16x8 __attribute__((__vector_size__(8 * sizeof(__bf16))));
typedef __bf16 bf16x2v __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void* wreg_lds_ptr_t;

constexpr int kWregThreads = 256;
constexpr int kWregWaves = 4;
constexpr int kWregNoLoad = int(0x80000000u);

// RB: 16-row weight blocks per wave; STB: LDS bytes of one activation stage;
// WG: work-groups per CU the registers are limited for.  INT4 batches have
// few rows per expert and few experts, so their tiles are half as wide
// (twice the work-groups) and one row block deep, which leaves registers for
// 16 waves a CU: its decoding is bound by instruction issue at 8 (64 experts
// x 1 row, K 2048: 52 -> 28 us).
template <int F> struct WregFmt;
template <> struct WregFmt<GRIM_FMT_MXFP4> {
    static constexpr int SEGK = 128, J = 4, RB = 4, STB = 32768, WG = 2;
    static constexpr bool kInt4 = false;
};
template <> struct WregFmt<GRIM_FMT_INT4> {
    static constexpr int SEGK = 128, J = 4, RB = 2, STB = 16384, WG = 4;
    static constexpr bool kInt4 = true;
};
template <> struct WregFmt<GRIM_FMT_INT4_F16> : WregFmt<GRIM_FMT_INT4> {};
template <> struct WregFmt<GRIM_FMT_BF16> {
    static constexpr int SEGK = 32, J = 1, RB = 4, STB = 32768, WG = 2;
    static constexpr bool kInt4 = false;
};

// Segments per stage: what the LDS stage and the registers hold (an item
// of 8 row blocks keeps 128 accumulators: one segment of 4-bit weights).
template <int F> constexpr int wreg_sp(int nt, int pl) {
    return WregFmt<F>::SEGK == 128 ? (nt * pl >= 8 ? 1 : 2) : (nt >= 8 ? 1 : nt >= 4 ? 2 : 4);
}

template <int... I, class Fn>
__device__ __forceinline__ void static_for_impl(std::integer_sequence<int, I...>, Fn&& f) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class Fn>
__device__ __forceinline__ void static_for(Fn&& f) {
    static_for_impl(std::make_integer_sequence<int, N>{}, std::forward<Fn>(f));
}

// One fragment from LDS byte address addr + OFF; the caller waits.
template <int OFF>
__device__ __forceinline__ void wreg_dsr(u32x4& v, uint32_t addr) {
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "n"(OFF));
}

__device__ __forceinline__ bf16x8 as_bf16x8(u32x4 v) {
    bf16x8 r;
    __builtin_memcpy(&r, &v, 16);
    return r;
}

// The operand of MFMA step j from a lane's 16 weight bytes.
template <int F>
__device__ __forceinline__ bf16x8 wreg_frag(u32x4 raw, float s, int j) {
    if constexpr (F == GRIM_FMT_BF16) {
        return as_bf16x8(raw);
    } else if constexpr (F == GRIM_FMT_MXFP4) {
        const uint32_t w = raw[j];
        const bf16x2v v[4] = {__builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, s, 0),
                              __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, s, 1),
                              __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, s, 2),
                              __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, s, 3)};
        bf16x8 r;
        __builtin_memcpy(&r, v, 16);
        return r;
    } else {
        // pairs (k, k + 4) of the word's eight codes: 16 + q each
        const uint32_t w = raw[j];
        // (both constants in vector registers: one v_bfi_b32 takes one scalar)
        uint32_t m = 0x00780078u, e = 0x41804180u;
        asm("" : "+v"(m), "+v"(e));
        u32x4 o;
        o[0] = (m & (w << 3)) | (~m & e);
        o[1] = (m & (w >> 1)) | (~m & e);
        o[2] = (m & (w >> 5)) | (~m & e);
        o[3] = (m & (w >> 9)) | (~m & e);
        return as_bf16x8(o);
    }
}

// What a tile of rows and a column tile of one expert need.
struct WregItem {
    int64_t wrow0;    // first weight row of the expert's block
    int r0, rows;     // first activation / output row, live rows
    int col;          // column tile
    bool sh;
};

template <int F, bool GU, int NT, int PL, bool HZ>
__device__ __forceinline__ void wreg_tile(const WregArgs& a, const WregItem& it, int planes, uint8_t* lds) {
    using T = WregFmt<F>;
    constexpr int SEGK = T::SEGK, J = T::J, RB = T::RB;
    constexpr int SP = wreg_sp<F>(NT, PL);
    constexpr int RBY = SP * SEGK * 2;                 // stage bytes of one activation row and plane
    constexpr int SL = RBY / 16;                       // its 16-byte slots
    constexpr int PLB = NT * 16 * RBY;                 // bytes of one plane
    constexpr int NI = PL * PLB / 1024 / kWregWaves;   // DMA instructions per wave and stage
    static_assert(PL * PLB <= T::STB && NI * kWregWaves * 1024 == PL * PLB, "stage");
    constexpr int NG = NT < 4 ? NT : NT == 8 ? 2 : 4;  // row blocks per read unit (registers)
    constexpr int NU = PL * (NT / NG);                 // units per step
    const int tid = threadIdx.x, lane = tid & 63, c = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int K = a.K, N = a.N;
    const WView& w = it.sh ? a.w_sh : a.w;
    const int Kp = (K + SEGK - 1) / SEGK * SEGK;
    const int64_t astride = int64_t(planes) * Kp * 2;  // bytes of an activation row
    const bool gather = GU && !it.sh;
    const int64_t a_rows = it.sh ? a.a_rows_sh : a.a_rows;
    const int64_t a_base = gather ? 0 : int64_t(it.r0) * astride;
    const int64_t a_left = a_rows * astride - a_base;
    const __amdgpu_buffer_rsrc_t rA = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<char*>(reinterpret_cast<const char*>(it.sh ? a.A_sh : a.A) + a_base), 0,
        int(a_left < 0x7FFFFFFF ? a_left : 0x7FFFFFFF), 0x00020000);
    const int slab = GU ? 2 * N : N;
    const __amdgpu_buffer_rsrc_t rW = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(w.payload + it.wrow0 * w.row_bytes), 0, int(slab * w.row_bytes), 0x00020000);
    constexpr int SB = F == GRIM_FMT_MXFP4 ? 1 : T::kInt4 ? 2 : 0;
    const __amdgpu_buffer_rsrc_t rS = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(static_cast<const uint8_t*>(w.scales) + it.wrow0 * w.row_scales * SB), 0,
        slab * w.row_scales * SB, 0x00020000);
    const __amdgpu_buffer_rsrc_t rZ = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(HZ ? w.zeros + it.wrow0 * w.row_scales : w.payload), 0, HZ ? slab * w.row_scales : 0,
        0x00020000);

    // weight rows of this wave (GU: two blocks of gate rows, the matching up rows)
    int woff[RB], soff[RB];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
        const int i = GU ? (it.col * kWregWaves + wave) * (RB * 8) + rb % (RB / 2) * 16 + c
                         : (it.col * kWregWaves + wave) * (RB * 16) + rb * 16 + c;
        const int row = (GU && rb >= RB / 2 ? N : 0) + (i < N ? i : N - 1);
        woff[rb] = row * int(w.row_bytes) + g * 16;
        soff[rb] = row * w.row_scales * SB;
    }
    // activation rows: DMA instruction ii of this wave fills stage bytes
    // [(wave NI + ii) 1024, + 1024), 16 bytes a lane: [plane][row][slot],
    // slot p of row t holding piece p ^ swz(t)
    auto swz = [](int t) { return SL >= 16 ? (t & 15) : SL == 8 ? (t & 7) : ((t >> 1) & 3); };
    int aoff[NI];
#pragma unroll
    for (int ii = 0; ii < NI; ++ii) {
        const int o = (wave * NI + ii) * 1024 + lane * 16;
        const int p = o / PLB, t = o % PLB / RBY, sl = o % RBY / 16;
        int rr = t < it.rows ? t : 0;
        if (gather) rr = a.map[it.r0 + rr];
        aoff[ii] = rr * int(astride) + p * Kp * 2 + (sl ^ swz(t)) * 16;
    }
    // fragment addresses: step j (4-bit) or segment s (bf16) picks the entry
    constexpr int NFO = J > 1 ? J : SP;
    uint32_t fo[NFO];
    const uint32_t lb = uint32_t(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) uint8_t*)(lds)));
#pragma unroll
    for (int q = 0; q < NFO; ++q) {
        const int slot = J > 1 ? g * J + q : q * 4 + g;
        fo[q] = lb + uint32_t(c * RBY + (slot ^ swz(c)) * 16);
    }

    struct Stage {
        u32x4 b[SP][RB];
    };
    const int nstg = (K + SP * SEGK - 1) / (SP * SEGK);
    // Side scales in chunks of 16 segments (2048 K): lane group g holds the
    // scales (and zero points) of segments 4 g + [0, 4) of its column's row,
    // so that a row's scales are whole 64-byte (MXFP4) pieces read once,
    // not a line per row touched at every stage: those lines, one per weight
    // row in flight, do not stay in the L2 (MXFP4, K 2880: 1.42x the weight
    // bytes fetched that way).  A window that would pass the row's end
    // starts `late` bytes early (settle), so none straddles the tensor's end.
    constexpr int CW = F == GRIM_FMT_MXFP4 ? 16 : T::kInt4 ? 8 : 0;   // window bytes per lane
    struct Side {
        uint32_t s[CW ? RB : 1][CW ? CW / 4 : 1];
        uint32_t z[T::kInt4 ? RB : 1];
    };
    Side side, next;
    int chunk = -1, chunk_n = -1;        // the chunks in side and next
    const int srow = w.row_scales * SB;  // scale bytes per row
    // stage st's activations into LDS buffer buf (stages past the last load nothing)
    auto load_a = [&](int st, int buf) __attribute__((always_inline)) {
        const int dead = st >= nstg ? kWregNoLoad : 0;
#pragma unroll
        for (int ii = 0; ii < NI; ++ii)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                rA, (wreg_lds_ptr_t)(lds + buf * T::STB + (wave * NI + ii) * 1024), 16, aoff[ii] | dead,
                st * RBY, 0, 0);
    };
    // stage st's weights (K past the row's end reads as zero), and its
    // chunk of scales when that is not the one at hand
    auto load_w = [&](Stage& S, int st) __attribute__((always_inline)) {
        // (row blocks outermost: the segments of a row one after the other, so
        // that the pieces of a memory line are requested together: MXFP4, 128
        // experts x 8 rows, K = N = 2880: 286 -> 259 us; K 4096, N 2048: 245
        // -> 228)
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
#pragma unroll
            for (int s = 0; s < SP; ++s) {
                const int seg = st * SP + s;
                const bool in = seg * SEGK + g * (SEGK / 4) < K;
                S.b[s][rb] = __builtin_amdgcn_raw_buffer_load_b128(rW, in ? woff[rb] : kWregNoLoad, seg * 64, 0);
            }
        if constexpr (CW != 0) {
            const int ch = st * SP / 16;
            if (st < nstg && ch != chunk_n) {   // uniform
                chunk_n = ch;
                const int at = min(ch * 4 * CW + g * CW, srow - CW);
#pragma unroll
                for (int rb = 0; rb < RB; ++rb) {
                    if constexpr (CW == 16) {
                        const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(rS, soff[rb] + at, 0, 0);
#pragma unroll
                        for (int q = 0; q < 4; ++q) next.s[rb][q] = v[q];
                    } else {
                        const auto v = __builtin_amdgcn_raw_buffer_load_b64(rS, soff[rb] + at, 0, 0);
                        next.s[rb][0] = v[0]; next.s[rb][1] = v[1];
                        if constexpr (HZ)
                            next.z[rb] = __builtin_amdgcn_raw_buffer_load_b32(
                                rZ, (soff[rb] >> 1) + min(ch * 16 + g * 4, w.row_scales - 4), 0, 0);
                    }
                }
            }
        }
    };
    // chunk ch becomes the one at hand, late windows moved to where the
    // others have their scales (bytes past the row become 0)
    auto settle = [&](int ch) __attribute__((always_inline)) {
        if constexpr (CW != 0) {
            if (ch == chunk) return;   // uniform
            chunk = ch;
            const int late = max(0, ch * 4 * CW + g * CW - (srow - CW));
#pragma unroll
            for (int rb = 0; rb < RB; ++rb) {
#pragma unroll
                for (int i = 0; i < CW / 4; ++i) {
                    uint32_t lo = 0, hi = 0;
#pragma unroll
                    for (int q = i; q < CW / 4; ++q) {
                        lo = q == i + (late >> 2) ? next.s[rb][q] : lo;
                        hi = q == i + (late >> 2) + 1 ? next.s[rb][q] : hi;
                    }
                    side.s[rb][i] = __builtin_amdgcn_alignbyte(hi, lo, late & 3);
                }
                // (late counts two bytes per group)
                if constexpr (HZ) side.z[rb] = late >= 8 ? 0u : next.z[rb] >> (late * 4);
            }
        }
    };
    // b where the uniform bit is set, else a (not a select: that would turn
    // the registers of side into an indexed array)
    auto pick = [](int bit, uint32_t a, uint32_t b) __attribute__((always_inline)) {
        const uint32_t m = bit ? ~0u : 0u;
        return (m & b) | (~m & a);
    };
    // the dword of side that holds segment seg's scales, from the lane group that has it
    auto from = [&](int seg, uint32_t v) __attribute__((always_inline)) {
        return uint32_t(__builtin_amdgcn_ds_bpermute((((seg >> 2) & 3) * 16 + c) * 4, int(v)));
    };

    f32x4 acc[RB][NT];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) acc[rb][nt] = f32x4{0.f, 0.f, 0.f, 0.f};

    // the products of stage st (weights S, activations in buffer BUF)
    auto compute = [&](Stage& S, int st, auto bufc) __attribute__((always_inline)) {
        constexpr int BUF = decltype(bufc)::value;
        static_for<SP>([&](auto sc) __attribute__((always_inline)) {
            constexpr int s = decltype(sc)::value;
            if ((st * SP + s) * SEGK >= K) return;     // uniform
            f32x4 gacc[T::kInt4 ? RB : 1][T::kInt4 ? NT : 1], sx[T::kInt4 ? NT : 1];
            const int seg = st * SP + s;
            float sb[RB];           // MXFP4: the scale of this lane's 32 elements; INT4: the group's
            float zoff[RB];         // INT4: -(16 + zero point)
            if constexpr (F == GRIM_FMT_MXFP4) {
#pragma unroll
                for (int rb = 0; rb < RB; ++rb) {
                    const uint32_t lo = pick(seg & 1, side.s[rb][0], side.s[rb][1]);
                    const uint32_t hi = pick(seg & 1, side.s[rb][2], side.s[rb][3]);
                    const uint32_t v = pick(seg & 2, lo, hi);
                    sb[rb] = e8m0_to_f32(uint8_t(from(seg, v) >> (8 * g)));
                }
            }
            if constexpr (T::kInt4) {
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) {
                    sx[nt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int rb = 0; rb < RB; ++rb) gacc[rb][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
                }
#pragma unroll
                for (int rb = 0; rb < RB; ++rb) {
                    const uint32_t v = from(seg, pick(seg & 2, side.s[rb][0], side.s[rb][1]));
                    const uint16_t sr = uint16_t(v >> (16 * (seg & 1)));
                    sb[rb] = F == GRIM_FMT_INT4 ? bf16_to_f32(sr) : f16_to_f32(sr);
                    if constexpr (HZ) {
                        // signed codes (zero point byte 0xFF): xor 8 makes
                        // them offset binary with zero point 8
                        const uint32_t z = (from(seg, side.z[rb]) >> (8 * (seg & 3))) & 0xFFu;
                        const uint32_t flip = z == 0xFFu ? 0x88888888u : 0u;
                        zoff[rb] = -float(16u + (z == 0xFFu ? 8u : z));
#pragma unroll
                        for (int q = 0; q < 4; ++q) S.b[s][rb][q] ^= flip;
                    } else {
                        zoff[rb] = -float(16 + w.default_zero);
                    }
                }
            }
            u32x4 fa[2][NG];
            auto reads = [&](auto uc) __attribute__((always_inline)) {
                constexpr int u = decltype(uc)::value;
                constexpr int j = u / NU, p = u % NU / (NT / NG), q0 = u % (NT / NG);
                static_for<NG>([&](auto ic) __attribute__((always_inline)) {
                    constexpr int i = decltype(ic)::value;
                    constexpr int OFF = BUF * T::STB + p * PLB + (q0 * NG + i) * 16 * RBY +
                                        (J > 1 ? s * SEGK * 2 : 0);
                    wreg_dsr<OFF>(fa[u & 1][i], fo[J > 1 ? j : s]);
                });
            };
            bf16x8 fb[RB];
            reads(std::integral_constant<int, 0>{});
            static_for<J * NU>([&](auto uc) __attribute__((always_inline)) {
                constexpr int u = decltype(uc)::value;
                constexpr int j = u / NU, q0 = u % (NT / NG);
                constexpr bool more = u + 1 < J * NU;
                if constexpr (more) reads(std::integral_constant<int, more ? u + 1 : 0>{});
                if constexpr (u % NU == 0) {
#pragma unroll
                    for (int rb = 0; rb < RB; ++rb) fb[rb] = wreg_frag<F>(S.b[s][rb], sb[rb], j);
                }
                // this unit's reads are in once only the next unit's are left
                if constexpr (NG == 1)
                    asm volatile("s_waitcnt lgkmcnt(%1)" : "+v"(fa[u & 1][0]) : "n"(more ? NG : 0));
                else if constexpr (NG == 2)
                    asm volatile("s_waitcnt lgkmcnt(%2)" : "+v"(fa[u & 1][0]), "+v"(fa[u & 1][1]) : "n"(more ? NG : 0));
                else
                    asm volatile("s_waitcnt lgkmcnt(%4)"
                                 : "+v"(fa[u & 1][0]), "+v"(fa[u & 1][1]), "+v"(fa[u & 1][2]), "+v"(fa[u & 1][3])
                                 : "n"(more ? NG : 0));
#pragma unroll
                for (int i = 0; i < NG; ++i) {
                    const bf16x8 av = as_bf16x8(fa[u & 1][i]);
#pragma unroll
                    for (int rb = 0; rb < RB; ++rb) {
                        f32x4& d = T::kInt4 ? gacc[T::kInt4 ? rb : 0][T::kInt4 ? q0 * NG + i : 0] : acc[rb][q0 * NG + i];
                        d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, fb[rb], d, 0, 0, 0);
                    }
                    if constexpr (T::kInt4) {
                        const u32x4 one = {0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u};
                        sx[q0 * NG + i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, as_bf16x8(one), sx[q0 * NG + i], 0, 0, 0);
                    }
                }
            });
            if constexpr (T::kInt4) {
#pragma unroll
                for (int rb = 0; rb < RB; ++rb) {
#pragma unroll
                    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                        for (int v = 0; v < 4; ++v)
                            acc[rb][nt][v] = __builtin_fmaf(sb[rb], __builtin_fmaf(zoff[rb], sx[nt][v], gacc[rb][nt][v]), acc[rb][nt][v]);
                }
            }
        });
    };
    // The stage's activations of this wave have landed (all but the NW
    // weight loads issued after them; loads return in order), then every
    // wave's.  The weights stay in flight until their first use.
    // (a chunk of scales after them only makes the wait stricter)
    constexpr int NW = SP * RB;
    static_assert(NW <= 63, "vmcnt holds 63");
    auto turn = [&]() __attribute__((always_inline)) {
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(NW) : "memory");
    };
    // keeps a stage's weight loads behind its activation loads
    auto order = []() __attribute__((always_inline)) { asm volatile("" ::: "memory"); };

    // Rows a power of two apart put every row's bytes at one K in the same
    // few memory channels: there the K walk starts at a stage of its own per
    // column tile, so that work-groups in step do not all queue on them (bf16
    // rows of 4096 bytes: 129 -> 109 us; rows of 1440 bytes are spread
    // already and lose the A rows' locality: 322 -> 329 us).
    const int k0 = w.row_bytes % 1024 ? 0 : it.col % nstg;
    auto at = [&](int i) { return i >= nstg ? nstg : i + k0 >= nstg ? i + k0 - nstg : i + k0; };
    Stage S0, S1;
    load_w(S0, at(0));
    load_a(at(0), 0);
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
    for (int i = 0; i < nstg; i += 2) {
        settle(at(i) * SP / 16);
        load_a(at(i + 1), 1);
        order();
        load_w(S1, at(i + 1));
        compute(S0, at(i), std::integral_constant<int, 0>{});
        turn();
        if (i + 1 < nstg) settle(at(i + 1) * SP / 16);
        load_a(at(i + 2), 0);
        order();
        load_w(S0, at(i + 2));
        compute(S1, at(i + 1), std::integral_constant<int, 1>{});   // no segments past the last stage
        turn();
    }

    // ---- results: lane (c, g) holds rows 4 g + v of each 16-row block, at
    // its weight row; rows past the tile's fall outside the buffers
    if constexpr (GU) {
        const int Ip = (N + SEGK - 1) / SEGK * SEGK;
        const __amdgpu_buffer_rsrc_t rO = __builtin_amdgcn_make_buffer_rsrc(
            (it.sh ? a.h_sh : a.h) + int64_t(it.r0) * 2 * Ip, 0, it.rows * 4 * Ip, 0x00020000);
#pragma unroll
        for (int rb = 0; rb < RB / 2; ++rb) {
            const int i = (it.col * kWregWaves + wave) * (RB * 8) + rb * 16 + c;
            // INT4: the order of the decoder's pairs within eight
            const int pos = T::kInt4 ? (i & ~7) | ((i & 3) << 1) | ((i >> 2) & 1) : i;
            const int off = i < Ip ? pos * 2 : kWregNoLoad;
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const float hv = i < N ? fast_silu(acc[rb][nt][v]) * acc[rb + RB / 2][nt][v] : 0.0f;
                    const uint16_t hi = f32_to_bf16(hv);
                    const int o = off + (nt * 16 + 4 * g + v) * 4 * Ip;
                    __builtin_amdgcn_raw_buffer_store_b16(hi, rO, o, 0, 0);
                    __builtin_amdgcn_raw_buffer_store_b16(f32_to_bf16(hv - bf16_to_f32(hi)), rO, o, 2 * Ip, 0);
                }
        }
    } else {
        const __amdgpu_buffer_rsrc_t rO = __builtin_amdgcn_make_buffer_rsrc(
            (it.sh ? a.y_sh : a.y) + int64_t(it.r0) * N, 0, it.rows * N * 4, 0x00020000);
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) {
            const int n = (it.col * kWregWaves + wave) * (RB * 16) + rb * 16 + c;
            const int off = n < N ? n * 4 : kWregNoLoad;
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    __builtin_amdgcn_raw_buffer_store_b32(f_bits(acc[rb][nt][v]), rO, off + (nt * 16 + 4 * g + v) * N * 4, 0, 0);
        }
    }
}

// One work-group per (row tile, column tile); the grid covers the bound of
// the tile count and work-groups past the live tiles end at once.
template <int F, bool GU>
__global__ __launch_bounds__(kWregThreads, WregFmt<F>::WG) void grouped_wreg_kernel(WregArgs a, int ncols) {
    __shared__ __attribute__((aligned(1024))) uint8_t lds[2 * WregFmt<F>::STB];
    constexpr bool kInt4 = WregFmt<F>::kInt4;
    constexpr int MC = wreg_mc(F, GU);
    const int ty = blockIdx.x / ncols;
    // (uniform values kept in scalar registers: buffer descriptors are
    // built from them)
    const int live = __builtin_amdgcn_readfirstlane(*a.n_live);
    WregItem it;
    it.col = blockIdx.x % ncols;
    if (ty < live) {
        const TileDesc d = a.tiles[ty];
        it.r0 = __builtin_amdgcn_readfirstlane(d.r0);
        it.rows = __builtin_amdgcn_readfirstlane(d.rows);
        it.wrow0 = int64_t(__builtin_amdgcn_readfirstlane(d.e)) * (GU ? 2 * a.N : a.N);
        it.sh = false;
        // work-groups are dealt over the eight XCDs: the tiles of an expert
        // read the same weight rows through the same L2
        it.col = (it.col + __builtin_amdgcn_readfirstlane(d.mb) * ncols % 8) % ncols;
    } else {
        it.r0 = (ty - live) * MC;
        it.rows = min(MC, a.T_sh - it.r0);
        it.wrow0 = 0;
        it.sh = true;
    }
    if (it.rows <= 0) return;
    const int planes = GU && !kInt4 ? 1 : 2;
    if constexpr (kInt4) {
        const bool hz = (it.sh ? a.w_sh : a.w).zeros != nullptr;
        bool two = true;
        if constexpr (GU) {
            // both halves of x only where some row of the tile has a low half
            const int t = int(threadIdx.x) & 63;
            int lo = 0;
            if (t < it.rows) lo = a.a_lo[it.sh ? it.r0 + t : a.map[it.r0 + t]];
            two = __ballot(lo != 0) != 0;
            if (!two) {
                if (hz) wreg_tile<F, GU, 1, 1, true>(a, it, planes, lds);
                else wreg_tile<F, GU, 1, 1, false>(a, it, planes, lds);
            }
        }
        if (two) {
            if (hz) wreg_tile<F, GU, 1, 2, true>(a, it, planes, lds);
            else wreg_tile<F, GU, 1, 2, false>(a, it, planes, lds);
        }
    } else if constexpr (GU) {
        if (it.rows <= 16) wreg_tile<F, GU, 1, 1, false>(a, it, planes, lds);
        else if (it.rows <= 32) wreg_tile<F, GU, 2, 1, false>(a, it, planes, lds);
        else if (it.rows <= 64) wreg_tile<F, GU, 4, 1, false>(a, it, planes, lds);
        else wreg_tile<F, GU, 8, 1, false>(a, it, planes, lds);
    } else {
        if (it.rows <= 16) wreg_tile<F, GU, 1, 2, false>(a, it, planes, lds);
        else if (it.rows <= 32) wreg_tile<F, GU, 2, 2, false>(a, it, planes, lds);
        else wreg_tile<F, GU, 4, 2, false>(a, it, planes, lds);
    }
}

// One x row as bf16 planes in the order the weights decode to, K padded
// with zeros.
template <bool INT4>
__device__ __forceinline__ void wreg_format_row(const float* __restrict__ x, int t, int H, int Kp,
                                                uint16_t* __restrict__ dst, int32_t* __restrict__ lo) {
    const float* xr = x + int64_t(t) * H;
    uint16_t* d = dst + int64_t(t) * (INT4 ? 2 : 1) * Kp;
    int any = 0;
    for (int k = threadIdx.x * 8; k < Kp; k += blockDim.x * 8) {
        float v[8];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const float4 f = k < H ? *reinterpret_cast<const float4*>(xr + k + 4 * q) : make_float4(0.f, 0.f, 0.f, 0.f);
            v[4 * q] = f.x; v[4 * q + 1] = f.y; v[4 * q + 2] = f.z; v[4 * q + 3] = f.w;
        }
        uint16_t hi[8], lw[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            hi[i] = f32_to_bf16(v[i]);
            lw[i] = f32_to_bf16(v[i] - bf16_to_f32(hi[i]));
            any |= lw[i] & 0x7FFF;
        }
        u32x4 a, b;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int e0 = INT4 ? i : 2 * i, e1 = INT4 ? i + 4 : 2 * i + 1;
            a[i] = uint32_t(hi[e0]) | (uint32_t(hi[e1]) << 16);
            b[i] = uint32_t(lw[e0]) | (uint32_t(lw[e1]) << 16);
        }
        *reinterpret_cast<u32x4*>(d + k) = a;
        if constexpr (INT4) *reinterpret_cast<u32x4*>(d + Kp + k) = b;
    }
    if constexpr (INT4) {
        const int r = __syncthreads_or(any);
        if (threadIdx.x == 0) lo[t] = r ? 1 : 0;
    }
}

// Work-group 0 (`route`): the top-k of up to 16 tokens, one wave each
// (topk_kernel's code, so the same bits; more tokens would share one CU),
// and the dispatch; the other work-groups format one token row each
// meanwhile.  One launch of 9.0 us for 16 tokens x top-4 where top-k, four
// dispatch launches and the formatting took 27.
template <bool INT4>
__global__ __launch_bounds__(kOneThreads) void wreg_route_kernel(const float* x, int H, int Kp, uint16_t* dst,
                                                                 int32_t* lo, TopkArgs tk, OneArgs oa, int route,
                                                                 int topk) {
    struct TopkLds {
        float gsel[kOneWaves][512];
        float gscore[kOneWaves][64];
        int32_t e[kOneWaves][16];
        float w[kOneWaves][16];
    };
    __shared__ union { OneLds one; TopkLds tk; } lds;
    if (int(blockIdx.x) >= route) {
        wreg_format_row<INT4>(x, int(blockIdx.x) - route, H, Kp, dst, lo);
        return;
    }
    if (!topk) {
        dispatch_one_block(oa, lds.one, [&](int r) { return tk.out_e[r]; });
        return;
    }
    const int wv = threadIdx.x / kWave, R = tk.T * tk.K;
    if (wv < tk.T)
        topk_wave(tk.logits + int64_t(wv) * tk.E, tk.E, tk.K, tk.mode, tk.normalize, tk.scaling, tk.bias16, tk.bias32,
                  tk.n_group, tk.topk_group, lds.tk.e[wv], lds.tk.w[wv], lds.tk.gsel[wv], lds.tk.gscore[wv]);
    __syncthreads();
    // (at most 16 tokens x 16 picks: one route per thread of the first waves)
    const int r = threadIdx.x;
    int pe = -1;
    if (r < R) {
        pe = lds.tk.e[r / tk.K][r % tk.K];
        tk.out_e[r] = pe;
        tk.out_w[r] = lds.tk.w[r / tk.K][r % tk.K];
    }
    __syncthreads();
    // with R <= 1024 the dispatch asks each thread for its own route only
    dispatch_one_block(oa, lds.one, [&](int) { return pe; });
}

static bool is_int4(int fmt) { return fmt == GRIM_FMT_INT4 || fmt == GRIM_FMT_INT4_F16; }

int wreg_kpad(int fmt, int K) {
    const int s = fmt == GRIM_FMT_BF16 ? 32 : 128;
    return (K + s - 1) / s * s;
}

int wreg_x_planes(int fmt) { return is_int4(fmt) ? 2 : 1; }

bool wreg_weight_ok(const grim_quant_weight& w, int rows_per_expert, int K) {
    if (K % 64) return false;
    const int64_t bits = w.fmt == GRIM_FMT_BF16 ? 16 : 4;
    if (w.row_bytes < K * bits / 8 || w.row_bytes % 16) return false;
    // 32-bit offsets inside an expert's block
    if (w.row_bytes * rows_per_expert >= 0x7FFFFFFF || int64_t(w.row_scales) * 2 * rows_per_expert >= 0x7FFFFFFF)
        return false;
    switch (w.fmt) {
    case GRIM_FMT_BF16: return true;
    case GRIM_FMT_MXFP4: return K >= 512 &&   // a 16-byte window
        w.row_scales >= K / 32;
    case GRIM_FMT_INT4:
    case GRIM_FMT_INT4_F16:
        // one scale group per 128-K segment, a window of four
        return K % 128 == 0 && K >= 512 && w.row_scales == K / 128;
    }
    return false;
}

bool wreg_one_dispatch(int T, int K, int E) { return int64_t(T) * K <= kOneMaxRoutes && E <= kOneMaxE; }
bool wreg_one_topk(int T) { return T <= kOneWaves; }

hipError_t wreg_route_launch(hipStream_t st, int fmt, const float* x, int H, uint16_t* dst, int32_t* lo,
                             const TopkArgs& tk, const DispatchArgs* d, bool topk) {
    if (tk.T <= 0) return hipSuccess;
    if (d && !wreg_one_dispatch(d->T, d->K, d->E)) return hipErrorInvalidValue;
    if (topk && (!d || !wreg_one_topk(tk.T) || tk.K > 16 || tk.E > 512 || tk.part1)) return hipErrorInvalidValue;
    OneArgs oa{};
    if (d)
        oa = OneArgs{d->T * d->K, d->E, d->K, d->counts, d->offsets, d->inverse, d->perm_token, d->lists,
                     nullptr, nullptr, 0, 0, nullptr};
    const int Kp = wreg_kpad(fmt, H), route = d ? 1 : 0;
    const dim3 grid(tk.T + route), block(d ? kOneThreads : 256);
    if (is_int4(fmt))
        hipLaunchKernelGGL(wreg_route_kernel<true>, grid, block, 0, st, x, H, Kp, dst, lo, tk, oa, route, int(topk));
    else
        hipLaunchKernelGGL(wreg_route_kernel<false>, grid, block, 0, st, x, H, Kp, dst, lo, tk, oa, route, int(topk));
    return hipGetLastError();
}

template <int F>
static hipError_t wreg_launch_fmt(hipStream_t st, const WregArgs& a, bool gate_up) {
    constexpr int CW = kWregWaves * WregFmt<F>::RB * 16;   // weight rows per column tile
    const int ncols = gate_up ? (a.N + CW / 2 - 1) / (CW / 2) : (a.N + CW - 1) / CW;
    const int mc = wreg_mc(F, gate_up);
    const int64_t tiles = int64_t(a.max_tiles) + (a.T_sh + mc - 1) / mc;
    if (tiles <= 0 || ncols <= 0) return hipSuccess;
    if (tiles * ncols >= 0x7FFFFFFF) return hipErrorInvalidValue;
    const dim3 grid(unsigned(tiles * ncols));
    if (gate_up)
        hipLaunchKernelGGL((grouped_wreg_kernel<F, true>), grid, dim3(kWregThreads), 0, st, a, ncols);
    else
        hipLaunchKernelGGL((grouped_wreg_kernel<F, false>), grid, dim3(kWregThreads), 0, st, a, ncols);
    return hipGetLastError();
}

hipError_t wreg_launch(hipStream_t st, int fmt, const WregArgs& a, bool gate_up) {
    switch (fmt) {
    case GRIM_FMT_BF16: return wreg_launch_fmt<GRIM_FMT_BF16>(st, a, gate_up);
    case GRIM_FMT_MXFP4: return wreg_launch_fmt<GRIM_FMT_MXFP4>(st, a, gate_up);
    case GRIM_FMT_INT4: return wreg_launch_fmt<GRIM_FMT_INT4>(st, a, gate_up);
    case GRIM_FMT_INT4_F16: return wreg_launch_fmt<GRIM_FMT_INT4_F16>(st, a, gate_up);
    }
    return hipErrorInvalidValue;
}

}  // namespace grim

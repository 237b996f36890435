// Device building blocks of the search, executed by a "group" of 32 lanes (half of a wave64; two groups per wave):
// the float forward transform, dead-zone quantizer, distortion and exact coefficient rate of one transform block,
// intra edge preparation and SATD.
//
// Arithmetic contract (shared with the CPU oracle, bit for bit): every forward-transform output is one fmaf chain in
// ascending k; sums over coefficients run on 32 virtual lanes (lane l takes elements l, l + 32, ... in order) combined
// by the xor butterfly 16, 8, 4, 2, 1; J = fmaf(lambda, bits, D).  Which physical lane computes a chain does not
// change a value, so the passes spread their chains over the group freely.
#pragma once
#include <type_traits>
#include <cstddef>
#include "av1m_common.h"

namespace av1m {

constexpr int GW = 32;   // lanes per group

constexpr int tx_of(int W, int H) {
    return W == H ? (W == 4 ? TX_4X4 : W == 8 ? TX_8X8 : W == 16 ? TX_16X16 : W == 32 ? TX_32X32 : TX_64X64)
         : (W == 4 && H == 8) ? TX_4X8 : (W == 8 && H == 4) ? TX_8X4 : (W == 8 && H == 16) ? TX_8X16 : (W == 16 && H == 8) ? TX_16X8
         : (W == 16 && H == 32) ? TX_16X32 : (W == 32 && H == 16) ? TX_32X16 : (W == 32 && H == 64) ? TX_32X64
         : (W == 64 && H == 32) ? TX_64X32 : (W == 4 && H == 16) ? TX_4X16 : (W == 16 && H == 4) ? TX_16X4
         : (W == 8 && H == 32) ? TX_8X32 : (W == 32 && H == 8) ? TX_32X8 : (W == 16 && H == 64) ? TX_16X64 : TX_64X16;
}

// global memory seen through its own address space: a generic pointer read back from LDS would go through flat
// instructions, which wait on the LDS counter too
template <typename T> using glb = __attribute__((address_space(1))) T;
// LDS view of a type: accesses through it compile to ds_* instructions, also inside functions the compiler keeps out
// of line (where a plain pointer would lose its address space and go through flat instructions)
template <typename T> using lds = __attribute__((address_space(3))) T;
// read-only global data seen through the constant address space: wave-uniform indices load through the scalar unit
template <typename T> using cst = __attribute__((address_space(4))) const T;
// the generic pointer to an LDS object (for library calls such as atomicAdd)
template <typename T> __device__ __forceinline__ T *gen(lds<T> *p) { return (T *)p; }
// p (the same value in every lane) as a wave-uniform constant-space pointer; pointers reach out-of-line functions in
// vector registers, so uniformity has to be restated for scalar loads
template <typename T> __device__ __forceinline__ cst<T> *uni(const T *p) {
    const uint64_t v = (uint64_t)p;
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return (cst<T> *)(((uint64_t)hi << 32) | lo);
}

// levels laid over the coefficients they come from: stores through this type may alias the float loads
typedef int16_t __attribute__((may_alias)) lev16;

__device__ __forceinline__ int glane() { return threadIdx.x & 31; }
__device__ __forceinline__ int gid() { return threadIdx.x >> 5; }
// the value of lane (this lane xor M) within the 32-lane group, every lane active, in vector registers only: M = 1, 2 by
// DPP quad permutes ([1,0,3,2], [2,3,0,1]), 4 as a mirror of 8 lanes (xor 7) and of 4 (xor 3), 8 as a rotation of the 16-lane
// row, 16 by swapping rows (v_permlane16_swap).  ds_swizzle, which reaches the same lanes, waits on the LDS unit each time.
template <int M>
__device__ __forceinline__ int lane_xor(int v) {
    static_assert(M == 1 || M == 2 || M == 4 || M == 8 || M == 16, "lane_xor: one lane bit of the 32-lane group");
    if constexpr (M == 1) return __builtin_amdgcn_update_dpp(0, v, 0xB1, 0xF, 0xF, false);
    else if constexpr (M == 2) return __builtin_amdgcn_update_dpp(0, v, 0x4E, 0xF, 0xF, false);
    else if constexpr (M == 4) return __builtin_amdgcn_update_dpp(0, __builtin_amdgcn_update_dpp(0, v, 0x141, 0xF, 0xF, false), 0x1B, 0xF, 0xF, false);
    else if constexpr (M == 8) return __builtin_amdgcn_update_dpp(0, v, 0x128, 0xF, 0xF, false);
    else {   // the pair after the swap: (even row's value, odd row's value) in every lane
        const auto p = __builtin_amdgcn_permlane16_swap((unsigned)v, (unsigned)v, false, false);
        return (int)((threadIdx.x & 16) ? p[0] : p[1]);
    }
}
template <int M>
__device__ __forceinline__ float lane_xorf(float v) { return __int_as_float(lane_xor<M>(__float_as_int(v))); }
template <int M>
__device__ __forceinline__ long long lane_xorl(long long v) {
    const unsigned lo = (unsigned)lane_xor<M>((int)(unsigned)(v & 0xFFFFFFFFll)), hi = (unsigned)lane_xor<M>((int)(v >> 32));
    return (long long)(((unsigned long long)hi << 32) | lo);
}
// orders the group's LDS accesses (one wave executes both groups in lockstep; this stops compiler reordering)
__device__ __forceinline__ void gsync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
// butterfly reductions over the 32 lanes of the group: partners lane xor 16, 8, 4, 2, 1 in that order, every lane ends
// with the result
__device__ __forceinline__ float gsum(float v) {
    v += lane_xorf<16>(v); v += lane_xorf<8>(v); v += lane_xorf<4>(v); v += lane_xorf<2>(v); v += lane_xorf<1>(v);
    return v;
}
__device__ __forceinline__ int gsumi(int v) {
    v += lane_xor<16>(v); v += lane_xor<8>(v); v += lane_xor<4>(v); v += lane_xor<2>(v); v += lane_xor<1>(v);
    return v;
}
__device__ __forceinline__ long long gsuml(long long v) {
    v += lane_xorl<16>(v); v += lane_xorl<8>(v); v += lane_xorl<4>(v); v += lane_xorl<2>(v); v += lane_xorl<1>(v);
    return v;
}
__device__ __forceinline__ int gmaxi(int v) {
    v = max(v, lane_xor<16>(v)); v = max(v, lane_xor<8>(v)); v = max(v, lane_xor<4>(v)); v = max(v, lane_xor<2>(v));
    v = max(v, lane_xor<1>(v));
    return v;
}
// index of the smallest (v, i) over the group, the lowest index among equal values; -1 if every v is INF
template <int M>
__device__ __forceinline__ void argmin_step(float &v, int &i) {
    const float ov = lane_xorf<M>(v);
    const int oi = lane_xor<M>(i);
    if (ov < v || (ov == v && oi < i)) { v = ov; i = oi; }
}
__device__ __forceinline__ int gargmin(float v, int i) {
    argmin_step<16>(v, i); argmin_step<8>(v, i); argmin_step<4>(v, i); argmin_step<2>(v, i); argmin_step<1>(v, i);
    return v < INF ? i : -1;
}

// inputs of one tx block evaluation; CP: pointer to the cost tables (global, or an LDS copy)
template <typename CP>
struct EvalInT {
    int txSz, txType, plane, dcQ, acQ, skipCtx, dcCtx, intraDir, bd;
    float dcRcp, acRcp;   // 1 / dcQ, 1 / acQ rounded to nearest
    float rnd, zbin, resEnergy;
    CP C;
};
using EvalIn = EvalInT<const CostTab *>;
struct EvalOut { float D, R; int eob; };

__device__ __forceinline__ int txsz_ctx(int t) { return (av1t::Tx_Size_Sqr[t] + av1t::Tx_Size_Sqr_Up[t] + 1) >> 1; }

// Indexes of the cost tables' entries of a transform-size context, tx size or plane kind: a table that holds one of them
// only (the analysis's LDS copy) has its own overloads that return 0.
template <typename CT> __device__ __forceinline__ int cost_i(const CT &, int i) { return i; }
// the eob position bits of an area class ms (16 << ms coefficients)
template <int MS, typename CT>
__device__ __forceinline__ float eob_pt_bits(const CT &C, int pt, int ec, int i) {
    return MS == 0 ? C.eob_pt16[pt][ec][i] : MS == 1 ? C.eob_pt32[pt][ec][i] : MS == 2 ? C.eob_pt64[pt][ec][i] : MS == 3 ? C.eob_pt128[pt][ec][i]
         : MS == 4 ? C.eob_pt256[pt][ec][i] : MS == 5 ? C.eob_pt512[pt][i] : C.eob_pt1024[pt][i];
}

// txb_skip, luma tx type and eob position bits of a tx block of size TSZ (no branch per lane: the terms that do not apply
// are read at clamped positions and dropped)
template <int TSZ, typename E>
__device__ __forceinline__ float base_bits(const E &e, int eob) {
    const auto &C = *e.C;
    constexpr int t = TSZ, ctx = txsz_ctx_of(t);
    const int pt = e.plane > 0;
    const float skip = C.txb_skip[cost_i(C, ctx)][e.skipCtx][eob == 0 ? 1 : 0];
    float b = skip;
    constexpr int set = tx_set_intra(t), sqr = av1t::Tx_Size_Sqr[t];
    if constexpr (set == TX_SET_INTRA_1) {
        int idx = 0;
#pragma unroll
        for (int i = 0; i < 7; i++) idx = av1t::Tx_Type_Intra_Inv_Set1[i] == e.txType ? i : idx;
        const float x = C.tx_set1[cost_i(C, sqr)][e.intraDir][idx];
        b += pt ? 0.f : x;
    } else if constexpr (set == TX_SET_INTRA_2) {
        int idx = 0;
#pragma unroll
        for (int i = 0; i < 5; i++) idx = av1t::Tx_Type_Intra_Inv_Set2[i] == e.txType ? i : idx;
        const float x = C.tx_set2[cost_i(C, sqr)][e.intraDir][idx];
        b += pt ? 0.f : x;
    }
    constexpr int lw = av1t::Tx_Width_Log2[t], lh = av1t::Tx_Height_Log2[t];
    constexpr int ms = (lw < 5 ? lw : 5) + (lh < 5 ? lh : 5) - 4;
    const int eobPt = eob <= 2 ? max(eob, 1) : 2 + (31 - __clz(eob - 1));
    const int ec = tx_class(e.txType) == TX_CLASS_2D ? 0 : 1;
    const float p = eob_pt_bits<ms>(C, pt, ec, eobPt - 1);
    b += p;
    const int x = max(eobPt - 3, 0), rem = eob - ((1 << (x + 1)) + 1);
    const float ex = C.eob_extra[cost_i(C, ctx)][cost_i(C, pt)][x][(rem >> x) & 1];
    b += eobPt >= 3 ? ex : 0.f;
    b += (float)x;
    return eob == 0 ? skip : b;
}

// The levels' magnitudes for the contexts: bytes min(|level|, 15) with four columns to the right and four rows below the
// block that stay 0, so a neighbour is one read at a fixed distance with neither bounds nor absolute value (against reading
// the levels: 45 of the 120 vector instructions per coefficient).  They are laid over the coefficients, which are all in
// registers by then.
template <int TW>
constexpr int lv_stride() { return TW + 4; }
__device__ __forceinline__ uint8_t *lv_of(float *p) { return (uint8_t *)p; }
__device__ __forceinline__ lds<uint8_t> *lv_of(lds<float> *p) { return (lds<uint8_t> *)p; }
typedef uint32_t __attribute__((may_alias)) word_a;
__device__ __forceinline__ void lv_zero(uint8_t *p) { *(word_a *)p = 0; }
__device__ __forceinline__ void lv_zero(lds<uint8_t> *p) { *(lds<word_a> *)p = 0; }
// a level's magnitude byte (a rounding offset below -1 makes levels of the other sign)
__device__ __forceinline__ uint8_t lv_byte(int l) { return (uint8_t)min(max(l, -l), 15); }
// the margins of a TW x TH block by NL lanes
template <int TW, int TH, int NL, typename LV>
__device__ __forceinline__ void lv_margins(LV lv, int lane) {
    constexpr int S = lv_stride<TW>(), NW = TH + S;   // words: one right of each row, S below
    static_assert(TW % 4 == 0, "the margins are whole words");
#pragma unroll
    for (int k = 0; k < NW; k += NL) {
        const int w = k + lane;
        if (w < NW) lv_zero(lv + (w < TH ? w * S + TW : TH * S + 4 * (w - TH)));
    }
}

// What the coefficients of one tx block share: the distances of the class's own three neighbours, (1,1) (0,2) (2,0) / (0,2) (0,3)
// (0,4) / (2,0) (3,0) (4,0) for sk 0 (2D) / 1 (HORIZ) / 2 (VERT), and the cost of the DC's sign
struct CoefIn {
    int sk, d2, d3, d4;
    float dcSign;
};
template <int TSZ, typename QP, typename E>
__device__ __forceinline__ CoefIn coef_in(QP q, const E &e, int sk) {
    constexpr int S = lv_stride<av1t::Tx_Width[av1t::Adjusted_Tx_Size[TSZ]]>();
    static_assert(av1t::Sig_Ref_Diff_Offset[0][2][0] == 1 && av1t::Sig_Ref_Diff_Offset[1][2][1] == 2 && av1t::Sig_Ref_Diff_Offset[2][4][0] == 4,
                  "neighbour order: right, below, then the class's own three");
    return CoefIn{sk, sk == 0 ? S + 1 : sk == 1 ? 2 : 2 * S, sk == 0 ? 2 : sk == 1 ? 3 : 3 * S, sk == 1 ? 4 : sk == 0 ? 2 * S : 4 * S,
                  (&(*e.C).dc_sign[cost_i(*e.C, e.plane > 0)][e.dcCtx][0])[q[0] < 0]};
}

// Bits of the coefficient at scan position c (< eob) of a tx block of size TSZ given its magnitudes lv and levels q (natural
// order, stride = adjusted width); in.sk: the scan and context class (0: 2D, default zig-zag scan dscan; 1: HORIZ, columns;
// 2: VERT, rows), always 0 for sizes with a side over 16; cbOff: Coeff_Base_Ctx_Offset[TSZ] (5 x 5).  One path for the three
// classes, whose neighbour positions differ in data only, so the lanes of a wave that evaluate different tx types do not
// run the classes one after the other; the five neighbours are read once for both contexts.
template <int TSZ, typename LV, typename QP, typename SP, typename OP, typename CT>
__device__ __forceinline__ float coeff_bits(int c, int eob, const CoefIn &in, LV lv, QP q, SP dscan, OP cbOff, int pt, const CT &C) {
    constexpr int ctx = txsz_ctx_of(TSZ), adj = av1t::Adjusted_Tx_Size[TSZ];
    constexpr int bwl = av1t::Tx_Width_Log2[adj], width = 1 << bwl, lbh = av1t::Tx_Height_Log2[adj], height = 1 << lbh, S = lv_stride<width>();
    constexpr bool only2d = width > 16 || height > 16;
    const int sk = in.sk;
    int pos = dscan[c];
    if constexpr (!only2d) pos = sk == 0 ? pos : sk == 1 ? ((c & (height - 1)) << bwl) + (c >> lbh) : c;
    const int row = pos >> bwl, col = pos & (width - 1);
    const auto at = lv + row * S + col;
    const int level = at[0], a0 = at[1], a1 = at[S];
    int a2, a3, a4;
    if constexpr (only2d) {
        a2 = at[S + 1]; a3 = at[2]; a4 = at[2 * S];
    } else {
        a2 = at[in.d2]; a3 = at[in.d3]; a4 = at[in.d4];
    }
    const int m5 = min(a0, 3) + min(a1, 3) + min(a2, 3) + min(a3, 3) + min(a4, 3);
    const int m = min((m5 + 1) >> 1, 4);
    int bctx = pos == 0 ? 0 : m + (int)cbOff[min(row, 4) * 5 + min(col, 4)];
    if constexpr (!only2d) {
        static_assert(av1t::Coeff_Base_Pos_Ctx_Offset[0] == 26 && av1t::Coeff_Base_Pos_Ctx_Offset[1] == 31 && av1t::Coeff_Base_Pos_Ctx_Offset[2] == 36,
                      "26 + 5 min(position, 2)");
        bctx = sk == 0 ? bctx : m + 26 + 5 * min(sk == 1 ? col : row, 2);
    }
    const int ectx = c == 0 ? 0 : c <= (height << bwl) / 8 ? 1 : c <= (height << bwl) / 4 ? 2 : 3;
    const auto *pb = c == eob - 1 ? &C.coeff_base_eob[cost_i(C, ctx)][cost_i(C, pt)][ectx][min(max(level, 1), 3) - 1] : &C.coeff_base[cost_i(C, ctx)][cost_i(C, pt)][bctx][min(level, 3)];
    float b = *pb, golomb = 0.f;
    if (level > 2) {
        const int mb = min((a0 + a1 + a2 + 1) >> 1, 6);
        bool near0 = row < 2 && col < 2;
        if constexpr (!only2d) near0 = sk == 0 ? near0 : sk == 1 ? col == 0 : row == 0;
        const auto *br = C.coeff_br[cost_i(C, min(ctx, (int)TX_32X32))][cost_i(C, pt)][pos == 0 ? mb : near0 ? mb + 7 : mb + 14];
        // up to four symbols of at most 3: n3 full ones, then the rest
        const int rem = level - 3, n3 = (rem * 11) >> 5;   // rem / 3 for 0 .. 12
        const float full = br[3], rest = br[rem - 3 * n3];
        const int qv = q[pos], v = max(qv, -qv);
#pragma unroll
        for (int i = 0; i < 4; i++) b += i < n3 ? full : i == n3 ? rest : 0.f;
        golomb = v > 14 ? (float)(2 * (31 - __clz(max(v - 14, 1))) + 1) : 0.f;
    }
    b += level ? (c == 0 ? in.dcSign : 1.0f) : 0.f;   // the sign, then the Golomb part (sums with 0 are exact)
    return b + golomb;
}

// eob and rate of the levels of a tx block of size TSZ, class sk, by the group (all lanes return both); last: the
// lane's share of the eob (1 + the largest scan index of a nonzero level among the positions the lane quantized)
template <int TSZ, typename LV, typename QP, typename SP, typename OP, typename E>
__device__ __forceinline__ void grp_rate(LV lv, QP q, SP dscan, OP cbOff, const E &e, int sk, int last, int &eobOut, float &bitsOut) {
    const int lane = glane();
    const int eob = gmaxi(last);
    const float base = base_bits<TSZ>(e, eob);
    const CoefIn in = coef_in<TSZ>(q, e, sk);
    float bits = lane == 0 ? base : 0.f;
    for (int c = lane; c < eob; c += GW) bits += coeff_bits<TSZ>(c, eob, in, lv, q, dscan, cbOff, e.plane > 0, *e.C);
    eobOut = eob;
    bitsOut = gsum(bits);
}

// the default scan and the base-context offsets of tx size TSZ (global tables; the closed loop reads LDS copies)
template <int TSZ>
__device__ __forceinline__ const uint16_t *dscan_ptr(const DevTables &) { return scan_of(TSZ, DCT_DCT); }
template <int TSZ>
__device__ __forceinline__ const uint8_t *cboff_ptr(const DevTables &) { return &av1t::Coeff_Base_Ctx_Offset[TSZ][0][0]; }
template <int TSZ>
__device__ __forceinline__ const uint16_t *iscan_ptr(const DevTables &T) { return T.iscan + dscan_off(av1t::Adjusted_Tx_Size[TSZ]); }

// Evaluation scratch of one group in LDS, for tx blocks of W x H up to 16 x 16
template <int W, int H>
struct EvalScr {
    int16_t res[W * H];
    float tmp[H * (W + 1)];
    int16_t q[W * H];
    __device__ std::nullptr_t lv() { return nullptr; }
};

template <int W, int H, typename FP, typename QP, typename E, typename TT, typename LV>
__device__ __forceinline__ EvalOut grp_qrate(FP tmp, int ts, QP q, const E &e, const TT &T, LV lvSep);

// Forward transform + quantization + distortion + rate of the residual res (W x H, row-major), by the 32 lanes of
// the calling group, with tmp (th x (W + 1) floats) as scratch.  Levels into q (natural order, tw x th).  All lanes
// return the same values.
template <int W, int H, typename RP, typename FP, typename QP, typename E, typename TT, typename LV = std::nullptr_t>
__device__ EvalOut grp_eval(RP res, FP tmp, QP q, const E &e, const TT &T, LV lvSep = nullptr) {
    constexpr int TW = W, TH = H, TS = W + 1;
    constexpr int LW = W == 4 ? 2 : W == 8 ? 3 : 4, LH = H == 4 ? 2 : H == 8 ? 3 : 4;
    const int lane = glane();
    const int rk = row_kind(e.txType), ck = col_kind(e.txType), fud = flip_ud(e.txType), flr = flip_lr(e.txType);
    // Outputs per item chosen so that a pass fills the group's 32 lanes where the block allows (at most 8 per item):
    // each output is one fmaf chain over k ascending whichever lane computes it.
    // ---- column pass: item = (column j, OC consecutive outputs) ----
    {
        constexpr int OCF = W * TH / GW, OC = OCF < 1 ? 1 : OCF > 8 ? 8 : OCF, NI = W * (TH / OC);
        const auto *FcT = T.fwdT + T.fwdOff[ck][LH];
        for (int it = lane; it < NI; it += GW) {
            const int j = it % W, i0 = (it / W) * OC, jj = flr ? W - 1 - j : j;
            float acc[OC];
            if (ck == K_IDT) {
#pragma unroll
                for (int o = 0; o < OC; o++) acc[o] = FcT[(i0 + o) * H + i0 + o] * (float)res[(fud ? H - 1 - (i0 + o) : i0 + o) * W + jj];
            } else {
#pragma unroll
                for (int o = 0; o < OC; o++) acc[o] = 0.f;
#pragma unroll 4
                for (int k = 0; k < H; k++) {
                    const float x = (float)res[(fud ? H - 1 - k : k) * W + jj];
                    const auto *f = FcT + k * H + i0;
#pragma unroll
                    for (int o = 0; o < OC; o++) acc[o] = fmaf(f[o], x, acc[o]);
                }
            }
#pragma unroll
            for (int o = 0; o < OC; o++) tmp[(i0 + o) * TS + j] = acc[o];
        }
    }
    gsync();
    // ---- row pass, in place: item = (row i, OR consecutive outputs); every lane reads its row whole before any writes ----
    {
        constexpr int ORF = TW * TH / GW, OR = ORF < 1 ? 1 : ORF > TW ? TW : ORF, NR = TH * (TW / OR);
        static_assert(NR <= GW, "one row item per lane");
        const auto *FrT = T.fwdT + T.fwdOff[rk][LW];
        const float scale = T.txScale[cost_i(T, e.txSz)];
        const int i = lane % TH, o0 = (lane / TH) * OR;
        auto *row = tmp + i * TS;
        float acc[OR];
        if (lane < NR) {
            if (rk == K_IDT) {
#pragma unroll
                for (int o = 0; o < OR; o++) acc[o] = FrT[(o0 + o) * W + o0 + o] * row[o0 + o];
            } else {
#pragma unroll
                for (int o = 0; o < OR; o++) acc[o] = 0.f;
#pragma unroll 2
                for (int k = 0; k < W; k++) {
                    const float x = row[k];
                    const auto *f = FrT + k * W + o0;
#pragma unroll
                    for (int o = 0; o < OR; o++) acc[o] = fmaf(f[o], x, acc[o]);
                }
            }
        }
        gsync();
        if (lane < NR) {
#pragma unroll
            for (int o = 0; o < OR; o++) row[o0 + o] = acc[o] * scale;
        }
    }
    gsync();
    return grp_qrate<W, H>(tmp, TS, q, e, T, lvSep);
}

// Quantization, distortion and rate of the coefficients of a W x H tx block held in tmp (row i of the kept tw x th
// region at tmp + i * ts), levels into q (natural order, tw x th).  All lanes of the group return the same values.
// lvSep: where the magnitudes go, or null: over the coefficients, which then all pass through registers (where a lane has
// eight of them and 168 registers that costs 40 in spills: the analysis of 16x16 keeps the two apart, 1.48 -> 1.14 ms on 12 MP).
template <int W, int H, typename FP, typename QP, typename E, typename TT, typename LV>
__device__ __forceinline__ EvalOut grp_qrate(FP tmp, int ts, QP q, const E &e, const TT &T, LV lvSep) {
    static_assert(W <= 16 && H <= 16 && W * H >= GW, "larger tx blocks: wave_qrate; smaller ones: half_qrate");
    static_assert((H + 4) * lv_stride<W>() <= H * (W + 1) * 4, "the magnitudes fit in the coefficients' space");
    constexpr int TW = W, TH = H;
    constexpr int LTW = TW == 4 ? 2 : TW == 8 ? 3 : 4;
    constexpr int N = TW * TH;
    const int lane = glane();
    constexpr int TSZ = tx_of(W, H);
    const int cls = tx_class(e.txType);
    // the scan of the rate: the default (2D) scan, rows (class VERT: raster order) or columns (class HORIZ)
    const int sk = cls == TX_CLASS_2D ? 0 : cls == TX_CLASS_HORIZ ? 1 : 2;
    const auto iscan = iscan_ptr<TSZ>(T);
    // ---- quantization + distortion (virtual lane = physical lane), and the eob ----
    const int den = dq_denom(e.txSz), dsh = den == 4 ? 2 : den == 2 ? 1 : 0;
    float dist = 0.f;
    int last = 0;
    constexpr int NE = N / GW;   // per lane
    constexpr bool SEP = !std::is_same_v<LV, std::nullptr_t>;
    auto coef = [&](int idx) -> float { return tmp[(idx >> LTW) * ts + (idx & (TW - 1))]; };
    float x[NE];
    if constexpr (!SEP) {
#pragma unroll
        for (int t = 0; t < NE; t++) x[t] = coef(lane + GW * t);
        gsync();
    }
    const auto lv = [&] { if constexpr (SEP) return lvSep; else return lv_of(tmp); }();
    lv_margins<TW, TH, GW>(lv, lane);
    constexpr int UNR = SEP ? 4 : NE;
#pragma unroll UNR
    for (int t = 0; t < NE; t++) {
        const int idx = lane + GW * t;
        const float v = SEP ? coef(idx) : x[t];
        const int step = idx == 0 ? e.dcQ : e.acQ;
        const float a = quot_step(fabsf(v) * (float)den, (float)step, idx == 0 ? e.dcRcp : e.acRcp);
        int l = a < e.zbin ? 0 : (int)(a + e.rnd);
        l = min(l, 16383);
        const int qv = v < 0 ? -l : l;
        q[idx] = (int16_t)qv;
        lv[(idx >> LTW) * lv_stride<TW>() + (idx & (TW - 1))] = lv_byte(l);
        const int c0 = (int)iscan[idx], c = sk == 0 ? c0 : sk == 1 ? (idx & (TW - 1)) * TH + (idx >> LTW) : idx;
        last = max(last, l ? c + 1 : 0);
        const float dq = (float)dequant(qv, step, dsh, e.bd);   // 0 for level 0
        const float d = v - dq;
        const float sq = d * d;
        dist = dist + sq;
    }
    const float distS = gsum(dist);
    gsync();
    const auto dscan = dscan_ptr<TSZ>(T);
    const auto cbOff = cboff_ptr<TSZ>(T);
    int eob;
    EvalOut o;
    grp_rate<TSZ>(lv, q, dscan, cbOff, e, sk, last, eob, o.R);
    const float g = T.txg[cost_i(T, e.txSz)][e.txType];
    o.D = g * distS;
    o.eob = eob;
    return o;
}

// ---- the same evaluation by half a group (16 lanes) for tx blocks of up to 64 coefficients ----
// Lane l of the half holds virtual lanes l and l + 16 of the 32-lane form: their partial sums stay apart, and the sums
// over the group add them first (the xor-16 step of gsum), then run the remaining butterfly steps across the 16 lanes,
// so every result is the 32-lane form's to the bit.  The two halves of a group run two evaluations at once.
__device__ __forceinline__ int hlane() { return threadIdx.x & 15; }
__device__ __forceinline__ float hsum2(float a, float b) {
    float v = a + b;
    v += lane_xorf<8>(v); v += lane_xorf<4>(v); v += lane_xorf<2>(v); v += lane_xorf<1>(v);
    return v;
}
__device__ __forceinline__ int hmaxi(int v) {
    v = max(v, lane_xor<8>(v)); v = max(v, lane_xor<4>(v)); v = max(v, lane_xor<2>(v)); v = max(v, lane_xor<1>(v));
    return v;
}

template <int W, int H, typename FP, typename QP, typename E, typename TT>
__device__ EvalOut half_qrate(FP tmp, int ts, QP q, const E &e, const TT &T) {
    static_assert(W <= 16 && H <= 16 && W * H <= 64, "half-group evaluation: up to 64 coefficients");
    constexpr int TW = W, TH = H, LTW = TW == 4 ? 2 : TW == 8 ? 3 : 4, N = TW * TH, TSZ = tx_of(W, H);
    const int lane = hlane();
    const int cls = tx_class(e.txType);
    const int sk = cls == TX_CLASS_2D ? 0 : cls == TX_CLASS_HORIZ ? 1 : 2;
    const auto iscan = iscan_ptr<TSZ>(T);
    const int den = dq_denom(e.txSz), dsh = den == 4 ? 2 : den == 2 ? 1 : 0;
    float dist[2] = {0.f, 0.f};
    int last = 0;
    float x[N / 16];
#pragma unroll
    for (int t = 0; t < N / 16; t++) {
        const int idx = lane + 16 * t;
        x[t] = tmp[(idx >> LTW) * ts + (idx & (TW - 1))];
    }
    gsync();
    const auto lv = lv_of(tmp);
    lv_margins<TW, TH, 16>(lv, lane);
#pragma unroll
    for (int t = 0; t < N / 16; t++) {   // virtual lane lane + 16 (t & 1)
        const int idx = lane + 16 * t;
        const float v = x[t];
        const int step = idx == 0 ? e.dcQ : e.acQ;
        const float a = quot_step(fabsf(v) * (float)den, (float)step, idx == 0 ? e.dcRcp : e.acRcp);
        int l = a < e.zbin ? 0 : (int)(a + e.rnd);
        l = min(l, 16383);
        const int qv = v < 0 ? -l : l;
        q[idx] = (int16_t)qv;
        lv[(idx >> LTW) * lv_stride<TW>() + (idx & (TW - 1))] = lv_byte(l);
        const int c0 = (int)iscan[idx], c = sk == 0 ? c0 : sk == 1 ? (idx & (TW - 1)) * TH + (idx >> LTW) : idx;
        last = max(last, l ? c + 1 : 0);
        const float dq = (float)dequant(qv, step, dsh, e.bd);
        const float d = v - dq;
        const float sq = d * d;
        dist[t & 1] = dist[t & 1] + sq;
    }
    const float distS = hsum2(dist[0], dist[1]);
    gsync();
    const auto dscan = dscan_ptr<TSZ>(T);
    const auto cbOff = cboff_ptr<TSZ>(T);
    const int eob = hmaxi(last);
    const float base = base_bits<TSZ>(e, eob);
    float b0 = lane == 0 ? base : 0.f, b1 = 0.f;
    const CoefIn in = coef_in<TSZ>(q, e, sk);
    // the lane's two virtual lanes side by side: their chains of reads overlap
    for (int c = lane; c < eob; c += GW) {
        const int d = c + 16 < N ? c + 16 : c;
        const float v0 = coeff_bits<TSZ>(c, eob, in, lv, q, dscan, cbOff, e.plane > 0, *e.C);
        const float v1 = coeff_bits<TSZ>(d, eob, in, lv, q, dscan, cbOff, e.plane > 0, *e.C);
        b0 += v0;
        if (c + 16 < eob) b1 += v1;
    }
    EvalOut o;
    o.R = hsum2(b0, b1);
    o.D = T.txg[cost_i(T, e.txSz)][e.txType] * distS;
    o.eob = eob;
    return o;
}

// grp_eval by half a group (W x H up to 64 coefficients): the same column / row passes, items spread over 16 lanes
template <int W, int H, typename RP, typename FP, typename QP, typename E, typename TT>
__device__ EvalOut half_eval(RP res, FP tmp, QP q, const E &e, const TT &T) {
    constexpr int TW = W, TH = H, TS = W + 1;
    constexpr int LW = W == 4 ? 2 : W == 8 ? 3 : 4, LH = H == 4 ? 2 : H == 8 ? 3 : 4;
    const int lane = hlane();
    const int rk = row_kind(e.txType), ck = col_kind(e.txType), fud = flip_ud(e.txType), flr = flip_lr(e.txType);
    // outputs per item chosen so that each pass fills the 16 lanes (as grp_eval does with 32)
    {
        constexpr int OCF = W * TH / 16, OC = OCF < 1 ? 1 : OCF > 8 ? 8 : OCF, NI = W * (TH / OC);
        const auto *FcT = T.fwdT + T.fwdOff[ck][LH];
        for (int it = lane; it < NI; it += 16) {
            const int j = it % W, i0 = (it / W) * OC, jj = flr ? W - 1 - j : j;
            float acc[OC];
            if (ck == K_IDT) {
#pragma unroll
                for (int o = 0; o < OC; o++) acc[o] = FcT[(i0 + o) * H + i0 + o] * (float)res[(fud ? H - 1 - (i0 + o) : i0 + o) * W + jj];
            } else {
#pragma unroll
                for (int o = 0; o < OC; o++) acc[o] = 0.f;
#pragma unroll 4
                for (int k = 0; k < H; k++) {
                    const float x = (float)res[(fud ? H - 1 - k : k) * W + jj];
                    const auto *f = FcT + k * H + i0;
#pragma unroll
                    for (int o = 0; o < OC; o++) acc[o] = fmaf(f[o], x, acc[o]);
                }
            }
#pragma unroll
            for (int o = 0; o < OC; o++) tmp[(i0 + o) * TS + j] = acc[o];
        }
    }
    gsync();
    {
        constexpr int ORF = TW * TH / 16, OR = ORF < 1 ? 1 : ORF > TW ? TW : ORF, NR = TH * (TW / OR);
        static_assert(NR <= 16, "one row item per lane");
        const auto *FrT = T.fwdT + T.fwdOff[rk][LW];
        const float scale = T.txScale[cost_i(T, e.txSz)];
        const int i = lane % TH, o0 = (lane / TH) * OR;
        auto *row = tmp + i * TS;
        float acc[OR];
        if (lane < NR) {
            if (rk == K_IDT) {
#pragma unroll
                for (int o = 0; o < OR; o++) acc[o] = FrT[(o0 + o) * W + o0 + o] * row[o0 + o];
            } else {
#pragma unroll
                for (int o = 0; o < OR; o++) acc[o] = 0.f;
#pragma unroll 2
                for (int k = 0; k < W; k++) {
                    const float x = row[k];
                    const auto *f = FrT + k * W + o0;
#pragma unroll
                    for (int o = 0; o < OR; o++) acc[o] = fmaf(f[o], x, acc[o]);
                }
            }
        }
        gsync();   // every read of the rows precedes the in-place writes
        if (lane < NR) {
#pragma unroll
            for (int o = 0; o < OR; o++) row[o0 + o] = acc[o] * scale;
        }
    }
    gsync();
    return half_qrate<W, H>(tmp, TS, q, e, T);
}

// ---- tx blocks with a side of 32 or 64 (DCT_DCT only), by a whole wave ----
// Each forward-transform output is one fmaf chain over ascending k, and so is each element of an FP32 MFMA: the 16x16x4
// instruction adds its four products in ascending k with a rounding per product (checked on MI355X against fmaf chains,
// 1.4 M elements over three value ranges, none different).  So both passes run on the matrix cores under the same
// arithmetic contract, at twice the FMA rate of the vector unit and without an operand load per product.
__device__ __forceinline__ int wlane() { return threadIdx.x & 63; }
// (the value of this 32-lane half's partner lane in the lower half, in the upper half), in every lane
struct Halves { float lo, hi; };
__device__ __forceinline__ Halves halves(float v) {
    const auto p = __builtin_amdgcn_permlane32_swap((unsigned)__float_as_int(v), (unsigned)__float_as_int(v), false, false);
    return Halves{__int_as_float((int)p[0]), __int_as_float((int)p[1])};
}
__device__ __forceinline__ int other_half(int v) {
    const auto p = __builtin_amdgcn_permlane32_swap((unsigned)v, (unsigned)v, false, false);
    return (int)((threadIdx.x & 32) ? p[0] : p[1]);
}
__device__ __forceinline__ int wsumi(int v) { v = gsumi(v); return v + other_half(v); }   // over the wave

typedef float f32x4 __attribute__((ext_vector_type(4)));

// the residual energy as 32 sequential float sums over the raster order (virtual lane v: elements v, v + 32, ...), for
// sums past 2^24, whose order of additions matters; res(i0, di, j, r) fills r with rows i0, i0 + di, ... of column j
template <int W, int H, typename Res>
__device__ __forceinline__ float wave_energy_seq(Res res) {
    const int v = threadIdx.x & 31;
    float e = 0.f;
    for (int k = 0; k < H; k++) {
        int r[1];
        if constexpr (W == 64) {
            res(k, 1, v, r);
            e = e + (float)(r[0] * r[0]);
            res(k, 1, v + 32, r);
            e = e + (float)(r[0] * r[0]);
        } else if constexpr (W == 32) {
            res(k, 1, v, r);
            e = e + (float)(r[0] * r[0]);
        } else {   // W = 16: element v + 32 t is column v & 15 of row 2 t + (v >> 4)
            if ((k & 1) == (v >> 4)) {
                res(k, 1, v & 15, r);
                e = e + (float)(r[0] * r[0]);
            }
        }
    }
    return e;
}

// Forward DCT of a W x H residual made on the fly by res (above), by the 64 lanes of the wave.  Column pass as Y^T = X^T
// Fc^T: lane l supplies rows k = 4 s + g (g = l / 16) of its column, so the prediction of a sample is made once, in the lane
// that feeds it to the matrix core; the columns of a 16-column tile go to the lanes in the order 4 (m % 4) + m / 4, which
// makes accumulator register r of lane group g column 4 r + g -- the operand the row pass (Y Fr^T) wants of that lane, so
// nothing moves between the passes.  The kept th x tw coefficients (scaled) land in tmp (row stride TS).  Returns the
// energy sum over the raster order where a side is 64, else 0.
template <int W, int H, int TS, typename FP, typename Res>
__device__ __forceinline__ float wave_fwd_dct(FP tmp, const DevTables &T, float scale, Res res) {
    constexpr int TW = W > 32 ? 32 : W, TH = H > 32 ? 32 : H;
    constexpr int LW = W == 8 ? 3 : W == 16 ? 4 : W == 32 ? 5 : 6, LH = H == 8 ? 3 : H == 16 ? 4 : H == 32 ? 5 : 6;
    constexpr int NJ = W < 16 ? 1 : W / 16, NI = TH < 16 ? 1 : TH / 16, NO = TW < 16 ? 1 : TW / 16, KS = H / 4, RS = W / 4, CH = KS < 8 ? KS : 8;
    constexpr bool E64 = W == 64 || H == 64;
    const int l = wlane(), n = l & 15, g = l >> 4, jm = 4 * (n & 3) + (n >> 2);
    const DevTables *TU = (const DevTables *)uni(&T);
    const glb<float> *const FcT0 = (const glb<float> *)TU->fwdT + TU->fwdOff[K_DCT][LH];
    const glb<float> *const FrT0 = (const glb<float> *)TU->fwdT + TU->fwdOff[K_DCT][LW];
    uint32_t en0 = 0, en1 = 0;   // squares of the even and the odd column tiles
    f32x4 z[NI][NO];
#pragma unroll
    for (int it = 0; it < NI; it++)
#pragma unroll
        for (int ot = 0; ot < NO; ot++) z[it][ot] = f32x4{0.f, 0.f, 0.f, 0.f};
    // a column tile at a time through both passes (the row pass's k are the columns in ascending order); rolled, since the
    // prediction's modes make it the larger part of the code
#pragma unroll 1
    for (int jt = 0; jt < NJ; jt++) {
        const int j = 16 * jt + jm;
        f32x4 y[NI];
#pragma unroll
        for (int it = 0; it < NI; it++) y[it] = f32x4{0.f, 0.f, 0.f, 0.f};
        // the matrix operands are read again for each run of rows (and candidate): hoisted out of the loops they would hold
        // 30-60 registers through the whole search and spill as many others
        const glb<float> *FrT = FrT0;
#pragma unroll 1
        for (int s0 = 0; s0 < KS; s0 += CH) {
            const glb<float> *FcT = FcT0;
            asm volatile("" : "+s"(FcT), "+s"(FrT));
            int r[CH];
            res(4 * s0 + g, 4, W < 16 ? j & (W - 1) : j, r);
            if constexpr (E64) {
                uint32_t q = 0;
#pragma unroll
                for (int s = 0; s < CH; s++) q += (uint32_t)(r[s] * r[s]);
                en0 += (jt & 1) ? 0u : q;
                en1 += (jt & 1) ? q : 0u;
            }
#pragma unroll
            for (int s = 0; s < CH; s++) {
                const float x = W < 16 && j >= W ? 0.f : (float)r[s];
#pragma unroll
                for (int it = 0; it < NI; it++) {
                    const int i = 16 * it + n;
                    float f = FcT[(4 * (s0 + s) + g) * H + (TH < 16 ? i & (TH - 1) : i)];
                    if constexpr (TH < 16) f = i < TH ? f : 0.f;
                    y[it] = __builtin_amdgcn_mfma_f32_16x16x4f32(x, f, y[it], 0, 0, 0);
                }
            }
        }
#pragma unroll
        for (int s = 0; s < (RS < 4 ? RS : 4); s++) {
#pragma unroll
            for (int ot = 0; ot < NO; ot++) {
                const int o = 16 * ot + n;
                float f = FrT[(16 * jt + 4 * s + g) * W + (TW < 16 ? o & (TW - 1) : o)];
                if constexpr (TW < 16) f = o < TW ? f : 0.f;
#pragma unroll
                for (int it = 0; it < NI; it++) z[it][ot] = __builtin_amdgcn_mfma_f32_16x16x4f32(y[it][s], f, z[it][ot], 0, 0, 0);
            }
        }
    }
#pragma unroll
    for (int it = 0; it < NI; it++)
#pragma unroll
        for (int ot = 0; ot < NO; ot++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int i = 16 * it + 4 * g + r, o = 16 * ot + n;
                if ((TH >= 16 || i < TH) && (TW >= 16 || o < TW)) tmp[i * TS + o] = z[it][ot][r] * scale;
            }
    gsync();
    if constexpr (E64) {
        // the virtual lanes' sums as integers: v = 16 (column tile parity) + column in the tile (W = 16: + 16 (row parity),
        // which is g & 1), each over the lanes of the other rows; a sum below 2^24 is what any order of float additions gives
        uint32_t a = en0, b = en1;
        float f;
        bool exact;
        if constexpr (W == 16) {
            a += (uint32_t)other_half((int)a);
            exact = a < (1u << 24);
            f = (float)a;
            f += lane_xorf<16>(f);
        } else {
            a += (uint32_t)lane_xor<16>((int)a); a += (uint32_t)other_half((int)a);
            b += (uint32_t)lane_xor<16>((int)b); b += (uint32_t)other_half((int)b);
            exact = a < (1u << 24) && b < (1u << 24);
            f = (float)a + (float)b;
        }
        if (__any(!exact)) return gsum(wave_energy_seq<W, H>(res));
        // the butterfly over the column bits: columns 4 (n % 4) + n / 4, so steps 8, 4, 2, 1 are lanes xor 2, 1, 8, 4
        f += lane_xorf<2>(f); f += lane_xorf<1>(f); f += lane_xorf<8>(f); f += lane_xorf<4>(f);
        return f;
    }
    return 0.f;
}

// Quantization, distortion and rate of those coefficients (row stride ts), levels into q (natural order; the front of tmp: every
// coefficient is read before the first level is written).  Each virtual lane v of the 32-lane form is two lanes here: the
// lower half's takes the first half of its elements, the upper half's the rest, and the sequential sums are handed over
// once; the rate's scan positions alternate between the two.  All lanes return the same values.
template <int W, int H, typename FP, typename QP, typename E, typename TT>
__device__ __forceinline__ EvalOut wave_qrate(FP tmp, int ts, QP q, const E &e, const TT &T) {
    constexpr int TW = W > 32 ? 32 : W, TH = H > 32 ? 32 : H;
    constexpr int LTW = TW == 8 ? 3 : TW == 16 ? 4 : 5;
    constexpr int N = TW * TH, NE = N / 64, TSZ = tx_of(W, H);
    static_assert(N * 2 + (TH + 4) * lv_stride<TW>() <= TH * (TW + 1) * 4, "levels and magnitudes fit in the coefficients' space");
    constexpr bool E64 = W == 64 || H == 64;
    const int v = threadIdx.x & 31, h = (threadIdx.x >> 5) & 1;
    const auto iscan = iscan_ptr<TSZ>(T);
    const int den = dq_denom(e.txSz), dsh = den == 4 ? 2 : den == 2 ? 1 : 0;
    float x[NE], sq[NE];
#pragma unroll
    for (int u = 0; u < NE; u++) {
        const int idx = v + 32 * (NE * h + u);
        x[u] = tmp[(idx >> LTW) * ts + (idx & (TW - 1))];
    }
    gsync();
    // the levels take the front of the coefficients' space, their magnitudes what follows
    const auto lv = lv_of(tmp) + N * 2;
    lv_margins<TW, TH, 64>(lv, wlane());
    int last = 0;
#pragma unroll
    for (int u = 0; u < NE; u++) {
        const int idx = v + 32 * (NE * h + u);
        const int step = idx == 0 ? e.dcQ : e.acQ;
        const float a = quot_step(fabsf(x[u]) * (float)den, (float)step, idx == 0 ? e.dcRcp : e.acRcp);
        int l = a < e.zbin ? 0 : (int)(a + e.rnd);
        l = min(l, 16383);
        const int qv = x[u] < 0 ? -l : l;
        q[idx] = (int16_t)qv;
        lv[(idx >> LTW) * lv_stride<TW>() + (idx & (TW - 1))] = lv_byte(l);
        last = max(last, l ? (int)iscan[idx] + 1 : 0);
        const float d = x[u] - (float)dequant(qv, step, dsh, e.bd);
        sq[u] = d * d;
    }
    float dist = 0.f, kept = 0.f;
#pragma unroll
    for (int u = 0; u < NE; u++) {
        dist = dist + sq[u];
        if constexpr (E64) kept = fmaf(x[u], x[u], kept);
    }
    dist = halves(dist).lo;
    if constexpr (E64) kept = halves(kept).lo;
#pragma unroll
    for (int u = 0; u < NE; u++) {
        dist = dist + sq[u];
        if constexpr (E64) kept = fmaf(x[u], x[u], kept);
    }
    const float distS = gsum(halves(dist).hi);
    gsync();
    const auto dscan = dscan_ptr<TSZ>(T);
    const auto cbOff = cboff_ptr<TSZ>(T);
    last = max(last, other_half(last));
    const int eob = __builtin_amdgcn_readfirstlane(gmaxi(last));
    const float base = base_bits<TSZ>(e, eob);
    const CoefIn in = coef_in<TSZ>(q, e, 0);
    float bits = v == 0 ? base : 0.f;
    for (int c0 = 0; c0 < eob; c0 += 64) {
        const int c = c0 + 32 * h + v;
        const float b = coeff_bits<TSZ>(min(c, N - 1), eob, in, lv, q, dscan, cbOff, e.plane > 0, *e.C);
        const Halves p = halves(c < eob ? b : 0.f);
        bits += p.lo;
        bits += p.hi;
    }
    EvalOut o;
    o.R = gsum(bits);
    const float g = T.txg[cost_i(T, e.txSz)][e.txType];
    o.D = g * distS;
    if constexpr (E64) {
        const float keptS = gsum(halves(kept).hi);
        o.D = o.D + fmaxf(0.f, fmaf(-g, keptS, e.resEnergy));
    }
    o.eob = eob;
    return o;
}

// ---- intra edge preparation by a group: av1g_edge_prepare's integer arithmetic (spec 7.11.2.4 step 4, 7.11.2.9-12)
// buf: AboveRow or LeftCol, index 0 = first sample (indices -2 .. 2 (w + h) used)
template <typename P>
__device__ void grp_edge_filter(P *buf, int sz, int strength) {
    if (!strength) return;
    const int lane = glane();
    // Intra_Edge_Kernel[strength - 1]: 0 4 8 4 0 / 0 5 6 5 0 / 2 4 4 4 2
    static_assert(av1t::Intra_Edge_Kernel[0][2] == 8 && av1t::Intra_Edge_Kernel[1][1] == 5 && av1t::Intra_Edge_Kernel[2][0] == 2, "edge kernel");
    const int k0 = strength == 3 ? 2 : 0, k1 = strength == 2 ? 5 : 4, k2 = 10 - 2 * strength;
    int v[5];
#pragma unroll
    for (int k = 0; k < 5; k++) {
        const int i = lane + 1 + GW * k;
        int s = 0;
        if (i < sz) {
#pragma unroll
            for (int j = 0; j < 5; j++) s += (j == 2 ? k2 : j == 1 || j == 3 ? k1 : k0) * buf[clip3(0, sz - 1, i - 2 + j) - 1];
        }
        v[k] = (s + 8) >> 4;
    }
    gsync();
#pragma unroll
    for (int k = 0; k < 5; k++)
        if (lane + 1 + GW * k < sz) buf[lane + GW * k] = v[k];
    gsync();
}
template <typename P>
__device__ void grp_edge_upsample(P *buf, int numPx, int bd) {   // numPx <= 16
    const int lane = glane();
    auto dup = [&](int k) -> int { return k == 0 ? buf[-1] : k == numPx + 2 ? buf[numPx - 1] : buf[k - 2]; };
    int s = 0, e = 0;
    if (lane < numPx) {
        s = clip3(0, (1 << bd) - 1, round2(-dup(lane) + 9 * dup(lane + 1) + 9 * dup(lane + 2) - dup(lane + 3), 4));
        e = dup(lane + 2);
    }
    const int c = buf[-1];
    gsync();
    if (lane < numPx) { buf[2 * lane - 1] = s; buf[2 * lane] = e; }
    if (lane == 0) buf[-2] = c;
    gsync();
}
// prepare directional-mode edges in place (A, L are the group's copies); returns the upsampling flags
template <typename P>
__device__ void grp_edge_prepare(int pa, int lw, int lh, int ft, int haveL, int haveA, int x, int y, int maxX, int maxY, P *A, P *L,
                                 int bd, int &upA, int &upL) {
    const int w = 1 << lw, h = 1 << lh;
    if (pa != 90 && pa != 180) {
        if (pa > 90 && pa < 180 && w + h >= 24) {
            if (glane() == 0) {
                const int c = round2(L[0] * 5 + A[-1] * 6 + A[0] * 5, 4);
                L[-1] = c;
                A[-1] = c;
            }
            gsync();
        }
        if (haveA) grp_edge_filter(A, min(w, maxX - x + 1) + (pa < 90 ? h : 0) + 1, edge_strength(w, h, ft, pa - 90));
        if (haveL) grp_edge_filter(L, min(h, maxY - y + 1) + (pa > 180 ? w : 0) + 1, edge_strength(w, h, ft, pa - 180));
    }
    upA = edge_upsample(w, h, ft, pa - 90);
    if (upA) grp_edge_upsample(A, w + (pa < 90 ? h : 0), bd);
    upL = edge_upsample(w, h, ft, pa - 180);
    if (upL) grp_edge_upsample(L, h + (pa > 180 ? w : 0), bd);
}

// build AboveRow / LeftCol [-1 .. w + h - 1] of the tx block at (x, y) of plane (pitch) by the group's lanes
template <typename SP, typename P>
__device__ void grp_build_edges(const SP *plane, int pitch, int x, int y, int lw, int lh, int haveL, int haveA, int haveAR, int haveBL,
                                int maxX, int maxY, P *A, P *L, int bd) {
    const int w = 1 << lw, h = 1 << lh, n = w + h;
    const int alim = min(x + (haveAR ? 2 * w : w) - 1, maxX), llim = min(y + (haveBL ? 2 * h : h) - 1, maxY);
    for (int i = glane(); i < n; i += GW) {
        int a, l;
        if (!haveA && haveL) a = plane[(size_t)y * pitch + x - 1];
        else if (!haveA) a = (1 << (bd - 1)) - 1;
        else a = plane[(size_t)(y - 1) * pitch + min(x + i, alim)];
        if (!haveL && haveA) l = plane[(size_t)(y - 1) * pitch + x];
        else if (!haveL) l = (1 << (bd - 1)) + 1;
        else l = plane[(size_t)min(y + i, llim) * pitch + x - 1];
        A[i] = a;
        L[i] = l;
    }
    if (glane() == 0) {
        int c;
        if (haveA && haveL) c = plane[(size_t)(y - 1) * pitch + x - 1];
        else if (haveA) c = plane[(size_t)(y - 1) * pitch + x];
        else if (haveL) c = plane[(size_t)y * pitch + x - 1];
        else c = 1 << (bd - 1);
        A[-1] = c;
        L[-1] = c;
    }
    gsync();
}
// DC value (spec 7.11.2.5) with the edge sums over the group
template <typename P>
__device__ int grp_dc_value(const P *A, const P *L, int haveL, int haveA, int lw, int lh, int bd) {
    const int w = 1 << lw, h = 1 << lh;
    int sa = 0, sl = 0;
    for (int k = glane(); k < w; k += GW) sa += A[k];
    for (int k = glane(); k < h; k += GW) sl += L[k];
    sa = gsumi(sa);
    sl = gsumi(sl);
    if (haveL && haveA) return (sa + sl + ((w + h) >> 1)) / (w + h);
    if (haveL) return clip3(0, (1 << bd) - 1, (sl + (h >> 1)) >> lh);
    if (haveA) return clip3(0, (1 << bd) - 1, (sa + (w >> 1)) >> lw);
    return 1 << (bd - 1);
}

// sum |4x4 Hadamard coefficients| of d
__device__ __forceinline__ int hadamard4(int *d) {
#pragma unroll
    for (int i = 0; i < 4; i++) {
        int *r = d + 4 * i;
        const int s0 = r[0] + r[1], s1 = r[0] - r[1], s2 = r[2] + r[3], s3 = r[2] - r[3];
        r[0] = s0 + s2; r[1] = s1 + s3; r[2] = s0 - s2; r[3] = s1 - s3;
    }
    int sum = 0;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int s0 = d[j] + d[4 + j], s1 = d[j] - d[4 + j], s2 = d[8 + j] + d[12 + j], s3 = d[8 + j] - d[12 + j];
        sum += abs(s0 + s2) + abs(s1 + s3) + abs(s0 - s2) + abs(s1 - s3);
    }
    return sum;
}

// sum over the SEG consecutive lanes of a segment (SEG a power of 2 up to 32), in every lane of it
template <int SEG>
__device__ __forceinline__ int seg_sumi(int v) {
    if constexpr (SEG >= 32) v += lane_xor<16>(v);
    if constexpr (SEG >= 16) v += lane_xor<8>(v);
    if constexpr (SEG >= 8) v += lane_xor<4>(v);
    if constexpr (SEG >= 4) v += lane_xor<2>(v);
    if constexpr (SEG >= 2) v += lane_xor<1>(v);
    return v;
}

// the same transform with one value of d per lane: lanes 16k .. 16k + 15 of the group hold one 4x4 block in raster
// order (lane bits 0-1: column, 2-3: row).  The butterflies are those of hadamard4 (rows, then columns), so the 16
// lanes return the absolute values of its 16 coefficients, whose sum is its result.  Every lane of the group calls it.
__device__ __forceinline__ int hadamard4_lanes(int v) {
    const int l = glane();
    int t = lane_xor<1>(v);
    v = (l & 1) ? t - v : v + t;
    t = lane_xor<2>(v);
    v = (l & 2) ? t - v : v + t;
    t = lane_xor<4>(v);
    v = (l & 4) ? t - v : v + t;
    t = lane_xor<8>(v);
    v = (l & 8) ? t - v : v + t;
    return abs(v);
}

// runtime tx-size dispatch to a template taking <W, H>
#define AV1M_TX_SWITCH(txSz, M)                                                                                   \
    switch (txSz) {                                                                                               \
    case TX_4X4: M(4, 4); break; case TX_8X8: M(8, 8); break; case TX_16X16: M(16, 16); break;                    \
    case TX_32X32: M(32, 32); break; case TX_64X64: M(64, 64); break; case TX_4X8: M(4, 8); break;                \
    case TX_8X4: M(8, 4); break; case TX_8X16: M(8, 16); break; case TX_16X8: M(16, 8); break;                    \
    case TX_16X32: M(16, 32); break; case TX_32X16: M(32, 16); break; case TX_32X64: M(32, 64); break;            \
    case TX_64X32: M(64, 32); break; case TX_4X16: M(4, 16); break; case TX_16X4: M(16, 4); break;                \
    case TX_8X32: M(8, 32); break; case TX_32X8: M(32, 8); break; case TX_16X64: M(16, 64); break;                \
    default: M(64, 16); break;                                                                                    \
    }

}  // namespace av1m

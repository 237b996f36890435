// Closed-loop decisions and reconstruction: one workgroup (groups of 32 lanes, RC_NT threads) per 64x64 superblock and plane
// kind (luma, or both chroma planes), from a persistent queue or one launch per wavefront step.  Inside the superblock the
// leaves run in decode order exactly as the decoder sees them: BlockDecoded state, real reconstructed edges, exact
// coefficient contexts from the 4x4 maps.  Reference: encoder/src/k_recon.cuh:1692-1808 (kernel), 822-1213 (luma),
// 1220-1686 (chroma), 139-197 (inverse + add), 203-238 (contexts), 685-730 (records).
//
// What bounds it: the latency of the chain of blocks.  A block's steps depend on each other and on the blocks before it,
// so a superblock keeps its workgroup's waves mostly waiting, and an image keeps about one superblock per wavefront
// column ready.  Two splits shorten the chain: luma needs nothing of chroma, so the two run as separate items beside each
// other; and progress published per block lets a superblock start beside its unfinished neighbours (recon_part).
// When the two came in, the closed loop of one 512 x 512 image went 48.7 -> 20.2 ms, 24 MP learned 115 -> 54 ms, 16 images
// of 12 MP 175 -> 94 ms; with all that the comments below name they take 10.6, 29 and 66 ms.
//
// Per block:
//   luma    every re-checked analysis candidate x every intra tx type of the set (tx blocks up to 16x16; DCT_DCT only
//           above), RD tasks spread over the groups, the first minimum of J = fmaf(lambda, R + mode bits, D) wins;
//   chroma  CfL alpha (least squares from the reconstructed luma, then +-1 by exact SSE), SATD screening of the 13 UV
//           modes and the deltas around the best directional one, top uvK (+ CfL) RD tasks for U and V, pick;
//   final   the winner re-quantized (the same levels), prediction, exact dequant + inverse transform + add with the
//           conformance repair, tx records, context maps, BlockDecoded, block record, 4x4 maps.
#pragma once
#ifndef AV1M_RC_THREADS
#error "the includer sets AV1M_RC_THREADS, the threads of a workgroup, and AV1M_RC_SPACE, the namespace of that instance"
#endif
#include "dev_eval.h"

namespace av1m {
namespace AV1M_RC_SPACE {

constexpr int RC_NT = AV1M_RC_THREADS, RC_NG = RC_NT / 32;
// transform teams for tx blocks with a side of 32 or 64: the waves
constexpr int RC_NTEAM = RC_NT / 64;

constexpr int RC_SMALL_RES = 14;   // 6 luma candidates, or 2 planes x 7 chroma candidates
// levels of every task of a tx block up to 16x16, packed by the block's size (task t at t * W * H): at most 6 candidates
// x 7 tx types of 128 coefficients, 6 x 5 of 256 (16x16: intra set 2), or 2 planes x 7 chroma candidates of 256
constexpr int RC_LEV_TOTAL = 7680;
// per-group scratch of the evaluations of transform blocks up to 16x16
struct RcGroup {
    float tmp[16 * 17];
    uint16_t ea[EDGE_LEN], el[EDGE_LEN];
};
// blocks up to 16x16: the residual of each candidate (luma) or task (chroma) and the levels of every task, kept until
// the decision so the winner is neither predicted nor quantized again
struct RcSmall {
    RcGroup g[RC_NG];
    int16_t res[RC_SMALL_RES][256];
    int16_t lev[RC_LEV_TOTAL];
};
// scratch of one wave evaluating a transform block with a side of 32 or 64 (DCT_DCT only): the kept coefficients, which the
// levels overlay, and the prepared edges
struct RcTeam {
    float tmp[32 * 33];
    uint16_t ea[EDGE_LEN], el[EDGE_LEN];
};
template <typename X> __device__ __forceinline__ lds<int16_t> *team_lev(X &t) { return (lds<int16_t> *)(lds<char> *)t.tmp; }
// The tables the evaluations and the decisions read, staged once per workgroup (the costs: per quantizer context of the
// images it meets).  An evaluation reads them in chains (level -> context -> cost) that nothing else hides in the few
// waves of one workgroup.  From the device tables they were about 480 flat loads per wave and block; when they moved to LDS,
// before the other steps named here, the closed loop of a 512 x 512 image went 52.7 -> 48.7 ms, of 16 12 MP images 191 ->
// 175 ms (two workgroups per CU still fit: the inverse's scratch and the levels share the evaluations' scratch).
struct RcTabs {
    float fwdT[3 * 336];     // DCT, ADST, identity for n = 4, 8, 16, transposed (offsets fwdOff)
    int fwdOff[3][7];
    float txScale[19];
    float txg[19][16];
    uint8_t cbOff[19][25];         // Coeff_Base_Ctx_Offset
    uint8_t scan8[SCAN8_TOTAL], iscan8[SCAN8_TOTAL];   // default scans of up to 256 coefficients and their inverses
    uint16_t step[90];             // Dr_Intra_Derivative
    uint8_t smooth[124];           // the smooth weights, n = 4, 8, .. 64 at n - 4
    const uint16_t *iscan;         // the larger ones' inverses (device tables; read through the caches)
    CostTab cost;                  // of the image's quantizer context
};
struct RcPredTables {
    const lds<RcTabs> &T;
    __device__ __forceinline__ int step(int pa) const { return T.step[pa]; }
    __device__ __forceinline__ const lds<uint8_t> *weights(int l) const { return T.smooth + (1 << l) - 4; }
};
using RcEvalIn = EvalInT<const lds<CostTab> *>;
template <int TSZ>
__device__ __forceinline__ auto dscan_ptr(const lds<RcTabs> &T) {
    constexpr int t = av1t::Adjusted_Tx_Size[TSZ];
    if constexpr (scan8_has(t)) return (const lds<uint8_t> *)(T.scan8 + scan8_off(t));
    else return scan_of(TSZ, DCT_DCT);
}
template <int TSZ>
__device__ __forceinline__ const lds<uint8_t> *cboff_ptr(const lds<RcTabs> &T) { return T.cbOff[TSZ]; }
template <int TSZ>
__device__ __forceinline__ auto iscan_ptr(const lds<RcTabs> &T) {
    constexpr int t = av1t::Adjusted_Tx_Size[TSZ];
    if constexpr (scan8_has(t)) return (const lds<uint8_t> *)(T.iscan8 + scan8_off(t));
    else return T.iscan + dscan_off(t);
}

struct RcBig {
    RcTeam t[RC_NTEAM];
    int16_t inv[64 * 64];    // inverse transform residual (the row pass clamps to 16 bits; the column outputs of a block
                             // passing the range checks are within 12)
};
union RcScr {
    RcSmall s;
    RcBig b;
};
struct BlockCand { uint8_t cand[MAXK], ncand, tx; };   // the tail of BlockRes
struct RcShared {
    RcScr u;
    RcTabs tab;
    uint16_t srcb[64 * 64];                  // source: the superblock's luma, or its chroma, U at 0 and V at 2048 (4:4:4: of
                                             // the current tx block only)
    int srcAt, srcSp;                        // the current block in it, and its row stride
    Img img;                                 // descriptor of the superblock's image
    SearchParams prm;                        // the launch's search parameters
    int dcQ, acQ;                            // its quantizer steps
    float dcRcp, acRcp;                      // 1 / dcQ, 1 / acQ
    uint16_t ea[3][EDGE_LEN], el[3][EDGE_LEN];   // unfiltered edges of the current tx block per plane
    int dcv[3], ft[3], hvL[3], hvA[3], px[3], py[3], mx[3], my[3];
    int skipCtx[3], dcCtx[3];
    int gup[RC_NG][2];                       // upsampling flags of each group's (team's) prepared edges
    uint8_t bdm[3][18][18];                  // BlockDecoded[plane][y + 1][x + 1]
    uint8_t taskC[64], taskT[64], taskP[64], taskK[64];   // candidate, tx type, plane, residual slot
    uint16_t taskE[64];                      // eob
    int candC[8], nCand;                     // luma: the re-checked candidates
    float taskJ[64];
    int nTask;
    float gBestJ[RC_NG];
    int gBestT[RC_NG];
    int win, winEob[3];
    int16_t cflL[32 * 32];                   // CfL luma (at most 8 x 1023)
    int cflAvg, cflAlpha[2];
    unsigned long long acc64[8];
    int satdI[32], uvc[32];
    float uvJ[32];                           // screening costs of the UV candidates
    int errFlag[2], nzFlag[2];               // range violations, nonzero levels left (luma or U, V)
    int flopsOn;                             // count the forward-transform work (Batch::flops set)
    unsigned long long flops;                // of the superblock so far
    int am, lm, mode, uvMode, uvDelta, nuv, bsize;
    int nSkip, nCfl;                         // skipped blocks and CfL blocks of the item
    uint32_t qItem;                          // persistent schedule: the item taken
    uint16_t leaf[MAX_LEAVES];               // the superblock's blocks: size | x4 << 5 | y4 << 9
    uint32_t cand[MAX_LEAVES][2];            // luma: their analysis candidates (6 bytes), count and tx type (BlockRes)
    uint32_t known[4];                       // last seen progress of the left, above and above-right superblock and of the
                                             // superblock's own luma; [0] bit 31: a wait failed
};

template <typename Px> __device__ __forceinline__ glb<Px> *rec_plane(const lds<Img> &I, int p) { return (glb<Px> *)I.rec[p]; }
template <typename Px> __device__ __forceinline__ const glb<Px> *src_plane(const lds<Img> &I, int p) { return (const glb<Px> *)I.src[p]; }
__device__ __forceinline__ glb<uint8_t> *map8(uint8_t *p) { return (glb<uint8_t> *)p; }
// get_filter_type (spec 7.11.2.8): 1 if the above or left block (chroma: the chroma-carrying one) uses a SMOOTH mode
__device__ int filter_type(const lds<Img> &I, int plane, int mi_row, int mi_col, int availU, int availL) {
    const glb<uint8_t> *m = map8(plane ? I.mUV : I.mY);
    auto smooth = [](int v) { return v == SMOOTH_PRED || v == SMOOTH_V_PRED || v == SMOOTH_H_PRED; };
    int a = 0, l = 0;
    if (availU) {
        int r = mi_row - 1, c = mi_col;
        if (plane > 0 && I.ss) { if (!(mi_col & 1)) c++; if (mi_row & 1) r--; }
        a = smooth(m[(size_t)r * I.MiCols + c]);
    }
    if (availL) {
        int r = mi_row, c = mi_col - 1;
        if (plane > 0 && I.ss) { if (mi_col & 1) c--; if (!(mi_row & 1)) r++; }
        l = smooth(m[(size_t)r * I.MiCols + c]);
    }
    return a || l;
}

// coefficient contexts of a tx block from the context maps (spec get_tx_block ctx), by the 32 lanes of the group:
// lane k reads the k-th 4x4 column above and row to the left
__device__ void grp_txb_ctx(const lds<Img> &I, int plane, int txSz, int x4, int y4, int bsize, int tx0, int ty0, lds<int> *skipCtx,
                            lds<int> *dcCtx) {
    const int lane = glane(), ss = plane ? I.ss : 0;
    const int stride = I.MiCols >> ss, maxX4 = I.MiCols >> ss, maxY4 = I.MiRows >> ss;
    const glb<uint8_t> *L = map8(I.cLvl[plane]), *D = map8(I.cDc[plane]);
    const bool hasA = y4 > ((ty0 >> 2) >> ss), hasL = x4 > ((tx0 >> 2) >> ss);
    const int w = tx_w(txSz), h = tx_h(txSz), w4 = w >> 2, h4 = h >> 2;
    int top = 0, left = 0, topAny = 0, leftAny = 0, sgn = 0;
    if (hasA && lane < w4 && x4 + lane < maxX4) {
        const int l = L[(size_t)(y4 - 1) * stride + x4 + lane], d = D[(size_t)(y4 - 1) * stride + x4 + lane];
        top = l; topAny = (l | d) != 0; sgn += d == 2 ? 1 : d == 1 ? -1 : 0;
    }
    if (hasL && lane < h4 && y4 + lane < maxY4) {
        const int l = L[(size_t)(y4 + lane) * stride + x4 - 1], d = D[(size_t)(y4 + lane) * stride + x4 - 1];
        left = l; leftAny = (l | d) != 0; sgn += d == 2 ? 1 : d == 1 ? -1 : 0;
    }
    top = gmaxi(top); left = gmaxi(left); topAny = gmaxi(topAny); leftAny = gmaxi(leftAny); sgn = gsumi(sgn);
    if (lane == 0) {
        if (plane == 0) {
            const int bw = 4 * bw4(bsize), bh = 4 * bh4(bsize);
            *skipCtx = (bw == w && bh == h) ? 0 : (top == 0 && left == 0) ? 1 : (top == 0 || left == 0) ? 2 + (max(top, left) > 3)
                     : max(top, left) <= 3 ? 4 : min(top, left) <= 3 ? 5 : 6;
        } else {
            const int ub = uv_bsize(bsize, I.ss);
            *skipCtx = topAny + leftAny + 7 + ((16 * bw4(ub) * bh4(ub) > w * h) ? 3 : 0);
        }
        *dcCtx = sgn < 0 ? 1 : sgn > 0 ? 2 : 0;
    }
}

// base edges of the tx block of plane p at (px, py) from the reconstruction (group g), DC value and filter type
template <typename Px>
// fA / fL: the block's AvailU / AvailL for the edge filter type where they differ from the tx block's edges (a further
// 4:4:4 chroma tx block inside its block); -1: the same
__device__ void rc_edges(lds<RcShared> &S, const lds<Img> &I, int p, int px, int py, int lw, int lh, int haveL, int haveA, int haveAR, int haveBL,
                         int mi_row, int mi_col, int fA = -1, int fL = -1) {
    const int ss = p ? I.ss : 0;
    const int maxX = ((I.MiCols * 4) >> ss) - 1, maxY = ((I.MiRows * 4) >> ss) - 1;
    lds<uint16_t> *A = S.ea[p] + EDGE_OFF, *L = S.el[p] + EDGE_OFF;
    grp_build_edges(rec_plane<Px>(I, p), I.pitch[p], px, py, lw, lh, haveL, haveA, haveAR, haveBL, maxX, maxY, A, L, I.bd);
    const int dcv = grp_dc_value(A, L, haveL, haveA, lw, lh, I.bd);
    if (glane() == 0) {
        S.dcv[p] = dcv; S.hvL[p] = haveL; S.hvA[p] = haveA; S.px[p] = px; S.py[p] = py; S.mx[p] = maxX; S.my[p] = maxY;
        S.ft[p] = I.edgeFilter ? filter_type(I, p, mi_row, mi_col, fA < 0 ? haveA : fA, fL < 0 ? haveL : fL) : 0;
    }
}

// prediction of candidate c (255 = CfL) of plane p for a W x H tx block (W, H <= 16), by the group, into res = src -
// pred (raster order: lane l makes samples l, l + 32, ..., i.e. column l % W, rows l / W + k * 32 / W, as one run of
// pred_col); the group's edge buffers receive the prepared (filtered) edges of directional modes.  S.gup[gid] = flags.
template <int W, int H>
__device__ void grp_residual(lds<RcShared> &S, lds<uint16_t> *gea, lds<uint16_t> *gel, int p, int c, const lds<uint16_t> *src, int sp,
                             lds<int16_t> *res, int bd) {
    constexpr int lw = W == 4 ? 2 : W == 8 ? 3 : 4, lh = H == 4 ? 2 : H == 8 ? 3 : 4;
    constexpr int NPX = W * H, CH = NPX >= GW ? NPX / GW : 1, DI = GW / W;
    const int lane = glane();
    const int m = c == 255 ? DC_PRED : cand_mode(c), pa = pangle(m, c == 255 ? 0 : cand_delta(c));
    const lds<uint16_t> *EA = S.ea[p] + EDGE_OFF, *EL = S.el[p] + EDGE_OFF;
    int upA = 0, upL = 0;
    const bool filt = c != 255 && is_dir(m) && gea != nullptr;
    if (filt) {
        for (int i = lane + EDGE_OFF - 2; i < EDGE_OFF + W + H + 2; i += GW) { gea[i] = S.ea[p][i]; gel[i] = S.el[p][i]; }   // the filled part
        gsync();
        grp_edge_prepare(pa, lw, lh, S.ft[p], S.hvL[p], S.hvA[p], S.px[p], S.py[p], S.mx[p], S.my[p], gea + EDGE_OFF, gel + EDGE_OFF, bd, upA,
                         upL);
        EA = gea + EDGE_OFF;
        EL = gel + EDGE_OFF;
    }
    const int dcv = S.dcv[p];
    if (lane < NPX) {
        const int i0 = lane >> lw, j = lane & (W - 1);
        int r[CH];
        if (c == 255) {
            const int alpha = S.cflAlpha[p - 1], avg = S.cflAvg;
#pragma unroll
            for (int k = 0; k < CH; k++) r[k] = clip3(0, (1 << bd) - 1, dcv + round2signed(alpha * (S.cflL[(i0 + k * DI) * W + j] - avg), 6));
        } else {
            pred_col(m, pa, dcv, i0, DI, j, lw, lh, EA, EL, upA, upL, r, RcPredTables{S.tab});
        }
#pragma unroll
        for (int k = 0; k < CH; k++) {
            const int i = i0 + k * DI;
            res[i * W + j] = (int16_t)((int)src[i * sp + j] - r[k]);
        }
    }
    if (lane == 0) { S.gup[gid()][0] = upA; S.gup[gid()][1] = upL; }
    gsync();
}

// one RD task (candidate c of plane p with tx type t) of a tx block up to 16x16 by the calling group: the residual
// res is ready; the levels go to lev
template <int W, int H>
__device__ EvalOut grp_task(lds<RcShared> &S, lds<RcGroup> &X, const lds<Img> &I, int p, int c, int t, const lds<int16_t> *res,
                            lds<int16_t> *lev, const lds<SearchParams> &P) {
    RcEvalIn e;
    e.txSz = tx_of(W, H); e.txType = t; e.plane = p;
    e.dcQ = S.dcQ; e.acQ = S.acQ; e.dcRcp = S.dcRcp; e.acRcp = S.acRcp;
    e.skipCtx = S.skipCtx[p]; e.dcCtx = S.dcCtx[p]; e.intraDir = p == 0 ? cand_mode(c) : 0; e.bd = I.bd;
    e.rnd = p ? P.rndC : P.rnd; e.zbin = p ? P.zbinC : P.zbin;
    e.resEnergy = 0.f;
    e.C = &S.tab.cost;
    return grp_eval<W, H>(res, X.tmp, lev, e, S.tab);
}
// the same task by half the group (blocks of up to 64 coefficients), with tmp its own part of the group's scratch
template <int W, int H>
__device__ EvalOut half_task(lds<RcShared> &S, lds<float> *tmp, const lds<Img> &I, int p, int c, int t, const lds<int16_t> *res,
                             lds<int16_t> *lev, const lds<SearchParams> &P) {
    RcEvalIn e;
    e.txSz = tx_of(W, H); e.txType = t; e.plane = p;
    e.dcQ = S.dcQ; e.acQ = S.acQ; e.dcRcp = S.dcRcp; e.acRcp = S.acRcp;
    e.skipCtx = S.skipCtx[p]; e.dcCtx = S.dcCtx[p]; e.intraDir = p == 0 ? cand_mode(c) : 0; e.bd = I.bd;
    e.rnd = p ? P.rndC : P.rnd; e.zbin = p ? P.zbinC : P.zbin;
    e.resEnergy = 0.f;
    e.C = &S.tab.cost;
    return half_eval<W, H>(res, tmp, lev, e, S.tab);
}

// one RD task (candidate c, 255 = CfL, of plane p; DCT_DCT) of a tx block with a side of 32 or 64 by the calling wave (its
// two groups prepare the same edges)
template <int W, int H>
__device__ EvalOut wave_task(lds<RcShared> &S, lds<RcTeam> &X, int team, const lds<Img> &I, const DevTables &T, int p, int c,
                             const lds<uint16_t> *src, int sp, const lds<SearchParams> &P) {
    constexpr int LW = W == 8 ? 3 : W == 16 ? 4 : W == 32 ? 5 : 6, LH = H == 8 ? 3 : H == 16 ? 4 : H == 32 ? 5 : 6;
    constexpr int TS = (W > 32 ? 32 : W) + 1;
    const int lane = glane(), bd = I.bd;
    const int m = c == 255 ? DC_PRED : cand_mode(c), pa = pangle(m, c == 255 ? 0 : cand_delta(c));
    const lds<uint16_t> *EA = S.ea[p] + EDGE_OFF, *EL = S.el[p] + EDGE_OFF;
    int upA = 0, upL = 0;
    if (c != 255 && is_dir(m) && I.edgeFilter) {
        for (int i = lane + EDGE_OFF - 2; i < EDGE_OFF + W + H + 2; i += GW) { X.ea[i] = S.ea[p][i]; X.el[i] = S.el[p][i]; }
        gsync();
        grp_edge_prepare(pa, LW, LH, S.ft[p], S.hvL[p], S.hvA[p], S.px[p], S.py[p], S.mx[p], S.my[p], X.ea + EDGE_OFF, X.el + EDGE_OFF, bd,
                         upA, upL);
        EA = X.ea + EDGE_OFF;
        EL = X.el + EDGE_OFF;
    }
    if (wlane() == 0) { S.gup[team][0] = upA; S.gup[team][1] = upL; }
    const int dcv = S.dcv[p], alpha = c == 255 ? S.cflAlpha[p - 1] : 0, cavg = S.cflAvg;
    auto res = [&](int i0, int di, int j, auto &r) {
        constexpr int CH = sizeof(r) / sizeof(r[0]);
        if (c == 255) {
#pragma unroll
            for (int k = 0; k < CH; k++) r[k] = clip3(0, (1 << bd) - 1, dcv + round2signed(alpha * (S.cflL[(i0 + k * di) * W + j] - cavg), 6));
        } else {
            pred_col(m, pa, dcv, i0, di, j, LW, LH, EA, EL, upA, upL, r, RcPredTables{S.tab});
        }
#pragma unroll
        for (int k = 0; k < CH; k++) r[k] = (int)src[(i0 + k * di) * sp + j] - r[k];
    };
    const int txSz = tx_of(W, H);
    RcEvalIn e;
    e.resEnergy = wave_fwd_dct<W, H, TS>(X.tmp, T, S.tab.txScale[txSz], res);
    e.txSz = txSz; e.txType = DCT_DCT; e.plane = p;
    e.dcQ = S.dcQ; e.acQ = S.acQ; e.dcRcp = S.dcRcp; e.acRcp = S.acRcp;
    e.skipCtx = S.skipCtx[p]; e.dcCtx = S.dcCtx[p]; e.intraDir = p == 0 ? cand_mode(c) : 0; e.bd = bd;
    e.rnd = p ? P.rndC : P.rnd; e.zbin = p ? P.zbinC : P.zbin;
    e.C = &S.tab.cost;
    return wave_qrate<W, H>(X.tmp, TS, (lds<lev16> *)team_lev(X), e, S.tab);
}

// ---- exact inverse transform + reconstruction by the workgroup (spec 7.13.3, 7.12.3 step 3) ----
// A row or a column per lane, bound by one wave's chain of rotations.  With 24-bit products, one range test per transform and
// 32-bit rounding (before: four 32-bit products at a quarter of the rate and two tests per rotation) the closed loop of a 12
// MP image went 29.8 -> 28.1 ms, of 16 of them 67.8 -> 65.9 ms.
template <int LW>
__device__ __forceinline__ uint32_t inv_row(int i, int W, int th, int tw, const lds<int16_t> *q, int dcQ, int acQ, int dsh, int bd, bool rect, int rk,
                            int rowShift, lds<int16_t> *res) {
    constexpr int N = 1 << LW;
    int32_t Tv[N];
#pragma unroll
    for (int j = 0; j < N; j++) {
        const int v = (i < th && j < tw) ? q[i * tw + j] : 0;
        Tv[j] = dequant(v, (i == 0 && j == 0) ? dcQ : acQ, dsh, bd);   // 0 for level 0
        if (rect) Tv[j] = Inv::rnd12(Inv::mul24(Tv[j], 2896));   // |Tv| <= 2^17: exact
    }
    uint32_t err = 0;
    Inv::run<LW>(Tv, rk, bd + 8, err);
    const int colR = bd + 6 > 16 ? bd + 6 : 16;
#pragma unroll
    for (int j = 0; j < N; j++) res[i * W + j] = (int16_t)clip3(-(1 << (colR - 1)), (1 << (colR - 1)) - 1, rowShift ? Inv::add(Tv[j], 1 << (rowShift - 1)) >> rowShift : Tv[j]);
    return err;
}
template <int LH>
__device__ __forceinline__ uint32_t inv_col(int j, int W, int ck, int bd, lds<int16_t> *res) {
    constexpr int N = 1 << LH;
    int32_t Tv[N];
#pragma unroll
    for (int i = 0; i < N; i++) Tv[i] = res[i * W + j];
    uint32_t err = 0;
    Inv::run<LH>(Tv, ck, bd + 6 > 16 ? bd + 6 : 16, err);
#pragma unroll
    for (int i = 0; i < N; i++) res[i * W + j] = (int16_t)(Inv::add(Tv[i], 8) >> 4);
    return err;
}

// The barrier that closes a block, before one wave publishes it (recon_part).  A workgroup barrier by itself does not wait
// for the waves' stores to global memory (its release is of workgroup scope, which the compute unit's order of
// accesses provides), and the publisher's agent-scope release waits for its own wave's stores only: another wave's store could
// reach the L2 after that write-back and a workgroup on another XCD, which sees the progress word, read the old sample.
// So every wave first waits until its stores have arrived in the L2; the publisher's release then writes them all back.
// The wait costs 0.6 % of the closed loop of a 512 x 512 image (one launch per step: 27.55 -> 27.72 ms); a release by every
// wave in its place, a write-back of the L2 each, made the whole encode of 16 images of 12 MP 142 -> 211 ms.
__device__ __forceinline__ void block_barrier() {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
}

// source of plane p in the staging buffer
__device__ __forceinline__ const lds<uint16_t> *stage_src(const lds<RcShared> &S, int p) { return S.srcb + S.srcAt + (p == 2 ? 2048 : 0); }

// Inlined into each per-shape leaf function (rc_luma / rc_chroma): as a call of its own it would run on the ~140
// registers outside the callee-saved ones and spill; inlined, the leaf function's one frame covers it.
// run S.taskC/T/P[0 .. nTask) on the RC_NG groups (the source staged in S.srcb, row stride S.srcSp); per task
// J = fmaf(lambda, R + extra, D) with extra = luma mode bits (plane 0) or 0; S.taskJ / taskE.  Then S.win = the first
// minimum over the tasks.  Blocks up to 16x16: luma tasks read the residual of their candidate (S.taskK), made by
// wg_luma_residuals; chroma tasks make their own in slot t; levels of task t go to S.u.s.lev[t].  Larger blocks:
// team g (tasks g, g + RC_NTEAM, ..., run in descending order) keeps the levels and prepared edges of task g.
template <int W, int H>
__device__ __forceinline__ void wg_run_tasks(lds<RcShared> &S, const lds<Img> &I, const DevTables &T, const lds<SearchParams> &P, float lambda, bool lumaBits,
                             bool pickWinner) {
    constexpr bool big = W > 16 || H > 16;
    constexpr int LW = W == 4 ? 2 : W == 8 ? 3 : W == 16 ? 4 : W == 32 ? 5 : 6, LH = H == 4 ? 2 : H == 8 ? 3 : H == 16 ? 4 : H == 32 ? 5 : 6;
    if constexpr (!big) {   // the packed levels hold every task: 6 luma candidates x the set's types, or 14 chroma tasks
        constexpr int set = tx_set_intra(tx_of(W, H));
        constexpr int nt = set == TX_SET_INTRA_1 ? 7 : set == TX_SET_INTRA_2 ? 5 : 1;
        static_assert((6 * nt > 14 ? 6 * nt : 14) * W * H <= RC_LEV_TOTAL, "the packed levels cannot hold every task");
    }
    const int g = gid(), lane = glane();
    const lds<CostTab> &C = S.tab.cost;
    // blocks of up to 64 coefficients: 2 RC_NG half groups, two tasks per group at once; luma residuals are ready, chroma
    // tasks first make theirs (one task per group, as below), then the halves evaluate
    constexpr bool halves = !big && W * H <= 64;
    if constexpr (halves) {
        if (!lumaBits) {
            for (int t = g; t < S.nTask; t += RC_NG)
                grp_residual<W, H>(S, I.edgeFilter ? S.u.s.g[g].ea : nullptr, S.u.s.g[g].el, S.taskP[t], S.taskC[t], stage_src(S, S.taskP[t]), S.srcSp,
                             S.u.s.res[t], I.bd);
            __syncthreads();
        }
        // slot -> task with the candidates of one tx type side by side (the luma tasks are candidate-major), so the four
        // halves of a wave mostly run the same kinds of pass
        const int h = lane >> 4, nc = lumaBits && S.nTask % S.nCand == 0 ? S.nCand : 1, nt = S.nTask / nc;
        for (int s = 2 * g + h; s < S.nTask; s += 2 * RC_NG) {
            const int t = (s % nc) * nt + s / nc;
            const int c = S.taskC[t], tt = S.taskT[t], p = S.taskP[t];
            const EvalOut o = half_task<W, H>(S, S.u.s.g[g].tmp + h * 136, I, p, c, tt, S.u.s.res[lumaBits ? S.taskK[t] : t], S.u.s.lev + t * (W * H), P);
            float J;
            if (lumaBits) {
                const int m = cand_mode(c);
                float mb = C.y_mode[S.am][S.lm][m];
                if (S.bsize >= BLOCK_8X8 && is_dir(m)) mb += C.angle_delta[m - V_PRED][cand_delta(c) + 3];
                J = fmaf(lambda, o.R + mb, o.D);
            } else {
                J = fmaf(lambda, o.R, o.D);
            }
            if ((lane & 15) == 0) { S.taskJ[t] = J; S.taskE[t] = o.eob; }
            gsync();
        }
    }
    // big tasks: one per team at a time.  A team keeps the levels and prepared edges of its last task only: it runs its
    // tasks in descending order, so the first tasks -- the analysis's best candidates, the likeliest winners -- are kept
    constexpr int NGT = big ? RC_NTEAM : RC_NG;
    const int me = big ? (int)(threadIdx.x >> 6) : g;
    const int tFirst = big ? (me < S.nTask ? me + ((S.nTask - 1 - me) / NGT) * NGT : -1) : me, tStep = big ? -NGT : NGT;
    if constexpr (!halves) for (int t = tFirst; t >= 0 && t < S.nTask; t += tStep) {
        int c = S.taskC[t], p = S.taskP[t];
        const int tt = S.taskT[t];
        if constexpr (big) { c = __builtin_amdgcn_readfirstlane(c); p = __builtin_amdgcn_readfirstlane(p); }   // the wave's task
        EvalOut o;
        if constexpr (big) {
            o = wave_task<W, H>(S, S.u.b.t[me], me, I, T, p, c, stage_src(S, p), S.srcSp, P);
        } else {
            if (!lumaBits)   // chroma: this task's own residual
                grp_residual<W, H>(S, I.edgeFilter ? S.u.s.g[g].ea : nullptr, S.u.s.g[g].el, p, c, stage_src(S, p), S.srcSp, S.u.s.res[t], I.bd);
            o = grp_task<W, H>(S, S.u.s.g[g], I, p, c, tt, S.u.s.res[lumaBits ? S.taskK[t] : t], S.u.s.lev + t * (W * H), P);
        }
        float J;
        if (lumaBits) {
            const int m = cand_mode(c);
            float mb = C.y_mode[S.am][S.lm][m];
            if (S.bsize >= BLOCK_8X8 && is_dir(m)) mb += C.angle_delta[m - V_PRED][cand_delta(c) + 3];
            J = fmaf(lambda, o.R + mb, o.D);
        } else {
            J = fmaf(lambda, o.R, o.D);
        }
        if (lane == 0) { S.taskJ[t] = J; S.taskE[t] = o.eob; }
        gsync();
    }
    __syncthreads();
    if (S.flopsOn && threadIdx.x < GW) {   // work accounting: the forward transforms of the tasks
        int f = 0;
        for (int t = lane; t < S.nTask; t += GW) f += (int)fwd_flops(W, H, S.taskT[t]);
        f = gsumi(f);
        if (lane == 0) S.flops += (unsigned long long)f;
    }
    if (pickWinner && threadIdx.x < GW) {   // the first minimum over the tasks (at most 64)
        const int n = S.nTask;
        float v = lane < n ? S.taskJ[lane] : INF;
        int i = lane;
        if (lane + GW < n && S.taskJ[lane + GW] < v) { v = S.taskJ[lane + GW]; i = lane + GW; }
        const int w = gargmin(v, i);
        if (lane == 0) S.win = w < 0 ? 0 : w;
    }
    __syncthreads();
}

// luma blocks up to 16x16: the residual of each candidate S.candC[k] into S.u.s.res[k] (group k)
template <int W, int H>
__device__ void wg_luma_residuals(lds<RcShared> &S, const lds<Img> &I) {
    constexpr int LW = W == 4 ? 2 : W == 8 ? 3 : 4, LH = H == 4 ? 2 : H == 8 ? 3 : 4;
    const int g = gid();
    if (g < S.nCand)
        grp_residual<W, H>(S, I.edgeFilter ? S.u.s.g[g].ea : nullptr, S.u.s.g[g].el, 0, S.candC[g], stage_src(S, 0), S.srcSp, S.u.s.res[g], I.bd);
    __syncthreads();
}

// The end of a tx block (luma: NP 1, plane p0 = 0; chroma: NP 2, U and V side by side in the halves of the workgroup, V's
// task t0 + 1 behind U's t0): the winner's levels and prepared edges (a larger block evaluates the task again if its team
// ran another after it), exact dequantization and inverse transform with the conformance repair (spec 7.13.3, 7.12.3
// step 3: halve the levels until no range is violated), prediction + residual written once, then the record: levels, txb
// entry (index txb, + txbStep for V), context maps, BlockDecoded, and what done(eob, lane) adds.  One wave of each half
// keeps the record, so the only barriers are those of the inverse and one at the end.  (px, py): the tx block's first sample in its planes.
template <int W, int H, int NP, typename Px, typename Done>
__device__ __forceinline__ void wg_finish(lds<RcShared> &S, const Batch &B, const lds<SearchParams> &P, const DevTables &T, uint32_t sb, const lds<Img> &I,
                                          int t0, int slot0, int txType, int px, int py, uint32_t txb, uint32_t txbStep, uint32_t coef, Done done) {
    constexpr bool big = W > 16 || H > 16;
    constexpr int LW = W == 4 ? 2 : W == 8 ? 3 : W == 16 ? 4 : W == 32 ? 5 : 6, LH = H == 4 ? 2 : H == 8 ? 3 : H == 16 ? 4 : H == 32 ? 5 : 6;
    constexpr int TW = W > 32 ? 32 : W, TH = H > 32 ? 32 : H, N = TW * TH, txSz = tx_of(W, H), NT = RC_NT / NP;
    static_assert(NP == 1 || (H <= NT && W <= NT && W * H <= 32 * 32), "U and V share the workgroup and the inverse's scratch");
    const int half = NP == 2 ? (int)threadIdx.x / NT : 0, tl = (int)threadIdx.x & (NT - 1);
    const int p = NP == 2 ? 1 + half : 0, t = t0 + half, slot = slot0 + half, bd = I.bd;
    const int team = t % (big ? RC_NTEAM : RC_NG);
    if constexpr (big) {
        if (t0 >= RC_NTEAM) {
            const int wv = (int)(threadIdx.x >> 6);
            const int tw = wv == t0 % RC_NTEAM ? t0 : NP == 2 && wv == (t0 + 1) % RC_NTEAM ? t0 + 1 : -1;
            if (tw >= 0) {
                const int tp = __builtin_amdgcn_readfirstlane(S.taskP[tw]), tc = __builtin_amdgcn_readfirstlane(S.taskC[tw]);
                wave_task<W, H>(S, S.u.b.t[wv], wv, I, T, tp, tc, stage_src(S, tp), S.srcSp, P);
            }
            __syncthreads();
        }
    }
    lds<int16_t> *q = big ? team_lev(S.u.b.t[team]) : S.u.s.lev + t * (W * H);
    static_assert(sizeof(RcGroup::tmp) >= 16 * 16 * 2, "the inverse's scratch of a small block: a group's");
    lds<int16_t> *inv = big ? S.u.b.inv + half * (32 * 32) : (lds<int16_t> *)(lds<char> *)S.u.s.g[half].tmp;
    int eob = S.taskE[t], fixes = 0;
    bool add = eob > 0;
    if (NP == 2 ? (S.taskE[t0] > 0 || S.taskE[t0 + 1] > 0) : add) {
        constexpr int den = (W == 64 && H >= 32) || (H == 64 && W >= 32) ? 4 : W * H > 256 ? 2 : 1;
        const int dsh = den == 4 ? 2 : den == 2 ? 1 : 0, rk = row_kind(txType), ck = col_kind(txType);
        constexpr bool rect = W == 2 * H || H == 2 * W;
        for (;;) {
            uint32_t err = 0;
            if (add && tl < H) err = inv_row<LW>(tl, W, TH, TW, q, S.dcQ, S.acQ, dsh, bd, rect, rk, av1t::Transform_Row_Shift[txSz], inv);
            if (err) atomicOr(gen(&S.errFlag[half]), (int)err);
            __syncthreads();
            err = 0;
            if (add && tl < W) err = inv_col<LH>(tl, W, ck, bd, inv);
            if (err) atomicOr(gen(&S.errFlag[half]), (int)err);
            __syncthreads();
            const int bad = S.errFlag[half];
            if (!(S.errFlag[0] | S.errFlag[1])) break;
            __syncthreads();
            if (tl == 0) { S.errFlag[half] = 0; S.nzFlag[half] = 0; }
            __syncthreads();
            if (bad) {
                fixes++;
                for (int i = tl; i < N; i += NT) {
                    q[i] = (int16_t)(q[i] / 2);
                    if (q[i]) S.nzFlag[half] = 1;
                }
            }
            __syncthreads();
            if (bad && !S.nzFlag[half]) add = false;
        }
        if (fixes && tl == 0) atomicAdd(&B.stats[3], 1u);
    }
    // prediction + residual
    {
        const int maxv = (1 << bd) - 1, fud = flip_ud(txType), flr = flip_lr(txType), pitch = I.pitch[p];
        glb<Px> *dst = rec_plane<Px>(I, p) + (size_t)py * pitch + px;
        if constexpr (big) {
            const int c = S.taskC[t], m = c == 255 ? DC_PRED : cand_mode(c), pa = pangle(m, c == 255 ? 0 : cand_delta(c));
            const bool filt = c != 255 && is_dir(m) && I.edgeFilter;
            const lds<uint16_t> *EA = (filt ? S.u.b.t[team].ea : S.ea[p]) + EDGE_OFF, *EL = (filt ? S.u.b.t[team].el : S.el[p]) + EDGE_OFF;
            const int upA = filt ? S.gup[team][0] : 0, upL = filt ? S.gup[team][1] : 0, dcv = S.dcv[p];
            for (int k = tl; k < W * H; k += NT) {
                const int i = k >> LW, j = k & (W - 1);
                int v;
                if (c == 255) v = clip3(0, maxv, dcv + round2signed(S.cflAlpha[p == 2] * (S.cflL[k] - S.cflAvg), 6));
                else if (m == DC_PRED) v = dcv;
                else v = pred_px(m, pa, i, j, LW, LH, EA, EL, upA, upL, RcPredTables{S.tab});
                if (add) v = clip3(0, maxv, v + inv[k]);   // DCT_DCT: no flips
                dst[(size_t)i * pitch + j] = (Px)v;
            }
        } else {
            const lds<uint16_t> *src = stage_src(S, p);
            const lds<int16_t> *res = S.u.s.res[slot];
            for (int k = tl; k < W * H; k += NT) {
                const int i = k >> LW, j = k & (W - 1);
                int v = (int)src[i * S.srcSp + j] - res[k];
                if (add) v = clip3(0, maxv, v + inv[((fud ? H - 1 - i : i) << LW) + (flr ? W - 1 - j : j)]);
                dst[(size_t)i * pitch + j] = (Px)v;
            }
        }
    }
    // record
    coef += half * (txbStep * N);
    {
        glb<uint32_t> *oc = (glb<uint32_t> *)((glb<int16_t> *)B.oCoeffs + (size_t)sb * B.coefCap + coef);   // coef: a multiple of 16
        const lds<uint32_t> *qw = (const lds<uint32_t> *)(const lds<char> *)q;
        for (int i = tl; i < N / 2; i += NT) oc[i] = qw[i];
    }
    if (tl < 64) {   // a wave
        int cul = 0, last = 0;   // the sum of |level| (before the eob, i.e. over every level: later ones are 0)
        for (int i = tl; i < N; i += 64) { const int v = q[i]; cul += max(v, -v); }
        cul = gsumi(cul);
        cul = min(cul + other_half(cul), 63);
        if (fixes) {   // the eob of the halved levels: 1 + the largest scan index of a nonzero one
            const auto isc = iscan_ptr<txSz>(S.tab);
            const int cls = tx_class(txType);
            for (int i = tl; i < N; i += 64)
                if (q[i]) last = max(last, 1 + (cls == TX_CLASS_2D ? (int)isc[i] : cls == TX_CLASS_VERT ? i : (i % TW) * TH + i / TW));
            last = gmaxi(last);
            eob = max(last, other_half(last));
        }
        const int dcCat = q[0] < 0 ? 1 : q[0] > 0 ? 2 : 0;
        const int ss = p ? I.ss : 0, stride = I.MiCols >> ss, rows = I.MiRows >> ss, x4 = px >> 2, y4 = py >> 2;
        const int r4 = y4 & ((16 >> ss) - 1), c4 = x4 & ((16 >> ss) - 1);
        constexpr int W4 = W / 4, H4 = H / 4, LW4 = LW - 2;
        for (int k = tl; k < W4 * H4; k += 64) {
            const int yy = k >> LW4, xx = k & (W4 - 1);
            if (y4 + yy < rows && x4 + xx < stride) {
                map8(I.cLvl[p])[(size_t)(y4 + yy) * stride + x4 + xx] = (uint8_t)(eob ? cul : 0);
                map8(I.cDc[p])[(size_t)(y4 + yy) * stride + x4 + xx] = (uint8_t)(eob ? dcCat : 0);
            }
            S.bdm[p][r4 + yy + 1][c4 + xx + 1] = 1;
        }
        if (tl == 0) {
            RecTxb r;
            r.coeff_off = coef; r.x4 = (uint16_t)x4; r.y4 = (uint16_t)y4; r.plane = (uint8_t)p; r.tx_size = (uint8_t)txSz;
            r.tx_type = (uint8_t)(p == 0 && eob == 0 ? DCT_DCT : txType); r.flags = 0; r.eob = (uint16_t)eob; r.reserved = 0;
            B.oTxb[(size_t)sb * B.txbCap + txb + half * txbStep] = r;
            S.winEob[p] = eob;
        }
        done(eob, tl);
    }
    block_barrier();
}

template <int W, int H, typename Px>
__device__ __noinline__ void rc_luma(lds<RcShared> &S, const Batch &B, const lds<SearchParams> &P, uint32_t sb, const lds<Img> &I, int bsize, int x, int y, int availU,
                        int availL, int tx0, int ty0, float lambda, int li, int hasC, uint32_t txb, uint32_t coef) {
    constexpr int LW = W == 4 ? 2 : W == 8 ? 3 : W == 16 ? 4 : W == 32 ? 5 : 6, LH = H == 4 ? 2 : H == 8 ? 3 : H == 16 ? 4 : H == 32 ? 5 : 6;
    const DevTables &T = *B.T;
    const int tid = threadIdx.x, txSz = tx_of(W, H);
    const int sbr4 = (y >> 2) & 15, sbc4 = (x >> 2) & 15, mi_row = y >> 2, mi_col = x >> 2;
    if (gid() == 0)
        rc_edges<Px>(S, I, 0, x, y, LW, LH, availL, availU, S.bdm[0][sbr4][sbc4 + (W >> 2) + 1], S.bdm[0][sbr4 + (H >> 2) + 1][sbc4],
                     mi_row, mi_col);
    if (gid() == 2) grp_txb_ctx(I, 0, txSz, mi_col, mi_row, bsize, tx0, ty0, &S.skipCtx[0], &S.dcCtx[0]);
    if (tid >= 128 && tid < 192) {   // wave 2: the tasks (candidate k, tx type t), k-major, types ascending
        const int w = tid - 128;
        const lds<BlockCand> &br = *(const lds<BlockCand> *)(const lds<char> *)S.cand[li];
        const int nc = max(1, min((int)br.ncand, P.Krecheck));
        const int set = tx_set_intra(txSz);
        if (w < nc) S.candC[w] = br.cand[w];
        if (w == 0) {
            S.am = av1t::Intra_Mode_Context[availU ? map8(I.mY)[(size_t)(mi_row - 1) * I.MiCols + mi_col] : DC_PRED];
            S.lm = av1t::Intra_Mode_Context[availL ? map8(I.mY)[(size_t)mi_row * I.MiCols + mi_col - 1] : DC_PRED];
            S.nCand = nc;
            S.bsize = bsize;
        }
        if (P.txAllCL && set != TX_SET_DCTONLY) {
            // every pair at once: with nt types in the set, pair (k, t) is task k * nt + (types of the set below t)
            uint32_t sm = 0;
            for (int t = 0; t < 16; t++) sm |= tx_in_set(set, t) ? 1u << t : 0u;
            const int nt = __popc(sm);
            for (int i = w; i < nc * 16; i += 64) {
                const int k = i >> 4, t = i & 15;
                if ((sm >> t) & 1) {
                    const int n = k * nt + __popc(sm & ((1u << t) - 1));
                    S.taskC[n] = br.cand[k]; S.taskT[n] = t; S.taskP[n] = 0; S.taskK[n] = k;
                }
            }
            if (w == 0) S.nTask = nc * nt;
        } else if (w == 0) {
            int n = 0;
            for (int k = 0; k < nc; k++) { S.taskC[n] = br.cand[k]; S.taskT[n] = DCT_DCT; S.taskP[n] = 0; S.taskK[n] = k; n++; }
            if (br.tx != DCT_DCT) { S.taskC[n] = br.cand[0]; S.taskT[n] = br.tx; S.taskP[n] = 0; S.taskK[n] = 0; n++; }
            S.nTask = n;
        }
    }
    __syncthreads();
    if constexpr (W <= 16 && H <= 16) wg_luma_residuals<W, H>(S, I);
    wg_run_tasks<W, H>(S, I, T, P, lambda, true, true);
    if (!(P.txAllCL && tx_set_intra(txSz) != TX_SET_DCTONLY) && P.txSearchCL && tx_set_intra(txSz) != TX_SET_DCTONLY) {
        // tx-type pass for the pass-1 winner (txAllCL off): the other types of the set
        if (tid == 0) {
            const int c0 = S.taskC[S.win], k0 = S.taskK[S.win], n0 = S.nTask;
            const lds<BlockCand> &br = *(const lds<BlockCand> *)(const lds<char> *)S.cand[li];
            int n = n0;
            for (int t = 1; t < 16; t++)
                if (tx_in_set(tx_set_intra(txSz), t) && !(c0 == br.cand[0] && t == br.tx)) {
                    S.taskC[n] = c0; S.taskT[n] = t; S.taskP[n] = 0; S.taskK[n] = k0; n++;
                }
            S.nTask = n;
        }
        __syncthreads();
        wg_run_tasks<W, H>(S, I, T, P, lambda, true, true);
    }
    const int win = S.win, yMode = cand_mode(S.taskC[win]), yDelta = cand_delta(S.taskC[win]);
    // the 4x4 maps and the block's record (the chroma item completes that of a block that carries chroma), with the tx
    // block's own record, so that the block ends at one barrier
    constexpr int W4 = W / 4, H4 = H / 4;
    auto each4x4 = [&](int l0, int dl, auto f) {
        for (int k = l0; k < W4 * H4; k += dl) {
            const int r = mi_row + (k >> (LW - 2)), c = mi_col + (k & (W4 - 1));
            if (r < I.MiRows && c < I.MiCols) f((size_t)r * I.MiCols + c);
        }
    };
    each4x4(tid, RC_NT, [&](size_t o) { map8(I.mY)[o] = (uint8_t)yMode; map8(I.mMiSize)[o] = (uint8_t)bsize; map8(I.mTx)[o] = (uint8_t)txSz; });
    wg_finish<W, H, 1, Px>(S, B, P, T, sb, I, win, S.taskK[win], S.taskT[win], x, y, txb, 0, coef, [&](int eob, int l) {
        const int skip = eob == 0;
        if (!hasC) each4x4(l, 64, [&](size_t o) { map8(I.mSkip)[o] = (uint8_t)skip; });
        if (l == 0) {
            RecBlock b;
            b.mi_row = (uint16_t)mi_row; b.mi_col = (uint16_t)mi_col; b.bsize = (uint8_t)bsize; b.skip = (uint8_t)skip; b.tx_depth = 0;
            b.y_mode = (uint8_t)yMode;
            b.angle_delta_y = (int8_t)(bsize >= BLOCK_8X8 && is_dir(yMode) ? yDelta : 0);
            b.uv_mode = 0; b.angle_delta_uv = 0; b.cfl_alpha_u = 0; b.cfl_alpha_v = 0;
            b.filter_intra = 0; b.cdef_idx = 0; b.sb_qindex = 0;
            B.oBlocks[(size_t)sb * MAX_LEAVES + li] = b;
            B.oBlockTxb[(size_t)sb * MAX_LEAVES + li] = (uint16_t)txb;
            if (skip && !hasC) S.nSkip++;
        }
    });
}

template <int W, int H, typename Px>
__device__ __noinline__ void rc_chroma(lds<RcShared> &S, const Batch &B, const lds<SearchParams> &P, uint32_t sb, const lds<Img> &I, int bsize, int mi_row, int mi_col,
                          int availUC, int availLC, int tx0, int ty0, float lambda, uint32_t txb, uint32_t coef, int nTxb) {
    constexpr int LW = W == 4 ? 2 : W == 8 ? 3 : W == 16 ? 4 : W == 32 ? 5 : 6, LH = H == 4 ? 2 : H == 8 ? 3 : H == 16 ? 4 : H == 32 ? 5 : 6;
    const DevTables &T = *B.T;
    const lds<CostTab> &C = S.tab.cost;
    const int tid = threadIdx.x, ss = I.ss, bd = I.bd, txSz = tx_of(W, H);
    const int cx = (mi_col >> ss) * 4, cy = (mi_row >> ss) * 4, x4 = cx >> 2, y4 = cy >> 2;
    const int sbr4 = (mi_row & 15) >> ss, sbc4 = (mi_col & 15) >> ss;
    if (gid() < 2) {
        const int p = 1 + gid();
        rc_edges<Px>(S, I, p, cx, cy, LW, LH, availLC, availUC, S.bdm[p][sbr4][sbc4 + (W >> 2) + 1], S.bdm[p][sbr4 + (H >> 2) + 1][sbc4],
                     mi_row, mi_col);
    }
    if (gid() == 2) grp_txb_ctx(I, 1, txSz, x4, y4, bsize, tx0, ty0, &S.skipCtx[1], &S.dcCtx[1]);
    if (gid() == 3) grp_txb_ctx(I, 2, txSz, x4, y4, bsize, tx0, ty0, &S.skipCtx[2], &S.dcCtx[2]);
    if (!ss) {   // (4:2:0: the superblock's chroma is there)
        const glb<Px> *gU = src_plane<Px>(I, 1) + (size_t)cy * I.spitch[1] + cx, *gV = src_plane<Px>(I, 2) + (size_t)cy * I.spitch[2] + cx;
        for (int q = tid; q < W * H; q += RC_NT) {
            S.srcb[q] = gU[(size_t)(q >> LW) * I.spitch[1] + (q & (W - 1))];
            S.srcb[2048 + q] = gV[(size_t)(q >> LW) * I.spitch[2] + (q & (W - 1))];
        }
    }
    if (tid < 32) S.satdI[tid] = 0;
    if (tid < 8) S.acc64[tid] = 0;
    if (tid < 13) S.uvc[tid] = cand_pack(tid, 0);
    // CfL of up to 256 samples: the last wave alone, up to 4 samples a lane.  Here their luma and its average; the alphas
    // while wave 0 chooses the deltas to screen (they are read from the ranking on).  Every sum fits in 32 bits: at 10 bits
    // |l| <= 8184 gives |l x residual| x 256 < 2^31; the squared deviations of values in 0 .. 8184 from their rounded mean
    // are at most 4092^2 + 1/4 on average, 256 of them < 2^32.  In steps of its own with 64-bit shuffles this took 20% of
    // a chroma block, and a 4:4:4 image waits for its chroma: closed loop of one of 1021 x 767, 10 bits, 20.2 -> 17.6 ms,
    // of nine 36.4 -> 31.8 ms.
    constexpr bool CFLW = W * H <= 256;
    constexpr int NPL = W * H <= 64 ? 1 : CFLW ? W * H / 64 : 1;
    const bool cflOk = P.cfl && cfl_allowed(bsize), cflWave = tid >= RC_NT - 64;
    const int cl = tid & 63;
    int cv[NPL], cavg = 0;
    if constexpr (CFLW) if (cflOk && cflWave) {
        const int lt = av1t::Max_Tx_Size_Rect[bsize], tw = tx_w(lt), th = tx_h(lt);
        int maxLumaW = 0, maxLumaH = 0;
        for (int ly = mi_row * 4; ly < mi_row * 4 + 4 * bh4(bsize); ly += th)
            for (int lx = mi_col * 4; lx < mi_col * 4 + 4 * bw4(bsize); lx += tw)
                if (lx < I.MiCols * 4 && ly < I.MiRows * 4) { maxLumaW = lx + tw; maxLumaH = ly + th; }
        const glb<Px> *luma = rec_plane<Px>(I, 0);
        const int lp = I.pitch[0];
        int sum = 0;
#pragma unroll
        for (int k = 0; k < NPL; k++) {
            const int q = cl + 64 * k, i = q >> LW, j = q & (W - 1);
            cv[k] = 0;
            if (W * H >= 64 || q < W * H) {
                if (ss) {
                    const int ly = min((cy + i) << 1, maxLumaH - 2), lx = min((cx + j) << 1, maxLumaW - 2);
                    const glb<Px> *r = luma + (size_t)ly * lp + lx;
                    cv[k] = ((int)r[0] + r[1] + r[lp] + r[lp + 1]) << 1;
                } else {
                    cv[k] = (int)luma[(size_t)min(cy + i, maxLumaH - 1) * lp + min(cx + j, maxLumaW - 1)] << 3;
                }
                S.cflL[q] = cv[k];
            }
            sum += cv[k];
        }
        cavg = round2(wsumi(sum), LW + LH);
    }
    __syncthreads();
    const int sp = S.srcSp;
    const lds<uint16_t> *srcU = stage_src(S, 1), *srcV = stage_src(S, 2);
    const float lamS = P.satdLambda * T.lamS[bd == 10][I.qindex];   // the luma lambda's screening weight
    const int yMode = S.mode;
    auto uvbits = [&](int m) -> float { return cfl_allowed(bsize) ? C.uv_cfl_yes[yMode][m] : C.uv_cfl_no[yMode][m < 13 ? m : 0]; };
    auto uvcbits = [&](int c) -> float {
        const int m = cand_mode(c);
        float b = uvbits(m);
        if (bsize >= BLOCK_8X8 && is_dir(m)) b += C.angle_delta[m - V_PRED][cand_delta(c) + 3];
        return b;
    };
    // ---- CfL: least-squares alpha, +-1 refinement by exact SSE ----
    auto wave_cfl = [&] {   // CFLW: by the last wave, from the samples it holds
        int nU = 0, nV = 0;
        uint32_t dd = 0;
#pragma unroll
        for (int k = 0; k < NPL; k++) {
            const int q = cl + 64 * k, i = q >> LW, j = q & (W - 1), l = cv[k] - cavg;
            if (W * H >= 64 || q < W * H) {
                nU += l * ((int)srcU[i * sp + j] - S.dcv[1]);
                nV += l * ((int)srcV[i * sp + j] - S.dcv[2]);
                dd += (uint32_t)(l * l);
            }
        }
        nU = wsumi(nU); nV = wsumi(nV); dd = (uint32_t)wsumi((int)dd);
        int alpha[2], sse[6] = {0, 0, 0, 0, 0, 0};
#pragma unroll
        for (int pl = 0; pl < 2; pl++) {
            const int a = dd > 0 ? (int)rintf(64.f * (float)(pl ? nV : nU) / (float)dd) : 0;
            alpha[pl] = max(-16, min(16, a));
        }
#pragma unroll
        for (int k = 0; k < NPL; k++) {
            const int q = cl + 64 * k, i = q >> LW, j = q & (W - 1), l = cv[k] - cavg;
            if (W * H >= 64 || q < W * H)
#pragma unroll
                for (int c = 0; c < 6; c++) {
                    const int pl = c / 3, a = max(-16, min(16, alpha[pl] + c % 3 - 1));
                    const int d = (int)(pl ? srcV : srcU)[i * sp + j] - clip3(0, (1 << bd) - 1, S.dcv[pl + 1] + round2signed(a * l, 6));
                    sse[c] += d * d;
                }
        }
#pragma unroll
        for (int c = 0; c < 6; c++) sse[c] = wsumi(sse[c]);
        if (cl == 0) {
            S.cflAvg = cavg;
#pragma unroll
            for (int pl = 0; pl < 2; pl++) {
                int bk = 1;
#pragma unroll
                for (int k = 0; k < 3; k++) if (sse[pl * 3 + k] < (bk == 0 ? sse[pl * 3] : sse[pl * 3 + 1])) bk = k;
                S.cflAlpha[pl] = max(-16, min(16, alpha[pl] + bk - 1));
            }
        }
    };
    if (tid == 0 && (!CFLW || !cflOk)) S.cflAlpha[0] = S.cflAlpha[1] = 0;
    if constexpr (!CFLW) if (cflOk) {
        const int lt = av1t::Max_Tx_Size_Rect[bsize], tw = tx_w(lt), th = tx_h(lt);
        int maxLumaW = 0, maxLumaH = 0;
        for (int ly = mi_row * 4; ly < mi_row * 4 + 4 * bh4(bsize); ly += th)
            for (int lx = mi_col * 4; lx < mi_col * 4 + 4 * bw4(bsize); lx += tw)
                if (lx < I.MiCols * 4 && ly < I.MiRows * 4) { maxLumaW = lx + tw; maxLumaH = ly + th; }
        const glb<Px> *luma = rec_plane<Px>(I, 0);
        const int lp = I.pitch[0];
        int sum = 0;
        for (int q = tid; q < W * H; q += RC_NT) {
            const int i = q >> LW, j = q & (W - 1);
            int v;
            if (ss) {
                const int ly = min((cy + i) << 1, maxLumaH - 2), lx = min((cx + j) << 1, maxLumaW - 2);
                v = ((int)luma[(size_t)ly * lp + lx] + luma[(size_t)ly * lp + lx + 1] + luma[(size_t)(ly + 1) * lp + lx] + luma[(size_t)(ly + 1) * lp + lx + 1]) << 1;
            } else {
                v = (int)luma[(size_t)min(cy + i, maxLumaH - 1) * lp + min(cx + j, maxLumaW - 1)] << 3;
            }
            S.cflL[q] = v;
            sum += v;
        }
        sum = gsumi(sum);
        if (glane() == 0) atomicAdd(gen(&S.satdI[31]), sum);
        __syncthreads();
        if (tid == 0) S.cflAvg = round2(S.satdI[31], LW + LH);
        __syncthreads();
        long long nU = 0, nV = 0, dd = 0;
        for (int q = tid; q < W * H; q += RC_NT) {
            const int i = q >> LW, j = q & (W - 1);
            const long long l = S.cflL[q] - S.cflAvg;
            nU += l * ((int)srcU[i * sp + j] - S.dcv[1]);
            nV += l * ((int)srcV[i * sp + j] - S.dcv[2]);
            dd += l * l;
        }
        nU = gsuml(nU); nV = gsuml(nV); dd = gsuml(dd);
        if (glane() == 0) {
            atomicAdd(gen(&S.acc64[0]), (unsigned long long)nU);
            atomicAdd(gen(&S.acc64[1]), (unsigned long long)nV);
            atomicAdd(gen(&S.acc64[2]), (unsigned long long)dd);
        }
        __syncthreads();
        if (tid == 0) {
            const long long d = (long long)S.acc64[2];
            for (int k = 0; k < 2; k++) {
                const long long n = (long long)S.acc64[k];
                const int a = d > 0 ? (int)rintf(64.f * (float)n / (float)d) : 0;
                S.cflAlpha[k] = max(-16, min(16, a));
            }
            for (int k = 0; k < 6; k++) S.acc64[2 + k] = 0;
        }
        __syncthreads();
        long long sse[6] = {0, 0, 0, 0, 0, 0};
        for (int q = tid; q < W * H; q += RC_NT) {
            const int i = q >> LW, j = q & (W - 1), l = S.cflL[q] - S.cflAvg;
#pragma unroll
            for (int pl = 0; pl < 2; pl++) {
                const int s = pl == 0 ? srcU[i * sp + j] : srcV[i * sp + j];
#pragma unroll
                for (int k = 0; k < 3; k++) {
                    const int a = max(-16, min(16, S.cflAlpha[pl] + k - 1));
                    const int d = s - clip3(0, (1 << bd) - 1, S.dcv[pl + 1] + round2signed(a * l, 6));
                    sse[pl * 3 + k] += (long long)d * d;
                }
            }
        }
#pragma unroll
        for (int k = 0; k < 6; k++) {
            const long long v = gsuml(sse[k]);
            if (glane() == 0) atomicAdd(gen(&S.acc64[2 + k]), (unsigned long long)v);
        }
        __syncthreads();
        if (tid == 0)
            for (int pl = 0; pl < 2; pl++) {
                int bk = 1;
                for (int k = 0; k < 3; k++) if ((long long)S.acc64[2 + pl * 3 + k] < (long long)S.acc64[2 + pl * 3 + bk]) bk = k;
                S.cflAlpha[pl] = max(-16, min(16, S.cflAlpha[pl] + bk - 1));
            }
        if (tid < 32) S.satdI[tid] = 0;
        __syncthreads();
    }
    // ---- SATD screening of the UV candidates over U and V (unfiltered edges) ----
    constexpr int NSUB = (W / 4) * (H / 4), NSX = W / 4;
    // screening of blocks of up to 16 4x4s: item = (candidate, plane, pixel or run of pixels), 16 lanes per 4x4 and the
    // Hadamard across them, so a wave holds at most two candidates (modes); larger blocks: item = (candidate, plane, 4x4).
    // A candidate's items are consecutive, so each segment of up to 32 lanes sums its costs across lanes before one LDS
    // atomic.
    auto screen = [&](int c0, int c1) {
        constexpr int NSY = NSUB / NSX;
        if constexpr (NSUB <= 16 && NSY >= 2) {
            // item = (candidate, plane, 4x4 column, pixel of the 4x4): each thread predicts a vertical run of pred_col
            // through the column's NSY 4x4s at its (row, column) = ((t >> 2) & 3, t & 3); each 4x4's Hadamard runs
            // across the 16 lanes holding it; a (candidate, plane) spans NSX x 16 consecutive threads (a whole wave
            // for 16-wide blocks), so a round holds few modes
            constexpr int TPC = NSX * 16, SEG = TPC < GW ? TPC : GW;
            const int items = (c1 - c0) * 2 * TPC;
            for (int base = 0; base < items; base += RC_NT) {
                const int it = base + tid;
                int d[NSY], ci = c0;
#pragma unroll
                for (int k = 0; k < NSY; k++) d[k] = 0;
                if (it < items) {
                    ci = c0 + it / (2 * TPC);
                    const int rr = it % (2 * TPC), p = 1 + rr / TPC, q = rr % TPC;
                    const int sx = (q >> 4) * 4 + (q & 3), sy0 = (q >> 2) & 3;
                    const int c = S.uvc[ci], m = cand_mode(c), pa = pangle(m, cand_delta(c));
                    const lds<uint16_t> *s = p == 1 ? srcU : srcV;
                    const lds<uint16_t> *A = S.ea[p] + EDGE_OFF, *L = S.el[p] + EDGE_OFF;
                    int pr[NSY];
                    pred_col(m, pa, S.dcv[p], sy0, 4, sx, LW, LH, A, L, 0, 0, pr, RcPredTables{S.tab});
#pragma unroll
                    for (int k = 0; k < NSY; k++) d[k] = (int)s[(sy0 + 4 * k) * sp + sx] - pr[k];
                }
                int v = 0;
#pragma unroll
                for (int k = 0; k < NSY; k++) v += hadamard4_lanes(d[k]);
                v = seg_sumi<SEG>(v);
                if (it < items && (it & (SEG - 1)) == 0) atomicAdd(gen(&S.satdI[ci]), v);
            }
            __syncthreads();
            return;
        }
        if constexpr (NSUB <= 16) {
            constexpr int PIX = NSUB * 16;
            const int items = (c1 - c0) * PIX * 2;
            for (int base = 0; base < items; base += RC_NT) {
                const int it = base + tid;
                int v = 0, ci = c0;
                if (it < items) {
                    ci = c0 + it / (2 * PIX);
                    const int rr = it % (2 * PIX), p = 1 + rr / PIX, px = rr % PIX, sbk = px >> 4;
                    const int sx = (sbk % NSX) * 4 + (px & 3), sy = (sbk / NSX) * 4 + ((px >> 2) & 3);
                    const int c = S.uvc[ci], m = cand_mode(c), pa = pangle(m, cand_delta(c));
                    const lds<uint16_t> *s = p == 1 ? srcU : srcV;
                    const lds<uint16_t> *A = S.ea[p] + EDGE_OFF, *L = S.el[p] + EDGE_OFF;
                    const int pr = m == DC_PRED ? S.dcv[p] : pred_px(m, pa, sy, sx, LW, LH, A, L, 0, 0, RcPredTables{S.tab});
                    v = (int)s[sy * sp + sx] - pr;
                }
                v = seg_sumi<GW>(hadamard4_lanes(v));
                if (it < items && (it & (GW - 1)) == 0) atomicAdd(gen(&S.satdI[ci]), v);
            }
            __syncthreads();
            return;
        }
        constexpr int SEG = 2 * NSUB < GW ? 2 * NSUB : GW;
        const int items = (c1 - c0) * NSUB * 2;
        for (int base = 0; base < items; base += RC_NT) {
            const int it = base + tid;
            int v = 0, ci = c0;
            if (it < items) {
                ci = c0 + it / (2 * NSUB);
                const int rr = it % (2 * NSUB), p = 1 + rr / NSUB, sbk = rr % NSUB;
                const int sx = (sbk % NSX) * 4, sy = (sbk / NSX) * 4, c = S.uvc[ci], m = cand_mode(c), pa = pangle(m, cand_delta(c));
                const lds<uint16_t> *s = p == 1 ? srcU : srcV;
                const lds<uint16_t> *A = S.ea[p] + EDGE_OFF, *L = S.el[p] + EDGE_OFF;
                int d[16], r[16];
                pred_4x4(m, pa, S.dcv[p], sy, sx, LW, LH, A, L, r, RcPredTables{S.tab});
#pragma unroll
                for (int i = 0; i < 4; i++)
#pragma unroll
                    for (int j = 0; j < 4; j++) d[i * 4 + j] = (int)s[(sy + i) * sp + sx + j] - r[i * 4 + j];
                v = hadamard4(d);
            }
            v = seg_sumi<SEG>(v);
            if (it < items && (it & (SEG - 1)) == 0) atomicAdd(gen(&S.satdI[ci]), v);
        }
        __syncthreads();
    };
    screen(0, 13);
    if (tid < GW) {   // the deltas around the best directional mode (first minimum of the screening cost)
        const bool dl = P.uvDeltas && bsize >= BLOCK_8X8;
        if (dl) {
            const float j = tid < 8 ? fmaf(lamS, uvcbits(cand_pack(V_PRED + tid, 0)), (float)S.satdI[V_PRED + tid] * 0.25f) : INF;
            const int bm = V_PRED + gargmin(j, tid);
            if (tid < 6) S.uvc[13 + tid] = cand_pack(bm, tid < 3 ? -(tid + 1) : tid - 2);
        }
        if (tid == 0) S.nuv = dl ? 19 : 13;
    }
    if constexpr (CFLW) if (cflOk && cflWave) wave_cfl();
    __syncthreads();
    if (S.nuv > 13) screen(13, 19);
    if (tid < GW) {   // the uvK candidates of smallest screening cost (first minimum each round), U and V tasks each
        // taken at once: a candidate's place in that order is its rank under (cost, index), so the ones of rank < K
        // (finite cost) are the rounds' picks and rank k fills tasks 2k (U) and 2k + 1 (V)
        const int l = tid, nuv = S.nuv, K = max(1, min(P.uvK, 6));
        const float js = l < nuv ? fmaf(lamS, uvcbits(S.uvc[l]), (float)S.satdI[l] * 0.25f) : INF;
        S.uvJ[l] = js;
        gsync();
        int rank = 0, fin = 0;
#pragma unroll
        for (int j = 0; j < 19; j++) {   // candidates past nuv are INF
            const float o = S.uvJ[j];
            rank += (o < js || (o == js && j < l)) ? 1 : 0;
            fin += o < INF ? 1 : 0;
        }
        if (js < INF && rank < K) {
            const int c = S.uvc[l], tt = chroma_tx_type(txSz, cand_mode(c));
            S.taskC[2 * rank] = c; S.taskT[2 * rank] = tt; S.taskP[2 * rank] = 1;
            S.taskC[2 * rank + 1] = c; S.taskT[2 * rank + 1] = tt; S.taskP[2 * rank + 1] = 2;
        }
        int n = 2 * min(K, fin);
        if (cflOk && (S.cflAlpha[0] || S.cflAlpha[1])) {
            if (l < 2) { S.taskC[n + l] = 255; S.taskT[n + l] = chroma_tx_type(txSz, UV_CFL_PRED); S.taskP[n + l] = 1 + l; }
            n += 2;
        }
        if (l == 0) S.nTask = n;
    }
    __syncthreads();
    wg_run_tasks<W, H>(S, I, T, P, lambda, false, false);
    if (tid < GW) {   // pick: the first minimum over the (U, V) task pairs of J_U + J_V + lambda * mode bits
        const int l = tid;
        float J = INF;
        if (2 * l + 1 < S.nTask) {
            const int t = 2 * l, c = S.taskC[t];
            J = S.taskJ[t] + S.taskJ[t + 1];
            if (c == 255) {
                const int aU = S.cflAlpha[0], aV = S.cflAlpha[1];
                const int sU = aU == 0 ? 0 : aU < 0 ? 1 : 2, sV = aV == 0 ? 0 : aV < 0 ? 1 : 2;
                float b = uvbits(UV_CFL_PRED) + C.cfl_sign[sU * 3 + sV - 1];
                if (sU) b += C.cfl_alpha[(sU - 1) * 3 + sV][abs(aU) - 1];
                if (sV) b += C.cfl_alpha[(sV - 1) * 3 + sU][abs(aV) - 1];
                J = fmaf(lambda, b, J);
            } else {
                J = fmaf(lambda, uvcbits(c), J);
            }
        }
        const int w = gargmin(J, l), bt = 2 * (w < 0 ? 0 : w);
        if (l == 0) {
            S.win = bt;
            const int c = S.taskC[bt];
            S.uvMode = c == 255 ? UV_CFL_PRED : cand_mode(c);
            S.uvDelta = c == 255 ? 0 : cand_delta(c);
        }
    }
    __syncthreads();
    // 4:4:4 blocks with a 64-sample side hold several chroma tx blocks per plane (raster order, U's then V's in the record):
    // the decision above is the first one's; each further one gets its edges from the reconstruction, its own contexts and
    // a closed-loop final quantization with the chosen mode, and is not coded outside the coded area
    const int win = S.win, uvTxType = S.taskT[win], winC = S.taskC[win];
    const uint32_t perPlane = (uint32_t)nTxb / 2;
    wg_finish<W, H, 2, Px>(S, B, P, T, sb, I, win, win, uvTxType, cx, cy, txb, perPlane, coef, [](int, int) {});
    // only a chroma tx block with a 32-sample side belongs to a 64-sided 4:4:4 block
    if constexpr (W == 32 || H == 32) if (perPlane > 1) {
        const int nTxX = (4 * bw4(bsize)) / W, nTxY = (4 * bh4(bsize)) / H;
        int eobU = S.winEob[1], eobV = S.winEob[2];
        uint32_t n = 0;
        for (int k = 1; k < nTxX * nTxY; k++) {
            const int ox = (k % nTxX) * W, oy = (k / nTxX) * H;
            if (x4 + (ox >> 2) >= I.MiCols || y4 + (oy >> 2) >= I.MiRows) continue;
            n++;
            const int r4 = sbr4 + (oy >> 2), c4 = sbc4 + (ox >> 2);
            if (gid() < 2) {
                const int p = 1 + gid();
                rc_edges<Px>(S, I, p, cx + ox, cy + oy, LW, LH, availLC || ox > 0, availUC || oy > 0, S.bdm[p][r4][c4 + (W >> 2) + 1],
                             S.bdm[p][r4 + (H >> 2) + 1][c4], mi_row, mi_col, availUC, availLC);
            }
            if (gid() == 2 || gid() == 3) {
                const int p = gid() - 1;
                grp_txb_ctx(I, p, txSz, x4 + (ox >> 2), y4 + (oy >> 2), bsize, tx0, ty0, &S.skipCtx[p], &S.dcCtx[p]);
            }
            for (int p = 1; p <= 2; p++) {
                lds<uint16_t> *sd = S.srcb + (p == 2 ? 2048 : 0);
                const glb<Px> *g = src_plane<Px>(I, p) + (size_t)(cy + oy) * I.spitch[p] + cx + ox;
                for (int i = tid; i < W * H; i += RC_NT) sd[i] = g[(size_t)(i >> LW) * I.spitch[p] + (i & (W - 1))];
            }
            if (tid < 2) { S.taskC[tid] = winC; S.taskT[tid] = uvTxType; S.taskP[tid] = 1 + tid; }
            if (tid == 0) S.nTask = 2;
            __syncthreads();
            wg_run_tasks<W, H>(S, I, T, P, lambda, false, false);
            wg_finish<W, H, 2, Px>(S, B, P, T, sb, I, 0, 0, uvTxType, cx + ox, cy + oy, txb + n, perPlane, coef + n * tx_ncoef(txSz), [](int, int) {});
            eobU |= S.winEob[1]; eobV |= S.winEob[2];
        }
        __syncthreads();
        if (tid == 0) { S.winEob[1] = eobU; S.winEob[2] = eobV; }
        __syncthreads();
    }
}

// stage the cost tables of quantizer context qctx (and, when first, the tables of every image) in LDS
__device__ void stage_tables(lds<RcShared> &S, const DevTables &T, const SearchParams &P, int qctx, bool first) {
    const int tid = threadIdx.x;
    static_assert(sizeof(CostTab) % 4 == 0, "the cost tables are floats");
    {
        const float *c = (const float *)&T.cost[qctx];
        lds<float> *d = (lds<float> *)(lds<char> *)&S.tab.cost;
        for (int k = tid; k < (int)(sizeof(CostTab) / 4); k += RC_NT) d[k] = c[k];
    }
    if (first) {
        if (tid == 0) S.tab.iscan = T.iscan;
        if (tid < (int)(sizeof(SearchParams) / 4)) ((lds<uint32_t> *)(lds<char> *)&S.prm)[tid] = ((const uint32_t *)&P)[tid];
        for (int k = tid; k < 3 * 336; k += RC_NT) {
            const int kind = k / 336, r = k % 336, ln = r < 16 ? 2 : r < 80 ? 3 : 4, e = r - (ln == 2 ? 0 : ln == 3 ? 16 : 80);
            S.tab.fwdT[k] = T.fwdT[T.fwdOff[kind][ln] + e];
        }
        if (tid < 21) S.tab.fwdOff[tid / 7][tid % 7] = (tid / 7) * 336 + ((tid % 7) == 3 ? 16 : (tid % 7) == 4 ? 80 : 0);
        if (tid < 19) S.tab.txScale[tid] = T.txScale[tid];
        for (int k = tid; k < 19 * 16; k += RC_NT) S.tab.txg[k / 16][k % 16] = T.txg[k / 16][k % 16];
        for (int k = tid; k < 19 * 25; k += RC_NT) S.tab.cbOff[k / 25][k % 25] = (&av1t::Coeff_Base_Ctx_Offset[0][0][0])[k];
        if (tid < 90) S.tab.step[tid] = av1t::Dr_Intra_Derivative[tid];
        if (tid >= 4 && tid < 128) S.tab.smooth[tid - 4] = sm_weights(31 - __clz(tid))[tid - (1 << (31 - __clz(tid)))];
        for (int k = tid; k < SCAN8_TOTAL; k += RC_NT) { S.tab.scan8[k] = T.scan8[k]; S.tab.iscan8[k] = T.iscan8[k]; }
    }
}

// number and coefficients of the chroma tx blocks of a block that carries chroma (4:4:4 blocks with a 64-sample side hold
// several per plane, coded where they start inside the coded area; the first always)
__device__ __forceinline__ void chroma_size(const lds<Img> &I, int bsize, int mi_row, int mi_col, int &nTxb, int &nCoef) {
    const int t = uv_tx_size(bsize, I.ss), w4 = tx_w(t) >> 2, h4 = tx_h(t) >> 2;
    int n = 1;
    if (!I.ss && (bw4(bsize) > w4 || bh4(bsize) > h4)) {
        n = 0;
        for (int y = 0; y < bh4(bsize); y += h4)
            for (int x = 0; x < bw4(bsize); x += w4) n += (x == 0 && y == 0) || (mi_col + x < I.MiCols && mi_row + y < I.MiRows);
    }
    nTxb = 2 * n;
    nCoef = 2 * n * tx_ncoef(t);
}

// wait (one thread) until the byte of progress word f at bit `shift` (16: the 16-bit block count) is at least need; the
// word last seen in seen; false when the wait ran out of time or another workgroup aborted
__device__ bool wait_progress(const uint32_t *f, int shift, uint32_t need, const RcQueue &Q, uint32_t &seen) {
    const uint32_t mask = shift == 16 ? 0x7FFFu : 0xFFu;
    const uint64_t t0 = wall_clock64();
    for (;;) {
        seen = __hip_atomic_load(f, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (((seen >> shift) & mask) >= need) break;
        if (__hip_atomic_load(Q.abort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return false;
        if (wall_clock64() - t0 > Q.spinTicks) {
            __hip_atomic_store(Q.abort, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            return false;
        }
        __builtin_amdgcn_s_sleep(2);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    return true;
}

// The closed loop of the luma (PL 0) or the chroma (PL 1) of superblock sb, by the workgroup (the tables staged for its
// image's quantizer context).  Luma reads nothing of chroma; chroma reads its own block's luma reconstruction, mode and
// end of block and, like luma, its own plane kind's neighbours, so the two are separate items whose chains run beside
// each other.  Q null: one launch per wavefront step (every neighbour complete, luma before chroma in one workgroup).
// Else, before each block on the superblock's left or upper edge the workgroup waits for the neighbours' samples that
// block can read (twice its size along the edge) and for chroma for its luma, and after every block it publishes its own
// progress; blocks along the right (bottom) edge of a superblock come in ascending row (column) order whatever the
// partition, so two counts tell how far an edge is.  False: a wait failed (the schedule is being aborted).
template <typename Px, int PL>
__device__ bool recon_part(lds<RcShared> &S, const Batch &B, uint32_t sb, const RcQueue *Q) {
    const int tid = threadIdx.x;
    const lds<SearchParams> &P = S.prm;
    {   // the image's descriptor, read in place in LDS from here on, and the blocks
        static_assert(sizeof(Img) % 4 == 0, "the descriptor is copied by words");
        const uint32_t *g = (const uint32_t *)&B.img[B.sbImg[sb]];
        lds<uint32_t> *d = (lds<uint32_t> *)(lds<char> *)&S.img;
        for (int k = tid; k < (int)(sizeof(Img) / 4); k += RC_NT) d[k] = g[k];
        static_assert(RC_NT >= MAX_LEAVES && BLOCK_INVALID <= 32, "a thread per block, 5 + 4 + 4 bits");
        if (tid < MAX_LEAVES) {
            const Leaf lf = B.leaves[(size_t)sb * MAX_LEAVES + tid];
            S.leaf[tid] = (uint16_t)(lf.bsize | lf.x4 << 5 | lf.y4 << 9);
        }
    }
    __syncthreads();
    const lds<Img> &I = S.img;
    const DevTables &T = *B.T;
    const uint32_t local = sb - I.sbBase;
    const int sbc = (int)(local % I.sbCols), sbr = (int)(local / I.sbCols), sbx = sbc * 64, sby = sbr * 64;
    const int nLeaves = B.leafCount[sb];
    // what the blocks will want of global memory whatever they decide: the source, and for luma the candidates
    if constexpr (PL == 0) {
        const glb<Px> *src = src_plane<Px>(I, 0) + (size_t)sby * I.spitch[0] + sbx;
        for (int k = tid; k < 64 * 64; k += RC_NT) S.srcb[k] = src[(size_t)(k >> 6) * I.spitch[0] + (k & 63)];
        if (tid < nLeaves) {
            const int lf = S.leaf[tid], bs = lf & 31, x4 = (lf >> 5) & 15, y4 = lf >> 9;
            static_assert(offsetof(BlockRes, cand) == 4 && sizeof(BlockRes) == 12, "candidates, count and type: the last two words");
            const glb<uint32_t> *r = (const glb<uint32_t> *)(B.blk + I.shOff[bs] + (uint32_t)((sby + 4 * y4) / (4 * bh4(bs))) * I.shNbx[bs] +
                                                             (sbx + 4 * x4) / (4 * bw4(bs)));
            S.cand[tid][0] = r[1];
            S.cand[tid][1] = r[2];
        }
    } else if (I.ss) {
        for (int k = tid; k < 2 * 32 * 32; k += RC_NT) {
            const int p = 1 + (k >> 10), y = (k >> 5) & 31, x = k & 31;
            S.srcb[(p - 1) * 2048 + (k & 1023)] = (src_plane<Px>(I, p) + (size_t)(sby / 2 + y) * I.spitch[p] + sbx / 2)[x];
        }
    }
    int tc = 0, tr = 0;
    while (tc + 1 < I.tileCols && sbx >= I.tileColStart[tc + 1] * 4) tc++;
    while (tr + 1 < I.tileRows && sby >= I.tileRowStart[tr + 1] * 4) tr++;
    const int tx0 = I.tileColStart[tc] * 4, ty0 = I.tileRowStart[tr] * 4;
    const int miColEnd = I.tileColStart[tc + 1], miRowEnd = I.tileRowStart[tr + 1];
    // clear_block_decoded_flags (spec 7.3.3)
    for (int k = tid; k < 3 * 18 * 18; k += RC_NT) {
        const int p = k / 324, yy = (k / 18) % 18 - 1, xx = k % 18 - 1;
        const int ss = p ? I.ss : 0;
        const int sbW4 = (miColEnd - sbc * 16) >> ss, sbH4 = (miRowEnd - sbr * 16) >> ss;
        uint8_t v = (yy < 0 && xx < sbW4) ? 1 : (xx < 0 && yy < sbH4) ? 1 : 0;
        if (yy == (16 >> ss) && xx == -1) v = 0;
        S.bdm[p][yy + 1][xx + 1] = v;
    }
    if (tid == 0) {
        S.flopsOn = B.flops != nullptr; S.flops = 0; S.dcQ = dc_q(I.qindex, I.bd); S.acQ = ac_q(I.qindex, I.bd);
        S.dcRcp = 1.f / (float)S.dcQ; S.acRcp = 1.f / (float)S.acQ;
        for (int k = 0; k < 4; k++) S.known[k] = 0;
        S.errFlag[0] = S.errFlag[1] = 0;
        S.nSkip = S.nCfl = 0;
    }
    __syncthreads();
    const float lambda = T.lambda[I.bd == 10][I.qindex] * P.lambdaMul;
    // the neighbours inside the tile and how much of them the coded area holds (units of 4 luma samples)
    uint32_t *const prog = Q ? Q->prog + (size_t)PL * Q->nSb + sb : nullptr;
    const bool hasLeft = sbx > tx0, hasUp = sby > ty0, hasUpR = hasUp && (sbc + 1) * 16 < miColEnd;
    const int inRows = min(16, I.MiRows - sbr * 16), inCols = min(16, I.MiCols - sbc * 16), inColsR = min(16, I.MiCols - sbc * 16 - 16);
    uint32_t knL = 0, knU = 0, knR = 0, knY = 0;
    uint32_t ownR = 0, ownB = 0;   // this superblock's edges so far
    int nTxb = 0, nCoef = 0;       // of the superblock before the block
    for (int li = 0; li < nLeaves; li++) {
        const int lf = __builtin_amdgcn_readfirstlane((int)S.leaf[li]);
        const int bsize = lf & 31, lx4 = (lf >> 5) & 15, ly4 = lf >> 9, x = sbx + lx4 * 4, y = sby + ly4 * 4, mi_row = y >> 2, mi_col = x >> 2;
        const int bw = bw4(bsize), bh = bh4(bsize), lbw = 31 - __clz(bw);
        auto inside = [&](int r, int c) { return c >= (tx0 >> 2) && c < miColEnd && r >= (ty0 >> 2) && r < miRowEnd; };
        const int hasC = has_chroma(bsize, mi_row, mi_col, I.mono, I.ss);
        const int txSz = av1t::Max_Tx_Size_Rect[bsize];
        int cTxb = 0, cCoef = 0;
        if (hasC) chroma_size(I, bsize, mi_row, mi_col, cTxb, cCoef);
        const int firstTxb = nTxb, firstCoef = nCoef;
        nTxb += 1 + cTxb;
        nCoef += tx_ncoef(txSz) + cCoef;
        if (PL && !hasC) continue;
        // the block's luma area in the superblock; chroma of a 4-sample side covers the block before it too
        const int ax = PL && I.ss && bw == 1 ? lx4 - 1 : lx4, ay = PL && I.ss && bh == 1 ? ly4 - 1 : ly4;
        const int aw = lx4 + bw - ax, ah = ly4 + bh - ay;
        if (Q) {
            const uint32_t needL = hasLeft && ax == 0 ? min(ay + 2 * ah, inRows) : 0;
            const uint32_t needU = hasUp && ay == 0 ? min(ax + 2 * aw, inCols) : 0;
            const uint32_t needR = hasUpR && ay == 0 && ax + 2 * aw > 16 ? min(ax + 2 * aw - 16, inColsR) : 0;
            if ((knL & 0xFF) < needL || ((knU >> 8) & 0xFF) < needU || ((knR >> 8) & 0xFF) < needR || (PL && (int)(knY >> 16) < li + 1)) {
                if (tid == 0) {
                    uint32_t l = knL, u = knU, r = knR, yp = knY;
                    bool ok = true;
                    if (needL) ok = wait_progress(prog - 1, 0, needL, *Q, l);
                    if (ok && needU) ok = wait_progress(prog - I.sbCols, 8, needU, *Q, u);
                    if (ok && needR) ok = wait_progress(prog - I.sbCols + 1, 8, needR, *Q, r);
                    if (ok && PL) ok = wait_progress(Q->prog + sb, 16, li + 1, *Q, yp);
                    S.known[0] = ok ? l & 0x7FFFFFFFu : 0x80000000u; S.known[1] = u; S.known[2] = r; S.known[3] = yp;
                }
                __syncthreads();
                knL = S.known[0]; knU = S.known[1]; knR = S.known[2]; knY = S.known[3];
                if (knL & 0x80000000u) return false;
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
            }
        }
        if (tid == 0) {
            S.srcAt = PL == 0 ? ly4 * 256 + lx4 * 4 : I.ss ? (ay >> 1) * 128 + (ax >> 1) * 4 : 0;
            S.srcSp = PL == 0 ? 64 : I.ss ? 32 : tx_w(uv_tx_size(bsize, 0));
        }
        if constexpr (PL == 0) {
            const int availU = inside(mi_row - 1, mi_col), availL = inside(mi_row, mi_col - 1);
#define RC_LUMA(w, h) rc_luma<w, h, Px>(S, B, P, sb, I, bsize, x, y, availU, availL, tx0, ty0, lambda, li, hasC, firstTxb, firstCoef)
            AV1M_TX_SWITCH(txSz, RC_LUMA)
#undef RC_LUMA
        } else {
            RecBlock *const rb = B.oBlocks + (size_t)sb * MAX_LEAVES + li;
            const int availUC = (I.ss && bh == 1) ? inside(mi_row - 2, mi_col) : inside(mi_row - 1, mi_col);
            const int availLC = (I.ss && bw == 1) ? inside(mi_row, mi_col - 2) : inside(mi_row, mi_col - 1);
            if (tid == 128) { S.mode = rb->y_mode; S.winEob[0] = !rb->skip; }   // read from the first barrier on
            const int uvTx = uv_tx_size(bsize, I.ss);
#define RC_CHROMA(w, h) rc_chroma<w, h, Px>(S, B, P, sb, I, bsize, mi_row, mi_col, availUC, availLC, tx0, ty0, lambda * P.lambdaCMul, \
                                                   firstTxb + 1, firstCoef + tx_ncoef(txSz), cTxb)
            switch (uvTx) {
            case TX_4X4: RC_CHROMA(4, 4); break; case TX_8X8: RC_CHROMA(8, 8); break; case TX_16X16: RC_CHROMA(16, 16); break;
            case TX_32X32: RC_CHROMA(32, 32); break; case TX_4X8: RC_CHROMA(4, 8); break; case TX_8X4: RC_CHROMA(8, 4); break;
            case TX_8X16: RC_CHROMA(8, 16); break; case TX_16X8: RC_CHROMA(16, 8); break; case TX_16X32: RC_CHROMA(16, 32); break;
            case TX_32X16: RC_CHROMA(32, 16); break; case TX_4X16: RC_CHROMA(4, 16); break; case TX_16X4: RC_CHROMA(16, 4); break;
            case TX_8X32: RC_CHROMA(8, 32); break; default: RC_CHROMA(32, 8); break;
            }
#undef RC_CHROMA
            __syncthreads();
            const int skip = S.winEob[0] == 0 && S.winEob[1] == 0 && S.winEob[2] == 0;
            const int uv = S.uvMode;
            for (int k = tid; k < bw * bh; k += RC_NT) {
                const int r = mi_row + (k >> lbw), c = mi_col + (k & (bw - 1));
                if (r < I.MiRows && c < I.MiCols) {
                    const size_t o = (size_t)r * I.MiCols + c;
                    map8(I.mUV)[o] = (uint8_t)uv;
                    map8(I.mSkip)[o] = (uint8_t)skip;
                }
            }
            if (tid == 0) {
                const bool cfl = uv == UV_CFL_PRED;
                rb->skip = (uint8_t)skip;
                rb->uv_mode = (uint8_t)uv;
                rb->angle_delta_uv = (int8_t)(bsize >= BLOCK_8X8 && is_dir(uv) ? S.uvDelta : 0);
                rb->cfl_alpha_u = (int8_t)(cfl ? S.cflAlpha[0] : 0);
                rb->cfl_alpha_v = (int8_t)(cfl ? S.cflAlpha[1] : 0);
                S.nSkip += skip;
                S.nCfl += cfl;
            }
            block_barrier();
        }
        if (ax + aw == 16) ownR = ay + ah;
        if (ay + ah == 16) ownB = ax + aw;
        // the block's stores have all arrived (block_barrier): one lane writes them back and publishes, in the last wave,
        // which has the least to do while the next block is set up
        if (Q && tid == RC_NT - 64) {
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
            __hip_atomic_store(prog, ownR | ownB << 8 | (uint32_t)(li + 1) << 16, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    if (tid == 0) {
        if constexpr (PL == 0) {
            SbOut o;
            o.nBlocks = (uint32_t)nLeaves; o.nTxb = (uint32_t)nTxb; o.nCoeffs = (uint32_t)nCoef; o.pad = 0;
            B.sbOut[sb] = o;
            atomicAdd(&B.stats[0], (uint32_t)nLeaves);
        } else if (S.nCfl) {
            atomicAdd(&B.stats[2], (uint32_t)S.nCfl);
        }
        if (S.nSkip) atomicAdd(&B.stats[1], (uint32_t)S.nSkip);
        if (S.flopsOn && S.flops) atomicAdd(&B.flops[32 + (sb & 31)], S.flops);
    }
    return true;
}

// Both instances run two waves per SIMD: two 256-thread workgroups per compute unit (batches: more superblocks in flight), or
// one of 512 threads, which spends them on the latency of one superblock (a single image, whose closed loop is bound by
// its chain of blocks).  The same results either way.  Closed loop on MI355X, 512 against 256 threads with a unit to
// itself: 512 x 512 image 11.2 / 14.0 ms, 12 MP 30.4 / 38.0, 24 MP learned 31.2 / 38.6; two narrow workgroups per unit against
// a wide one on 16 images of 12 MP: 69.0 / 77.5 ms, on 16 of 0.18-2 MP 30.8 / 25.6.
#define AV1M_RC_KERNEL __global__ void __launch_bounds__(RC_NT) __attribute__((amdgpu_waves_per_eu(2, 2)))

// The kernels' one parameter, read in place in the kernarg segment (it is the segment's first argument): handing a
// reference to a by-value kernel parameter to the out-of-line superblock code would make the compiler copy it into
// every lane's scratch, and every read of a field a per-lane scratch load.
struct RcQueueArgs {
    Batch B;
    SearchParams P;
    RcQueue Q;
};
template <typename A> __device__ __forceinline__ const A &kernel_args() { return *(const A *)__builtin_amdgcn_kernarg_segment_ptr(); }

// Persistent schedule: every workgroup pulls items (a superblock's luma or chroma) from the queue, the anti-diagonal
// wavefront order of all images of the batch, and runs it beside what it depends on: its left, above and above-right
// neighbours of the same plane kind inside its tile and, for chroma, its own luma (recon_part waits block by block).  An
// item's dependencies stand before it in the queue, so they were taken earlier by a running workgroup and the waits
// always end; a wait that exceeds the time limit raises the abort flag, which makes every workgroup stop taking items and
// return.
template <typename Px>
AV1M_RC_KERNEL k_recon_queue(RcQueueArgs) {
    extern __shared__ __align__(16) char smraw[];
    lds<RcShared> &S = *(lds<RcShared> *)(lds<char> *)smraw;
    const RcQueueArgs &A = kernel_args<RcQueueArgs>();
    const Batch &B = A.B;
    const RcQueue &Q = A.Q;
    const int tid = threadIdx.x;
    int staged = -1;
    for (;;) {
        if (tid == 0) {
            uint32_t it = Q.n;
            if (!__hip_atomic_load(Q.abort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
                it = __hip_atomic_fetch_add(Q.head, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            S.qItem = it < Q.n ? Q.order[it] : 0xFFFFFFFFu;
        }
        __syncthreads();
        const uint32_t item = S.qItem;
        if (item == 0xFFFFFFFFu) break;
        const uint32_t sb = item & ~RC_CHROMA;
        const int qctx = B.img[B.sbImg[sb]].qctx;
        if (qctx != staged) {
            stage_tables(S, *B.T, A.P, qctx, staged < 0);
            staged = qctx;
        }
        __syncthreads();
        const bool ok = (item & RC_CHROMA) ? recon_part<Px, 1>(S, B, sb, &Q) : recon_part<Px, 0>(S, B, sb, &Q);
        if (!ok) break;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
        __syncthreads();
        if (tid == 0)   // complete: both edges and every block
            __hip_atomic_store(Q.prog + ((item & RC_CHROMA) ? Q.nSb : 0) + sb, 0x7FFF1010u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

static_assert(sizeof(RcShared) * (512 / RC_NT) <= 160 * 1024, "the closed loop's LDS exceeds a compute unit's 160 KiB");

}  // namespace AV1M_RC_SPACE
}  // namespace av1m

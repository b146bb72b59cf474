// Row plan of one 64-row tile, shared by the forward's row_plan kernel and the selection's
// sel_norms launch (which can compute the plan alongside the norms).
//
// Head-independent preparation read by the forward and dQ kernels.  Within each 64-row
// tile the rows are ordered by window start lo_i (ties by row; rows past the end last), so
// the 16 rows a wave takes have close window starts: the wave's key range [min lo, max i]
// and its count of masked subtiles shrink.  Each 16-row group's {min lo, max lo, max i,
// min i} is recorded, with the tile's largest clamped window (whose maximum over a sequence
// bounds the key-parallel backward sweep).
#pragma once

#include "common.h"

namespace dsalt {

struct PlanOut {
    uint8_t* perm;   // [S * n_tiles * 64] row offset within the tile
    int* bounds;     // [S * n_tiles * 4 * 4]
    int* wmax;       // [S * n_tiles]
};

// The plan of one tile in the registers of a wave (every lane calls it; lane l holds sorted
// position l): the row offset at that position, its 16-row group's bounds, and the tile's largest
// window.  The forward's blocks compute it themselves where a call is too small to hide the
// plan's own launch.
struct PlanRegs {
    int perm, lo, lomax, hi, himin, wmax;
};
__device__ __forceinline__ PlanRegs plan_regs(const int32_t* w, int st, int len, int r0, int l) {
    const int i = r0 + l;
    int lo = 0x7fffffff, wcl = 0;
    if (i < len) {
        const int wi = max(w[st + i], 1);
        lo = max(i - wi + 1, 0);
        wcl = min(wi, len);
    }
    int rank = 0;  // by (lo, row)
#pragma unroll 8
    for (int j = 0; j < 64; ++j) {
        const int jlo = __builtin_amdgcn_readlane(lo, j);
        rank += (jlo < lo || (jlo == lo && j < l)) ? 1 : 0;
    }
    PlanRegs r;
    r.perm = __builtin_amdgcn_ds_permute(rank * 4, l);
    const bool rv = r0 + r.perm < len;
    const int slo = __shfl(lo, r.perm);
    r.lo = row_min16(rv ? slo : 0x7fffffff);
    r.lomax = row_max16(rv ? slo : (int)0x80000000);
    r.hi = row_max16(rv ? r0 + r.perm : -1);
    r.himin = row_min16(rv ? r0 + r.perm : 0x7fffffff);
    r.wmax = wave_max(wcl);
    return r;
}
// writes it where row_plan_tile would (one wave)
__device__ __forceinline__ void plan_store(const PlanRegs& r, int64_t tile, int l, const PlanOut& o) {
    o.perm[tile * 64 + l] = (uint8_t)r.perm;
    if ((l & 15) == 0) {
        int* b = o.bounds + (tile * 4 + (l >> 4)) * 4;
        b[0] = r.lo;
        b[1] = r.lomax;
        b[2] = r.hi;
        b[3] = r.himin;
    }
    if (l == 0) o.wmax[tile] = r.wmax;
}

// One wave (lane l) plans tile `tile` (= s * n_tiles + t) when `active`; sp, slo: 64 ints
// of LDS each, private to the wave.  Every thread of the block must call it once (one
// block barrier inside); nothing is written for an inactive tile.
__device__ __forceinline__ void row_plan_tile(const int32_t* w, const int32_t* cu, int total_len, int max_seqlen,
                                              int n_tiles, int tile, bool active, int l, int* sp, int* slo,
                                              const PlanOut& o) {
    const int s = active ? tile / n_tiles : 0, t = active ? tile % n_tiles : 0;
    int st = 0, len = 0;
    if (active) seq_bounds(cu, s, total_len, max_seqlen, st, len);
    const int r0 = t * 64;
    const int i = r0 + l;
    const bool valid = active && i < len;
    int lo = 0x7fffffff, wcl = 0;
    if (valid) {
        const int wi = max(w[st + i], 1);
        lo = max(i - wi + 1, 0);
        wcl = min(wi, len);
    }
    const uint32_t khi = (uint32_t)lo >> 26, klo = ((uint32_t)lo << 6) | (uint32_t)l;  // key lo * 64 + l
    int rank = 0;
    for (int j = 0; j < 64; ++j) {
        const uint32_t jhi = (uint32_t)__builtin_amdgcn_readlane((int)khi, j);
        const uint32_t jlo = (uint32_t)__builtin_amdgcn_readlane((int)klo, j);
        rank += (jhi < khi || (jhi == khi && jlo < klo)) ? 1 : 0;
    }
    sp[rank] = l;
    slo[l] = lo;
    __syncthreads();
    const int pl = sp[l];  // row offset at sorted position l
    const int ri = r0 + pl;
    const bool rv = active && ri < len;
    int rlo = 0x7fffffff, rlmax = (int)0x80000000, rhi = -1, rhmin = 0x7fffffff;
    if (rv) {
        rlo = slo[pl];
        rlmax = rlo;
        rhi = ri;
        rhmin = ri;
    }
    rlo = row_min16(rlo);
    rlmax = row_max16(rlmax);
    rhi = row_max16(rhi);
    rhmin = row_min16(rhmin);
    const int m = row_max16(wcl);
    const int tm = max(max(__builtin_amdgcn_readlane(m, 0), __builtin_amdgcn_readlane(m, 16)),
                       max(__builtin_amdgcn_readlane(m, 32), __builtin_amdgcn_readlane(m, 48)));
    if (!active) return;
    o.perm[(int64_t)tile * 64 + l] = (uint8_t)pl;
    if ((l & 15) == 0) {
        int* b = o.bounds + ((int64_t)tile * 4 + (l >> 4)) * 4;
        b[0] = rlo;
        b[1] = rlmax;
        b[2] = rhi;
        b[3] = rhmin;
    }
    if (l == 0) o.wmax[tile] = tm;
}

}  // namespace dsalt

// Where the slots of a chunk lie in the grid, as a wavefront sees a 64-slot tile.
#pragma once
#include "bsa_common.h"

namespace bsa {

constexpr int kTileSlots = 64;

__device__ __forceinline__ void keep_if(uint4& x, bool keep) {
    const uint32_t m = keep ? ~0u : 0u;
    x.x &= m; x.y &= m; x.z &= m; x.w &= m;
}

// The 64 slots of a tile as a wavefront sees them, one per lane: grid position, token row (-1: padding), and the word of
// the real ones.
struct Slots {
    int token, loc;        // loc: position inside the chunk, ti | hi << 8 | wi << 16
    uint64_t word;
};
__device__ __forceinline__ Slots slots_of(const Grid3& g, int blk, int sub, int lane) {
    const int nw = blk % g.Nw, nh = (blk / g.Nw) % g.Nh, nt = blk / (g.Nw * g.Nh);
    const int r = sub * kTileSlots + lane;
    int wi, hi, ti;
    if (((g.w & (g.w - 1)) | (g.h & (g.h - 1))) == 0) {           // the usual chunks: shifts instead of three divisions
        const int ws = __builtin_ctz(g.w), hs = __builtin_ctz(g.h);
        wi = r & (g.w - 1); hi = (r >> ws) & (g.h - 1); ti = r >> (ws + hs);
    } else {
        wi = r % g.w; hi = (r / g.w) % g.h; ti = r / (g.w * g.h);
    }
    const int tt = nt * g.t + ti, hh = nh * g.h + hi, ww = nw * g.w + wi;
    const bool ok = tt < g.T && hh < g.H && ww < g.W;
    Slots s;
    s.token = ok ? (tt * g.H + hh) * g.W + ww : -1;
    s.loc = ti | (hi << 8) | (wi << 16);
    s.word = __ballot(ok);
    return s;
}

// The same where the real slots of the chunk come first, in their order, and the padding behind them.
__device__ __forceinline__ Slots packed_slots_of(const Grid3& g, int blk, int sub, int lane) {
    const int nw = blk % g.Nw, nh = (blk / g.Nw) % g.Nh, nt = blk / (g.Nw * g.Nh);
    const int ew = min(g.w, g.W - nw * g.w), eh = min(g.h, g.H - nh * g.h), et = min(g.t, g.T - nt * g.t);
    const int rows = et * eh * ew;
    if (rows == g.chunk()) return slots_of(g, blk, sub, lane);
    const int r = sub * kTileSlots + lane, plane = r / ew, ti = plane / eh;
    const int wi = r - plane * ew, hi = plane - ti * eh;
    Slots s;
    s.token = r < rows ? ((nt * g.t + ti) * g.H + nh * g.h + hi) * g.W + nw * g.w + wi : -1;
    s.loc = ti | (hi << 8) | (wi << 16);
    s.word = __ballot(r < rows);
    return s;
}
// Halves of 32 slots that then hold real ones.
__device__ __forceinline__ int live_halves(const Grid3& g, int blk) {
    return (chunk_rows(g, blk / (g.Nw * g.Nh), (blk / g.Nw) % g.Nh, blk % g.Nw) + 31) / 32;
}

}  // namespace bsa

// dispatch_one.hpp -- the whole dispatch of a batch of at most kOneMaxRoutes
// routes by one work-group: counts, offsets, row tiles and the stable ranks
// of dispatch.hip's launches, the same integers.
//
// Wave w takes the routes [w C, (w + 1) C) in batches of 64, one per lane.  A
// batch finds the earlier lanes with the same expert by ballots over the
// expert index's bits and reads, then advances, the wave's own count of that
// expert in LDS: the route's rank inside its wave, in route order.  After one
// barrier a thread per expert turns the waves' counts into bases and a scan
// over the experts gives the offsets; rank + base + offset is the row.
#pragma once

#include "common.hpp"
#include "dispatch.hpp"

namespace grim {

constexpr int kOneThreads = 1024;
constexpr int kOneWaves = kOneThreads / kWave;
constexpr int kOneBatches = 8;                             // route batches per wave, at most
constexpr int kOneMaxRoutes = kOneThreads * kOneBatches;
constexpr int kOneMaxE = 512;

struct OneLds {
    int32_t hist[kOneWaves][kOneMaxE];
    int32_t wsum[kOneWaves][3];
};

struct OneArgs {
    int R, E, K;
    int32_t *counts, *offsets, *inverse, *perm_token;      // perm_token may be null
    TileLists lists;                                       // or (n null) the tile table:
    int32_t *tile_e, *tile_mb;                             // -1 padded to tmax, or null
    int tmax, mc;
    int32_t* n_tiles;                                      // its live length, or null
};

// id_at(r): the expert of route r < R (out of [0, E): the route is skipped).
template <class IdAt>
__device__ __forceinline__ void dispatch_one_block(const OneArgs& a, OneLds& s, IdAt id_at) {
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wv = tid / kWave;
    const int E = a.E, nb = (a.R + kOneThreads - 1) / kOneThreads;   // batches per wave
    for (int e = lane; e < E; e += kWave) s.hist[wv][e] = 0;
    volatile int32_t* hist = s.hist[wv];
    const int r0 = wv * nb * kWave + lane;
    int id[kOneBatches], rank[kOneBatches];
#pragma unroll
    for (int b = 0; b < kOneBatches; ++b) {
        const int r = r0 + b * kWave;
        int v = -1;
        if (b < nb && r < a.R) v = id_at(r);
        id[b] = v >= 0 && v < E ? v : -1;
    }
#pragma unroll
    for (int b = 0; b < kOneBatches; ++b) {
        rank[b] = 0;
        if (b >= nb) continue;   // uniform
        const bool on = id[b] >= 0;
        uint64_t m = __ballot(on);
#pragma unroll
        for (int bit = 0; bit < 9; ++bit) {
            const uint64_t q = __ballot((id[b] >> bit) & 1);
            m &= (id[b] >> bit) & 1 ? q : ~q;
        }
        static_assert(kOneMaxE == 512, "nine bits of an expert index");
        const int below = __popcll(m & ((1ull << lane) - 1));
        const int at = on ? id[b] : 0;
        const int base = hist[at];
        rank[b] = base + below;
        // the last lane of each expert's advances the count (LDS operations
        // of a wave stay in order)
        if (on && (m >> lane) == 1) hist[at] = base + below + 1;
    }
    __syncthreads();
    int c = 0;
    if (tid < E)
#pragma unroll
        for (int w = 0; w < kOneWaves; ++w) {
            const int v = s.hist[w][tid];
            s.hist[w][tid] = c;
            c += v;
        }
    const bool lists = a.lists.n != nullptr;
    const int mc0 = lists ? a.lists.mc[0] : a.mc, mc1 = lists ? a.lists.mc[1] : 0;
    const int nt0 = mc0 > 0 ? (c + mc0 - 1) / mc0 : 0, nt1 = mc1 > 0 ? (c + mc1 - 1) / mc1 : 0;
    int v[3] = {c, nt0, nt1};
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1)
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            const int u = __shfl_up(v[q], off, kWave);
            if (lane >= off) v[q] += u;
        }
    if (lane == kWave - 1)
#pragma unroll
        for (int q = 0; q < 3; ++q) s.wsum[wv][q] = v[q];
    __syncthreads();
    int tot[3] = {0, 0, 0};
    for (int w = 0; w < kOneWaves; ++w)
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            const int u = s.wsum[w][q];
            v[q] += w < wv ? u : 0;
            tot[q] += u;
        }
    const int off_e = v[0] - c;
    if (tid < E) {
        a.counts[tid] = c;
        a.offsets[tid] = off_e;
#pragma unroll
        for (int w = 0; w < kOneWaves; ++w) s.hist[w][tid] += off_e;
        const int t0 = v[1] - nt0, t1 = v[2] - nt1;
        if (lists) {
            for (int i = 0; i < nt0; ++i)
                a.lists.d[0][t0 + i] = TileDesc{tid, off_e + i * mc0, min(mc0, c - i * mc0), i};
            for (int i = 0; i < nt1; ++i)
                a.lists.d[1][t1 + i] = TileDesc{tid, off_e + i * mc1, min(mc1, c - i * mc1), i};
        } else if (a.tile_e) {
            for (int i = 0; i < nt0; ++i)
                if (t0 + i < a.tmax) { a.tile_e[t0 + i] = tid; a.tile_mb[t0 + i] = i; }
        }
    }
    if (lists) {
        if (tid < 2) a.lists.n[tid] = tid ? tot[2] : tot[1];
    } else {
        if (a.tile_e)
            for (int t = tot[1] + tid; t < a.tmax; t += kOneThreads) { a.tile_e[t] = -1; a.tile_mb[t] = 0; }
        if (tid == 0 && a.n_tiles) *a.n_tiles = tot[1];
    }
    __syncthreads();
#pragma unroll
    for (int b = 0; b < kOneBatches; ++b) {
        const int r = r0 + b * kWave;
        if (b >= nb || r >= a.R) continue;
        const int p = id[b] >= 0 ? s.hist[wv][id[b]] + rank[b] : -1;
        a.inverse[r] = p;
        if (p >= 0 && a.perm_token) a.perm_token[p] = r / a.K;
    }
}

}  // namespace grim

// Tiled triangular sweeps (tile_sweep.h): set-up of the tiles on the device
// and the fused forward and backward sweep.
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <cstdio>
#include <cstdlib>

#include "pcg.h"
#include "pcg_common.h"
#include "sweep_merge.h"
#include "tile_grid.h"
#include "tile_sweep.h"

namespace astg {

namespace {

// Rows per tile. With positions: about 2048 asked for, before the boxes' shape
// is chosen (tile_grid.h). Fewer rows a tile mean more boundary crossings on the
// dependency chain, more rows a longer queue of chunks per wavefront; measured
// flat between about 1300 and 2400 (FP64 forward / backward us: n = 63 k, 27
// tiles 41 / 43, 48 tiles 40 / 43, 8 tiles 55 / 58; n = 456 k, 252 tiles 73 / 79,
// 64 tiles 92 / 94). Without, the tiles are index ranges, whose boundary a
// grid's chain crosses once per tile, so as few as the LDS holds (n = 152 k, ms
// per solve: 16 tiles 8.5, 32 10.1, 64 12.9, 128 13.4, merged sweeps 15.3; other
// sizes, us per FP64 iteration at the tiles that this gives, at fewer and more,
// and merged: 28^3 3 tiles 80, 2 86, 5 79, merged 162; 36^3 5 tiles 99, 3 114,
// 8 99, merged 201; 150^2 3 tiles 146, 2 140, 8 160, merged 472; 400^2 17 tiles
// 378, 9 354, 34 424, merged 1232; 61^3 24 tiles 183, 32 200, merged 336).
constexpr int kTileRows = 2048;
constexpr int kTileRangeRows = 9600;

// Index ranges cut an order of few wide levels (a colouring) everywhere: its
// tiles import as many values as they hold rows, by 128 lanes, while merged
// sweeps take it in a few steps over the whole chip. From 125 systems of boxes
// and grids in ten orders, alone and in batches, FP64, ns per forward and
// backward sweep: a level costs merged sweeps about 850 more than tiles, and the
// second launch 8000; a tile costs 1.5 per row and 9 per imported value. us per
// iteration tiled / merged: red-black 20^3 43 / 34, 2 x 30^3 in a batch 90 / 47;
// blocks of 4 in 8 colours 28^3 83 / 69, 24 x 20^3 100 / 106, of 8 28^3 87 / 114;
// natural order 28^3 80 / 161, 47 x 53 x 61 150 / 297; the form taken is at most
// 9 % behind the other (one of the 250 in both precisions over 5 %). Boxes'
// surfaces are small whatever the order: tiles cut by positions are not asked.
inline bool rangesPay(int depth, int S, int halo) {
    return 850ll * depth + 8000 >= 3ll * S / 2 + 9ll * halo;
}

inline int blocks(long n) { return (int)((n + BS - 1) / BS); }

// ---------------------------------------------------------------------------
// set-up
// ---------------------------------------------------------------------------
// Row coordinates are packed z << 36 | y << 18 | x (18 bits each).
__global__ void k_coord_key(int n, const unsigned long long* coord, int shift, const int* idx, int parts, int* key,
                            int* val) {
    const int q = blockIdx.x * BS + threadIdx.x;
    if (q >= n) return;
    const int i = idx ? idx[q] : q;
    const int part = idx ? (int)((long long)q * parts / n) : 0;
    key[q] = (part << 18) | (int)((coord[i] >> shift) & 0x3FFFF);
    val[q] = i;
}
// Tile of the row at rank q of the partition order: K tiles of equal count.
__global__ void k_tile_of(int n, const int* idx, int K, int* tile) {
    const int q = blockIdx.x * BS + threadIdx.x;
    if (q < n) tile[idx ? idx[q] : q] = (int)((long long)q * K / n);
}
// Rows by tile, then level, then number of lower entries (rows of one
// width side by side: less padding in the chunks' entries).
constexpr int kWidthBits = 5;
static_assert(kMaxDeps < (1 << kWidthBits), "row width in the sort key");
__global__ void k_tile_key(int n, const int* tile, const int* lev, int depth, const int* rs, const int* lend,
                           unsigned int* key, int* val) {
    const int i = blockIdx.x * BS + threadIdx.x;
    if (i >= n) return;
    key[i] = ((unsigned int)(tile[i] * depth + lev[i]) << kWidthBits) | (unsigned int)(lend[i] - rs[i]);
    val[i] = i;
}
__global__ void k_tile_fill_i32(int n, int v, int* p) {
    const int i = blockIdx.x * BS + threadIdx.x;
    if (i < n) p[i] = v;
}
// Rows sorted by tile to their positions: tile b starts at b S.
__global__ void k_tile_place(int n, const int* rows, int K, int S, int* order, int* pos) {
    const int q = blockIdx.x * BS + threadIdx.x;
    if (q >= n) return;
    const int b = (int)((long long)q * K / n);
    const int first = (int)(((long long)b * n + K - 1) / K);
    const int t = b * S + (q - first);
    order[t] = rows[q];
    pos[rows[q]] = t;
}
// A tile imports a row of another tile once, however many of its own rows read
// it, at the need of the first of them to be worked on: forward the reader of
// the lowest level and position, backward the highest. The passes below go
// over the rows whose values are exported (their entries of the other
// triangle: upper ones in the forward direction) and over the reading rows.
struct TilePattern {
    int P, S;
    const int *order, *pos, *rs, *lend, *ubeg, *col, *tpos, *lev;
};
template <int DIR>
__device__ inline void exportRange(const TilePattern& M, int i, int& p0, int& p1) {
    p0 = DIR == 0 ? M.ubeg[i] : M.rs[i];
    p1 = DIR == 0 ? M.rs[i + 1] : M.lend[i];
}
// Calls f(entry of the first reader, tile) for every other tile that reads row i.
template <int DIR, class F>
__device__ inline void forReaders(const TilePattern& M, int i, int own, F f) {
    int p0, p1;
    exportRange<DIR>(M, i, p0, p1);
    for (int p = p0; p < p1; ++p) {
        const int tile = M.pos[M.col[p]] / M.S;
        if (tile == own) continue;
        bool seen = false;
        for (int q = p0; q < p && !seen; ++q) seen = M.pos[M.col[q]] / M.S == tile;
        if (seen) continue;
        int best = p;
        for (int q = p + 1; q < p1; ++q) {
            const int c = M.col[q], d = M.col[best];
            if (M.pos[c] / M.S != tile) continue;
            const bool before = M.lev[c] != M.lev[d] ? M.lev[c] < M.lev[d] : M.pos[c] < M.pos[d];
            if (DIR == 0 ? before : !before) best = q;
        }
        f(best, tile);
    }
}
// Per exported row: the number of tiles that read it; their first readers'
// entries are marked 1 (entryHalo starts as zero).
template <int DIR>
__global__ void __launch_bounds__(BS) k_tile_mark(TilePattern M, int* exports, int* entryHalo) {
    const int t = blockIdx.x * BS + threadIdx.x;
    if (t >= M.P) return;
    const int i = M.order[t];
    int k = 0;
    if (i >= 0)
        forReaders<DIR>(M, i, t / M.S, [&](int p, int) {
            entryHalo[M.tpos[p]] = 1;
            ++k;
        });
    exports[t] = k;
}
// Per position: imports of both directions and the rank of the row's level in
// the chunk; per chunk: the entry pairs of the widest row of each direction.
__global__ void __launch_bounds__(BS) k_tile_count(TilePattern M, const int* entryHalo, int* impF, int* impB,
                                                   uint8_t* step, int* wF, int* wB) {
    const int t = blockIdx.x * BS + threadIdx.x;
    if (t >= M.P) return;  // P is a multiple of 64: whole wavefronts
    const int i = M.order[t];
    int nl = 0, nu = 0, el = 0, eu = 0;
    if (i >= 0) {
        nl = M.lend[i] - M.rs[i];
        nu = M.rs[i + 1] - M.ubeg[i];
        for (int p = M.rs[i]; p < M.lend[i]; ++p) el += entryHalo[p];
        for (int p = M.ubeg[i]; p < M.rs[i + 1]; ++p) eu += entryHalo[p];
    }
    impF[t] = el;
    impB[t] = eu;
    // padding (behind the last row of a tile) counts to the level before it
    const int lane = threadIdx.x & 63, lv = i >= 0 ? M.lev[i] : -1, before = __shfl_up(lv, 1, 64);
    const unsigned long long steps = __ballot(lane > 0 && lv >= 0 && lv != before);
    const int rank = __popcll(steps & ((2ull << lane) - 1ull));
    step[t] = (uint8_t)rank;
    for (int o = 32; o > 0; o >>= 1) {
        nl = max(nl, __shfl_xor(nl, o, 64));
        nu = max(nu, __shfl_xor(nu, o, 64));
    }
    if ((threadIdx.x & 63) == 0) {
        wF[t >> 6] = (nl + 1) / 2;
        wB[t >> 6] = (nu + 1) / 2;
    }
}
// Largest halo and export list of a tile.
__global__ void k_tile_max(int K, int S, const int* hF, const int* hB, const int* xF, const int* xB, int* out) {
    const int b = blockIdx.x * BS + threadIdx.x;
    if (b >= K) return;
    const int p0 = b * S, p1 = p0 + S;
    atomicMax(out, max(hF[p1] - hF[p0], hB[p1] - hB[p0]));
    atomicMax(out + 1, max(xF[p1] - xF[p0], xB[p1] - xB[p0]));
}
// Marked entries to their halo entries, in the order of the reading rows.
template <int DIR>
__global__ void __launch_bounds__(BS) k_tile_halo(TilePattern M, const int* hstart, int* entryHalo) {
    const int t = blockIdx.x * BS + threadIdx.x;
    if (t >= M.P) return;
    const int i = M.order[t];
    if (i < 0) return;
    int h = hstart[t];
    const int p0 = DIR == 0 ? M.rs[i] : M.ubeg[i], p1 = DIR == 0 ? M.lend[i] : M.rs[i + 1];
    for (int p = p0; p < p1; ++p)
        if (entryHalo[p] == 1) entryHalo[p] = h++;
}
// Exports, and the halo entry of every reader.
template <int DIR>
__global__ void __launch_bounds__(BS) k_tile_exports(TilePattern M, int* entryHalo, const int* xstart,
                                                     uint16_t* xslot, int* xdest) {
    const int t = blockIdx.x * BS + threadIdx.x;
    if (t >= M.P) return;
    const int i = M.order[t], b = t / M.S;
    if (i < 0) return;
    int x = xstart[t], p0, p1;
    exportRange<DIR>(M, i, p0, p1);
    forReaders<DIR>(M, i, b, [&](int p, int tile) {
        const int h = entryHalo[M.tpos[p]];
        xslot[x] = (uint16_t)(t - b * M.S);
        xdest[x++] = h;
        for (int q = p0; q < p1; ++q)
            if (M.pos[M.col[q]] / M.S == tile) entryHalo[M.tpos[q]] = h;
    });
}
template <int DIR>
__global__ void __launch_bounds__(BS) k_tile_slots(TilePattern M, int zero, const int* sell, const int* hstart,
                                                   const int* entryHalo, uint32_t* slot) {
    const int t = blockIdx.x * BS + threadIdx.x;
    if (t >= M.P) return;
    const int i = M.order[t], b = t / M.S, lane = t & 63;
    const int base = sell[t >> 6], w = sell[(t >> 6) + 1] - base;
    int p0 = 0, nd = 0;
    if (i >= 0) {
        p0 = DIR == 0 ? M.rs[i] : M.ubeg[i];
        nd = (DIR == 0 ? M.lend[i] : M.rs[i + 1]) - p0;
    }
    const int h0 = hstart[b * M.S];
    auto at = [&](int k) {
        if (k >= nd) return zero;
        const int pc = M.pos[M.col[p0 + k]];
        return pc / M.S == b ? pc - b * M.S : M.S + (entryHalo[p0 + k] - h0);
    };
    for (int k = 0; k < w; ++k)
        slot[((size_t)base + k) * 64 + lane] = (uint32_t)at(2 * k) | (uint32_t)at(2 * k + 1) << 16;
}

template <typename T>
struct Pair {
    T a, b;
};
// Entry coefficients from the factor, in the chunks' layout.
template <typename T, int DIR>
__global__ void __launch_bounds__(BS) k_tile_coef(int P, const int* order, const int* rs, const int* lend,
                                                  const int* ubeg, const double* F, const int* sell,
                                                  Pair<T>* coef) {
    const int t = blockIdx.x * BS + threadIdx.x;
    if (t >= P) return;
    const int i = order[t], lane = t & 63;
    const int base = sell[t >> 6], w = sell[(t >> 6) + 1] - base;
    int p0 = 0, nd = 0;
    if (i >= 0) {
        p0 = DIR == 0 ? rs[i] : ubeg[i];
        nd = (DIR == 0 ? lend[i] : rs[i + 1]) - p0;
    }
    for (int k = 0; k < w; ++k) {
        Pair<T> c;
        c.a = 2 * k < nd ? (T)F[p0 + 2 * k] : (T)0;
        c.b = 2 * k + 1 < nd ? (T)F[p0 + 2 * k + 1] : (T)0;
        coef[((size_t)base + k) * 64 + lane] = c;
    }
}

// ---------------------------------------------------------------------------
// the sweep
// ---------------------------------------------------------------------------
// Largest wait of any loop below, in ticks of the 100 MHz wall clock: 3 s. A
// healthy sweep takes well under a millisecond; a workgroup that was not
// resident, or a device busy with other work for longer, ends the sweep with
// an error bit instead of a wait without end.
constexpr long long kTileTicks = 300000000ll;

template <typename T>
__device__ inline typename Sentinel<T>::bits_t lds_load(const T* p) {
    typedef typename Sentinel<T>::bits_t B;
    return __hip_atomic_load(reinterpret_cast<const B*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
template <typename T>
__device__ inline void lds_store(T* p, typename Sentinel<T>::bits_t v) {
    typedef typename Sentinel<T>::bits_t B;
    __hip_atomic_store(reinterpret_cast<B*>(p), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ inline double from_bits(unsigned long long b) { return Sentinel<double>::val(b); }
__device__ inline float from_bits(unsigned int b) { return Sentinel<float>::val(b); }
__device__ inline unsigned long long to_bits(double v) { return (unsigned long long)__double_as_longlong(v); }
__device__ inline unsigned int to_bits(float v) { return __float_as_uint(v); }

// Every 256 rounds of a waiting loop: another wave has given up, or this one
// does now. Wave-uniform.
__device__ inline bool tile_stop(int spins, long long t0, int* err, int bit) {
    if ((spins & 255) != 255) return false;
    if (ld_agent_i32(err) != 0) return true;
    if (wall_clock64() - t0 > kTileTicks) {
        atomicOr(err, bit);
        return true;
    }
    return false;
}

// The tile's imports. The list is in the order the tile's rows need the values:
// a lane that waits for a value can then hold up only values that rows of the
// same or a later level wait for, so the values that the least finished level
// needs are always being polled. Lane `lane` of the importing wavefronts takes
// entries lane, lane + L, ... (the backward sweep from the list's end); each is
// polled in memory and copied to its slot when it appears. One entry in flight
// per lane: with two and four a round takes longer and the sweeps are slower.
template <typename T, int DIR>
__device__ inline void tile_import(const TileDir& D, int p0, int S, const T* in, T* halo, int lane, long long t0,
                                   int* err, int bit) {
    typedef typename Sentinel<T>::bits_t B;
    constexpr int L = kTileImport * 64;
    const int h0 = D.hstart[p0], cnt = D.hstart[p0 + S] - h0;
    auto at = [&](int k) { return DIR == 0 ? k : cnt - 1 - k; };
    int e = lane;
    for (int spins = 0; __any(e < cnt); ++spins) {
        B b = Sentinel<T>::value;
        if (e < cnt) b = Sentinel<T>::load(&in[h0 + at(e)]);
        if (b != Sentinel<T>::value) {
            lds_store<T>(&halo[at(e)], b);
            e += L;
        }
        if (tile_stop(spins, t0, err, bit)) break;
    }
}

// The tile's exports: values that other tiles read, stored from their slots to
// the halo entries they fill as they appear. The computing wavefronts hold no
// store in flight but their chunk's last, so that waiting for the next chunk's
// loads never means waiting for stores to memory.
template <typename T, int DIR>
__device__ inline void tile_export(const TileDir& D, const uint16_t* xslot, const int* xdest, int p0, int S,
                                   const T* lds, T* outbox, int lane, long long t0, int* err, int bit) {
    constexpr int L = kTileExport * 64;
    const int cnt = D.xstart[p0 + S] - D.xstart[p0];
    // past the end, the last entry again (not stored)
    auto at = [&](int k) { return DIR == 0 ? min(k, cnt - 1) : max(cnt - 1 - k, 0); };
    int e = lane, sl = 0, dst = 0, waits = 0;
    if (cnt > 0) {
        sl = xslot[at(e)];
        dst = xdest[at(e)];
    }
    while (__any(e < cnt)) {
        // the value and the entry behind it, all LDS reads of a round in flight together
        const auto b = lds_load<T>(&lds[sl]);
        const int nsl = xslot[at(e + L)], ndst = xdest[at(e + L)];
        const bool got = e < cnt && b != Sentinel<T>::value;
        if (got) {
            Sentinel<T>::store(&outbox[dst], from_bits(b));
            e += L;
            sl = nsl;
            dst = ndst;
        }
        if (!__any(got)) {
            __builtin_amdgcn_s_sleep(1);
            if (tile_stop(waits++, t0, err, bit)) break;
        }
    }
}

// Forms of the sweep: vectors by position; the same with a timeline of every
// row; r, z and the pivots by row (batched solves).
enum TileMode { kTilePlain, kTileTrace, kTileByRow };

// A 64-row chunk's data in registers.
template <typename T>
struct TileChunk {
    Pair<T> f[kMaxDeps / 2];
    uint32_t sl[kMaxDeps / 2];
    T y, inv, r;
    int step, w, t, v;  // v: the row (kTileByRow), -1 padding
    int done;           // the row's system has finished (kTileByRow)
};
template <typename T, int DIR, int MODE>
__device__ inline void tile_load(TileChunk<T>& C, const TileView& V, const Pair<T>* coef, const T* invd, const T* r,
                                 const T* y, int chunk, int base, int w, bool some) {
    const int lane = threadIdx.x & 63;
    C.w = w;
    C.t = chunk * 64 + lane;
    const size_t q = (size_t)base * 64 + lane;
#pragma unroll
    for (int k = 0; k < kMaxDeps / 2; ++k)
        if (k < C.w) {
            C.sl[k] = V.d[DIR].slot[q + (size_t)k * 64];
            C.f[k] = coef[q + (size_t)k * 64];
        }
    if constexpr (MODE == kTileByRow) {
        C.v = V.order[C.t];
        const int s = some ? V.sys[C.t] : 0;
        C.r = C.inv = (T)0;  // padding: the row's value is zero
        C.done = 0;
        if (C.v >= 0) {
            C.r = r[C.v];
            C.inv = invd[C.v];
            if (some) C.done = V.sysDone[s * kSysStride];
        }
    } else {
        C.r = r[C.t];
        C.inv = invd[C.t];
    }
    if (DIR == 1) C.y = y[C.t];
    C.step = V.step[C.t];
}
// The chunk's loads have arrived: waited for here, once, and not at their uses
// inside the loop of tile_rows.
template <int DIR, typename T>
__device__ inline void tile_arrived(TileChunk<T>& C) {
#pragma unroll
    for (int k = 0; k < kMaxDeps / 2; ++k)
        if (k < C.w) asm volatile("" : "+v"(C.sl[k]), "+v"(C.f[k].a), "+v"(C.f[k].b));
    if (DIR == 1) asm volatile("" : "+v"(C.y));
    asm volatile("" : "+v"(C.inv), "+v"(C.r), "+v"(C.step));
}

// One chunk of W entry pairs: rows publish acc - sum f v, times the pivot, in
// their slots, in the order of their levels. A row of the chunk's k-th level
// first looks at its values in round k, when the chunk's earlier levels are
// done unless they wait for another wavefront; it then looks again in every
// round. A value not there yet is a NaN and makes the sum one, so the values
// themselves are looked at only when the sum is a NaN. v: the row's value;
// seen: the wall clock of its round (kTileTrace).
template <typename T, int DIR, int W, int MODE>
__device__ inline bool tile_rows(const TileChunk<T>& C, T* lds, T* own, T& v, long long& seen, long long t0, int* err,
                                 int bit) {
    typedef typename Sentinel<T>::bits_t B;
    int step = C.step;
    if (DIR == 1) step = __shfl(step, 63, 64) - step;
    if (MODE == kTileByRow && C.done) step = 0;
    const T* lo[W + 1];
    const T* hi[W + 1];
#pragma unroll
    for (int k = 0; k < W; ++k) {
        lo[k] = lds + (C.sl[k] & 0xFFFF);
        hi[k] = lds + (C.sl[k] >> 16);
    }
    bool pending = true;
    int waits = 0;
    for (int round = 0;; ++round) {
        bool ready = false;
        if (pending && step <= round) {
            B b[2 * W + 1];
#pragma unroll
            for (int k = 0; k < W; ++k) {
                b[2 * k] = lds_load<T>(lo[k]);
                b[2 * k + 1] = lds_load<T>(hi[k]);
            }
            T a = DIR == 0 ? C.r : C.y;
#pragma unroll
            for (int k = 0; k < W; ++k) {
                a -= C.f[k].a * from_bits(b[2 * k]);
                a -= C.f[k].b * from_bits(b[2 * k + 1]);
            }
            ready = true;
            if (a != a)
#pragma unroll
                for (int k = 0; k < 2 * W; ++k) ready &= b[k] != Sentinel<T>::value;
            if (ready) {
                v = a * C.inv;
                lds_store<T>(own, to_bits(v));
                if (MODE == kTileTrace) seen = wall_clock64();
                pending = false;
            }
        }
        if (!__any(pending)) return true;
        if (!__any(ready)) {
            // waiting for another wavefront: leave the LDS to it
            __builtin_amdgcn_s_sleep(1);
            if (tile_stop(waits++, t0, err, bit)) return false;
        }
    }
}

// One direction over a wavefront's chunks: of the tile's, in level order (DIR 1:
// reversed), every kTileWaves-th from the wavefront's own, so that a chunk's
// data is loaded while the chunks before it are worked on. out: y or z; dot: the
// backward sweep's z.r; some: a system with rows in the tile has finished.
template <typename T, int DIR, int MODE>
__device__ inline void tile_chunks(const TileView& V, const Pair<T>* coef, const T* invd, const T* r, const T* y,
                                   T* out, double& dot, int p0, int wave, T* lds, long long t0, int* err, int bit,
                                   bool some) {
    const int chunks = V.S / 64, first = p0 / 64 + wave, count = (chunks - wave + kTileWaves - 1) / kTileWaves;
    if (count <= 0) return;
    const int zero = V.slots - 1;
    // the chunks' entry starts and ends, in the lanes of two registers
    static_assert(kTileLdsBytes / sizeof(float) / 64 / kTileWaves < 64, "chunks of a wavefront");
    const int lane = threadIdx.x & 63;
    auto chunk = [&](int j) { return first + kTileWaves * (DIR == 0 ? j : count - 1 - j); };
    const int c0 = chunk(min(lane, count - 1));
    const int* sell = V.d[DIR].sell;
    int s0 = sell[c0], e0 = sell[c0 + 1];
    // waited for here: a wait at a chunk's first use of them would also be one for
    // the store of the chunk before (192^3 FP64 87.4 instead of 83.6 ms a projection)
    asm volatile("" : "+v"(s0), "+v"(e0));
    auto load = [&](TileChunk<T>& C, int j) {
        const int base = __builtin_amdgcn_readlane(s0, j), end = __builtin_amdgcn_readlane(e0, j);
        tile_load<T, DIR, MODE>(C, V, coef, invd, r, y, chunk(j), base, end - base, some);
    };
    auto work = [&](TileChunk<T>& C) {
        if constexpr (MODE == kTileByRow) {
            // a row of a finished system takes no part: a zero that waits for
            // nothing (only its own system reads it). FP64 batches whose deepest
            // system finishes in the first iterations, ms per solve without and
            // with: a 20000-row chain and four 20^3 boxes 144 / 9.3, a 56^3 box and
            // four red-black 20^3 boxes 10.3 / 4.7; six boxes that finish about
            // together 9.31 / 9.32 (mixed).
            if (C.done) {
                C.v = -1;
                C.r = C.inv = (T)0;
                if (DIR == 1) C.y = (T)0;
#pragma unroll
                for (int k = 0; k < kMaxDeps / 2; ++k) C.sl[k] = (uint32_t)zero | (uint32_t)zero << 16;
            }
        }
        T v = (T)0;
        long long seen = 0;
        T* own = &lds[C.t - p0];
        bool ok = false;
#define ASTG_TILE_ROWS(W) \
    case W: ok = tile_rows<T, DIR, W, MODE>(C, lds, own, v, seen, t0, err, bit); break;
        switch (C.w) {
            ASTG_TILE_ROWS(0)
            ASTG_TILE_ROWS(1)
            ASTG_TILE_ROWS(2)
            ASTG_TILE_ROWS(3)
            ASTG_TILE_ROWS(4)
            ASTG_TILE_ROWS(5)
            ASTG_TILE_ROWS(6)
            ASTG_TILE_ROWS(7)
            ASTG_TILE_ROWS(8)
        }
#undef ASTG_TILE_ROWS
        static_assert(kMaxDeps == 16, "one case per width");
        if constexpr (DIR == 1 && MODE == kTileByRow) {
            if (C.v >= 0) out[C.v] = v;
        } else {
            out[C.t] = v;
        }
        if (DIR == 1) dot += (double)v * (double)C.r;
        if (MODE == kTileTrace && V.order[C.t] >= 0) {
            long long* tr = V.trace + 3 * (long)V.order[C.t];
            tr[0] = t0;
            tr[1] = seen;
            tr[2] = wall_clock64();
        }
        return ok;
    };
    if constexpr (sizeof(T) == 4) {
        // FP32: registers for the wavefront's next chunk too (5 % at the most
        // rows a tile holds; in FP64 it spills)
        TileChunk<T> A, B;
        load(A, 0);
        for (int j = 0; j < count; j += 2) {
            tile_arrived<DIR>(A);
            if (j + 1 < count) load(B, j + 1);
            if (!work(A) || j + 1 >= count) return;
            tile_arrived<DIR>(B);
            if (j + 2 < count) load(A, j + 2);
            if (!work(B)) return;
        }
    } else {
        for (int j = 0; j < count; ++j) {
            TileChunk<T> A;
            load(A, j);
            tile_arrived<DIR>(A);
            if (!work(A)) return;
        }
    }
}

// y = L^-1 r, then z = L^-T y and the partial dot z.r (one per tile). phases:
// 1 forward, 2 backward, 3 both (single phases are for timing one sweep).
// Bound by the latency of the dependency chain, and at the most rows a tile
// holds by the stream of coefficients. Measured us, forward / backward, merged
// sweeps before and tiles now: FP64 reference order n = 63 k (71 levels) 69 / 89
// and 41 / 43, 456 k (133) 140 / 175 and 73 / 79; FP32 block colours 198 k (61)
// 108 / 104 and 46 / 47, 3.5 M (67) 144 / 147 and 65 / 80 (FP64, 262 levels,
// 312 / 381 and 213 / 238).
// xF / xB: the halo entries of this sweep (armed by the sweep before), nF / nB:
// those of the next one, armed here. A position is worked on by the
// same lane in both sweeps, so y needs no hand-over.
constexpr int kTileThreads = 64 * (kTileWaves + kTileImport + kTileExport);
template <typename T, int MODE>
__global__ void __launch_bounds__(kTileThreads) k_tile_sweep(TileView V, const Pair<T>* coefF, const Pair<T>* coefB,
                                                             const T* invd, const T* r, T* y, T* z, T* xF, T* xB,
                                                             T* nF, T* nB, Parts Pt, int* cnt, double* scal, int mode,
                                                             int it, int maxIt, int norm, double tolRel,
                                                             int parityOut, int phases) {
    constexpr int NT = kTileThreads;
    extern __shared__ __align__(16) unsigned char tile_lds[];
    T* lds = reinterpret_cast<T*>(tile_lds);
    int* xdest = reinterpret_cast<int*>(lds + V.slots);
    uint16_t* xslot = reinterpret_cast<uint16_t*>(xdest + V.exports);
    const bool some = MODE == kTileByRow && V.finished[blockIdx.x] != 0;  // changes between launches only
    if (sweep_stopped(scal, cnt)) return;
    const int S = V.S, p0 = blockIdx.x * S, zero = V.slots - 1;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int* err = &cnt[C_ERR];
    double dot = 0.0;
    // the tile's slots and halo wait for values, and the next sweep's halo; the export list
    auto arm = [&](const TileDir& D, T* next) {
        const int h0 = D.hstart[p0], h = D.hstart[p0 + S] - h0, x0 = D.xstart[p0], x = D.xstart[p0 + S] - x0;
        for (int s = threadIdx.x; s < S + h; s += NT) Sentinel<T>::storeSent(&lds[s]);
        for (int s = threadIdx.x; s < h; s += NT) Sentinel<T>::storeSent(&next[h0 + s]);
        for (int s = threadIdx.x; s < x; s += NT) {
            xslot[s] = D.xslot[x0 + s];
            xdest[s] = D.xdest[x0 + s];
        }
    };
    if (threadIdx.x == 0) lds[zero] = (T)0;
    if (phases & 1) {
        arm(V.d[0], nF);
        if (mode != 2 && fwd_prologue<NT>(Pt, scal, mode, it, maxIt, norm, tolRel)) return;
        __syncthreads();
        const long long t0 = wall_clock64();
        if (wave < kTileWaves)
            tile_chunks<T, 0, MODE>(V, coefF, invd, r, y, y, dot, p0, wave, lds, t0, err, E_FWD, some);
        else if (wave < kTileWaves + kTileImport)
            tile_import<T, 0>(V.d[0], p0, S, xF, lds + S, threadIdx.x - kTileWaves * 64, t0, err, E_FWD);
        else
            tile_export<T, 0>(V.d[0], xslot, xdest, p0, S, lds, xF,
                              threadIdx.x - (kTileWaves + kTileImport) * 64, t0, err, E_FWD);
        __syncthreads();
    }
    if (!(phases & 2)) return;
    arm(V.d[1], nB);
    __syncthreads();
    const long long t0 = wall_clock64();
    if (wave < kTileWaves)
        tile_chunks<T, 1, MODE>(V, coefB, invd, r, y, z, dot, p0, wave, lds, t0, err, E_BWD, some);
    else if (wave < kTileWaves + kTileImport)
        tile_import<T, 1>(V.d[1], p0, S, xB, lds + S, threadIdx.x - kTileWaves * 64, t0, err, E_BWD);
    else
        tile_export<T, 1>(V.d[1], xslot, xdest, p0, S, lds, xB,
                          threadIdx.x - (kTileWaves + kTileImport) * 64, t0, err, E_BWD);
    const double s = block_reduce<false, NT>(dot);
    if (threadIdx.x == 0) (parityOut ? Pt.rho1 : Pt.rho0)[blockIdx.x] = s;
}

}  // namespace

bool PcgDevice::tilesFit(int width) const { return tileLds(width) <= kTileLdsBytes; }
size_t PcgDevice::tileLds(int width) const { return (size_t)f_->tileSlots * width + (size_t)f_->tileExports * 6; }

// The system of every position of the batched form's tiles (0 at padding).
static __global__ void k_tile_sys(int P, const int* order, const int* chunkSeg, int* sys) {
    const int t = blockIdx.x * BS + threadIdx.x;
    if (t < P) sys[t] = order[t] >= 0 ? chunkSeg[order[t] / BS] : 0;
}
int PcgDevice::tileSystems(std::string& err) {
    HIPCHK(f_->tileSys.alloc((size_t)f_->PS * 4));
    HIPCHK(tileFin_.alloc((size_t)f_->tileK * 4));
    k_tile_sys<<<blocks(f_->PS), BS, 0, stream_>>>(f_->PS, f_->sorder.as<int>(), chunkSeg_.as<int>(), f_->tileSys.as<int>());
    HIPCHK(hipGetLastError());
    return ASTG_OK;
}

bool PcgDevice::mayTile(long long n, int width) {
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
        return true;
    return (n + cus - 1) / std::max(1, cus) * width <= (long long)kTileLdsBytes;
}

int PcgDevice::tileSetup(int width, bool& used, std::string& err) {
    used = false;
    const int n = n_;
    const bool placed = coordExt_[0] > 0 && coordN_ == n;
    // a batch's chains end at its systems' boundaries, so its ranges are half as long
    // (6 systems of 12^3 to 56^3, FP32, ms per solve: 12 tiles 10.7, 16 9.7, 24 9.2, 48 9.6;
    // other batches, us per FP64 iteration at the tiles that this gives, at fewer and more:
    // 24 x 20^3 41 tiles 106, 21 129, 82 99; 2 x 30^3 12 tiles 112, 6 133, 24 117; 8 x 40^3
    // 107 tiles 171, 54 199, 214 185)
    const int range = rowOrderForced_ ? kTileRangeRows / 2 : kTileRangeRows;
    int K = std::min(cus_, placed ? std::max(1, n / kTileRows) : (n + range - 1) / range);
    if (tilesAsked_ == 0) return ASTG_OK;
    if (tilesAsked_ > 0) K = std::min(tilesAsked_, cus_);
    int kk[3] = {1, 1, K};  // tiles per axis
    if (placed) {
        tileGrid(K, n, cus_, coordExt_, kk);
        K = kk[0] * kk[1] * kk[2];
    }
    if (K > n) return ASTG_OK;
    const long long S64 = (((long long)n + K - 1) / K + 63) / 64 * 64;
    // rows alone that do not fit: nothing is set up
    if (S64 >= 65535 || S64 * width > (long long)kTileLdsBytes || ((long long)K * depth_ << kWidthBits) >= (1ll << 32) ||
        S64 * K >= (1ll << 31) - 64)
        return ASTG_OK;
    const int S = (int)S64, P = K * S, nch = P / 64;
    const size_t n4 = (size_t)n * 4, P4 = (size_t)P * 4;
    HIPCHK(tileKey_.alloc(n4));
    HIPCHK(tileKey2_.alloc(n4));
    HIPCHK(tileVal_.alloc(n4));
    HIPCHK(tileVal2_.alloc(n4));
    HIPCHK(tileOf_.alloc(n4));
    int* key = tileKey_.as<int>();
    int* key2 = tileKey2_.as<int>();
    int* val = tileVal_.as<int>();
    int* val2 = tileVal2_.as<int>();
    auto bits = [](long long m) {  // bits that hold values below m
        int b = 1;
        while ((1ll << b) < m) ++b;
        return b;
    };
    auto sortPairs = [&](int nbits) -> hipError_t {
        unsigned int *k1 = (unsigned int*)key, *k2 = (unsigned int*)key2;
        size_t tb = 0;
        hipError_t e = hipcub::DeviceRadixSort::SortPairs(nullptr, tb, k1, k2, val, val2, n, 0, nbits, stream_);
        if (e == hipSuccess) e = planTmp_.alloc(tb);
        if (e != hipSuccess) return e;
        return hipcub::DeviceRadixSort::SortPairs(planTmp_.p, tb, k1, k2, val, val2, n, 0, nbits, stream_);
    };
    const int nb = blocks(n);
    const int* idx = nullptr;
    if (placed) {
        // equal-count cuts along z, then y inside each slab, then x
        const unsigned long long* co = rowCoord_.as<unsigned long long>();
        int parts = 1;
        for (int a = 2; a >= 0; --a) {
            if (kk[a] == 1) continue;
            k_coord_key<<<nb, BS, 0, stream_>>>(n, co, 18 * a, idx, parts, key, val);
            HIPCHK(sortPairs(18 + (parts > 1 ? bits(parts) : 0)));
            idx = val2;
            parts *= kk[a];
        }
    }
    k_tile_of<<<nb, BS, 0, stream_>>>(n, idx, K, tileOf_.as<int>());
    k_tile_key<<<nb, BS, 0, stream_>>>(n, tileOf_.as<int>(), lev_.as<int>(), depth_, rs_.as<int>(), lend_.as<int>(),
                                       (unsigned int*)key, val);
    HIPCHK(sortPairs(bits((long long)K * depth_) + kWidthBits));
    HIPCHK(f_->sorder.alloc(P4));
    HIPCHK(f_->pos.alloc(n4));
    k_tile_fill_i32<<<blocks(P), BS, 0, stream_>>>(P, -1, f_->sorder.as<int>());
    k_tile_place<<<nb, BS, 0, stream_>>>(n, val2, K, S, f_->sorder.as<int>(), f_->pos.as<int>());
    // counts and their prefix sums
    HIPCHK(tileCnt_.alloc(4 * P4 + 2 * (size_t)nch * 4));
    HIPCHK(f_->tileStep.alloc((size_t)P));
    HIPCHK(entryHalo_.alloc((size_t)nnz_ * 4));
    int* eh = entryHalo_.as<int>();
    int* cnt[2][2];
    int* wid[2];
    for (int d = 0; d < 2; ++d) {
        cnt[d][0] = tileCnt_.as<int>() + 2 * d * (size_t)P;  // imports
        cnt[d][1] = cnt[d][0] + P;                           // exports
        wid[d] = tileCnt_.as<int>() + 4 * (size_t)P + d * nch;
    }
    const TilePattern M{P, S, f_->sorder.as<int>(), f_->pos.as<int>(), rs_.as<int>(), lend_.as<int>(), ubeg_.as<int>(),
                        col_.as<int>(), tpos_.as<int>(), lev_.as<int>()};
    const int pb = blocks(P);
    k_tile_fill_i32<<<blocks(nnz_), BS, 0, stream_>>>((int)nnz_, 0, eh);
    k_tile_mark<0><<<pb, BS, 0, stream_>>>(M, cnt[0][1], eh);
    k_tile_mark<1><<<pb, BS, 0, stream_>>>(M, cnt[1][1], eh);
    k_tile_count<<<pb, BS, 0, stream_>>>(M, eh, cnt[0][0], cnt[1][0], f_->tileStep.as<uint8_t>(), wid[0], wid[1]);
    auto scan = [&](const int* in, DevBuf& out, int m) -> hipError_t {  // out[0] = 0, out[k + 1] = in[0] + .. + in[k]
        size_t tb = 0;
        hipError_t e = out.alloc(((size_t)m + 1) * 4);
        if (e == hipSuccess) e = hipcub::DeviceScan::InclusiveSum(nullptr, tb, in, out.as<int>() + 1, m, stream_);
        if (e == hipSuccess) e = planTmp_.alloc(tb);
        if (e == hipSuccess) e = hipcub::DeviceScan::InclusiveSum(planTmp_.p, tb, in, out.as<int>() + 1, m, stream_);
        k_tile_fill_i32<<<1, BS, 0, stream_>>>(1, 0, out.as<int>());
        return e;
    };
    for (int d = 0; d < 2; ++d) {
        HIPCHK(scan(cnt[d][0], f_->tile[d].hstart, P));
        HIPCHK(scan(cnt[d][1], f_->tile[d].xstart, P));
        HIPCHK(scan(wid[d], f_->tile[d].sell, nch));
    }
    HIPCHK(tileMax_.alloc(8));
    k_tile_fill_i32<<<1, BS, 0, stream_>>>(2, 0, tileMax_.as<int>());
    k_tile_max<<<blocks(K), BS, 0, stream_>>>(K, S, f_->tile[0].hstart.as<int>(), f_->tile[1].hstart.as<int>(),
                                              f_->tile[0].xstart.as<int>(), f_->tile[1].xstart.as<int>(),
                                              tileMax_.as<int>());
    HIPCHK(hipGetLastError());
    int* h = reinterpret_cast<int*>(hplan_);
    for (int d = 0; d < 2; ++d) {
        HIPCHK(hipMemcpyAsync(h + 2 * d, f_->tile[d].hstart.as<int>() + P, 4, hipMemcpyDeviceToHost, stream_));
        HIPCHK(hipMemcpyAsync(h + 2 * d + 1, f_->tile[d].sell.as<int>() + nch, 4, hipMemcpyDeviceToHost, stream_));
    }
    HIPCHK(hipMemcpyAsync(h + 4, tileMax_.p, 8, hipMemcpyDeviceToHost, stream_));
    HIPCHK(hipStreamSynchronize(stream_));
    const long long slots = (long long)S + h[4] + 1;
    if (getenv("ASTG_TIMING"))
        fprintf(stderr, "[astg timing] tiles: n %d depth %d K %d (%d x %d x %d) S %d halo %d exports %d entries "
                "%lld %lld\n", n, depth_, K, kk[0], kk[1], kk[2], S, h[4], h[5], (long long)h[1] * 128,
                (long long)h[3] * 128);
    // slots are named by 16 bits; the values and the export list share the LDS
    f_->tileExports = h[5];
    f_->tileSlots = (int)std::min<long long>(slots, 65537);
    if (slots > 65536 || !tilesFit(width)) return ASTG_OK;
    if (!placed && tilesAsked_ < 0 && !rangesPay(depth_, S, h[4])) return ASTG_OK;
    f_->tileK = K;
    f_->tileS = S;
    for (int d = 0; d < 2; ++d) {
        DevTile& D = f_->tile[d];
        D.E = (long long)h[2 * d + 1] * 128;
        D.halo = h[2 * d];
        // every halo entry is one export of another tile
        HIPCHK(D.slot.alloc(std::max<size_t>(4, (size_t)D.E * 2)));
        HIPCHK(D.inbox.alloc(std::max<size_t>(16, (size_t)D.halo * 16)));
        HIPCHK(D.xslot.alloc(std::max<size_t>(4, (size_t)D.halo * 2)));
        HIPCHK(D.xdest.alloc(std::max<size_t>(4, (size_t)D.halo * 4)));
        auto kh = d == 0 ? k_tile_halo<0> : k_tile_halo<1>;
        auto kx = d == 0 ? k_tile_exports<0> : k_tile_exports<1>;
        auto ks = d == 0 ? k_tile_slots<0> : k_tile_slots<1>;
        kh<<<pb, BS, 0, stream_>>>(M, D.hstart.as<int>(), eh);
        kx<<<pb, BS, 0, stream_>>>(M, eh, D.xstart.as<int>(), D.xslot.as<uint16_t>(), D.xdest.as<int>());
        ks<<<pb, BS, 0, stream_>>>(M, (int)slots - 1, D.sell.as<int>(), D.hstart.as<int>(), eh,
                                   D.slot.as<uint32_t>());
    }
    HIPCHK(hipGetLastError());
    f_->PS = P;
    used = true;
    return ASTG_OK;
}

TileView PcgDevice::tileView() const {
    TileView v;
    for (int d = 0; d < 2; ++d) {
        v.d[d].sell = f_->tile[d].sell.as<int>();
        v.d[d].slot = f_->tile[d].slot.as<uint32_t>();
        v.d[d].hstart = f_->tile[d].hstart.as<int>();
        v.d[d].xstart = f_->tile[d].xstart.as<int>();
        v.d[d].xslot = f_->tile[d].xslot.as<uint16_t>();
        v.d[d].xdest = f_->tile[d].xdest.as<int>();
    }
    v.step = f_->tileStep.as<uint8_t>();
    v.order = f_->sorder.as<int>();
    // the upper word of each system's B_DONE
    static_assert(kSysStride == 2 * B_COUNT, "state of a system");
    v.sys = K_ ? f_->tileSys.as<int>() : nullptr;
    v.finished = K_ ? tileFin_.as<int>() : nullptr;
    v.sysDone = K_ ? bst_.as<int>() + 2 * B_DONE + 1 : nullptr;
    v.S = f_->tileS;
    v.slots = f_->tileSlots;
    v.exports = f_->tileExports;
    v.trace = trace_;
    return v;
}

bool PcgDevice::isTileKernel(const void* f) const {
    return f == (const void*)k_tile_sweep<double, kTilePlain> || f == (const void*)k_tile_sweep<float, kTilePlain> ||
           f == (const void*)k_tile_sweep<double, kTileByRow> || f == (const void*)k_tile_sweep<float, kTileByRow>;
}

template <typename T>
int PcgDevice::tileCoef(std::string& err) {
    for (int d = 0; d < 2; ++d) {
        DevBuf& c = sizeof(T) == 8 ? f_->tile[d].coef : f_->tile[d].coef32;
        HIPCHK(c.alloc(std::max<size_t>(16, (size_t)f_->tile[d].E * sizeof(T))));
        auto k = d == 0 ? k_tile_coef<T, 0> : k_tile_coef<T, 1>;
        k<<<blocks(f_->PS), BS, 0, stream_>>>(f_->PS, f_->sorder.as<int>(), rs_.as<int>(), lend_.as<int>(), ubeg_.as<int>(),
                                           F_.as<double>(), f_->tile[d].sell.as<int>(), c.as<Pair<T>>());
    }
    HIPCHK(hipGetLastError());
    return ASTG_OK;
}

template <typename T>
int PcgDevice::launchTile(const T* invd, const T* r, T* z, int k, int mode, int it, int maxIt, int norm,
                          double tolRel, int phases, std::string& err) {
    const TileMode form = !perm_ ? kTileByRow : trace_ ? kTileTrace : kTilePlain;
    const auto kernel = form == kTileByRow   ? k_tile_sweep<T, kTileByRow>
                        : form == kTileTrace ? k_tile_sweep<T, kTileTrace>
                                             : k_tile_sweep<T, kTilePlain>;
    const size_t lds = tileLds(sizeof(T));
    bool& raised = tileLds_[sizeof(T) == 8][form];
    if (!raised) {
        HIPCHK(hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                                   (int)kTileLdsBytes));
        raised = true;
    }
    TileView V = tileView();
    const Pair<T>* cF = (const Pair<T>*)(sizeof(T) == 8 ? f_->tile[0].coef.p : f_->tile[0].coef32.p);
    const Pair<T>* cB = (const Pair<T>*)(sizeof(T) == 8 ? f_->tile[1].coef.p : f_->tile[1].coef32.p);
    T* y = y_.as<T>();
    T* xF = f_->tile[0].inbox.as<T>() + (size_t)(k & 1) * f_->tile[0].halo;
    T* nF = f_->tile[0].inbox.as<T>() + (size_t)((k + 1) & 1) * f_->tile[0].halo;
    T* xB = f_->tile[1].inbox.as<T>() + (size_t)(k & 1) * f_->tile[1].halo;
    T* nB = f_->tile[1].inbox.as<T>() + (size_t)((k + 1) & 1) * f_->tile[1].halo;
    Parts Pt = parts(f_->tileK);
    int* cnt = cnt_.as<int>();
    double* scal = scal_.as<double>();
    int parity = k & 1;
    if (!coop_) {
        kernel<<<f_->tileK, kTileThreads, lds, stream_>>>(V, cF, cB, invd, r, y, z, xF, xB, nF, nB, Pt, cnt, scal, mode,
                                                       it, maxIt, norm, tolRel, parity, phases);
        HIPCHK(hipGetLastError());
    } else {
        void* args[] = {&V,  &cF, &cB,  &invd, &r,    &y,    &z,  &xF,    &xB,   &nF,     &nB,
                        &Pt, &cnt, &scal, &mode, &it, &maxIt, &norm, &tolRel, &parity, &phases};
        HIPCHK(hipLaunchCooperativeKernel((const void*)kernel, dim3(f_->tileK), dim3(kTileThreads), args,
                                          (unsigned)lds, stream_));
    }
    return ASTG_OK;
}

template int PcgDevice::tileCoef<double>(std::string&);
template int PcgDevice::tileCoef<float>(std::string&);
template int PcgDevice::launchTile<double>(const double*, const double*, double*, int, int, int, int, int, double,
                                           int, std::string&);
template int PcgDevice::launchTile<float>(const float*, const float*, float*, int, int, int, int, int, double, int,
                                          std::string&);

}  // namespace astg

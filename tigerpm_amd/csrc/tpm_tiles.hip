// tpm_tiles.hip -- the direct kernel's work items.
//
// The reference takes its sinks in buckets of a per-cell tree (<= 128,
// tree.cpp:216-245) and compacts the active ones inside the kernel
// (kick_treepm.cu:476-503).  Here every kick makes tiles of <= ts active
// sinks of one chain cell, ts the tuning's tile size:
//   count:  active particles per cell -> tiles per cell;
//   scan:   tile offsets and their number (on the device, no wait);
//   build:  per cell, the active particles' order and the tiles.
// The order splits a cell's active particles in halves at the median of the
// longest axis until <= ts remain, so a tile's box is near a cube: at 512^3
// 16-sink tiles stage 1580 sources instead of 1930 with runs of the Morton
// order (a CPU model of the boxes).  Count and build take 0.05 + 0.52 ms at
// 256^3 and 0.32 + 3.7 ms at 512^3; the pair kernel went from 22.2 to 19.0 ms at 256^3.
// Tiles of active sinks only: with an eighth of 256^3 particles active the
// kernel has an eighth of the tiles (11.9 -> 4.8 ms).
#include "tpm_tiles.hpp"
#include "tpm_tile_order.hpp"

#include <algorithm>
#include <climits>
#include <type_traits>

namespace {

__device__ __forceinline__ unsigned count_below(unsigned long long m) {
    return __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
}

// What a cell's wave needs of its box.
struct CellBox {
    int box, cell0, C, min_rung;
    int64_t n;
    uint32_t w;
};
__device__ __forceinline__ CellBox cell_box(const tpm_tile_args& a, int c) {
    if (!a.boxes) return CellBox{0, 0, a.C, a.min_rung, a.n, a.cell_w};
    const int b = tpm_upper_index(a.nbox, c, [&](int k) { return (int64_t)a.boxes[k].cell0; });
    return CellBox{b, a.boxes[b].cell0, a.boxes[b].C, a.boxes[b].min_rung, a.boxes[b].n, a.boxes[b].cell_w};
}

// Counts the active particles of [i, e) from i on, in pieces that end at
// multiples of 16, while at least COUNT_STEP particles are left and the count cannot
// exceed most; i moves to the first particle not counted.  Four 16-byte loads
// are in flight per lane (a cell of 10^5 particles: 28 us, 314 with one byte a lane).
constexpr int COUNT_STEP = 4096;
__device__ __forceinline__ int count_active(const int8_t* __restrict__ rung, int& i, int e, int most, int lane,
                                            int min_rung) {
    int n = 0;
    while (true) {
        const int i0 = i & ~15;
        if (i0 + COUNT_STEP > e || COUNT_STEP > most - n) break;
        int4 v[4];
#pragma unroll
        for (int p = 0; p < 4; p++) v[p] = *reinterpret_cast<const int4*>(rung + i0 + 1024 * p + 16 * lane);
        int mine = 0;
#pragma unroll
        for (int p = 0; p < 4; p++) {
            const int w[4] = {v[p].x, v[p].y, v[p].z, v[p].w};
#pragma unroll
            for (int k = 0; k < 16; k++) {
                const int r = (int)(int8_t)(w[k / 4] >> (8 * (k % 4)));
                mine += r >= min_rung && (p > 0 || 16 * lane + k >= i - i0) ? 1 : 0;
            }
        }
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) mine += __shfl_xor(mine, o);
        n += __builtin_amdgcn_readfirstlane(mine);
        i = i0 + COUNT_STEP;
    }
    return n;
}

// The active particles of [b, e), counted by a wave.
__device__ __forceinline__ int cell_active(const tpm_tile_args& a, int b, int e, int lane, int min_rung) {
    int i = b, n = count_active(a.rung, i, e, INT_MAX, lane, min_rung);
    for (; i < e; i += 64) n += __popcll(__ballot(i + lane < e && a.rung[min(i + lane, e - 1)] >= min_rung));
    return n;
}

// Whether cell c's sinks are wanted (in [lo, hi)), and its place in the tile
// list.
__device__ __forceinline__ bool cell_wanted(const tpm_tile_args& a, int c, int* rank) {
    *rank = c;
    if (a.boxes) return true;
    *rank = tile_rank((uint32_t)c, (uint32_t)a.C);
    const int x = c % a.C, y = (c / a.C) % a.C, z = c / (a.C * a.C);
    return x >= a.lo.x && x < a.hi.x && y >= a.lo.y && y < a.hi.y && z >= a.lo.z && z < a.hi.z;
}

// Number of tiles per cell, ceil(active / ts) (zero outside [lo, hi)): one
// wave per cell, where cells have few particles one lane, and the wave for a
// cell of more than 64.
template <bool LANE>
__global__ __launch_bounds__(256, 8) void tile_count_kernel(tpm_tile_args a) {
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)((blockIdx.x * (int64_t)blockDim.x + threadIdx.x) >> 6));
    const int nwave = (int)(((int64_t)gridDim.x * blockDim.x) >> 6);
    if constexpr (LANE) {
        for (int64_t c0 = (int64_t)wave * 64; c0 < a.ncell; c0 += (int64_t)nwave * 64) {
            const int c = (int)c0 + lane;
            int b = 0, e = 0, r = 0, min_rung = 0, n = 0;
            if (c < a.ncell) {
                b = a.cell_begin[c];
                e = cell_wanted(a, c, &r) ? a.cell_begin[c + 1] : b;
                if (b < e) min_rung = cell_box(a, c).min_rung;
            }
            if (a.all)
                n = e - b;
            else if (e - b <= 64)
                for (int i = b; i < e; i++) n += a.rung[i] >= min_rung ? 1 : 0;
            for (unsigned long long m = __ballot(!a.all && e - b > 64); m; m &= m - 1) {
                const int l = __builtin_ctzll(m);
                const int k = cell_active(a, __builtin_amdgcn_readlane(b, l), __builtin_amdgcn_readlane(e, l), lane,
                                          __builtin_amdgcn_readlane(min_rung, l));
                if (lane == l) n = k;
            }
            if (c < a.ncell) a.cnt[r] = (n + a.ts - 1) / a.ts;
        }
    } else {
        for (int c = wave; c < a.ncell; c += nwave) {
            int r, n = 0;
            if (cell_wanted(a, c, &r)) {
                const int b = a.cell_begin[c], e = a.cell_begin[c + 1];
                n = a.all ? e - b : cell_active(a, b, e, lane, cell_box(a, c).min_rung);
            }
            if (lane == 0) a.cnt[r] = (n + a.ts - 1) / a.ts;
        }
    }
}

__global__ void order_positions_kernel(int64_t n, const uint32_t* __restrict__ order, const uint32_t* __restrict__ x,
                                       const uint32_t* __restrict__ y, const uint32_t* __restrict__ z,
                                       uint32_t* __restrict__ ox, uint32_t* __restrict__ oy,
                                       uint32_t* __restrict__ oz) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const uint32_t j = order[i];
        ox[i] = x[j];
        oy[i] = y[j];
        oz[i] = z[j];
    }
}

// The order and the tiles of a chunk of a cell's active particles, by one
// wave: KD_CHUNK of them in chain-mesh order, whose Morton codes keep them
// together, half as many in boxes below KD_SMALL particles, where the waves
// are few and the splits of a chunk, one after the other, are the kernel's
// time.  a.per_cell waves share a cell's first KD_RUN a.per_cell chunks; the
// chunks beyond, of cells far more crowded than the average, are found one by
// one from the tile list by further waves (tile_slot_chunk), so that a halo's
// cell is made by the whole chip: one cell of 10^5 particles among 64^3
// uniform ones takes 0.10 ms (11^3 cells) and 0.13 ms (45^3), where its chunks
// were the work of one wave or two 3.9 and 7.5 ms.  A
// segment of len particles that makes m tiles is split m / 2 : m - m / 2, at
// the position whose lower side has len (m / 2) / m particles (full tiles: ts
// (m / 2)), found by
// bisection of the coordinate with ballot counts; ties go by position, so the
// split is exact and depends on nothing but the cell's particles.
constexpr int KD_CHUNK = 256;
constexpr int KD_SMALL = 1 << 19;
constexpr int KD_RUN = 4;
constexpr int KD_SLOTS = 8;  // slots of the tile list that a wave looks at
constexpr int KD_STACK = 8;  // pending segments: one per level of at most log2(256 / 8), and the current one

struct KdWave {
    uint32_t p[3][KD_CHUNK];  // offsets from the cell's centre, + 2^31
    uint32_t id[KD_CHUNK];    // particles of the chunk
    uint32_t ord[KD_CHUNK];   // their order
    int stack[KD_STACK][9];   // first, len, tiles, box
};

// The LDS words of a KdWave are written and read by the lanes of one wave,
// whose LDS operations complete in order: the compiler keeps the order, and
// nothing waits for the tiles' global stores, as a fence would.
__device__ __forceinline__ void kd_sync() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_wave_barrier();
}

// Minimum and maximum of a wave: DPP within the rows of 16, the rows by
// scalar operations.
template <class Op>
__device__ __forceinline__ uint32_t wave_reduce(uint32_t v, Op op) {
    const auto dpp = [](uint32_t x, auto ctrl) {
        return (uint32_t)__builtin_amdgcn_update_dpp((int)x, (int)x, decltype(ctrl)::value, 0xf, 0xf, false);
    };
    v = op(v, dpp(v, std::integral_constant<int, 0xB1>{}));
    v = op(v, dpp(v, std::integral_constant<int, 0x4E>{}));
    v = op(v, dpp(v, std::integral_constant<int, 0x141>{}));
    v = op(v, dpp(v, std::integral_constant<int, 0x140>{}));
    const uint32_t a = (uint32_t)__builtin_amdgcn_readlane((int)v, 0), b = (uint32_t)__builtin_amdgcn_readlane((int)v, 16),
                   c = (uint32_t)__builtin_amdgcn_readlane((int)v, 32), d = (uint32_t)__builtin_amdgcn_readlane((int)v, 48);
    return op(op(a, b), op(c, d));
}
__device__ __forceinline__ uint32_t wave_umin(uint32_t v) {
    return wave_reduce(v, [](uint32_t a, uint32_t b) { return a < b ? a : b; });
}
__device__ __forceinline__ uint32_t wave_umax(uint32_t v) {
    return wave_reduce(v, [](uint32_t a, uint32_t b) { return a > b ? a : b; });
}

// Splits a.ord[s .. s + len) so that its first `left` entries are the `left`
// smallest along an axis; returns the split coordinate.  PER: entries per
// lane, at least len / 64 (most segments have at most 64 entries).
template <int PER>
__device__ __forceinline__ uint32_t kd_split(KdWave& w, int lane, int s, int len, int left, int axis, uint32_t lo,
                                             uint32_t hi) {
    uint32_t e[PER], key[PER];
#pragma unroll
    for (int i = 0; i < PER; i++) {
        e[i] = 0u;
        key[i] = ~0u;
        const int k = lane + 64 * i;
        if (k < len) {
            e[i] = w.ord[s + k];
            key[i] = w.p[axis][e[i]];
        }
    }
    const auto below = [&](uint32_t t) {
        int n = 0;
#pragma unroll
        for (int i = 0; i < PER; i++)
            n += __popcll(__ballot(key[i] < t));
        return n;
    };
    // below(a) <= left < below(b) or the exact split; keys lie in [lo, hi],
    // hi < 2^32 - 1 (offsets span less than half the box), so padding keys
    // are above every threshold
    uint32_t a = lo, b = hi + 1u, t = a;
    int nt = 0;
    while (b - a > 1u) {
        t = a + (b - a) / 2u;
        nt = below(t);
        if (nt == left) break;
        if (nt < left)
            a = t;
        else
            b = t;
    }
    if (nt != left) {
        t = a;
        nt = below(t);
    }
    // keys equal to t fill the lower side up in order
    int need = left - nt, nl = 0, nr = 0;
    uint32_t dst[PER];
#pragma unroll
    for (int i = 0; i < PER; i++) {
        const bool have = lane + 64 * i < len;
        const unsigned long long me = __ballot(have && key[i] == t);
        const bool lower = have && (key[i] < t || (key[i] == t && (int)count_below(me) < need));
        need = max(need - __popcll(me), 0);
        const unsigned long long ml = __ballot(lower), mr = __ballot(have && !lower);
        dst[i] = (uint32_t)(lower ? nl + (int)count_below(ml) : left + nr + (int)count_below(mr));
        nl += __popcll(ml);
        nr += __popcll(mr);
    }
    kd_sync();
#pragma unroll
    for (int i = 0; i < PER; i++)
        if (lane + 64 * i < len) w.ord[s + (int)dst[i]] = e[i];
    return t;
}

__device__ __forceinline__ int kd_chunk_size(int64_t n) { return n < KD_SMALL ? KD_CHUNK / 2 : KD_CHUNK; }

// A cell whose tiles are made.
struct KdCell {
    int c, b, e, chunk, first_tile;
    CellBox B;
    uint32_t q[3];  // its centre - 2^31
};
__device__ __forceinline__ KdCell kd_cell(const tpm_tile_args& a, int c, int first_tile) {
    KdCell x;
    x.c = c;
    x.b = a.cell_begin[c];
    x.e = a.cell_begin[c + 1];
    x.B = cell_box(a, c);
    x.chunk = kd_chunk_size(x.B.n);
    x.first_tile = first_tile;
    const uint32_t l = (uint32_t)(c - x.B.cell0), C = (uint32_t)x.B.C;
    x.q[0] = (l % C) * x.B.w + x.B.w / 2 - 0x80000000u;
    x.q[1] = ((l / C) % C) * x.B.w + x.B.w / 2 - 0x80000000u;
    x.q[2] = (l / (C * C)) * x.B.w + x.B.w / 2 - 0x80000000u;
    return x;
}

// Chunk k of a cell.  seen: active particles before particle i0 of the cell,
// at most those before the chunk; both move on.
__device__ __forceinline__ void kd_chunk(const tpm_tile_args& a, KdWave& w, int lane, const KdCell& x, int k, int& seen,
                                         int& i0) {
    const int ts = a.ts, e = x.e;
    const int first = k * x.chunk;  // active particles before the chunk
    int tile = x.first_tile + k * (x.chunk / ts);
    const int out = x.b + first;  // its place in the order
    if (a.all) {
        seen = first;
        i0 = out;
    }
    seen += count_active(a.rung, i0, e, first - seen, lane, x.B.min_rung);
    int n = 0;
    while (i0 < e && n < x.chunk) {
        const int i = i0 + lane;
        bool act = i < e && (a.all || a.rung[min(i, e - 1)] >= x.B.min_rung);
        const unsigned long long m = __ballot(act);
        const int rank = seen + (int)count_below(m) - first;
        act = act && rank >= 0 && rank < x.chunk;
        const unsigned long long mt = __ballot(act);
        if (act) {
            w.id[rank] = (uint32_t)i;
            w.ord[rank] = (uint32_t)rank;
            w.p[0][rank] = a.x[i] - x.q[0];
            w.p[1][rank] = a.y[i] - x.q[1];
            w.p[2][rank] = a.z[i] - x.q[2];
        }
        n += __popcll(mt);
        if (n == x.chunk) break;  // the next chunk may begin inside this group
        seen += __popcll(m);
        i0 += 64;
    }
    if (n == 0) return;
    kd_sync();
    const int m0 = (n + ts - 1) / ts;
    int sp = 1;
    uint32_t lo[3], hi[3];
    if (m0 > 1) {
        // the chunk's box; from there on halves of it
#pragma unroll
        for (int d = 0; d < 3; d++) {
            uint32_t mn = ~0u, mx = 0u;
            for (int k = lane; k < n; k += 64) {
                const uint32_t v = w.p[d][k];
                mn = min(mn, v);
                mx = max(mx, v);
            }
            lo[d] = wave_umin(mn);
            hi[d] = wave_umax(mx);
        }
    } else {
        lo[0] = lo[1] = lo[2] = hi[0] = hi[1] = hi[2] = 0u;
    }
    if (lane == 0) {
        w.stack[0][0] = 0;
        w.stack[0][1] = n;
        w.stack[0][2] = m0;
#pragma unroll
        for (int d = 0; d < 3; d++) {
            w.stack[0][3 + d] = (int)lo[d];
            w.stack[0][6 + d] = (int)hi[d];
        }
    }
    kd_sync();
    while (sp > 0) {
        sp--;
        const int s = __builtin_amdgcn_readfirstlane(w.stack[sp][0]);
        const int len = __builtin_amdgcn_readfirstlane(w.stack[sp][1]);
        const int m = __builtin_amdgcn_readfirstlane(w.stack[sp][2]);
        if (m == 1) {
            if (lane == 0 && a.tiles) a.tiles[tile] = make_int4(x.c, out + s, out + s + len, x.B.box);
            tile++;
            continue;
        }
#pragma unroll
        for (int d = 0; d < 3; d++) {
            lo[d] = (uint32_t)__builtin_amdgcn_readfirstlane(w.stack[sp][3 + d]);
            hi[d] = (uint32_t)__builtin_amdgcn_readfirstlane(w.stack[sp][6 + d]);
        }
        int axis = 0;
        uint32_t span = hi[0] - lo[0], l0 = lo[0], h0 = hi[0];
        if (hi[1] - lo[1] > span) {
            axis = 1;
            span = hi[1] - lo[1];
            l0 = lo[1];
            h0 = hi[1];
        }
        if (hi[2] - lo[2] > span) {
            axis = 2;
            l0 = lo[2];
            h0 = hi[2];
        }
        const int m1 = m / 2, left = a.full ? ts * m1 : len * m1 / m;
        const uint32_t t = len <= 64    ? kd_split<1>(w, lane, s, len, left, axis, l0, h0)
                           : len <= 128 ? kd_split<2>(w, lane, s, len, left, axis, l0, h0)
                                        : kd_split<KD_CHUNK / 64>(w, lane, s, len, left, axis, l0, h0);
        kd_sync();
        if (lane == 0) {
            // the upper side waits below the lower one
            int* up = w.stack[sp];
            int* dn = w.stack[sp + 1];
            up[0] = s + left;
            up[1] = len - left;
            up[2] = m - m1;
            dn[0] = s;
            dn[1] = left;
            dn[2] = m1;
#pragma unroll
            for (int d = 0; d < 3; d++) {
                dn[3 + d] = (int)lo[d];
                up[6 + d] = (int)hi[d];
                up[3 + d] = (int)(d == axis ? t : lo[d]);
                dn[6 + d] = (int)(d == axis ? t : hi[d]);
            }
        }
        sp += 2;
        kd_sync();
    }
    for (int i = lane; i < n; i += 64) a.order[out + i] = w.id[w.ord[i]];
    kd_sync();
}

__global__ __launch_bounds__(256, 7) void tile_build_kernel(tpm_tile_args a) {
    __shared__ KdWave s_wave[4];
    const int lane = threadIdx.x & 63;
    KdWave& w = s_wave[__builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6)];
    const int wave = __builtin_amdgcn_readfirstlane((int)((blockIdx.x * (int64_t)blockDim.x + threadIdx.x) >> 6));
    const int nwave = (int)(((int64_t)gridDim.x * blockDim.x) >> 6);
    const int run = KD_RUN * a.per_cell;
    const int cell_units = a.group ? (a.ncell + a.group - 1) / a.group : a.ncell * a.per_cell;
    for (int u = wave; u < cell_units + a.slot_waves; u += nwave) {
        // Lanes with k < k1 have every per_cell-th chunk of [k, k1) of cell c,
        // whose rank is r, for the wave to make.
        int c = 0, r = 0, k = 0, k1 = 0;
        if (u >= cell_units) {
            // slots apart by the number of these waves, so that neighbouring
            // chunks of a cell go to different ones
            const int space = KD_CHUNK / 2 / a.ts;
            const int64_t v = (u - cell_units) + (int64_t)lane * a.slot_waves;
            if (lane < KD_SLOTS && v * space < a.off[a.ncell]) {
                r = tpm_upper_index(a.ncell, v * space, [&](int j) { return (int64_t)a.off[j]; });
                c = a.boxes ? r : tile_cell((uint32_t)r, (uint32_t)a.C);
                k = tile_slot_chunk(v, space, kd_chunk_size(cell_box(a, c).n) / a.ts, a.off[r], a.off[r + 1]);
                k1 = k >= run ? k + 1 : k;
            }
        } else if (a.group) {
            // a lane makes the tile of its cell when there is one, of at most
            // 64 particles; the wave makes the others
            c = u * a.group + lane;
            if (lane < a.group && c < a.ncell) {
                r = a.boxes ? c : tile_rank((uint32_t)c, (uint32_t)a.C);
                const int ntile = a.cnt[r];
                if (ntile > 0) {
                    const int b = a.cell_begin[c], e = a.cell_begin[c + 1];
                    const CellBox B = cell_box(a, c);
                    if (ntile == 1 && e - b <= 64) {
                        int n = 0;
                        for (int i = b; i < e; i++)
                            if (a.all || a.rung[i] >= B.min_rung) a.order[b + n++] = (uint32_t)i;
                        if (a.tiles) a.tiles[a.off[r]] = make_int4(c, b, b + n, B.box);
                    } else {
                        const int chunk = kd_chunk_size(B.n);
                        k1 = min(run, (ntile * a.ts + chunk - 1) / chunk);
                    }
                }
            }
        } else {
            c = u / a.per_cell;
            r = a.boxes ? c : tile_rank((uint32_t)c, (uint32_t)a.C);
            const int ntile = a.cnt[r];
            if (ntile > 0 && lane == 0) {
                const int chunk = kd_chunk_size(cell_box(a, c).n);
                k = u - c * a.per_cell;
                k1 = min(run, (ntile * a.ts + chunk - 1) / chunk);
            }
        }
        for (unsigned long long m = __ballot(k < k1); m; m &= m - 1) {
            const int l = __builtin_ctzll(m);
            const KdCell x = kd_cell(a, __builtin_amdgcn_readlane(c, l), a.off[__builtin_amdgcn_readlane(r, l)]);
            const int end = __builtin_amdgcn_readlane(k1, l);
            int seen = 0, i0 = x.b;
            for (int j = __builtin_amdgcn_readlane(k, l); j < end; j += a.per_cell) kd_chunk(a, w, lane, x, j, seen, i0);
        }
    }
}

}  // namespace

// Workgroups of 4 waves, up to a grid that fills the chip many times over.
static unsigned wave_grid(int64_t waves) { return (unsigned)std::min<int64_t>((waves + 3) / 4, 65536); }

tpm_status tpm_order_positions(std::string& err, hipStream_t s, int64_t n, const tpm_tile_args& a, uint32_t* x,
                               uint32_t* y, uint32_t* z) {
    order_positions_kernel<<<grid_for(n, 256), 256, 0, s>>>(n, a.order, a.x, a.y, a.z, x, y, z);
    TPM_HIPE(err, hipGetLastError());
    return TPM_OK;
}

// Where the count takes a lane per cell: below COUNT_LANE_MEAN particles per
// cell and from COUNT_LANE_CELLS cells on, when a wave per cell is more than
// one round of the chip (4913 cells: 5 us a wave per cell, 7 a lane).
// Where the build's waves take several cells each, of which a lane makes
// those with one tile: where a wave per cell would be more than GROUP_WAVES
// waves (the chip holds 7168 of them).
// us, count + build, a wave per cell / so: 32^3 particles in 91^3 cells 426 / 27,
// 180^3 737 / 78, 200^3 769 / 146, 256^3 1015 / 660, 320^3 1328 / 1025; 64^3 in 45^3
// 108 / 27, 100^3 117 / 54, 160^3 188 / 152, 256^3 515 / 539.
constexpr int COUNT_LANE_MEAN = 48, COUNT_LANE_CELLS = 8192, GROUP_WAVES = 16384;

tpm_status tpm_tiles_make(std::string& err, hipStream_t s, tpm_tile_args a) {
    if (a.ncell == 0) return TPM_OK;
    if (a.n_all < COUNT_LANE_MEAN * (int64_t)a.ncell && a.ncell > COUNT_LANE_CELLS)
        tile_count_kernel<true><<<wave_grid(((int64_t)a.ncell + 63) / 64), 256, 0, s>>>(a);
    else
        tile_count_kernel<false><<<wave_grid(a.ncell), 256, 0, s>>>(a);
    TPM_HIPE(err, hipGetLastError());
    TPM_TRY(tpm_scan_i32(err, s, a.cnt, a.ncell, a.part, a.off));
    // as many waves as an average cell has chunks
    a.per_cell = (int)std::min<int64_t>(std::max<int64_t>(a.n_all / a.ncell / (KD_CHUNK / 2), 1), 32);
    const int64_t slots = (a.n_all / a.ts + std::min<int64_t>(a.ncell, a.n_all)) / (KD_CHUNK / 2 / a.ts) + 1;
    a.slot_waves = (int)((slots + KD_SLOTS - 1) / KD_SLOTS);
    a.group = 0;
    if (a.per_cell == 1)
        for (a.group = 1; a.group < 64 && a.ncell / (2 * a.group) >= GROUP_WAVES;) a.group *= 2;
    const int64_t units = a.group ? ((int64_t)a.ncell + a.group - 1) / a.group : (int64_t)a.ncell * a.per_cell;
    tile_build_kernel<<<wave_grid(units + a.slot_waves), 256, 0, s>>>(a);
    TPM_HIPE(err, hipGetLastError());
    return TPM_OK;
}
